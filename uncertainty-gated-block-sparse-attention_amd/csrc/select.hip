// Kernel 2 compile unit: the bf16 selection kernels (select.h) and the
// element-format dispatch.
#include "select.h"

namespace ugbsa {

hipError_t launch_select(const uint16_t* q, int64_t sq_b, int64_t sq_h, int64_t sq_m,
                         const uint16_t* planes, int B, int H, int Hk, int M, int N, int D,
                         int elem, int mode, float scaling, int k_base, int k_slots,
                         int want_sigma, int32_t* kv_idx, float* sigma, float* tile_score,
                         hipStream_t stream, const SelectAux* aux) {
  if (elem == ElemF16::code)
    return launch_select_f16(q, sq_b, sq_h, sq_m, planes, B, H, Hk, M, N, D, mode, scaling,
                             k_base, k_slots, want_sigma, kv_idx, sigma, tile_score, stream, aux);
  return launch_select_e<ElemBf16>(q, sq_b, sq_h, sq_m, planes, B, H, Hk, M, N, D, mode, scaling,
                                   k_base, k_slots, want_sigma, kv_idx, sigma, tile_score, stream,
                                   aux);
}

}  // namespace ugbsa
