// Kernel 1: per-block K summaries for block scoring (HBM-bound, K read once).
//
// Restates src/sparse_attention.py:618-622, 636-637, 646 of the reference on
// the GQA key tensor [B, Hk, N, D] (the reference works on the repeat_kv'd
// copy; the summaries of repeated heads are identical).  Rows past N count as
// zeros, as F.pad does for the last partial block.
//
// Output "planes", the operand layout of the scoring kernel:
//  * Quest: [B, Hk, NB, 2, D] in K's 16-bit format (bf16 or fp16): K-max,
//    K-min — input values, exact.
//  * mean, for both formats: [B, Hk, NB, 2, D] fp16, then [B, Hk, NB] fp32.
//    The fp32 mean m of a block is scaled by 2^e, e = 141 - (the fp32
//    exponent field of max_d |m_d|), so that max_d |m_d| 2^e lies in
//    [2^14, 2^15), and stored as the unevaluated sum hi + lo of two fp16
//    values (hi = fp16(m 2^e), lo = fp16(m 2^e - hi)); the fp32 array holds
//    2^-e.  hi + lo carries 22-23 significant bits of each m_d 2^e: the sum
//    is within 2^-23 |m_d| 2^e + 2^-25 of it (the second term where lo falls
//    in fp16's subnormal range, i.e. 2^-39 of the block's largest |m_d|).
//    The scoring kernel multiplies fp16 Q (scaled by a power of two per
//    tile, exact) by both planes on the fp16 MFMA — two contractions per
//    block instead of the three that a bf16 hi + mid + lo split of the fp32
//    mean takes — and undoes both scales exactly on the fp32 result.
#include "common.h"
#include "kv_operand.h"
#include "launch.h"

namespace ugbsa {

// A thread's running sum, minimum and maximum of its 8 dims: chunk c = thread %
// (D / 8) of every (256 / (D / 8))-th row of the block.
struct SummaryAcc {
  float s[8], mn[8], mx[8];
  __device__ __forceinline__ SummaryAcc() {
#pragma unroll
    for (int j = 0; j < 8; ++j) { s[j] = 0.f; mn[j] = INFINITY; mx[j] = -INFINITY; }
  }
  template <typename E>
  __device__ __forceinline__ void add(u32x4 raw) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float lo = E::to_f32(raw[j] & 0xFFFFu);
      const float hi = E::to_f32(raw[j] >> 16);
      s[2 * j] += lo; s[2 * j + 1] += hi;
      mn[2 * j] = fminf(mn[2 * j], lo); mn[2 * j + 1] = fminf(mn[2 * j + 1], hi);
      mx[2 * j] = fmaxf(mx[2 * j], lo); mx[2 * j + 1] = fmaxf(mx[2 * j + 1], hi);
    }
  }
};

// LDS floats of the workgroup's reduction: the three statistics of each row
// group, D + 1 apart.
__host__ __device__ constexpr int summary_red(int D) { return 3 * (256 / (D / 8)) * (D + 1); }

// The planes (and the pooled means) of block blk of (b, h) from the
// workgroup's accumulators, through red (summary_red(D) floats) and wmax.
template <int D, typename E>
__device__ __forceinline__ void summary_store(const SummaryAcc& acc, float* red, uint32_t* wmax,
                                              int b, int h, int blk, int B, int Hk, int NB,
                                              int mode, uint16_t* __restrict__ planes,
                                              uint16_t* __restrict__ pool, int rep) {
  constexpr int CH = D / 8;        // 16-byte chunks per row
  constexpr int RG = 256 / CH;     // row groups
  const int c = threadIdx.x % CH, rg = threadIdx.x / CH;
  auto at = [&](int stat, int g, int d) -> float& { return red[(stat * RG + g) * (D + 1) + d]; };
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    at(0, rg, c * 8 + j) = acc.s[j];
    at(1, rg, c * 8 + j) = acc.mn[j];
    at(2, rg, c * 8 + j) = acc.mx[j];
  }
  __syncthreads();

  if (mode == kModeQuest) {
    uint16_t* out = planes + ((static_cast<int64_t>(b) * Hk + h) * NB + blk) * 2 * D;
    for (int d = threadIdx.x; d < D; d += 256) {
      float a = -INFINITY, z = INFINITY;
      for (int g = 0; g < RG; ++g) { a = fmaxf(a, at(2, g, d)); z = fminf(z, at(1, g, d)); }
      out[d] = E::from_f32(a);          // exact: an input value (or 0)
      out[D + d] = E::from_f32(z);
    }
    return;
  }
  // mean: one d per thread (D <= 256 threads), the block's largest |mean|
  // over d through LDS, then the scaled two-term fp16 split
  const int d = threadIdx.x;
  float mean = 0.f;
  if (d < D) {
    float sum = 0.f;
    for (int g = 0; g < RG; ++g) sum += at(0, g, d);
    mean = sum * (1.0f / kBlock);
  }
  uint32_t mb = __float_as_uint(mean) & 0x7FFFFFFFu;     // |mean| orders as its bits
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) mb = max(mb, static_cast<uint32_t>(__shfl_xor(static_cast<int>(mb), m, 64)));
  if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = mb;
  __syncthreads();
  const uint32_t bmax = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
  const int e = bmax == 0u ? 0 : 141 - static_cast<int>(bmax >> 23);
  const int64_t bid = (static_cast<int64_t>(b) * Hk + h) * NB + blk;
  if (d < D) {
    uint16_t* out = planes + bid * 2 * D;
    const float x = ldexpf(mean, e);                   // exact
    const uint16_t hi = ElemF16::from_f32(x);
    const uint16_t lo = ElemF16::from_f32(x - ElemF16::to_f32(hi));
    out[d] = hi;
    out[D + d] = lo;
    if (pool != nullptr) {
      // the mean the planes hold, in K's format, once per query head
      const float m = (ElemF16::to_f32(hi) + ElemF16::to_f32(lo)) * ldexpf(1.0f, -e);
      const uint16_t m16 = static_cast<uint16_t>(E::pack2(m, 0.f) & 0xFFFFu);
      for (int r = 0; r < rep; ++r)
        pool[(((static_cast<int64_t>(b) * Hk + h) * rep + r) * NB + blk) * D + d] = m16;
    }
  }
  if (threadIdx.x == 0) {
    float* descale = reinterpret_cast<float*>(planes + static_cast<int64_t>(B) * Hk * NB * 2 * D);
    descale[bid] = ldexpf(1.0f, -e);
  }
}

template <int D, typename E>
__global__ __launch_bounds__(256) void block_summary_kernel(
    const uint16_t* __restrict__ k, int64_t sk_b, int64_t sk_h, int64_t sk_n,
    int B, int Hk, int N, int NB, int mode, uint16_t* __restrict__ planes,
    uint16_t* __restrict__ pool, int rep) {
  constexpr int CH = D / 8;        // 16-byte chunks per row
  constexpr int RG = 256 / CH;     // row groups
  constexpr int RPG = kBlock / RG; // rows per group
  __shared__ float red[summary_red(D)];
  __shared__ uint32_t wmax[4];
  const int blk = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int c = threadIdx.x % CH, rg = threadIdx.x / CH;
  const uint16_t* base = k + b * sk_b + h * sk_h + static_cast<int64_t>(c) * 8;
  SummaryAcc acc;
#pragma unroll
  for (int r = 0; r < RPG; ++r) {
    const int row = blk * kBlock + r * RG + rg;
    u32x4 raw = {0u, 0u, 0u, 0u};
    if (row < N) raw = *reinterpret_cast<const u32x4*>(base + row * sk_n);
    acc.template add<E>(raw);
  }
  summary_store<D, E>(acc, red, wmax, b, h, blk, B, Hk, NB, mode, planes, pool, rep);
}

// The summary of a block and its K / V operand copies (kv_operand.h) in one
// pass: K is read once instead of twice, and a layer takes one launch less (4 us
// of 48 at 2K tokens; the accumulators see the rows in block_summary_kernel's
// order, so the planes are the same bits).  The reduction reuses the tiles' LDS.
template <int D, typename E>
__global__ __launch_bounds__(256) void summary_operand_kernel(
    const uint16_t* __restrict__ k, int64_t sk_b, int64_t sk_h, int64_t sk_n,
    const uint16_t* __restrict__ v, int64_t sv_b, int64_t sv_h, int64_t sv_n, int B, int Hk, int N,
    int NB, int mode, uint16_t* __restrict__ planes, uint16_t* __restrict__ kop,
    uint16_t* __restrict__ vop) {
  constexpr int CH = D / 8, RG = 256 / CH, RPG = kBlock / RG, ROW = D + 8;
  constexpr bool ONE = D > 128;    // K and V pass through one tile in turn
  constexpr int TILE = kBlock * ROW * 2, TILES = (ONE ? 1 : 2) * TILE;
  constexpr int BYTES = TILES > summary_red(D) * 4 ? TILES : summary_red(D) * 4;
  __shared__ __align__(16) unsigned char smem[BYTES];
  __shared__ uint32_t wmax[4];
  uint16_t (*kt)[ROW] = reinterpret_cast<uint16_t (*)[ROW]>(smem);
  uint16_t (*vt)[ROW] = reinterpret_cast<uint16_t (*)[ROW]>(smem + (ONE ? 0 : TILE));
  const int blk = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int c = threadIdx.x % CH, rg = threadIdx.x / CH;
  const uint16_t* kb = k + b * sk_b + h * sk_h + static_cast<int64_t>(c) * 8;
  const uint16_t* vb = v + b * sv_b + h * sv_h + static_cast<int64_t>(c) * 8;
  const int64_t base = ((static_cast<int64_t>(b) * Hk + h) * NB + blk) * kBlock * D;
  // rows past N are zeros
  auto row_of = [&](const uint16_t* p, int64_t stride, int r) -> u32x4 {
    const int64_t row = blk * kBlock + r * RG + rg;
    u32x4 x = {0u, 0u, 0u, 0u};
    if (row < N) x = *reinterpret_cast<const u32x4*>(p + row * stride);
    return x;
  };
  SummaryAcc acc;
#pragma unroll
  for (int r = 0; r < RPG; ++r) {
    const u32x4 x = row_of(kb, sk_n, r);
    acc.template add<E>(x);
    *reinterpret_cast<u32x4*>(&kt[r * RG + rg][c * 8]) = x;
    if constexpr (!ONE) *reinterpret_cast<u32x4*>(&vt[r * RG + rg][c * 8]) = row_of(vb, sv_n, r);
  }
  __syncthreads();
  write_k_slabs<D>(kt, kop + base);
  if constexpr (ONE) {
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RPG; ++r)
      *reinterpret_cast<u32x4*>(&vt[r * RG + rg][c * 8]) = row_of(vb, sv_n, r);
    __syncthreads();
  }
  write_vt_slabs<D>(vt, vop + base);
  __syncthreads();                 // the tiles are read: their LDS is the reduction's
  summary_store<D, E>(acc, reinterpret_cast<float*>(smem), wmax, b, h, blk, B, Hk, NB, mode, planes,
                      nullptr, 1);
}

template <typename E>
static hipError_t launch_block_summary_e(const uint16_t* k, int64_t sk_b, int64_t sk_h,
                                         int64_t sk_n, int B, int Hk, int N, int D, int mode,
                                         uint16_t* planes, uint16_t* pool, int rep,
                                         hipStream_t stream) {
  const int NB = (N + kBlock - 1) / kBlock;
  dim3 grid(NB, Hk, B);
  switch (D) {
    case 64:
      block_summary_kernel<64, E><<<grid, 256, 0, stream>>>(k, sk_b, sk_h, sk_n, B, Hk, N, NB, mode, planes, pool, rep);
      break;
    case 128:
      block_summary_kernel<128, E><<<grid, 256, 0, stream>>>(k, sk_b, sk_h, sk_n, B, Hk, N, NB, mode, planes, pool, rep);
      break;
    case 256:
      block_summary_kernel<256, E><<<grid, 256, 0, stream>>>(k, sk_b, sk_h, sk_n, B, Hk, N, NB, mode, planes, pool, rep);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_block_summary(const uint16_t* k, int64_t sk_b, int64_t sk_h, int64_t sk_n,
                                int B, int Hk, int N, int D, int elem, int mode,
                                uint16_t* planes, hipStream_t stream, uint16_t* pool,
                                int rep) {
  if (elem == ElemF16::code)
    return launch_block_summary_e<ElemF16>(k, sk_b, sk_h, sk_n, B, Hk, N, D, mode, planes, pool, rep, stream);
  return launch_block_summary_e<ElemBf16>(k, sk_b, sk_h, sk_n, B, Hk, N, D, mode, planes, pool, rep, stream);
}

// One launch for launch_block_summary and launch_attn_prepare (64-row tiles).
hipError_t launch_summary_operand(const uint16_t* k, int64_t sk_b, int64_t sk_h, int64_t sk_n,
                                  const uint16_t* v, int64_t sv_b, int64_t sv_h, int64_t sv_n,
                                  int B, int Hk, int N, int D, int elem, int mode,
                                  uint16_t* planes, uint16_t* ws, hipStream_t stream) {
  const int NB = (N + kBlock - 1) / kBlock;
  uint16_t* vop = ws + static_cast<int64_t>(B) * Hk * NB * kBlock * D;
  const dim3 grid(NB, Hk, B);
#define UGBSA_SO(E_, D_)                                                                          \
  summary_operand_kernel<D_, E_><<<grid, 256, 0, stream>>>(k, sk_b, sk_h, sk_n, v, sv_b, sv_h, sv_n, \
                                                           B, Hk, N, NB, mode, planes, ws, vop)
  if (elem == ElemF16::code) {
    if (D == 64) UGBSA_SO(ElemF16, 64);
    else if (D == 128) UGBSA_SO(ElemF16, 128);
    else if (D == 256) UGBSA_SO(ElemF16, 256);
    else return hipErrorInvalidValue;
  } else {
    if (D == 64) UGBSA_SO(ElemBf16, 64);
    else if (D == 128) UGBSA_SO(ElemBf16, 128);
    else if (D == 256) UGBSA_SO(ElemBf16, 256);
    else return hipErrorInvalidValue;
  }
#undef UGBSA_SO
  return hipGetLastError();
}

}  // namespace ugbsa
