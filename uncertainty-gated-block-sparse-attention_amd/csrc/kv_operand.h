// The K / V operand order of the pipelined attention kernel, shared by the
// kernels that write it (256-thread workgroups, one 64-key block each).
#pragma once

#include "common.h"

namespace ugbsa {

// K and V of one 64-key block in the pipelined kernel's operand order: for
// each 32-key half block, K as 2 (mt) x KS 1 KiB slabs and V^T as DT 1 KiB
// slabs, where lane L's 16 bytes sit at 16 * L of its slab.  K slab (mt, ks)
// lane (g4, r16) = K[key 8 * (r16 >> 2) + 4 * mt + (r16 & 3)][32 * ks + 8 * g4 ..];
// V^T slab dt lane (g4, r16) = V[keys 8 * g4 .. 8 * g4 + 7][16 * dt + r16].
// Every operand load of the attention loop is then one contiguous KiB.
template <int D>
__device__ __forceinline__ void write_k_slabs(const uint16_t (*kt)[D + 8], uint16_t* __restrict__ dst) {
  constexpr int KS = D / 32;
  // K: 2 halves x 2 mt x KS slabs x 64 lanes
#pragma unroll 2
  for (int i = threadIdx.x; i < 2 * 2 * KS * 64; i += 256) {
    const int lane = i & 63, slab = i >> 6;
    const int ks = slab % KS, mt = (slab / KS) & 1, half = slab / (2 * KS);
    const int g4 = lane >> 4, r16 = lane & 15;
    const int key = 32 * half + 8 * (r16 >> 2) + 4 * mt + (r16 & 3);
    *reinterpret_cast<u32x4*>(dst + static_cast<int64_t>(i) * 8) =
        *reinterpret_cast<const u32x4*>(&kt[key][32 * ks + 8 * g4]);
  }
}

template <int D>
__device__ __forceinline__ void write_vt_slabs(const uint16_t (*vt)[D + 8], uint16_t* __restrict__ dst) {
  constexpr int DT = D / 16;
  // V^T: 2 halves x DT slabs x 64 lanes
#pragma unroll 2
  for (int i = threadIdx.x; i < 2 * DT * 64; i += 256) {
    const int lane = i & 63, slab = i >> 6;
    const int dt = slab % DT, half = slab / DT;
    const int g4 = lane >> 4, r16 = lane & 15;
    i16x8 w;
#pragma unroll
    for (int j = 0; j < 8; ++j) w[j] = static_cast<short>(vt[32 * half + 8 * g4 + j][16 * dt + r16]);
    *reinterpret_cast<i16x8*>(dst + static_cast<int64_t>(i) * 8) = w;
  }
}

}  // namespace ugbsa
