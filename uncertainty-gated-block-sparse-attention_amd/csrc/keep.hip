// keep mask -> per-tile kv_idx and row masks (the v1 path's compaction).
//
// Restates _compute_kv_idx (src/triton_block_attn.py:125-146): per (b, h,
// Q tile of block_m rows) the blocks that any row of the tile keeps, in
// ascending order, padded with the sentinel NB, and their count (the host
// takes the maximum, as the reference's MAX_KEPT).  Rows past M are the
// reference's F.pad rows and keep nothing.  Beside each listed block it
// writes the mask of the tile rows that keep it (bit r: row t * block_m + r)
// — the per-row keep test of the reference kernel (:87-103), read by the
// attention kernels once per block instead of once per row.
//
// One workgroup per tile, a wavefront per 8 of its rows (eight or four): a lane
// owns WB consecutive blocks (one WB-byte word per row, the eight words requested
// together) and leaves its rows' bits of each block in LDS, a byte of the block's
// mask.  Then the workgroup compacts the section 64 blocks a wavefront at a time.
// Latency-bound at the per-row lengths seen (64 to 512 blocks).  GPU us, 64-row
// tiles, by a wavefront a tile (8 rows at a time, its 8-byte words leaving 56
// lanes idle at 64 blocks) / four wavefronts of 16 rows / eight of 8: 28 heads x
// 4K rows x 64 blocks 22.0 / 9.2 / 8.6; 8 x 10007 x 157 27.2 / 16.3 / 11.1; 40 x
// 20000 x 313 325 / 364 / 225; 64 x 16384 x 256 96.7 / 102 / 92.5 (the 16 words
// of 16 rows cost registers, three wavefronts a SIMD).  32-row tiles, with
// four of 16 rows (two without rows) / four of 8: 40 x 6000 x 94 36.0 / 52.8 /
// 22.5; 2 x 8 x 20000 x 313 111 / 190 / 69.
#include "common.h"
#include "launch.h"

namespace ugbsa {

constexpr int kKeepSection = 1024;    // blocks whose masks LDS holds at once

// WB bytes (blocks) per lane and row: 8 or 4 where rows and the mask are
// multiples of it and the row is long enough to give most lanes a word, else 1.
// BM: rows per tile, 64 or 32.
template <int WB, int BM>
__global__ __launch_bounds__(8 * BM) void keep_kv_idx_kernel(
    const uint8_t* __restrict__ keep, int64_t tiles, int M, int NB, int Qt,
    int32_t* __restrict__ kv_idx, uint64_t* __restrict__ rowmask, int32_t* __restrict__ counts) {
  constexpr int RW = 8, NW = BM / RW;    // rows per wavefront, wavefronts
  using Mask = std::conditional_t<BM == 64, uint64_t, uint32_t>;
  __shared__ __align__(8) uint8_t s_mask[kKeepSection][NW];   // one Mask per block
  __shared__ int s_cnt[NW];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t unit = static_cast<int64_t>(blockIdx.y) * gridDim.x + blockIdx.x;
  if (unit >= tiles) return;
  const int64_t bh = unit / Qt;
  const int t = static_cast<int>(unit % Qt);
  const int rows = min(BM, M - t * BM);
  const int r0 = wave * RW;
  const uint8_t* kb = keep + (bh * M + static_cast<int64_t>(t) * BM + r0) * NB;
  int32_t* out = kv_idx + unit * NB;
  uint64_t* rm = rowmask != nullptr ? rowmask + unit * NB : nullptr;
  const uint64_t lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  int cnt = 0;
  for (int base = 0; base < NB; base += kKeepSection) {
    const int n = min(kKeepSection, NB - base);
    if (base > 0) __syncthreads();       // the section before is compacted
    for (int c = WB * lane; c < n; c += 64 * WB) {
      uint32_t mk[WB];
#pragma unroll
      for (int i = 0; i < WB; ++i) mk[i] = 0u;
      uint64_t w[RW];
#pragma unroll
      for (int r = 0; r < RW; ++r) {
        const uint8_t* src = kb + static_cast<int64_t>(r) * NB + base + c;
        w[r] = 0ull;
        if (r0 + r < rows) {
          if constexpr (WB == 8) w[r] = *reinterpret_cast<const uint64_t*>(src);
          else if constexpr (WB == 4) w[r] = *reinterpret_cast<const uint32_t*>(src);
          else w[r] = *src;
        }
      }
#pragma unroll
      for (int r = 0; r < RW; ++r)
#pragma unroll
        for (int i = 0; i < WB; ++i)
          mk[i] |= static_cast<uint32_t>(((w[r] >> (8 * i)) & 0xFFull) != 0) << r;
#pragma unroll
      for (int i = 0; i < WB; ++i) s_mask[c + i][wave] = static_cast<uint8_t>(mk[i]);
    }
    __syncthreads();
    for (int c = 0; c < n; c += 64 * NW) {
      const int i = c + threadIdx.x;
      const uint64_t mask = i < n ? *reinterpret_cast<const Mask*>(s_mask[i]) : 0u;
      const uint64_t bal = __ballot(mask != 0ull);
      if (c > 0) __syncthreads();        // the counts of the step before are read
      if (lane == 0) s_cnt[wave] = __popcll(bal);
      __syncthreads();
      int pos = cnt + __popcll(bal & lt_mask);
#pragma unroll
      for (int v = 0; v < NW; ++v) {
        pos += v < wave ? s_cnt[v] : 0;
        cnt += s_cnt[v];
      }
      if (mask != 0ull) {
        out[pos] = base + i;
        if (rm != nullptr) rm[pos] = mask;
      }
    }
  }
  for (int s = cnt + threadIdx.x; s < NB; s += 64 * NW) {
    out[s] = NB;
    if (rm != nullptr) rm[s] = 0ull;
  }
  if (threadIdx.x == 0) counts[unit] = cnt;
}

template <int BM>
static void launch_keep_t(const uint8_t* keep, int B, int H, int M, int NB, int32_t* kv_idx,
                          uint64_t* rowmask, int32_t* counts, hipStream_t stream) {
  const int Qt = (M + BM - 1) / BM;
  const int64_t tiles = static_cast<int64_t>(B) * H * Qt;
  // rows of 2^20 workgroups: a launch dimension holds less than 2^32 threads
  const int64_t per_row = tiles < (1 << 20) ? tiles : 1 << 20;
  const dim3 grid(static_cast<unsigned>(per_row), static_cast<unsigned>((tiles + per_row - 1) / per_row));
  const uintptr_t at = reinterpret_cast<uintptr_t>(keep);
  if (NB % 8 == 0 && at % 8 == 0 && NB >= 256)
    keep_kv_idx_kernel<8, BM><<<grid, 8 * BM, 0, stream>>>(keep, tiles, M, NB, Qt, kv_idx, rowmask, counts);
  else if (NB % 4 == 0 && at % 4 == 0 && NB >= 128)
    keep_kv_idx_kernel<4, BM><<<grid, 8 * BM, 0, stream>>>(keep, tiles, M, NB, Qt, kv_idx, rowmask, counts);
  else
    keep_kv_idx_kernel<1, BM><<<grid, 8 * BM, 0, stream>>>(keep, tiles, M, NB, Qt, kv_idx, rowmask, counts);
}

hipError_t launch_keep_kv_idx(const uint8_t* keep, int B, int H, int M, int NB, int block_m,
                              int32_t* kv_idx, uint64_t* rowmask, int32_t* counts,
                              hipStream_t stream) {
  if (block_m == 64) launch_keep_t<64>(keep, B, H, M, NB, kv_idx, rowmask, counts, stream);
  else if (block_m == 32) launch_keep_t<32>(keep, B, H, M, NB, kv_idx, rowmask, counts, stream);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace ugbsa
