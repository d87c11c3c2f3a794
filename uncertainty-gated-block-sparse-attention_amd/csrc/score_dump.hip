// Score-noise estimate of the score dump (tau_hat per (b, h)).
//
// Restates src/dump_block_scores.py:181-194 of the reference: for
// n_pairs = min(1024, M - 1) adjacent query-row pairs (i, i + 1) with
// i = min(p * max(1, (M - 1) / n_pairs), M - 2), the per-row block scores
// S[i, blk] (the selection's row score of :638-648, over every one of the NB
// blocks, no causal mask) give
//     tau_hat = sqrt(max(0, 0.5 * mean_{pairs, blk} (S[i + 1, blk] - S[i, blk])^2)),
// and 0 when M < 2.
//
// A wavefront takes 8 * MT pairs at a time as an MFMA A operand of 16 * MT
// rows ordered (lo, hi) per pair, so that a 16 x 16 accumulator tile holds a
// pair's two rows in lane elements (0, 1) and (2, 3): the differences need no
// lane exchange.  (Mean planes: fp16 Q scaled per wave pass and the blocks'
// scales undone on the sums, as in the selection kernel.)
//
// A workgroup is kTauWaves such wavefronts (pair groups) of one (b, h) over
// one range of the blocks; the ranges are as many as fill the chip.  The KV
// head's summary planes pass through LDS for all of its wavefronts, a chunk
// fetched into registers while the one before is scored.  28 heads, 32K
// tokens, Quest planes: one workgroup per (b, h), which left 228 of 256 CUs
// idle, 233 us; split over the chip with every wavefront reading the planes
// from L2 (64-byte pieces of 16 rows an instruction) 41 us; through LDS 25 us
// (0.6 PFLOP/s, launch ramp included).  Squares are summed per lane in fp64,
// then over lanes and waves; the workgroup's fp64 sum goes whole, as its upper
// and lower 32 bits, to part_hi / part_lo, and score_tau_reduce_kernel adds the
// sums in a fixed order, so the result is deterministic.
#include "common.h"
#include "launch.h"

namespace ugbsa {

constexpr int kTauWaves = 8;
constexpr int kTauMaxPairs = 1024;   // n_pairs cap of the reference
constexpr int kTauTarget = 512;      // workgroups that fill the chip

// Blocks per LDS chunk: 16 KiB of planes (8 at head_dim 64).
__host__ __device__ constexpr int tau_chunk(int D) { return D > 128 ? 16 : 32; }

template <typename E, int D, bool QUEST, int MT>
__global__ __launch_bounds__(64 * kTauWaves) void score_tau_kernel(
    const uint16_t* __restrict__ q, int64_t sq_b, int64_t sq_h, int64_t sq_m,
    const uint16_t* __restrict__ planes, const float* __restrict__ bscale, int Hk, int M, int NB,
    int grp, int n_pairs, int stride, float scaling, int nb_range, int64_t part_stride,
    uint32_t* __restrict__ part_hi, uint32_t* __restrict__ part_lo) {
  constexpr int KS = D / 32;
  constexpr int P = 2;
  constexpr int QSETS = QUEST ? 2 : 1;
  using EM = std::conditional_t<QUEST, E, ElemF16>;
  constexpr int PAIRS = 8 * MT;                     // pairs per pass
  constexpr int CH = tau_chunk(D), NT = CH / 16;    // blocks per chunk
  constexpr int STRIDE = P * D + 8;                 // elements per chunk row in LDS
  constexpr int PPB = P * D / 8;                    // 16-byte pieces per block
  constexpr int STAGE = CH * PPB / (64 * kTauWaves);
  static_assert(STAGE * 64 * kTauWaves == CH * PPB, "whole pieces per thread");
  __shared__ double part[kTauWaves];
  __shared__ __align__(16) uint16_t chunk[2][CH * STRIDE];

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int g4 = lane >> 4, r16 = lane & 15;
  const int64_t bh = blockIdx.x;
  const int H = Hk * grp;
  const int b = static_cast<int>(bh / H), h = static_cast<int>(bh % H);
  const uint16_t* qb = q + b * sq_b + h * sq_h;
  const uint16_t* pl = planes + (static_cast<int64_t>(b) * Hk + h / grp) * NB * P * D;
  const float* bs = QUEST ? nullptr : bscale + (static_cast<int64_t>(b) * Hk + h / grp) * NB;

  const int pass = blockIdx.y * kTauWaves + wave;   // pairs past n_pairs score 0 on both rows
  bf16x8 qf[QSETS][MT][KS];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int pair = pass * PAIRS + 8 * mt + (r16 >> 1);
    const bool live = pair < n_pairs;
    const int row = live ? min(pair * stride, M - 2) + (r16 & 1) : 0;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const bf16x8 x = live ? load_bf16x8(qb + row * sq_m + 32 * ks + 8 * g4) : zero_bf16x8();
      if constexpr (QUEST) {
        qf[0][mt][ks] = bf16_pos(x);
        qf[QSETS - 1][mt][ks] = bf16_neg(x);
      } else {
        qf[0][mt][ks] = x;
      }
    }
  }
  float tdesc = 1.f;
  if constexpr (!QUEST) tdesc = q_tile_to_f16<E, MT * KS>(&qf[0][0][0], lane);

  const int nb0 = blockIdx.z * nb_range, nb1 = min(NB, nb0 + nb_range);
  u32x4 stage[STAGE];
  auto fetch = [&](int n0) {
#pragma unroll
    for (int j = 0; j < STAGE; ++j) {
      const int pi = threadIdx.x + j * 64 * kTauWaves;
      const int blk = n0 + pi / PPB;
      stage[j] = u32x4{0u, 0u, 0u, 0u};    // blocks past the range score 0
      if (blk < nb1)
        stage[j] = *reinterpret_cast<const u32x4*>(pl + static_cast<int64_t>(blk) * P * D + pi % PPB * 8);
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int j = 0; j < STAGE; ++j) {
      const int pi = threadIdx.x + j * 64 * kTauWaves;
      *reinterpret_cast<u32x4*>(&chunk[buf][pi / PPB * STRIDE + pi % PPB * 8]) = stage[j];
    }
  };
  double sum = 0.0;
  fetch(nb0);
  store(0);
  __syncthreads();
  int buf = 0;
  for (int n0 = nb0; n0 < nb1; n0 += CH, buf ^= 1) {
    const bool more = n0 + CH < nb1;
    if (more) fetch(n0 + CH);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int blk = n0 + 16 * nt + r16;
      const uint16_t* src = &chunk[buf][(16 * nt + r16) * STRIDE + 8 * g4];
      f32x4 acc[MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const bf16x8 bfr = *reinterpret_cast<const bf16x8*>(src + p * D + 32 * ks);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            acc[mt] = EM::mfma(qf[QUEST ? p : 0][mt][ks], bfr, acc[mt]);
        }
      // the exact factor from the sums to the scores of this lane's block
      const float cs = QUEST ? 1.f : (blk < nb1 ? bs[blk] : 0.f) * tdesc;
      // rows (4 g4 + 0, 4 g4 + 1) and (4 g4 + 2, 4 g4 + 3) are (lo, hi) of
      // two pairs
      float s2 = 0.f;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const float d0 = (acc[mt][1] * cs) * scaling - (acc[mt][0] * cs) * scaling;
        const float d1 = (acc[mt][3] * cs) * scaling - (acc[mt][2] * cs) * scaling;
        s2 += d0 * d0 + d1 * d1;
      }
      sum += static_cast<double>(s2);
    }
    if (more) store(buf ^ 1);    // last read before the previous barrier
    __syncthreads();
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) sum += __shfl_xor(sum, m, 64);
  if (lane == 0) part[wave] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    double tot = 0.0;
    for (int w = 0; w < kTauWaves; ++w) tot += part[w];
    const uint64_t bits = __builtin_bit_cast(uint64_t, tot);
    const int64_t at = bh * part_stride + blockIdx.z * gridDim.y + blockIdx.y;
    part_hi[at] = static_cast<uint32_t>(bits >> 32);
    part_lo[at] = static_cast<uint32_t>(bits);
  }
}

// tau_hat of one (b, h) from its workgroups' sums, added in their order.
__global__ __launch_bounds__(64) void score_tau_reduce_kernel(
    const uint32_t* __restrict__ part_hi, const uint32_t* __restrict__ part_lo,
    int64_t part_stride, int parts, int n_pairs, int NB, float* __restrict__ tau_hat) {
  if (threadIdx.x != 0) return;
  double tot = 0.0;
  const int64_t at = blockIdx.x * part_stride;
#pragma unroll 8
  for (int i = 0; i < parts; ++i)
    tot += __builtin_bit_cast(double, static_cast<uint64_t>(part_hi[at + i]) << 32 | part_lo[at + i]);
  float tau = 0.f;
  if (n_pairs > 0) {
    const float mean = static_cast<float>(tot / (static_cast<double>(n_pairs) * NB));
    const float tsq = 0.5f * mean;
    tau = sqrtf(tsq > 0.f ? tsq : 0.f);
  }
  tau_hat[blockIdx.x] = tau;
}

template <typename E, int D, bool QUEST>
static hipError_t launch_tau_t(const uint16_t* q, int64_t sq_b, int64_t sq_h, int64_t sq_m,
                               const uint16_t* planes, int B, int H, int Hk, int M, int N,
                               float scaling, float* scratch_a, float* scratch_b, float* tau_hat,
                               hipStream_t stream) {
  // A operands of 4 m-tiles while they fit in 128 VGPRs, else 2
  constexpr int MT = (QUEST ? 2 : 1) * 4 * (D / 32) * 4 <= 128 ? 4 : 2;
  const int NB = (N + kBlock - 1) / kBlock;
  const int n_pairs = M >= 2 ? (M - 1 < kTauMaxPairs ? M - 1 : kTauMaxPairs) : 0;
  const int stride = n_pairs > 0 ? ((M - 1) / n_pairs > 1 ? (M - 1) / n_pairs : 1) : 1;
  // groups of kTauWaves passes x ranges of the blocks (whole chunks):
  // as many ranges as make kTauTarget workgroups.  Each workgroup's sum has a
  // place among the (b, h)'s Qt scratch values: groups <= Qt, as a pass of
  // 8 MT >= 16 pairs spans at least 16 of the M - 1 rows.
  const int Qt = (M + kBlock - 1) / kBlock;
  uint32_t* part_hi = reinterpret_cast<uint32_t*>(scratch_a);
  uint32_t* part_lo = reinterpret_cast<uint32_t*>(scratch_b);
  const int groups = n_pairs > 0 ? ((n_pairs + 8 * MT - 1) / (8 * MT) + kTauWaves - 1) / kTauWaves : 0;
  int ranges = 1;
  if (groups > 0) {
    const int steps = (NB + tau_chunk(D) - 1) / tau_chunk(D);
    const int64_t wgs = static_cast<int64_t>(B) * H * groups;
    int64_t want = (kTauTarget + wgs - 1) / wgs;
    if (want > steps) want = steps;
    if (want > Qt / groups) want = Qt / groups;
    if (want < 1) want = 1;
    const int per = (steps + static_cast<int>(want) - 1) / static_cast<int>(want);
    ranges = (steps + per - 1) / per;
    score_tau_kernel<E, D, QUEST, MT><<<dim3(static_cast<unsigned>(B * H), groups, ranges),
                                        64 * kTauWaves, 0, stream>>>(
        q, sq_b, sq_h, sq_m, planes, QUEST ? nullptr : mean_descale(planes, B, Hk, NB, D), Hk, M,
        NB, H / Hk, n_pairs, stride, scaling, tau_chunk(D) * per, Qt, part_hi, part_lo);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  score_tau_reduce_kernel<<<dim3(static_cast<unsigned>(B * H)), 64, 0, stream>>>(
      part_hi, part_lo, Qt, groups * ranges, n_pairs, NB, tau_hat);
  return hipGetLastError();
}

template <typename E>
static hipError_t launch_score_tau_e(const uint16_t* q, int64_t sq_b, int64_t sq_h,
                                     int64_t sq_m, const uint16_t* planes, int B, int H, int Hk,
                                     int M, int N, int D, int mode, float scaling,
                                     float* scratch_a, float* scratch_b, float* tau_hat,
                                     hipStream_t stream) {
  const bool quest = mode == kModeQuest;
#define UGBSA_TAU(D_)                                                                          \
  return quest ? launch_tau_t<E, D_, true>(q, sq_b, sq_h, sq_m, planes, B, H, Hk, M, N, scaling,   \
                                        scratch_a, scratch_b, tau_hat, stream)                                        \
               : launch_tau_t<E, D_, false>(q, sq_b, sq_h, sq_m, planes, B, H, Hk, M, N, scaling,   \
                                        scratch_a, scratch_b, tau_hat, stream)
  if (D == 64) UGBSA_TAU(64);
  if (D == 128) UGBSA_TAU(128);
  if (D == 256) UGBSA_TAU(256);
#undef UGBSA_TAU
  return hipErrorInvalidValue;
}

hipError_t launch_score_tau(const uint16_t* q, int64_t sq_b, int64_t sq_h, int64_t sq_m,
                            const uint16_t* planes, int B, int H, int Hk, int M, int N, int D,
                            int elem, int mode, float scaling, float* scratch_a,
                            float* scratch_b, float* tau_hat, hipStream_t stream) {
  if (elem == ElemF16::code)
    return launch_score_tau_e<ElemF16>(q, sq_b, sq_h, sq_m, planes, B, H, Hk, M, N, D, mode,
                                       scaling, scratch_a, scratch_b, tau_hat, stream);
  return launch_score_tau_e<ElemBf16>(q, sq_b, sq_h, sq_m, planes, B, H, Hk, M, N, D, mode,
                                      scaling, scratch_a, scratch_b, tau_hat, stream);
}

}  // namespace ugbsa
