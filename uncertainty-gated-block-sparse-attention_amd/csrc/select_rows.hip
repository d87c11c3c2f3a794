// v1 per-row selection (src/sparse_attention.py:245-295, 299-325 for the
// margin) over a buffer of per-row block scores.
//
// One wavefront takes kRowsPerWave consecutive query rows.  A row's visible
// scores (blocks 0 .. row / 64, M == N) sit in registers as order-preserving
// keys, RK consecutive blocks per lane, RK the smallest power of two that
// holds the row.  The K-th best key is found by building it bit by bit from
// the top: a candidate threshold is kept when at least K keys reach it, counted
// by one compare per register and the scalar unit's bit counts, and the search
// ends as soon as exactly K do.  The kept blocks are then the keys at or
// above the threshold; when more than K are (ties at the cut), the first of the
// equal ones in block order.  No histogram, no sort and no LDS for the top-k
// policies: this kernel is bound by instruction issue (one row of 64 blocks is
// a few dozen VALU instructions).  Beside the kept set the margin needs only
// three ranks: the best key, the smallest key of the k_eff best and the
// largest of the rest.
//
// count = k_bud, or for belief clamp(#{j : cumsum_j < top_p} + 1, k_min,
// k_max) over the sorted softmax probabilities (the K best keys are compacted
// into LDS and sorted, 32-bit keys only); then ranks past the visible blocks
// take the lowest invisible blocks (the total order's -inf ties), and the sink
// and the row's own block are forced.
//
// 28 heads x 4096 rows x 64 blocks: 35 us (a radix select through LDS
// histograms, a 64-bit sort and LDS flags took 119); 8 x 10007 x 157, belief:
// 91 us (117).
#include "common.h"
#include "launch.h"

namespace ugbsa {

constexpr int kRowsPerWave = 4;     // divides 64: the rows of a wave share their visible blocks
constexpr int kRowsWaves = 4;       // wavefronts per workgroup

struct KeyCut {
  uint32_t t;      // the largest threshold that at least K keys reach
  int n_ge;        // keys at or above it (more than K: ties at the cut)
};

// The cut of the K best of the wavefront's keys (K < their number; unused
// slots hold key 0, below every score's).
template <int RK>
__device__ __forceinline__ KeyCut key_cut(const uint32_t (&key)[RK], int K) {
  KeyCut r{0u, 64 * RK};
  for (int bit = 31; bit >= 0; --bit) {
    const uint32_t c = r.t | (1u << bit);
    int n = 0;
#pragma unroll
    for (int j = 0; j < RK; ++j) n += __popcll(__ballot(key[j] >= c));
    if (n >= K) {
      r.t = c;
      r.n_ge = n;
      if (n == K) break;
    }
  }
  return r;
}

// Descending bitonic sort of the first KP keys of v, element e = lane + 64 r.
template <int KP, int RT>
__device__ __forceinline__ void bitonic_keys(uint32_t (&v)[RT], int lane) {
  constexpr int R = KP / 64;
  constexpr int LOG_KP = KP == 64 ? 6 : KP == 128 ? 7 : KP == 256 ? 8 : 9;
  static_assert((1 << LOG_KP) == KP && R <= RT, "KP is a power of two within v");
  static_for<LOG_KP>([&](auto lk) {
    constexpr int kk = 2 << decltype(lk)::value;
    static_for<decltype(lk)::value + 1>([&](auto lj) {
      constexpr int j = (kk >> 1) >> decltype(lj)::value;
      uint32_t nv[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int e = lane + 64 * r;
        uint32_t other;
        if constexpr (j >= 64) other = v[r ^ (j >> 6)];
        else other = xor_lanes<j>(v[r], lane);
        const bool keep_max = ((e & j) == 0) == ((e & kk) == 0);
        nv[r] = keep_max ? max(v[r], other) : min(v[r], other);
      }
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = nv[r];
    });
  });
}

// Sorts the n keys of v (the rest are 0), as few of its registers as hold them
// (rows of up to 64 blocks have a body of their own).
template <int KP>
__device__ __forceinline__ void sort_keys(uint32_t (&v)[KP / 64], int n, int lane) {
  if constexpr (KP > 128) {
    if (n <= 128) return bitonic_keys<128>(v, lane);
  }
  if constexpr (KP > 256) {
    if (n <= 256) return bitonic_keys<256>(v, lane);
  }
  bitonic_keys<KP>(v, lane);
}

// Key of rank e (0 = best) of a sorted v.
template <int R>
__device__ __forceinline__ uint32_t sorted_key(const uint32_t (&v)[R], int e) {
  uint32_t x = 0;
#pragma unroll
  for (int r = 0; r < R; ++r)
    if (r == (e >> 6)) x = v[r];
  return static_cast<uint32_t>(__shfl(static_cast<int>(x), e & 63, 64));
}

// The belief budget of a row: its K best keys sorted, and the clamp of (sorted
// probabilities whose running sum stays below top_p) + 1.  Leaves the key of
// rank count - 1 in cut.t.
template <int RK, int KP>
__device__ __forceinline__ int belief_count(const RowsArgs& a, const float (&x)[RK],
                                            const uint32_t (&key)[RK], int n_vis, uint32_t* cand,
                                            int lane, uint32_t& cut_key) {
  constexpr int R = KP / 64;
  const int n_sel = min(n_vis, a.K);
  // the K best keys (any order; of those equal at the cut, any) into cand
  KeyCut kc{1u, n_vis};
  if (n_vis > a.K) kc = key_cut<RK>(key, a.K);
  int at = 0;
#pragma unroll
  for (int j = 0; j < RK; ++j) {
    const bool take = kc.n_ge == n_sel ? key[j] >= kc.t : key[j] > kc.t;
    const uint64_t bal = __ballot(take);
    if (take) cand[at + lanes_below(bal)] = key[j];
    at += __popcll(bal);
  }
  for (int e = at + lane; e < n_sel; e += 64) cand[e] = kc.t;   // ties at the cut
  wave_lds_sync();
  uint32_t v[R];
#pragma unroll
  for (int r = 0; r < R; ++r) v[r] = lane + 64 * r < n_sel ? cand[lane + 64 * r] : 0u;
  wave_lds_sync();
  sort_keys<KP>(v, n_sel, lane);

  // softmax over the visible blocks (max-subtracted, fp32), then the
  // cumulative mass of the sorted probabilities
  const float mx = key_float(sorted_key<R>(v, 0));
  float z = 0.f;
#pragma unroll
  for (int j = 0; j < RK; ++j) z += RK * lane + j < n_vis ? expf(x[j] - mx) : 0.f;
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) z += shfl_xor_f(z, m);
  float carry = 0.f;
  int cnt = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int e = lane + 64 * r;
    float c = e < n_sel ? expf(key_float(v[r]) - mx) / z : 0.f;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const float o = __shfl_up(c, d, 64);
      if (lane >= d) c += o;
    }
    c += carry;
    carry = __shfl(c, 63, 64);
    cnt += __popcll(__ballot(e < a.K && c < a.top_p));
  }
  // ranks past the sorted keys (none visible) add no mass: all of them count, or none
  if (a.K > KP && carry < a.top_p) cnt += a.K - KP;
  int count = cnt + 1;
  if (count < a.k_min) count = a.k_min;
  if (count > a.k_max) count = a.k_max;
  if (count >= 1 && count < n_vis) cut_key = sorted_key<R>(v, count - 1);
  return count;
}

// RK scores of a row per lane from blk0 on (0 past n): 16-byte loads where rows
// are 16-byte multiples.
template <int RK>
__device__ __forceinline__ void load_scores(const float* src, int blk0, int n, bool wide,
                                            float (&x)[RK]) {
  if constexpr (RK >= 4) {
    if (wide) {
#pragma unroll
      for (int j = 0; j < RK; j += 4) {
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
        if (blk0 + j < n) v = *reinterpret_cast<const f32x4*>(src + blk0 + j);   // row end: NB % 4 == 0
#pragma unroll
        for (int i = 0; i < 4; ++i) x[j + i] = v[i];
      }
      return;
    }
  }
#pragma unroll
  for (int j = 0; j < RK; ++j) x[j] = blk0 + j < n ? src[blk0 + j] : 0.f;
}

// Rows row0 .. row0 + kRowsPerWave - 1 of (b, h) = bh (those below M).
template <int RK, bool BELIEF, int KP>
__device__ __forceinline__ void rows_body(const RowsArgs& a, int64_t bh, int row0, int n_vis,
                                          uint32_t* cand, int lane) {
  // rows loaded at once (the belief body is long: one)
  constexpr int BATCH = BELIEF ? 1 : RK <= 4 ? kRowsPerWave : RK <= 16 ? 2 : 1;
  const int NB = a.NB;
  const int blk0 = RK * lane;
  const bool wide = NB % 4 == 0 && (reinterpret_cast<uintptr_t>(a.scores) & 15) == 0;
  const int self = row0 / kBlock;
  const float* src0 = a.scores + (bh * a.nrows + (row0 - a.r0)) * NB;
#pragma unroll 1
  for (int rb = 0; rb < kRowsPerWave; rb += BATCH) {
    float xs[BATCH][RK];
#pragma unroll
    for (int i = 0; i < BATCH; ++i)
      if (row0 + rb + i < a.M)
        load_scores<RK>(src0 + static_cast<int64_t>(rb + i) * NB, blk0, n_vis, wide, xs[i]);
#pragma unroll
    for (int i = 0; i < BATCH; ++i) {
      const int row = row0 + rb + i;
      if (row >= a.M) return;
      float (&x)[RK] = xs[i];
      if (a.penalty != nullptr && row == a.M - 1) {
        const float* pen = a.penalty + (bh % a.H) * NB;
#pragma unroll
        for (int j = 0; j < RK; ++j)
          if (blk0 + j < n_vis) x[j] -= pen[blk0 + j];
      }
      uint32_t key[RK];
#pragma unroll
      for (int j = 0; j < RK; ++j) key[j] = blk0 + j < n_vis ? float_key(x[j]) : 0u;

      int count = a.k_bud;
      KeyCut cut{1u, n_vis};               // every visible block
      if constexpr (BELIEF) {
        // (RK 1: at most 64 visible blocks, so 64 sorted keys, whatever K is)
        count = belief_count<RK, RK == 1 ? 64 : KP>(a, x, key, n_vis, cand, lane, cut.t);
        if (count < n_vis) {
          cut.n_ge = 0;
#pragma unroll
          for (int j = 0; j < RK; ++j) cut.n_ge += __popcll(__ballot(key[j] >= cut.t));
        }
      } else if (n_vis > count) {
        cut = key_cut<RK>(key, count);
      }

      // keep bytes of the lane's RK blocks
      uint32_t flag[RK];
      if (cut.n_ge <= count) {
#pragma unroll
        for (int j = 0; j < RK; ++j) flag[j] = key[j] >= cut.t ? 1u : 0u;
      } else {                             // ties: the first of the equal keys in block order
        uint32_t eq = 0;
        int n_eq = 0;
#pragma unroll
        for (int j = 0; j < RK; ++j) {
          eq += key[j] == cut.t ? 1u : 0u;
          n_eq += __popcll(__ballot(key[j] == cut.t));
        }
        const int need = count - (cut.n_ge - n_eq);
        int at = static_cast<int>(wave_excl_scan(eq, lane));
#pragma unroll
        for (int j = 0; j < RK; ++j) {
          const bool e = key[j] == cut.t;
          flag[j] = key[j] > cut.t || (e && at < need) ? 1u : 0u;
          at += e ? 1 : 0;
        }
      }
      uint8_t* kr = a.keep + (bh * a.M + row) * NB;
#pragma unroll
      for (int j = 0; j < RK; ++j) {
        const int blk = blk0 + j;
        if (blk == 0 || blk == self || (blk >= n_vis && blk < count)) flag[j] = 1u;
      }
      constexpr int U = RK < 8 ? RK : 8;   // bytes per store
      if (NB % U == 0 && (reinterpret_cast<uintptr_t>(a.keep) & (U - 1)) == 0) {
#pragma unroll
        for (int j = 0; j < RK; j += U) {
          if (blk0 + j >= NB) break;
          if constexpr (U == 8) {
            uint2 w = {0u, 0u};
#pragma unroll
            for (int i2 = 0; i2 < 4; ++i2) {
              w.x |= flag[j + i2] << (8 * i2);
              w.y |= flag[j + 4 + i2] << (8 * i2);
            }
            *reinterpret_cast<uint2*>(kr + blk0 + j) = w;
          } else if constexpr (U == 4) {
            *reinterpret_cast<uint32_t*>(kr + blk0) = flag[0] | flag[1] << 8 | flag[2] << 16 | flag[3] << 24;
          } else if constexpr (U == 2) {
            *reinterpret_cast<uint16_t*>(kr + blk0) = static_cast<uint16_t>(flag[0] | flag[1] << 8);
          } else {
            kr[blk0] = static_cast<uint8_t>(flag[0]);
          }
        }
      } else {
#pragma unroll
        for (int j = 0; j < RK; ++j)
          if (blk0 + j < NB) kr[blk0 + j] = static_cast<uint8_t>(flag[j]);
      }
      // blocks past the lanes' (none visible): those below count, else zero
      if (NB % 8 == 0 && (reinterpret_cast<uintptr_t>(a.keep) & 7) == 0) {
        for (int b0 = 64 * RK + 8 * lane; b0 < NB; b0 += 512) {
          uint64_t w = 0;
#pragma unroll
          for (int i2 = 0; i2 < 8; ++i2) w |= static_cast<uint64_t>(b0 + i2 < count) << (8 * i2);
          *reinterpret_cast<uint64_t*>(kr + b0) = w;
        }
      } else {
        for (int blk = 64 * RK + lane; blk < NB; blk += 64) kr[blk] = blk < count ? 1 : 0;
      }

      if (a.margin != nullptr) {
        // (s[k_eff - 1] - s[k_eff]) / max(s[0] - s[k_eff], 1e-6), -inf at
        // ranks past the visible blocks; NaN kept
        uint32_t top = 0, low = 0xFFFFFFFFu, rest = 0;
        KeyCut mc{1u, n_vis};
        if (n_vis > a.k_eff) mc = !BELIEF && a.k_eff == count ? cut : key_cut<RK>(key, a.k_eff);
#pragma unroll
        for (int j = 0; j < RK; ++j) {
          top = max(top, key[j]);
          if (key[j] >= mc.t) low = min(low, key[j]);
          else rest = max(rest, key[j]);
        }
        const float s_top = key_float(wave_max_u32(top, lane));
        float s_km1 = -INFINITY, s_k = -INFINITY;
        if (n_vis > a.k_eff) {
          // more than k_eff keys at the cut value or above: ranks k_eff - 1
          // and k_eff both hold it
          const bool tie = mc.n_ge > a.k_eff;
          const uint32_t lo = ~wave_max_u32(~low, lane), hi = wave_max_u32(rest, lane);
          s_km1 = key_float(tie ? mc.t : lo);
          s_k = key_float(tie ? mc.t : hi);
        } else if (n_vis == a.k_eff) {
          s_km1 = key_float(~wave_max_u32(~low, lane));
        }
        float spread = s_top - s_k;
        if (spread < 1e-6f) spread = 1e-6f;
        const float mg = (s_km1 - s_k) / spread;
        if (lane == 0) a.margin[bh * a.M + row] = mg;
      }
    }
  }
}

// Wavefronts per SIMD: the belief body's keys and scores of long rows would leave
// one or two. Held to two at 64 keys a lane it spills 28-68 bytes and is the
// faster all the same (1 head x 200K tokens 5.29 -> 3.84 ms; three at 32, 2 heads x
// 131K 2.19 -> 1.77).
constexpr int rows_eu_waves(int rkmax, bool belief) {
  return !belief ? 1 : rkmax == 64 ? 2 : rkmax == 32 ? 3 : 1;
}

template <int RKMAX, bool BELIEF, int KP>
__global__ __launch_bounds__(64 * kRowsWaves, rows_eu_waves(RKMAX, BELIEF)) void select_rows_kernel(const RowsArgs a) {
  __shared__ uint32_t s_cand[BELIEF ? kRowsWaves * KP : 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // one wave-uniform group of rows: row indices and branches stay scalar
  const int64_t gid = static_cast<int64_t>(blockIdx.x) * kRowsWaves +
                      __builtin_amdgcn_readfirstlane(wave);
  const int per_bh = a.nrows / kRowsPerWave;
  if (gid >= static_cast<int64_t>(a.B) * a.H * per_bh) return;
  const int64_t bh = gid / per_bh;
  const int row0 = a.r0 + static_cast<int>(gid % per_bh) * kRowsPerWave;
  if (row0 >= a.M) return;
  const int n_vis = row0 / kBlock + 1;      // the same for the wave's rows
  uint32_t* cand = s_cand + (BELIEF ? wave * KP : 0);
  if (RKMAX == 1 || n_vis <= 64) return rows_body<1, BELIEF, KP>(a, bh, row0, n_vis, cand, lane);
  if constexpr (RKMAX >= 2) {
    if (RKMAX == 2 || n_vis <= 128) return rows_body<2, BELIEF, KP>(a, bh, row0, n_vis, cand, lane);
  }
  if constexpr (RKMAX >= 4) {
    if (RKMAX == 4 || n_vis <= 256) return rows_body<4, BELIEF, KP>(a, bh, row0, n_vis, cand, lane);
  }
  if constexpr (RKMAX >= 8) {
    if (RKMAX == 8 || n_vis <= 512) return rows_body<8, BELIEF, KP>(a, bh, row0, n_vis, cand, lane);
  }
  if constexpr (RKMAX >= 16) {
    if (RKMAX == 16 || n_vis <= 1024) return rows_body<16, BELIEF, KP>(a, bh, row0, n_vis, cand, lane);
  }
  if constexpr (RKMAX >= 32) {
    if (RKMAX == 32 || n_vis <= 2048) return rows_body<32, BELIEF, KP>(a, bh, row0, n_vis, cand, lane);
  }
  if constexpr (RKMAX >= 64) rows_body<64, BELIEF, KP>(a, bh, row0, n_vis, cand, lane);
}

template <int RKMAX, bool BELIEF, int KP>
static hipError_t launch_rows_t(const RowsArgs& a, hipStream_t stream) {
  const int64_t waves = static_cast<int64_t>(a.B) * a.H * (a.nrows / kRowsPerWave);
  const int64_t wgs = (waves + kRowsWaves - 1) / kRowsWaves;
  select_rows_kernel<RKMAX, BELIEF, KP>
      <<<dim3(static_cast<unsigned>(wgs)), 64 * kRowsWaves, 0, stream>>>(a);
  return hipGetLastError();
}

// The kernel of the row length: short rows keep fewer registers live, so more
// wavefronts share a SIMD.
template <bool BELIEF, int KP>
static hipError_t launch_rows_k(const RowsArgs& a, hipStream_t stream) {
  static_assert(kStreamBlocksRows <= 64 * 64, "the longest row fits 64 keys per lane");
  if (a.NB <= 128) return launch_rows_t<2, BELIEF, KP>(a, stream);
  if (a.NB <= 512) return launch_rows_t<8, BELIEF, KP>(a, stream);
  if (a.NB <= 1024) return launch_rows_t<16, BELIEF, KP>(a, stream);
  if (a.NB <= 2048) return launch_rows_t<32, BELIEF, KP>(a, stream);
  if (a.NB <= kStreamBlocksRows) return launch_rows_t<64, BELIEF, KP>(a, stream);
  return hipErrorInvalidValue;
}

hipError_t launch_select_rows(const RowsArgs& a, hipStream_t stream) {
  if (a.K > 512 || a.nrows % kBlock != 0) return hipErrorInvalidValue;
  if (!a.belief) return launch_rows_k<false, 64>(a, stream);
  // as many sorted keys as ranks are asked for (the default k_max, 112: 128): 8
  // heads x 10007 rows, k_max 200: 223 us with 512, 131 with 256; k_max 40: 111
  // with 128, 98 with 64
  if (a.K <= 64) return launch_rows_k<true, 64>(a, stream);
  if (a.K <= 128) return launch_rows_k<true, 128>(a, stream);
  if (a.K <= 256) return launch_rows_k<true, 256>(a, stream);
  return launch_rows_k<true, 512>(a, stream);
}

}  // namespace ugbsa
