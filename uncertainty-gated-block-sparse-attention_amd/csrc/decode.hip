// Decode attention: one query row per head against the whole K/V of its KV
// head (the dispatcher's Q == 1 branch, src/sparse_attention.py:757-767).
//
// Memory-bound: every K and V element is read once for the G = H / Hk query
// heads that share it.  A workgroup of four wavefronts takes one contiguous
// key range ("split") of one (b, KV head) and up to 16 of its query heads; a
// wavefront takes every fourth 32-key step of the range and computes
//     S^T[key, head] = K . Q^T      (A = K rows as they lie in memory)
//     O^T[d, head]  += V^T . P^T    (A = V^T, from V rows by register permutes)
// on 16x16x32 MFMAs with the heads as the 16 columns, so K/V go straight from
// global memory into operand registers: no LDS staging, no operand copy and
// no barrier in the loop.  Keys are labelled inside a step so that a lane's
// eight P^T values are the eight keys of its V^T operand (P stays in its
// lane, rounded to the element format as the flash kernels do), and the row
// maximum and sum of a head live in the head's lanes.
//
// V^T: lane (g4, r16) loads V[key 8 g4 + i][dims ...], i = 0 .. 7, with the 16
// lanes of a g4 group covering whole rows, and pairs the eight keys of each of
// its dims with v_perm: DPL operand fragments of four registers.
//
// The splits' partial (O, m, l) meet in decode_combine_kernel; a single split
// writes the output itself.  One call over 32K keys, 28/4 heads, head_dim 128
// (67 MB, 13 us at the rate of a large copy): 17 us; 131K keys 44 us (6.1
// TB/s).  The library's flash kernel, one workgroup per query head, takes
// 1151 us at 32K.
#include "common.h"
#include "launch.h"
#include "../../include/ugbsa.h"

namespace ugbsa {

constexpr int kDecWaves = 4;      // wavefronts per workgroup
constexpr int kDecStep = 32;      // keys per wavefront step
// Query heads per workgroup: the 16 MFMA columns; 8 at head_dim 256, where the
// wavefronts' O of 16 heads would take 66 KiB of LDS.
__host__ __device__ constexpr int dec_heads(int D) { return D > 128 ? 8 : 16; }

template <typename E, int D>
__global__ __launch_bounds__(64 * kDecWaves) void decode_kernel(
    const uint16_t* __restrict__ q, int64_t sq_b, int64_t sq_h, const uint16_t* __restrict__ k,
    int64_t sk_b, int64_t sk_h, int64_t sk_n, const uint16_t* __restrict__ v, int64_t sv_b,
    int64_t sv_h, int64_t sv_n, int Hk, int N, int grp, int chunks, int splits, int keys_per_split,
    float scale_log2, uint16_t* __restrict__ out, int64_t so_b, int64_t so_h,
    float* __restrict__ part, float* __restrict__ ml) {
  constexpr int KS = D / 32, DT = D / 16, NH = dec_heads(D);
  // dims a lane loads per key: DPL = D / 16, as VL loads of VW dims each
  constexpr int DPL = D / 16, VW = D == 64 ? 4 : 8, VL = DPL / VW;
  __shared__ float s_o[kDecWaves][NH][D + 4];
  __shared__ float s_ml[kDecWaves][NH][2];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g4 = lane >> 4, r16 = lane & 15;
  const int split = blockIdx.x, c = blockIdx.y % chunks, g = blockIdx.y / chunks, b = blockIdx.z;
  const int heads = min(NH, grp - c * NH);   // live columns
  const int h0 = g * grp + c * NH;

  // Q^T columns (heads past the group are zero and never written)
  bf16x8 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
    qf[ks] = r16 < heads ? load_bf16x8(q + b * sq_b + (h0 + r16) * sq_h + 32 * ks + 8 * g4)
                         : zero_bf16x8();

  const int k0 = split * keys_per_split;
  const int k1 = min(N, k0 + keys_per_split);
  const uint16_t* kb = k + b * sk_b + g * sk_h + 8 * g4;
  const uint16_t* vb = v + b * sv_b + g * sv_h + VW * r16;
  // MFMA row R of S^T tile mt is key 8 (R >> 2) + 4 mt + (R & 3) of the step:
  // the lane then holds keys 8 g4 + 4 mt + i
  const int krow = 8 * (r16 >> 2) + (r16 & 3);

  bf16x8 kf[2][KS];
  uint32_t vr[8][DPL / 2];       // V[8 g4 + i][the lane's dims], pairs of dims
  // rows past N - 1 read row N - 1 (in bounds); their P is zero and their V cleared
  auto load_k = [&](int base) {
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      const uint16_t* row = kb + static_cast<int64_t>(min(base + krow + 4 * mt, N - 1)) * sk_n;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) kf[mt][ks] = load_bf16x8(row + 32 * ks);
    }
  };
  auto load_v = [&](int base) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint16_t* row = vb + static_cast<int64_t>(min(base + 8 * g4 + i, N - 1)) * sv_n;
#pragma unroll
      for (int l = 0; l < VL; ++l) {
        if constexpr (VW == 8) {
          const u32x4 x = *reinterpret_cast<const u32x4*>(row + 128 * l);
#pragma unroll
          for (int j = 0; j < 4; ++j) vr[i][4 * l + j] = x[j];
        } else {
          const uint2 x = *reinterpret_cast<const uint2*>(row);
          vr[i][0] = x.x;
          vr[i][1] = x.y;
        }
      }
    }
  };

  f32x4 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;    // of head r16; l over this lane's keys

  int base = k0 + wave * kDecStep;
  if (base < k1) {
    load_k(base);
    load_v(base);
  }
  for (; base < k1; base += kDecWaves * kDecStep) {
    const int next = base + kDecWaves * kDecStep;
    f32x4 s[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) s[mt] = E::mfma(kf[mt][ks], qf[ks], s[mt]);
    if (next < k1) load_k(next);
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = s[e >> 2][e & 3] * scale_log2;
    if (base + kDecStep > N) {       // the last step: keys past the end
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (base + 8 * g4 + e >= N) {
          x[e] = -INFINITY;
#pragma unroll
          for (int j = 0; j < DPL / 2; ++j) vr[e][j] = 0u;
        }
    }
    float mx = x[0];
#pragma unroll
    for (int e = 1; e < 8; ++e) mx = fmaxf(mx, x[e]);
    const float m_new = fmaxf(m, quad_rows_max(mx));
    // every score so far -inf: weights 0 (the total then is 0 / 0, as softmax gives)
    const float off = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = __builtin_amdgcn_exp2f(m - off);
    m = m_new;
    float p[8], sum = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      p[e] = __builtin_amdgcn_exp2f(x[e] - off);
      sum += p[e];
    }
    l = l * alpha + sum;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt] *= alpha;
    u32x4 pw;
#pragma unroll
    for (int j = 0; j < 4; ++j) pw[j] = E::pack2(p[2 * j], p[2 * j + 1]);
    const bf16x8 pb = __builtin_bit_cast(bf16x8, pw);
    // operand dt: the lane's dim dt of the eight keys
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      u32x4 a;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        a[j] = __builtin_amdgcn_perm(vr[2 * j + 1][dt / 2], vr[2 * j][dt / 2],
                                     dt & 1 ? 0x07060302u : 0x05040100u);
      o[dt] = E::mfma(__builtin_bit_cast(bf16x8, a), pb, o[dt]);
    }
    if (next < k1) load_v(next);
  }
  l = quad_rows_sum(l);

  // O^T row R = 4 g4 + i of operand dt is dim VW (4 g4 + i) + dt % VW of load
  // dt / VW (128 dims a load)
  if (r16 < heads) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        s_o[wave][r16][128 * (dt / VW) + VW * (4 * g4 + i) + dt % VW] = o[dt][i];
    if (g4 == 0) {
      s_ml[wave][r16][0] = m;
      s_ml[wave][r16][1] = l;
    }
  }
  __syncthreads();

  const int H = Hk * grp;
  for (int i = threadIdx.x; i < heads * D; i += 64 * kDecWaves) {
    const int hh = i / D, d = i % D;
    float mm = s_ml[0][hh][0];
#pragma unroll
    for (int w = 1; w < kDecWaves; ++w) mm = fmaxf(mm, s_ml[w][hh][0]);
    const float off = mm == -INFINITY ? 0.f : mm;
    float acc = 0.f, ll = 0.f;
#pragma unroll
    for (int w = 0; w < kDecWaves; ++w) {
      const float f = __builtin_amdgcn_exp2f(s_ml[w][hh][0] - off);
      acc += s_o[w][hh][d] * f;
      ll += s_ml[w][hh][1] * f;
    }
    const int64_t bh = static_cast<int64_t>(b) * H + h0 + hh;
    if (splits == 1) {
      out[b * so_b + (h0 + hh) * so_h + d] = static_cast<uint16_t>(E::pack2(acc / ll, 0.f) & 0xFFFFu);
    } else {
      part[(bh * splits + split) * D + d] = acc;
      if (d == 0) {
        ml[(bh * splits + split) * 2] = mm;
        ml[(bh * splits + split) * 2 + 1] = ll;
      }
    }
  }
}

// out of one (b, head) from its splits: 512 threads, 512 / D runs of splits a
// dim each, their sums through LDS.
constexpr int kDecMaxSplits = 512;
constexpr int kDecCombineThreads = 512;
template <typename E, int D>
__global__ __launch_bounds__(kDecCombineThreads) void decode_combine_kernel(
    const float* __restrict__ part, const float* __restrict__ ml, int H, int splits,
    uint16_t* __restrict__ out, int64_t so_b, int64_t so_h) {
  constexpr int RUNS = kDecCombineThreads / D;
  __shared__ float s_w[kDecMaxSplits];
  __shared__ float s_red[kDecCombineThreads / 64][2];
  __shared__ float s_acc[RUNS][D];
  const int64_t bh = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float* mlb = ml + bh * splits * 2;
  // splits <= the thread count: one split's (m, l) a thread
  const float ms = tid < splits ? mlb[2 * tid] : -INFINITY;
  const float ls = tid < splits ? mlb[2 * tid + 1] : 0.f;
  float mx = ms;
#pragma unroll
  for (int s = 32; s >= 1; s >>= 1) mx = fmaxf(mx, __shfl_xor(mx, s, 64));
  if (lane == 0) s_red[wave][0] = mx;
  __syncthreads();
  mx = s_red[0][0];
#pragma unroll
  for (int w = 1; w < kDecCombineThreads / 64; ++w) mx = fmaxf(mx, s_red[w][0]);
  const float off = mx == -INFINITY ? 0.f : mx;
  const float wgt = __builtin_amdgcn_exp2f(ms - off);
  if (tid < splits) s_w[tid] = wgt;
  float lt = ls * wgt;
#pragma unroll
  for (int s = 32; s >= 1; s >>= 1) lt += __shfl_xor(lt, s, 64);
  if (lane == 0) s_red[wave][1] = lt;
  __syncthreads();
  float total = 0.f;
#pragma unroll
  for (int w = 0; w < kDecCombineThreads / 64; ++w) total += s_red[w][1];

  const int run = tid / D, d = tid % D;
  const float* pb = part + bh * splits * D + d;
  float acc = 0.f;
#pragma unroll 8
  for (int s = run; s < splits; s += RUNS) acc += pb[static_cast<int64_t>(s) * D] * s_w[s];
  s_acc[run][d] = acc;
  __syncthreads();
  if (tid < D) {
#pragma unroll
    for (int r = 1; r < RUNS; ++r) acc += s_acc[r][tid];
    out[(bh / H) * so_b + (bh % H) * so_h + tid] =
        static_cast<uint16_t>(E::pack2(acc / total, 0.f) & 0xFFFFu);
  }
}

// Key ranges per (b, KV head, head chunk): enough workgroups that every CU
// holds two (one at head_dim 256, whose 256 VGPRs leave one wavefront per
// SIMD), as long as each wavefront keeps a whole step.  Graph replays, us, at
// 28/4 heads, head_dim 128, 4K / 32K / 131K keys: 256 workgroups 7.6 / 16.1 /
// 44.2, 512 7.6 / 16.8 / 44.2, 1024 7.6 / 19.3 / 45.8; 4 sequences of 32K 44.2 /
// 43.1 / 43.7; 16/2 heads, head_dim 256, 32K / 131K: 256 20.3 / 46.3, 512 27.6 /
// 52.6.  At least two or four steps per wavefront instead of one is slower up
// to 8K keys (4K: 9.6 / 11.1), and so is one split there from 1K keys on (12.2
// against 7.7): the second launch costs less than a longer chain of steps.
// At 512 keys the two are level (7.2 / 7.9 us on the GPU), and below, one split
// spares the caller a workspace and a launch (10 against 14 us of host time).
int decode_splits(int B, int H, int Hk, int N, int D) {
  const int64_t units = static_cast<int64_t>(B) * Hk * ((H / Hk + dec_heads(D) - 1) / dec_heads(D));
  int64_t want = (D > 128 ? 256 : 512) / units;
  const int64_t most = N < UGBSA_DECODE_ONE_SPLIT ? 1 : N / (kDecWaves * kDecStep);
  if (want > most) want = most;
  if (want > kDecMaxSplits) want = kDecMaxSplits;
  if (want < 1) want = 1;
  // whole 32-key steps per split, and no empty split
  const int64_t steps = (N + kDecStep - 1) / kDecStep;
  const int64_t per = (steps + want - 1) / want;
  return static_cast<int>((steps + per - 1) / per);
}

template <typename E, int D>
static hipError_t launch_decode_t(const uint16_t* q, int64_t sq_b, int64_t sq_h, const uint16_t* k,
                                  int64_t sk_b, int64_t sk_h, int64_t sk_n, const uint16_t* v,
                                  int64_t sv_b, int64_t sv_h, int64_t sv_n, int B, int H, int Hk,
                                  int N, float scale, uint16_t* out, int64_t so_b, int64_t so_h,
                                  float* ws, hipStream_t stream) {
  const int grp = H / Hk, chunks = (grp + dec_heads(D) - 1) / dec_heads(D);
  const int splits = decode_splits(B, H, Hk, N, D);
  const int steps = (N + kDecStep - 1) / kDecStep;
  const int keys = (steps + splits - 1) / splits * kDecStep;
  float* part = ws;
  float* ml = ws + static_cast<int64_t>(B) * H * splits * D;
  decode_kernel<E, D><<<dim3(splits, Hk * chunks, B), 64 * kDecWaves, 0, stream>>>(
      q, sq_b, sq_h, k, sk_b, sk_h, sk_n, v, sv_b, sv_h, sv_n, Hk, N, grp, chunks, splits, keys,
      scale * kLog2e, out, so_b, so_h, part, ml);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || splits == 1) return e;
  decode_combine_kernel<E, D><<<dim3(B * H), kDecCombineThreads, 0, stream>>>(part, ml, H, splits,
                                                                             out, so_b, so_h);
  return hipGetLastError();
}

hipError_t launch_decode(const uint16_t* q, int64_t sq_b, int64_t sq_h, const uint16_t* k,
                         int64_t sk_b, int64_t sk_h, int64_t sk_n, const uint16_t* v, int64_t sv_b,
                         int64_t sv_h, int64_t sv_n, int B, int H, int Hk, int N, int D, int elem,
                         float scale, uint16_t* out, int64_t so_b, int64_t so_h, float* ws,
                         hipStream_t stream) {
#define UGBSA_DEC(E_, D_)                                                                        \
  return launch_decode_t<E_, D_>(q, sq_b, sq_h, k, sk_b, sk_h, sk_n, v, sv_b, sv_h, sv_n, B, H, \
                                 Hk, N, scale, out, so_b, so_h, ws, stream)
  if (elem == ElemF16::code) {
    if (D == 64) UGBSA_DEC(ElemF16, 64);
    if (D == 128) UGBSA_DEC(ElemF16, 128);
    if (D == 256) UGBSA_DEC(ElemF16, 256);
  } else {
    if (D == 64) UGBSA_DEC(ElemBf16, 64);
    if (D == 128) UGBSA_DEC(ElemBf16, 128);
    if (D == 256) UGBSA_DEC(ElemBf16, 256);
  }
#undef UGBSA_DEC
  return hipErrorInvalidValue;
}

}  // namespace ugbsa
