// fp32 attention on the fp32 matrix unit (v_mfma_f32_16x16x4_f32, gfx950),
// head_dim 64, shared by the T5 and DeBERTa entry points. Every product, sum
// and probability stays in 32 bits.
//
// Work split: a workgroup of four waves owns 16 query rows of one (batch,
// head); wave w takes the 64-key chunks w, w + 4, ... and keeps its own
// running max, row sum and output, merged through LDS at the end. Splitting
// the keys over the waves rather than the queries keeps the short sequences
// of this type (a few hundred keys, a few dozen heads) from leaving most of
// the chip idle: 2 x 8 heads x 256 rows give 256 workgroups, where one thread
// per query row gave 64 single waves.
//
// Layouts (lane l, c = l % 16, g = l / 16; A = [16 x 4], B = [4 x 16]):
//   S^T = K Q^T : the 16 k-steps of a 16-key block may take d in any order
//                 that both operands share; step 4 i + e takes d = 16 i + 4 g
//                 + e, so a lane's operands are four 16-byte loads of row c
//                 of K and Q straight into registers, the four lanes of a row
//                 reading 64 contiguous bytes. The even and the odd i go to
//                 two accumulators, added at the end (a shorter sum).
//                 Result: query c, keys 4 g + r (r < 4).
//   O^T = V^T P^T: k-step r of a key block takes keys 4 g + r, so the B
//                 operand is the S^T register r as it stands. Output block j
//                 holds d = 4 c + j: a lane's four A operands are the 16
//                 bytes at d = 4 c of row 4 g + r of V. Result: query c,
//                 d = 16 g + 4 r + j.
//
// Bound: a 64-key chunk is 128 matrix instructions of 32 cycles on one SIMD
// beside 32 operand loads of 1 KiB a wave, so the texture units of a CU are
// nearly as busy as its matrix units. Two query tiles a wave (half the K and V
// loads) measured slower: the second tile's scores, biases and gather
// addresses leave fewer than two waves a SIMD.
//
// Measured against one thread per query row (T5, key mask): 2 x 8 heads x 256
// rows 467 -> 22 us, 8 x 16 x 599 2474 -> 200 us (66 TFLOP/s over all pairs).
// DeBERTa: 4 x 12 x 300 652 -> 46 us, 16 x 16 x 512 2609 -> 452 us, there
// bound by the gathers of the position rows. Errors against 64 bits fell by
// 1.2 to 2 times (shorter sums, and bias and score added with one rounding).
#pragma once

#include "vfk_common.h"

namespace vfk {

constexpr int kF32Rows = 16;       // query rows per workgroup
constexpr int kF32Waves = 4;
constexpr int kF32Pad = 68;        // floats per merged output row (64 + 4)
constexpr int kF32MaxLut = 2048;   // largest saturation distance kept as an LDS table
// Workgroups of one launch, whose threads must stay below 2^32. A call of more
// (16 rows take the 256 threads that 256 rows take at one thread each) goes in
// several launches.
constexpr int64_t kF32MaxGrid = ((1ll << 32) - 1) / (64 * kF32Waves);

struct F32Args {
  const float *q, *k, *v;  // row 0 of this (batch, head)
  float* o;
  int64_t qs, ks, vs, os;  // row strides
  int q0;                  // first query row of the workgroup
  int nq;                  // rows below this are computed (q0 < nq)
  int nstore;              // rows nq .. nstore - 1 are written as zeros
  int kend;                // keys 0 .. kend - 1
  int coff;                // causal: key j is seen by row i when j <= i + coff
};

// Distance from which a bucket step function is constant.
inline int step_saturates_at(const StepFn& s) {
  const int last = s.nthr > 0 ? s.thr[s.nthr - 1] : 0;
  return last > s.a0 ? last : s.a0;
}

// step_eval with the thresholds in LDS.
__device__ inline int step_eval_lds(const StepFn& s, const int16_t* thr, int a) {
  if (a < s.a0) return a;
  int lo = 0, hi = s.nthr;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if ((int)thr[mid] <= a) lo = mid + 1; else hi = mid;
  }
  return s.f0 + lo;
}

// Four floats that may lie on any 4-byte boundary (one 16-byte access).
struct __attribute__((packed, aligned(4))) F32Run {
  f32x4_t x;
};
__device__ inline f32x4_t ld4(const float* p) { return reinterpret_cast<const F32Run*>(p)->x; }

// Max / sum over the four lanes c, c + 16, c + 32, c + 48 of a query.
__device__ inline float quad_rows_max(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_int(v), __float_as_int(v), false, false);
  v = fmaxf(__int_as_float(r[0]), __int_as_float(r[1]));
  const auto u = __builtin_amdgcn_permlane32_swap(__float_as_int(v), __float_as_int(v), false, false);
  return fmaxf(__int_as_float(u[0]), __int_as_float(u[1]));
}
__device__ inline float quad_rows_sum(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_int(v), __float_as_int(v), false, false);
  v = __int_as_float(r[0]) + __int_as_float(r[1]);
  const auto u = __builtin_amdgcn_permlane32_swap(__float_as_int(v), __float_as_int(v), false, false);
  return __int_as_float(u[0]) + __int_as_float(u[1]);
}

__device__ inline f32x4_t mfma4(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Merge buffer of a workgroup.
struct F32Merge {
  float o[kF32Waves][kF32Rows][kF32Pad];
  float m[kF32Waves][kF32Rows];
  float l[kF32Waves][kF32Rows];
};

// Output part of non-finite V values, for a causal chunk: a row must not meet
// the V of a key it does not see (its probability there is 0, and 0 x inf is
// NaN). Non-finite values leave v; per output the seen keys that hold +inf or
// -inf with some weight, and those that give NaN (a NaN, or an infinity with
// weight 0), are counted by products of their own.
__device__ inline void split_nonfinite_v(f32x4_t (&v)[4][4], const f32x4_t (&p)[4],
                                         const bool (&seen)[4][4], f32x4_t (&o)[4]) {
  float fin = 0.f;
#pragma unroll
  for (int kb = 0; kb < 4; ++kb)
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int j = 0; j < 4; ++j) fin = __builtin_fmaf(v[kb][r][j], 0.f, fin);
  if (__builtin_amdgcn_ballot_w64(fin != 0.f) == 0ull) return;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    f32x4_t up = {}, down = {}, nan = {};
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float x = v[kb][r][j];
        const bool isnan = x != x, isinf = x == INFINITY || x == -INFINITY;
        const float some = p[kb][r] > 0.f ? 1.f : 0.f;
        const float none = seen[kb][r] && p[kb][r] == 0.f ? 1.f : 0.f;
        up = mfma4(x == INFINITY ? 1.f : 0.f, some, up);
        down = mfma4(x == -INFINITY ? 1.f : 0.f, some, down);
        nan = mfma4(isnan ? 1.f : 0.f, seen[kb][r] ? 1.f : 0.f, nan);
        nan = mfma4(isinf ? 1.f : 0.f, none, nan);
        if (isnan || isinf) v[kb][r][j] = 0.f;
      }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (up[r] > 0.f) o[j][r] += INFINITY;
      if (down[r] > 0.f) o[j][r] -= INFINITY;
      if (nan[r] > 0.f) o[j][r] = NAN;
    }
  }
}

// Bias policy P: chunk(key0) prepares a 64-key chunk and says whether it holds
// a key with any weight; load(kb, bias) fills bias[r] for the lane's query and
// keys key0 + 16 kb + 4 g + r (which may lie past kend) before the scores are
// known; score(s, bias) turns a raw score into log2 units.
template <bool CAUSAL, class P>
__device__ inline void f32_attend(const F32Args& a, P& pol, F32Merge& sm) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, c = lane & 15, g = lane >> 4;
  f32x4_t q[4];
  {
    const float* row = a.q + (int64_t)min(a.q0 + c, a.nq - 1) * a.qs + 4 * g;
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = ld4(row + 16 * i);
  }
  f32x4_t o[4] = {};
  float m = -INFINITY, l = 0.f;
  const int vis = CAUSAL ? min(a.kend - 1, a.q0 + c + a.coff) : a.kend - 1;

  for (int key0 = 64 * w; key0 < a.kend; key0 += 64 * kF32Waves) {
    if (!pol.chunk(key0)) continue;  // uniform in the wave
    const bool tail = key0 + 64 > a.kend;
    // the chunk holds a key that some row of the workgroup does not see
    const bool diag = CAUSAL && key0 + 63 > a.q0 + a.coff;
    f32x4_t bias[4], k[4][4], v[4][4], s[4], s2[4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const float* row = a.k + (int64_t)min(key0 + 16 * kb + c, a.kend - 1) * a.ks + 4 * g;
#pragma unroll
      for (int i = 0; i < 4; ++i) k[kb][i] = ld4(row + 16 * i);
    }
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      pol.load(kb, key0 + 16 * kb + 4 * g, bias[kb]);
      s[kb] = f32x4_t{};
      s2[kb] = f32x4_t{};
    }
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = key0 + 16 * kb + 4 * g + r;
        v[kb][r] = ld4(a.v + (int64_t)min(j, a.kend - 1) * a.vs + 4 * c);
        // a repeated last row must not reach the sums (0 x inf)
        if (tail && j >= a.kend) v[kb][r] = f32x4_t{};
      }
#pragma unroll
    for (int i = 0; i < 4; i += 2)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
          s[kb] = mfma4(k[kb][i][e], q[i][e], s[kb]);
          s2[kb] = mfma4(k[kb][i + 1][e], q[i + 1][e], s2[kb]);
        }
    bool seen[4][4];
    float mx = m;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        seen[kb][r] = !(tail || diag) || key0 + 16 * kb + 4 * g + r <= vis;
        s[kb][r] = pol.score(s[kb][r] + s2[kb][r], bias[kb][r]);
        if (seen[kb][r]) mx = fmaxf(mx, s[kb][r]);
      }
    mx = quad_rows_max(mx);
    const float ref = mx == -INFINITY ? 0.f : mx;
    const float alpha = exp2f(m - ref);  // m = -inf: 0
    m = mx;
    float sum = 0.f;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s[kb][r] = seen[kb][r] ? exp2f(s[kb][r] - ref) : 0.f;
        sum += s[kb][r];
      }
    l = l * alpha + sum;
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] *= alpha;
    if (CAUSAL && diag) split_nonfinite_v(v, s, seen, o);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = mfma4(v[kb][r][j], s[kb][r], o[j]);
  }

  const float lt = quad_rows_sum(l);
  if (g == 0) {
    sm.m[w][c] = m;
    sm.l[w][c] = lt;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
    *reinterpret_cast<f32x4_t*>(&sm.o[w][c][16 * g + 4 * r]) = f32x4_t{o[0][r], o[1][r], o[2][r], o[3][r]};
  __syncthreads();
  // 16 threads a row, four values each
  const int r = t >> 4, d = 4 * (t & 15), i = a.q0 + r;
  if (i >= a.nstore) return;
  float mm = sm.m[0][r];
#pragma unroll
  for (int u = 1; u < kF32Waves; ++u) mm = fmaxf(mm, sm.m[u][r]);
  float ls = 0.f;
  f32x4_t x = {};
#pragma unroll
  for (int u = 0; u < kF32Waves; ++u) {
    const float f = sm.m[u][r] == mm ? 1.f : exp2f(sm.m[u][r] - mm);
    ls += f * sm.l[u][r];
    x += f * *reinterpret_cast<const f32x4_t*>(&sm.o[u][r][d]);
  }
  // a row with keys whose sum is 0 has only scores of -inf (or NaN): NaN, as
  // the softmax gives; a row without keys is zero
  const bool keys = a.kend > 0 && (!CAUSAL || i + a.coff >= 0);
  const float inv = ls > 0.f ? 1.0f / ls : NAN;
  x = keys && i < a.nq ? x * inv : f32x4_t{};
  float* orow = a.o + (int64_t)i * a.os + d;
  reinterpret_cast<F32Run*>(orow)->x = x;
}

// Writes the rows of a workgroup that computes none as zeros.
__device__ inline void f32_zero_rows(const F32Args& a) {
  for (int e = threadIdx.x; e < kF32Rows * 64; e += 64 * kF32Waves) {
    const int i = a.q0 + (e >> 6);
    if (i < a.nstore) a.o[(int64_t)i * a.os + (e & 63)] = 0.f;
  }
}

}  // namespace vfk
