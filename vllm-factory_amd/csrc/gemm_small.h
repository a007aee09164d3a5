// Projections x W^T of few tokens (bf16 / fp16 on v_mfma_f32_32x32x16, gfx950):
// plain, or with the GLU product act(input) * gate as epilogue, and with the
// residual add and LayerNorm that precede them as prologue.
//
// Large tiles (256 tokens) give ceil(M / 256) rows of workgroups: 9 workgroups
// for the GLU projection of one query of 32 tokens and 18 for a document of
// 500 at I = 1152, each of which walks all of K alone while the rest of the
// chip idles. Here a workgroup owns 32 WM tokens x 32 WN NB weight rows (GLU:
// NB = 2, the input and the gate rows of 32 WN features), four waves as WM x
// WN x WK: the same calls give 36 and 144 workgroups, and three stages keep two
// steps of loads in flight, so that the time is about a memory latency plus
// the slices. GLU: 19.9 -> 5.5 us and 24.3 -> 7.3 us (six stages of 64 x 64,
// one workgroup a CU instead of two: 8.3 us).
//
// A step is WK consecutive 64-wide K slices, one for each of the WK wave
// groups; wave group wk multiplies slice WK s + wk, and the groups' partial
// sums meet in LDS at the end. Each LDS row is 128 bytes whose 16-byte chunks
// are XOR-swizzled by swz(row); a stage holds the x rows of all groups, then
// their weight rows.
//
// NORM: the workgroup normalises its 32 rows itself while its first weight
// rows arrive, and keeps them in LDS for all of K (the feature tiles repeat
// that work; at these sizes it costs less than a launch). The column of
// workgroups with feature tile 0 writes the new residual stream. 32 tokens, K =
// 768: Wqkv with the norm 7.7 us, 5.5 without it beside 3.8 for the norm.
#pragma once

#include "activation.h"
#include "attn_core.h"
#include "launch_util.h"

namespace vfk {

constexpr int kActPlain = -1;   // no GLU: out = x W^T
constexpr int kNormMaxK = 1024;
constexpr int kStages = 3;      // LDS stages of a product

struct SmallArgs {
  const uint16_t* x;
  const uint16_t* w;
  uint16_t* out;
  int64_t M;
  int K, I;       // I output features (GLU: w has 2I rows)
  int xs2, ws2;   // row strides of x and w in bytes
  int64_t os;     // row stride of out in elements
  int mt, nt;
  // NORM: x := LayerNorm(x + res) * nw; res == nullptr: of x alone, no sum
  const uint16_t* res;
  uint16_t* sum;
  const uint16_t* nw;
  int64_t rs, ss;  // row strides of res and sum in elements
  float eps;
};

template <int N>
__device__ inline void step_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"i"(N) : "memory");
}

// 64 lanes' 16 bytes at r + vo + so into the 1 KiB block at lds.
__device__ inline void lds_load16(rsrc_t r, char* lds, int vo, int so) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void_t*)lds, 16, vo, so, 0, 0);
}

// Rows t0 .. t0 + 31 of LayerNorm(x + res) * nw into the LDS rows at dst
// (slice s of row r at s * 4096 + r * 128). Half a wave holds a row: chunk c <
// CH of lane i is its columns 8 (32 c + i) .. +7, CH = ceil(K / 256). Statistics
// as in the LayerNorm kernel: mean, then the squared differences from it, in
// fp32. One wave a SIMD runs this, so its vector instructions are its time
// beside one memory latency: every load of the four rows comes before any use,
// only the last chunk is masked, and the four rows' reductions interleave.
template <typename E, int CH>
__device__ inline void norm_rows32_ch(const SmallArgs& a, int64_t t0, bool write_sum, char* dst) {
  const int l = threadIdx.x & 31, hw = threadIdx.x >> 5;  // half-wave of eight
  const int nch = a.K >> 3;
  const bool last_ok = 32 * (CH - 1) + l < nch;
  u32x4_t wv[CH], xv[4][CH], uv[4][CH];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 8 * i + hw;
    const int64_t t = t0 + r < a.M ? t0 + r : a.M - 1;
    const uint16_t* xr = a.x + t * (a.xs2 >> 1);
    const uint16_t* rr = a.res ? a.res + t * a.rs : xr;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int at = 8 * min(32 * c + l, nch - 1);
      xv[i][c] = *reinterpret_cast<const u32x4_t*>(xr + at);
      uv[i][c] = *reinterpret_cast<const u32x4_t*>(rr + at);
    }
  }
#pragma unroll
  for (int c = 0; c < CH; ++c)
    wv[c] = *reinterpret_cast<const u32x4_t*>(a.nw + 8 * min(32 * c + l, nch - 1));
  float v[4][CH][8], s[4], s2[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    s[i] = 0.f;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      unpack8<E>(xv[i][c], v[i][c]);
      if (a.res) {
        float u[8];
        unpack8<E>(uv[i][c], u);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[i][c][e] += u[e];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) s[i] += c < CH - 1 || last_ok ? v[i][c][e] : 0.f;
    }
  }
  if (write_sum) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int c = 0; c < CH; ++c)
        if (t0 + 8 * i + hw < a.M && (c < CH - 1 || last_ok))
          *reinterpret_cast<u32x4_t*>(a.sum + (t0 + 8 * i + hw) * a.ss + 8 * (32 * c + l)) = pack8<E>(v[i][c]);
  }
  const float n = (float)a.K;
#pragma unroll
  for (int i = 0; i < 4; ++i) s[i] = group_sum<32>(s[i]) / n;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    s2[i] = 0.f;
#pragma unroll
    for (int c = 0; c < CH; ++c)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        v[i][c][e] -= s[i];
        const float d = c < CH - 1 || last_ok ? v[i][c][e] : 0.f;
        s2[i] = __builtin_fmaf(d, d, s2[i]);
      }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) s2[i] = 1.0f / sqrtf(group_sum<32>(s2[i]) / n + a.eps);
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    float g[8];
    unpack8<E>(wv[c], g);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 8 * i + hw, ch = 32 * c + l;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[i][c][e] = v[i][c][e] * s2[i] * g[e];
      if (c < CH - 1 || last_ok)
        *reinterpret_cast<u32x4_t*>(dst + (ch >> 3) * 4096 + r * 128 + 16 * ((ch & 7) ^ swz(r))) =
            pack8<E>(v[i][c]);
    }
  }
}

template <typename E>
__device__ inline void norm_rows32(const SmallArgs& a, int64_t t0, bool write_sum, char* dst) {
  switch ((a.K + 255) >> 8) {
    case 1: norm_rows32_ch<E, 1>(a, t0, write_sum, dst); break;
    case 2: norm_rows32_ch<E, 2>(a, t0, write_sum, dst); break;
    case 3: norm_rows32_ch<E, 3>(a, t0, write_sum, dst); break;
    default: norm_rows32_ch<E, 4>(a, t0, write_sum, dst); break;
  }
}

template <typename E, int ACT, bool NORM, int NB, int WM, int WN, int WK>
__global__ __launch_bounds__(256) void gemm_small_kernel(SmallArgs a) {
  constexpr bool GLU = ACT != kActPlain;
  constexpr int TM = 32 * WM, TF = 32 * WN, TW = NB * TF;  // tokens, features, weight rows
  constexpr int kX = NORM ? 0 : WK * TM * 128, kStage = kX + WK * TW * 128;
  constexpr int NX = NORM ? 0 : WK * TM / 32, NW = WK * TW / 32;  // 8-row loads of a wave per stage
  constexpr int L = NX + NW;
  constexpr int kNorm = NORM ? kNormMaxK * 64 : 0;  // normalised rows, after the stages
  static_assert(WM * WN * WK == 4 && (kStages - 2) * L <= 63, "shape");
  static_assert((!GLU || NB == 2) && (!NORM || WK == 4), "form");
  static_assert(kStages * kStage >= NB * 16384, "the partial sums of the K groups");
  __shared__ __attribute__((aligned(1024))) char smem[kStages * kStage + kNorm];
  const int l = threadIdx.x & 63, c = l & 31, h = l >> 5;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wk = WK == 4 ? w : 0, wm = WK == 4 ? 0 : w / WN, wn = WK == 4 ? 0 : w % WN;
  // neighbours on one XCD share the operand of which each XCD then needs all;
  // the larger one is split over the XCDs
  const int work = xcd_remap(blockIdx.x, gridDim.x);
  const bool tok_fast = a.M <= (GLU ? 2 : 1) * (int64_t)a.I;
  const int mi = tok_fast ? work % a.mt : work / a.nt;
  const int ni = tok_fast ? work / a.mt : work % a.nt;
  const int64_t t0 = (int64_t)mi * TM;
  const int f0 = ni * (GLU ? TF : TW);
  const int hs = GLU ? a.I : TF;  // weight rows from one block of TF to the next
  const int nk = a.K >> 6, steps = (nk + WK - 1) / WK;

  // rows past the end of x or w read as zeros (GLU features past I of the
  // input half read gate rows, whose products are not stored); slices stay
  // inside K (k_slice): the range check takes the scalar offset off a
  // resource's size, which for a tile of one or two rows is below the offset
  // of a slice past K
  const int64_t xrows = a.M - t0 < TM ? a.M - t0 : TM;
  const rsrc_t xr = uniform_rsrc(a.x + t0 * (a.xs2 >> 1), (int)(xrows - 1) * a.xs2 + 2 * a.K);
  const rsrc_t wr = uniform_rsrc(a.w, ((GLU ? 2 : 1) * a.I - 1) * a.ws2 + 2 * a.K);
  int vx[NX > 0 ? NX : 1], vw[NW];
#pragma unroll
  for (int j = 0; j < NX; ++j) {
    const int row = 8 * (4 * j + w) + (l >> 3);  // of the stage's x region
    vx[j] = (row % TM) * a.xs2 + 16 * ((l & 7) ^ swz(row));
  }
#pragma unroll
  for (int j = 0; j < NW; ++j) {
    const int row = 8 * (4 * j + w) + (l >> 3), r = row % TW;
    vw[j] = (f0 + (r / TF) * hs + r % TF) * a.ws2 + 16 * ((l & 7) ^ swz(row));
  }
  auto load = [&](int s, char* st) {
#pragma unroll
    for (int j = 0; j < NX; ++j)
      lds_load16(xr, st + (4 * j + w) * 1024, vx[j], k_slice(s, 32 * j / TM, WK, nk) * 128);
#pragma unroll
    for (int j = 0; j < NW; ++j)
      lds_load16(wr, st + kX + (4 * j + w) * 1024, vw[j], k_slice(s, 32 * j / TW, WK, nk) * 128);
  };
#pragma unroll
  for (int s = 0; s < kStages - 1; ++s)
    if (s < steps) load(s, smem + s * kStage);
  if (NORM) {
    norm_rows32<E>(a, t0, ni == 0 && a.sum, smem + kStages * kStage);
    // the loop's waits count loads, which return in order; stores need not
    if (ni == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }

  f32x16_t acc[NB] = {};
  int xo[4], wo[4];
#pragma unroll
  for (int ds = 0; ds < 4; ++ds) {
    const int o = 128 * c + 16 * ((2 * ds + h) ^ swz(c));
    xo[ds] = o + (wk * TM + 32 * wm) * 128;
    wo[ds] = o + kX + (wk * TW + 32 * wn) * 128;
  }
  int cur = 0, nxt = (kStages - 1) * kStage;  // stage offsets of step s and of step s + kStages - 1
  for (int s = 0; s < steps; ++s) {
    // step s has landed in every wave, and every wave is done with step s - 1;
    // the loads of step s + 1, if there is one, stay in flight
    if (s + 1 < steps) step_barrier<L>(); else step_barrier<0>();
    const char* st = smem + cur;
    const char* xs = NORM ? smem + kStages * kStage + s * WK * 4096 : st;
    u32x4_t xf[4], wf[NB][4];
#pragma unroll
    for (int ds = 0; ds < 4; ++ds) {
      xf[ds] = *reinterpret_cast<const u32x4_t*>(xs + xo[ds]);
#pragma unroll
      for (int g = 0; g < NB; ++g)
        wf[g][ds] = *reinterpret_cast<const u32x4_t*>(st + wo[ds] + g * TF * 128);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (s + kStages - 1 < steps) load(s + kStages - 1, smem + nxt);
    cur = cur == (kStages - 1) * kStage ? 0 : cur + kStage;
    nxt = nxt == (kStages - 1) * kStage ? 0 : nxt + kStage;
    if (WK == 1 || s * WK + wk < nk) {  // uniform in the wave
#pragma unroll
      for (int ds = 0; ds < 4; ++ds)
#pragma unroll
        for (int g = 0; g < NB; ++g) acc[g] = E::mfma32(wf[g][ds], xf[ds], acc[g]);
    }
  }
  // lane: token t0 + 32 wm + c; feature f0 + 32 wn + 8 j + 4 h + e in register
  // 4 j + e of acc[0], of acc[1] its gate (GLU) or the feature TF further on
  const int64_t t = t0 + 32 * wm + c;
  uint16_t* orow = a.out + t * a.os;
  const int fl = f0 + 32 * wn + 4 * h;
  auto put = [&](int j, const f32x4_t (&y)[NB]) {
    if (t >= a.M) return;
#pragma unroll
    for (int g = 0; g < (GLU ? 1 : NB); ++g) {
      const int f = fl + 8 * j + g * TF;
      if (f >= a.I) continue;
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = GLU ? act_f<GLU ? ACT : 0>(y[0][e]) * y[NB - 1][e] : y[g][e];
      *reinterpret_cast<u32x2_t*>(orow + f) = u32x2_t{E::pack2(v[0], v[1]), E::pack2(v[2], v[3])};
    }
  };
  if (WK == 1) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f32x4_t y[NB];
#pragma unroll
      for (int g = 0; g < NB; ++g)
        y[g] = f32x4_t{acc[g][4 * j], acc[g][4 * j + 1], acc[g][4 * j + 2], acc[g][4 * j + 3]};
      put(j, y);
    }
    return;
  }
  // partial sums of the four K groups through LDS: wave w adds up registers
  // 4 w .. 4 w + 3 of each block
  __syncthreads();  // every wave has read its last operands
  f32x4_t* red = reinterpret_cast<f32x4_t*>(smem);  // [block][j][wave][lane]
#pragma unroll
  for (int g = 0; g < NB; ++g)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      red[((g * 4 + j) * 4 + w) * 64 + l] =
          f32x4_t{acc[g][4 * j], acc[g][4 * j + 1], acc[g][4 * j + 2], acc[g][4 * j + 3]};
  __syncthreads();
  f32x4_t y[NB];
#pragma unroll
  for (int g = 0; g < NB; ++g) {
    y[g] = red[((g * 4 + w) * 4) * 64 + l];
#pragma unroll
    for (int u = 1; u < 4; ++u) y[g] += red[((g * 4 + w) * 4 + u) * 64 + l];
  }
  put(w, y);
}

template <typename E, int ACT, bool NORM, int NB, int WM, int WN, int WK>
inline void launch_gemm_small(SmallArgs& a, hipStream_t st) {
  const int tf = 32 * WN * (ACT != kActPlain ? 1 : NB);
  a.mt = (int)((a.M + 32 * WM - 1) / (32 * WM));
  a.nt = (a.I + tf - 1) / tf;
  gemm_small_kernel<E, ACT, NORM, NB, WM, WN, WK><<<a.mt * a.nt, 256, 0, st>>>(a);
}

inline int compute_units() {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      cus < VFK_NUM_XCD)
    cus = 256;
  return cus;
}

// Whether 32 x 32 tiles have a CU each (they take most of a CU's LDS).
inline bool tiles32_fit(int64_t M, int64_t I, int cus) {
  return ((M + 31) / 32) * ((I + 31) / 32) <= cus;
}

}  // namespace vfk
