// One ModernBERT layer for few tokens, as one entry point that enqueues all of
// its kernels (gfx950): models/modernbert/modernbert_encoder.py:289-352 with
// the attention over packed sequences.
//
// A layer of a few hundred tokens is 20 to 60 us of device work, less than
// seven separate calls take to issue, three of them library products at 20 us
// of host time each. Here the products run on the tiles of gemm_small.h; where
// their 32 x 32 tiles fit the chip, the residual add and the LayerNorm in
// front of Wqkv and Wi are done by those products themselves, so that a layer
// is six launches instead of eight. 22 layers of width 768 with the embedding,
// 32 tokens: 2.57 ms as separate calls, 0.71 as one call a layer; on the device
// alone 0.87 and 0.69 (1.34 with the 256 x 128 GLU tiles). With the ColBERT
// head, one query: 0.78 ms, its kernels 0.74, the host 0.57.
#include <math.h>

#include "gemm_small.h"

using namespace vfk;

namespace {

int64_t round256(int64_t b) { return (b + 255) / 256 * 256; }

// Bytes of the layer's own buffers: x1, h, qkv, att, o, g.
struct LayerBuffers {
  int64_t rows, x1, h, qkv, att, o, g, attn, total;
  LayerBuffers(int64_t M, int64_t D, int64_t I, int64_t attn_bytes) {
    int64_t at = 0;
    const auto take = [&](int64_t cols) {
      const int64_t p = at;
      at += round256(M * cols * 2);
      return p;
    };
    rows = M;
    x1 = take(D); h = take(D); qkv = take(3 * D); att = take(D); o = take(D); g = take(I);
    attn = at;
    total = at + attn_bytes;
  }
};

vfk_tensor rows2(void* p, int dt, int64_t M, int64_t N) {
  vfk_tensor t = {};
  t.data = p; t.dtype = dt; t.ndim = 2;
  t.size[0] = M; t.size[1] = N; t.size[2] = t.size[3] = 1;
  t.stride[0] = N; t.stride[1] = 1;
  return t;
}

vfk_tensor heads3(void* p, int dt, int64_t M, int64_t row, int64_t H) {
  vfk_tensor t = {};
  t.data = p; t.dtype = dt; t.ndim = 3;
  t.size[0] = M; t.size[1] = H; t.size[2] = 64; t.size[3] = 1;
  t.stride[0] = row; t.stride[1] = 64; t.stride[2] = 1;
  return t;
}

// out = x w^T on the 32 x 32 tiles or the 64 x 128 ones.
template <typename E>
void project(SmallArgs a, bool small, hipStream_t st) {
  if (small) launch_gemm_small<E, kActPlain, false, 1, 1, 1, 4>(a, st);
  else launch_gemm_small<E, kActPlain, false, 2, 2, 2, 1>(a, st);
}

// out = LayerNorm(x + res) w^T, or its GLU, on the 32 x 32 tiles.
template <typename E, int ACT>
void project_norm(SmallArgs a, hipStream_t st) {
  launch_gemm_small<E, ACT, true, ACT == kActPlain ? 1 : 2, 1, 1, 4>(a, st);
}

SmallArgs small_args(const void* x, int64_t xs, const vfk_tensor* w, void* out, int64_t os, int64_t M,
                     int64_t I) {
  SmallArgs a = {};
  a.x = static_cast<const uint16_t*>(x);
  a.w = static_cast<const uint16_t*>(w->data);
  a.out = static_cast<uint16_t*>(out);
  a.M = M; a.K = (int)w->size[1]; a.I = (int)I;
  a.xs2 = (int)(2 * xs); a.ws2 = (int)(2 * w->stride[0]); a.os = os;
  return a;
}

int check_weight(const vfk_tensor* w, const char* name, int dt, int64_t N, int64_t K) {
  int rc = check_tensor(w, name, 2);
  if (rc) return rc;
  if (w->dtype != dt || w->size[0] != N || w->size[1] != K || w->stride[1] != 1 || w->stride[0] < K ||
      w->stride[0] % 8 || !aligned16(w->data) || (N + 128) * w->stride[0] * 2 >= (1ll << 31))
    return set_error(VFK_ERR_INVALID, "modernbert_layer: %s must be [%lld, %lld] of x's dtype with "
                     "16-byte aligned rows", name, (long long)N, (long long)K);
  return VFK_OK;
}

int check_rows(const vfk_tensor* t, const char* name, int dt, int64_t M, int64_t D) {
  int rc = check_tensor(t, name, 2);
  if (rc) return rc;
  if (t->dtype != dt || t->size[0] != M || t->size[1] != D || t->stride[1] != 1 || t->stride[0] != D ||
      !aligned16(t->data))
    return set_error(VFK_ERR_INVALID, "modernbert_layer: %s must be a contiguous [%lld, %lld] of x's dtype",
                     name, (long long)M, (long long)D);
  return VFK_OK;
}

int check_norm(const vfk_tensor* t, const char* name, int dt, int64_t D) {
  int rc = check_tensor(t, name, 1);
  if (rc) return rc;
  if (t->dtype != dt || t->size[0] != D || t->stride[0] != 1 || !aligned16(t->data))
    return set_error(VFK_ERR_INVALID, "modernbert_layer: %s must be a contiguous [%lld] of x's dtype", name,
                     (long long)D);
  return VFK_OK;
}

}  // namespace

extern "C" int64_t vfk_modernbert_layer_workspace_bytes(int32_t dtype, int64_t tokens, int32_t hidden,
                                                        int32_t inter, int32_t num_seqs,
                                                        int32_t max_seqlen) {
  if (tokens <= 0 || hidden <= 0 || inter <= 0) return 0;
  return LayerBuffers(tokens, hidden, inter,
                      vfk_varlen_attn_workspace_bytes(dtype, tokens, hidden / 64, 1, num_seqs, max_seqlen))
      .total;
}

extern "C" int vfk_modernbert_layer_fwd(const vfk_tensor* x, const vfk_tensor* pending,
                                        const vfk_tensor* attn_norm, const vfk_tensor* wqkv,
                                        const vfk_tensor* wo, const vfk_tensor* mlp_norm,
                                        const vfk_tensor* wi, const vfk_tensor* wo_mlp, float eps,
                                        const int32_t* cu_seqlens, int32_t num_seqs, int32_t max_seqlen,
                                        int32_t window, const float* rope_cos_sin, int32_t rope_positions,
                                        const uint8_t* key_valid, float softmax_scale, void* workspace,
                                        int64_t workspace_bytes, vfk_tensor* x_out,
                                        vfk_tensor* pending_out, void* stream) {
  const char* nm = "modernbert_layer";
  int rc = check_tensor(x, "x", 2);
  if (rc) return rc;
  const int dt = x->dtype;
  if (dt != VFK_BF16 && dt != VFK_F16) return set_error(VFK_ERR_UNSUPPORTED, "%s: bf16 or fp16 only", nm);
  const int64_t M = x->size[0], D = x->size[1];
  if (D < 64 || D % 64 || D > 16384) return set_error(VFK_ERR_UNSUPPORTED, "%s: hidden %lld", nm, (long long)D);
  if ((rc = check_tensor(wi, "wi", 2))) return rc;
  const int64_t I = wi->size[0] / 2;
  if (I < 64 || I % 64 || I > 65536 || wi->size[0] != 2 * I)
    return set_error(VFK_ERR_UNSUPPORTED, "%s: intermediate %lld", nm, (long long)I);
  if ((rc = check_rows(x, "x", dt, M, D)) || (rc = check_rows(x_out, "x_out", dt, M, D)) ||
      (rc = check_rows(pending_out, "pending_out", dt, M, D)) ||
      (rc = check_weight(wqkv, "wqkv", dt, 3 * D, D)) || (rc = check_weight(wo, "wo", dt, D, D)) ||
      (rc = check_weight(wi, "wi", dt, 2 * I, D)) || (rc = check_weight(wo_mlp, "wo_mlp", dt, D, I)) ||
      (rc = check_norm(mlp_norm, "mlp_norm", dt, D)))
    return rc;
  const bool has_pending = present(pending), has_norm = present(attn_norm);
  if (has_pending && (rc = check_rows(pending, "pending", dt, M, D))) return rc;
  if (has_norm && (rc = check_norm(attn_norm, "attn_norm", dt, D))) return rc;
  if (has_pending && !has_norm)
    return set_error(VFK_ERR_UNSUPPORTED, "%s: a pending output needs attn_norm", nm);
  if (!rope_cos_sin) return set_error(VFK_ERR_INVALID, "%s: rope table missing", nm);
  // the column of workgroups that writes x_out runs beside others that read x
  if (x_out->data == x->data) return set_error(VFK_ERR_INVALID, "%s: x_out must not be x", nm);
  if (x_out->data == pending_out->data)
    return set_error(VFK_ERR_INVALID, "%s: x_out must not be pending_out", nm);
  if (M > (1 << 20)) return set_error(VFK_ERR_UNSUPPORTED, "%s: too many tokens", nm);
  if (M == 0) return VFK_OK;
  const LayerBuffers buf(M, D, I,
                         vfk_varlen_attn_workspace_bytes(dt, M, (int32_t)(D / 64), 1, num_seqs, max_seqlen));
  if (!workspace || workspace_bytes < buf.total || !aligned16(workspace))
    return set_error(VFK_ERR_INVALID, "%s: workspace needs %lld 16-byte aligned bytes", nm, (long long)buf.total);
  char* ws = static_cast<char*>(workspace);
  const int64_t H = D / 64;
  uint16_t* qkv = reinterpret_cast<uint16_t*>(ws + buf.qkv);
  const vfk_tensor q = heads3(qkv, dt, M, 3 * D, H), k = heads3(qkv + D, dt, M, 3 * D, H),
                   v = heads3(qkv + 2 * D, dt, M, 3 * D, H);
  vfk_tensor att = heads3(ws + buf.att, dt, M, D, H);
  if ((rc = varlen_attn_check(&q, &k, &v, cu_seqlens, num_seqs, max_seqlen, window, rope_cos_sin,
                              rope_positions, softmax_scale, &att, nm)))
    return rc;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int cus = compute_units();
  const bool norm_fits = D <= kNormMaxK;
  vfk_tensor x1 = rows2(ws + buf.x1, dt, M, D), h = rows2(ws + buf.h, dt, M, D);
  vfk_tensor o = rows2(ws + buf.o, dt, M, D), g = rows2(ws + buf.g, dt, M, I);

  // q | k | v of h = LayerNorm(x + pending); x1 = x + pending
  {
    const bool small = tiles32_fit(M, 3 * D, cus), fused = small && has_norm && norm_fits;
    SmallArgs a = small_args(x->data, D, wqkv, ws + buf.qkv, 3 * D, M, 3 * D);
    if (fused) {
      a.res = has_pending ? static_cast<const uint16_t*>(pending->data) : nullptr;
      a.rs = D; a.ss = D; a.eps = eps;
      a.sum = has_pending ? static_cast<uint16_t*>(x1.data) : nullptr;
      a.nw = static_cast<const uint16_t*>(attn_norm->data);
    } else if (has_norm) {
      if ((rc = vfk_layernorm_fwd(has_pending ? pending : x, has_pending ? x : nullptr, attn_norm, nullptr,
                                  eps, &h, has_pending ? &x1 : nullptr, stream)))
        return rc;
      a.x = static_cast<const uint16_t*>(h.data);
    }
    if (!has_pending) x1.data = x->data;
    if (fused && dt == VFK_BF16) project_norm<BF16, kActPlain>(a, st);
    else if (fused) project_norm<F16, kActPlain>(a, st);
    else if (dt == VFK_BF16) project<BF16>(a, small, st);
    else project<F16>(a, small, st);
    if ((rc = launch_status(nm))) return rc;
  }
  // The direct form sums the split keys in another order than one chain does,
  // as the products that split K do (Wqkv up to this line, Wi and Wo up to
  // theirs further on). It is taken only with all of them: past this line the
  // attention gives the bits of a large pack and the products' sums alone make
  // a difference, past Wo's line (320 tokens at width 768) nothing does.
  if (tiles32_fit(M, 3 * D, cus) && vfk_varlen_attn_direct(dt, (int32_t)H, num_seqs, max_seqlen)) {
    if ((rc = vfk_varlen_attn_direct_fwd(&q, &k, &v, cu_seqlens, num_seqs, max_seqlen, window, rope_cos_sin,
                                         rope_positions, key_valid, softmax_scale, &att, stream)))
      return rc;
  } else if ((rc = vfk_varlen_attn_fwd(&q, &k, &v, cu_seqlens, num_seqs, max_seqlen, window, rope_cos_sin,
                                rope_positions, key_valid, softmax_scale, ws + buf.attn,
                                buf.total - buf.attn, &att, stream))) {
    return rc;
  }
  const bool narrow = tiles32_fit(M, D, cus);
  {
    const SmallArgs a = small_args(att.data, D, wo, o.data, D, M, D);
    if (dt == VFK_BF16) project<BF16>(a, narrow, st);
    else project<F16>(a, narrow, st);
    if ((rc = launch_status(nm))) return rc;
  }
  // g = GELU(input) * gate of LayerNorm(x1 + o); x_out = x1 + o
  if (tiles32_fit(M, I, cus) && norm_fits) {
    SmallArgs a = small_args(x1.data, D, wi, g.data, I, M, I);
    a.res = static_cast<const uint16_t*>(o.data);
    a.rs = D; a.ss = D; a.eps = eps;
    a.sum = static_cast<uint16_t*>(x_out->data);
    a.nw = static_cast<const uint16_t*>(mlp_norm->data);
    if (dt == VFK_BF16) project_norm<BF16, VFK_ACT_GELU_ERF>(a, st);
    else project_norm<F16, VFK_ACT_GELU_ERF>(a, st);
    if ((rc = launch_status(nm))) return rc;
  } else {
    if ((rc = vfk_layernorm_fwd(&o, &x1, mlp_norm, nullptr, eps, &h, x_out, stream)) ||
        (rc = vfk_glu_linear_fwd(VFK_ACT_GELU_ERF, &h, wi, &g, stream)))
      return rc;
  }
  const SmallArgs a = small_args(g.data, I, wo_mlp, pending_out->data, D, M, D);
  if (dt == VFK_BF16) project<BF16>(a, narrow, st);
  else project<F16>(a, narrow, st);
  return launch_status(nm);
}
