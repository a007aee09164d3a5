"""ModernBERT encoder forward on the packed (varlen) stream.

Follows models/modernbert/modernbert_encoder.py (embeddings :102-128, layer
:289-352, model :430-480): tok_embeddings -> LayerNorm; 22 x [attn_norm
(Identity in layer 0) -> Wqkv -> RoPE attention -> Wo -> + residual ->
mlp_norm -> Wi -> GELU(input) * gate -> Wo -> + residual]; final LayerNorm.
The Wi projection and the GELU gate run as one kernel (glu_linear), which
rounds the GLU output once where the reference rounds the projection first.
Wqkv and the rotary step of k run as one kernel (qkv_rope_projection), which
rotates the fp32 projection sums of k and rounds once; the attention then
reads that rotated k (varlen_rope_attention_krot) with no separate k pass.
Up to _SMALL_TOKENS tokens a layer is one call (vfk_modernbert_layer_fwd) that
enqueues the library's own products, norms and attention. Its products of few
rows split K over four waves: a call of up to 320 tokens (width 768) agrees with
its rows in a larger pack to rounding, longer calls bit for bit.
Global layers (layer_id % 3 == 0) attend inside each sequence with RoPE theta
160000, local layers within |i - j| <= 64 with theta 10000; tokens with id
50284 are hidden as keys (:456-460).

Differences from the reference, all by construction of the packed path:
sequences are given by cu_seqlens instead of position resets and dense
[T, T] masks; each residual add is fused into the LayerNorm that follows it
(vfk_layernorm_fwd with a residual); a query row that sees no key at all
(every key of its sequence is token 50284) returns zeros where the reference's
finite mask would average over the stream.
"""
from __future__ import annotations

import math
from dataclasses import dataclass, field
from typing import List, Optional

import torch
import torch.nn.functional as F

from kernels import _lib
from kernels.colbert_head import colbert_head
from kernels.dense_layernorm import dense_add_layernorm
from kernels.fused_glu_mlp import fused_gelu_mul_dropout, glu_linear
from kernels.fused_layernorm import fused_add_layernorm, fused_layernorm
from kernels.weight_pack import packed_weight
from kernels.varlen_attention import (qkv_rope_projection, rope_table, token_positions,
                                      varlen_from_positions, varlen_rope_attention,
                                      varlen_rope_attention_krot)

MASK_TOKEN_ID = 50284


@dataclass
class ModernBertLayerWeights:
    wqkv: torch.Tensor       # [3 * hidden, hidden]
    wo: torch.Tensor         # [hidden, hidden]
    wi: torch.Tensor         # [2 * inter, hidden] (input rows, then gate rows)
    wo_mlp: torch.Tensor     # [hidden, inter]
    attn_norm: Optional[torch.Tensor]   # [hidden]; None in layer 0 (Identity)
    mlp_norm: torch.Tensor   # [hidden]


@dataclass
class ModernBertWeights:
    hidden: int
    heads: int
    inter: int
    emb: torch.Tensor        # [vocab, hidden]
    emb_norm: torch.Tensor
    layers: List[ModernBertLayerWeights] = field(default_factory=list)
    final_norm: Optional[torch.Tensor] = None
    global_every: int = 3
    window: int = 64
    theta_global: float = 160000.0
    theta_local: float = 10000.0
    eps: float = 1e-5

    def to(self, device=None, dtype=None) -> "ModernBertWeights":
        def mv(t):
            return None if t is None else t.to(device=device, dtype=dtype)
        return ModernBertWeights(
            self.hidden, self.heads, self.inter, mv(self.emb), mv(self.emb_norm),
            [ModernBertLayerWeights(mv(l.wqkv), mv(l.wo), mv(l.wi), mv(l.wo_mlp), mv(l.attn_norm),
                                    mv(l.mlp_norm)) for l in self.layers],
            mv(self.final_norm), self.global_every, self.window, self.theta_global,
            self.theta_local, self.eps)


def random_weights(num_layers: int = 22, hidden: int = 768, heads: int = 12, inter: int = 1152,
                   vocab: int = 50368, seed: int = 1005, std: float = 0.02,
                   dtype=torch.bfloat16) -> ModernBertWeights:
    """Random-init weights ~ N(0, std) (CPU, seeded), LayerNorm weights 1."""
    g = torch.Generator().manual_seed(seed)

    def rnd(*shape):
        return (torch.randn(*shape, generator=g) * std).to(dtype)

    ones = torch.ones(hidden, dtype=dtype)
    layers = [ModernBertLayerWeights(rnd(3 * hidden, hidden), rnd(hidden, hidden),
                                     rnd(2 * inter, hidden), rnd(hidden, inter),
                                     None if i == 0 else ones.clone(), ones.clone())
              for i in range(num_layers)]
    return ModernBertWeights(hidden, heads, inter, rnd(vocab, hidden), ones.clone(), layers,
                             ones.clone())


def _glu_fusable(wi: torch.Tensor, h: torch.Tensor) -> bool:
    """Whether the Wi projection and GELU gate run as one kernel (glu_linear:
    16-bit weights, hidden a multiple of 64, intermediate of 8)."""
    return (wi.dtype in (torch.bfloat16, torch.float16) and h.dtype == wi.dtype
            and wi.shape[1] % 64 == 0 and (wi.shape[0] // 2) % 8 == 0)


def _qkv_fusable(wqkv: torch.Tensor, h: torch.Tensor, head_dim: int) -> bool:
    """Whether the Wqkv projection and the rotary step of k run as one kernel
    (qkv_rope_projection: 16-bit weights, head_dim 64, hidden a multiple of
    64)."""
    return (wqkv.dtype in (torch.bfloat16, torch.float16) and h.dtype == wqkv.dtype
            and head_dim == 64 and wqkv.shape[1] % 64 == 0 and h.dim() == 2)


def _dense_ln_fusable(wo: torch.Tensor) -> bool:
    """Wo + residual + mlp_norm as one kernel (dense_add_layernorm with the sum
    output): 16-bit weights, a square projection of width 256..1024."""
    N, K = wo.shape
    return wo.dtype in (torch.bfloat16, torch.float16) and N == K and N in (256, 512, 768, 1024)


# Token count up to which a layer runs as one call on the library's own small
# tiles (vfk_modernbert_layer_fwd) instead of seven separate calls. 22 layers of
# width 768, ms, seven calls / one call a layer, as eager calls and on the
# device alone (replays of a captured graph, which pay no host time):
#     32 tokens  2.57 / 0.71  device 0.87 / 0.69
#    512         2.57 / 1.23         1.08 / 1.21
#   1024         2.67 / 1.42         1.47 / 1.41
#   2048         2.68 / 1.84         1.90 / 1.85
#   2880         2.70 / 2.19         2.10 / 2.16
#   4096         2.70 / 2.57         2.44 / 2.56
#   4608         2.70 / 2.80         2.57 / 2.79
#   5549         2.99 / 3.31         2.98 / 3.29
#   7853         4.38 / 4.06         4.35 / 4.08
#  13090         5.22 / 6.12         5.22 / 6.07
# The line is that of eager calls, which the host bounds up to some 5000 tokens
# (seven calls issue in 2.6 to 2.9 ms); on the device alone the two are within 6 %
# of each other from 1000 tokens up to it, and both below the 2.31 and 2.69 ms
# of 2048 and 4096 tokens with the 256 x 128 GLU tiles alone. The tiles go over
# the chip in rounds, so the crossing is not monotone: one call is ahead again
# where the library products begin a round (7853).
_SMALL_TOKENS = 4096
# Wider layers reach that point earlier: what the seven calls cost the host is
# the same, what the small tiles take grows with a token's products. 28 layers
# of width 1024, intermediate 2624, ms, seven calls / one call a layer: 1536
# tokens 3.68 / 3.02 (device 3.01 / 2.98), 2048 3.66 / 3.49 (3.48 / 3.45), 2560
# 3.79 / 4.01 (3.76 / 3.97); the line lies at 1676.
_SMALL_WORK = _SMALL_TOKENS * (4 * 768 * 768 + 3 * 768 * 1152)
_PLAIN = (torch.Tensor, torch.nn.Parameter)
# Bytes of wi (4 I D) from which the entry point's 32-bit offsets, which reach
# one tile of rows past a weight, do not hold it; with hidden <= 16384 they hold
# the other weights.
_MAX_WEIGHT = (1 << 31) - 256 * 16384


def _small_layers(x: torch.Tensor, cu_seqlens: torch.Tensor, w: ModernBertWeights, n: int) -> bool:
    """Whether the layers take vfk_modernbert_layer_fwd: few tokens, 16-bit
    weights of x's type on its device with aligned rows, heads of 64, rotary
    embedding in every layer, no autocast (which would choose another type for
    the products)."""
    D, dt, dev = w.hidden, x.dtype, x.device
    if (not 0 < x.shape[0] <= _SMALL_TOKENS
            or x.shape[0] * D * (4 * D + 3 * w.inter) > _SMALL_WORK or dt not in (torch.bfloat16, torch.float16)
            or not (w.theta_global > 0 and w.theta_local > 0)  # 0: no rotation
            or torch.is_autocast_enabled() or D != 64 * w.heads or w.inter % 64 or w.inter < 64
            or D > 16384 or w.inter > 65536 or 4 * D * w.inter >= _MAX_WEIGHT
            or not x.is_contiguous() or x.data_ptr() % 16
            or cu_seqlens.dtype != torch.int32 or cu_seqlens.dim() != 1 or cu_seqlens.device != dev
            or not cu_seqlens.is_contiguous() or cu_seqlens.numel() < 2 or n <= 0):
        return False
    shapes = ((3 * D, D), (D, D), (2 * w.inter, D), (D, w.inter), (D,), (D,))
    for i in range(n):
        lw = w.layers[i]
        if lw.attn_norm is None and i:
            return False
        for t, shape in zip((lw.wqkv, lw.wo, lw.wi, lw.wo_mlp, lw.mlp_norm, lw.attn_norm), shapes):
            if t is None:
                continue
            # a subclass (a quantised weight) has its own linear
            if (type(t) not in _PLAIN or t.dtype != dt or t.shape != shape or not t.is_contiguous() or t.data_ptr() % 16
                    or t.device != dev):
                return False
    return True


def _encode_small(x: torch.Tensor, cu_seqlens: torch.Tensor, max_seqlen: int, key_valid: torch.Tensor,
                  w: ModernBertWeights, n: int):
    """The first n layers, one call each; returns (pending, x) as _encode."""
    T, D = x.shape
    dev, seqs, max_len = x.device, int(cu_seqlens.numel() - 1), int(max_seqlen)
    code, ref, desc = _lib.dtype_code(x.dtype), _lib.ref, _lib.desc
    size = int(_lib.load().vfk_modernbert_layer_workspace_bytes(code, T, D, w.inter, seqs, max_len))
    ws = torch.empty(size, dtype=torch.uint8, device=dev)
    valid = key_valid.view(torch.uint8)
    tables = [rope_table(t, max_len, dev) for t in (w.theta_global, w.theta_local)]
    # the residual stream alternates between two buffers; the MLP output is
    # read by the next layer before it is written again
    xs = (torch.empty_like(x), torch.empty_like(x) if n > 1 else None)
    out = torch.empty_like(x)
    xd, od, pending = ref(desc(x)), ref(desc(out)), None
    scale = 1.0 / math.sqrt(D // w.heads)
    for i in range(n):
        lw = w.layers[i]
        glob = i % w.global_every == 0
        tab = tables[0 if glob else 1]
        x = xs[i % 2]
        xo = ref(desc(x))
        _lib.on_device("vfk_modernbert_layer_fwd", dev, xd, pending, ref(desc(lw.attn_norm)),
                       ref(desc(lw.wqkv)), ref(desc(lw.wo)), ref(desc(lw.mlp_norm)), ref(desc(lw.wi)),
                       ref(desc(lw.wo_mlp)), float(w.eps), cu_seqlens.data_ptr(), seqs, max_len,
                       -1 if glob else int(w.window), tab.data_ptr(), int(tab.shape[0]), valid.data_ptr(),
                       scale, ws.data_ptr(), size, xo, od)
        xd, pending = xo, od
    return out, x


def _encode(ids: torch.Tensor, cu_seqlens: torch.Tensor, max_seqlen: int, w: ModernBertWeights,
            num_layers: Optional[int], fuse_qkv_rope: bool = False, fuse_dense_ln: bool = False):
    """Embeddings and layers; returns (pending MLP output or None, residual
    stream) before the final LayerNorm. fuse_qkv_rope: Wqkv and the k rotation
    as one kernel (qkv_rope_projection) where the weights allow it; off by
    default, since hipBLASLt plus the k pass measures about 5 % faster per
    layer at 163 736 tokens. fuse_dense_ln: the attention output's Wo, residual add
    and mlp_norm as one kernel (dense_add_layernorm, which also writes the
    new residual stream) where _dense_ln_fusable allows it; off by default:
    the 22-layer forward at 163 736 tokens takes 52.21 ms with it and
    52.25-52.33 ms without, within the run-to-run spread."""
    T = ids.shape[0]
    d = w.hidden // w.heads
    key_valid = ids != MASK_TOKEN_ID
    x = fused_layernorm(w.emb[ids], w.hidden, w.emb_norm, None, w.eps)
    pending = None  # MLP output not yet added to the residual stream x
    n = len(w.layers) if num_layers is None else num_layers
    if not (fuse_qkv_rope or fuse_dense_ln) and max_seqlen > 0 and _small_layers(x, cu_seqlens, w, n):
        return _encode_small(x, cu_seqlens, max_seqlen, key_valid, w, n)
    positions = None  # rotary position of each token, for the fused q | k | v projection
    for i in range(n):
        lw = w.layers[i]
        if pending is None:
            h = x if lw.attn_norm is None else fused_layernorm(x, w.hidden, lw.attn_norm, None, w.eps)
        else:
            h, x = fused_add_layernorm(pending, x, lw.attn_norm, None, w.eps)
        is_global = i % w.global_every == 0
        window = -1 if is_global else w.window
        theta = w.theta_global if is_global else w.theta_local
        if fuse_qkv_rope and _qkv_fusable(lw.wqkv, h, d):
            # Wqkv with the rotary step of k in the GEMM epilogue; the attention
            # reads the rotated k from its workspace (no k pass)
            if positions is None:
                positions = token_positions(cu_seqlens, T)
            res = qkv_rope_projection(h, lw.wqkv, w.heads, positions, max_seqlen, theta,
                                      1.0 / math.sqrt(d))
            att = varlen_rope_attention_krot(res, cu_seqlens, max_seqlen, window, key_valid)
        else:
            qkv = F.linear(h, lw.wqkv).view(T, 3, w.heads, d)
            att = varlen_rope_attention(qkv[:, 0], qkv[:, 1], qkv[:, 2], cu_seqlens, max_seqlen,
                                        window, theta, 1.0 / math.sqrt(d), key_valid)
        if fuse_dense_ln and _dense_ln_fusable(lw.wo):
            h, x = dense_add_layernorm(att.view(T, w.hidden), None, None, x, lw.mlp_norm, None,
                                       w.eps, packed_weight=packed_weight(lw.wo), return_sum=True)
        else:
            o = F.linear(att.view(T, w.hidden), lw.wo)
            h, x = fused_add_layernorm(o, x, lw.mlp_norm, None, w.eps)
        if _glu_fusable(lw.wi, h):
            g = glu_linear(h, lw.wi, "gelu")
        else:
            y = F.linear(h, lw.wi)
            g = fused_gelu_mul_dropout(y[:, :w.inter], y[:, w.inter:], "gelu")
        pending = F.linear(g, lw.wo_mlp)
    return pending, x


def modernbert_forward(ids: torch.Tensor, cu_seqlens: torch.Tensor, max_seqlen: int,
                       w: ModernBertWeights, num_layers: Optional[int] = None,
                       fuse_qkv_rope: bool = False, fuse_dense_ln: bool = False) -> torch.Tensor:
    """ids [T] (device, int64), cu_seqlens int32 [n + 1] -> last hidden state [T, hidden]."""
    pending, x = _encode(ids, cu_seqlens, max_seqlen, w, num_layers, fuse_qkv_rope, fuse_dense_ln)
    if pending is None:
        return fused_layernorm(x, w.hidden, w.final_norm, None, w.eps)
    out, _ = fused_add_layernorm(pending, x, w.final_norm, None, w.eps)
    return out


def modernbert_colbert_forward(ids: torch.Tensor, cu_seqlens: torch.Tensor, max_seqlen: int,
                               w: ModernBertWeights, proj_weight: torch.Tensor,
                               proj_bias: Optional[torch.Tensor] = None,
                               num_layers: Optional[int] = None) -> torch.Tensor:
    """ModernBERT + ColBERT head (plugins/moderncolbert/model.py:220-267 with a
    single Dense layer): the last residual add, the final LayerNorm, the
    projection [colbert_dim, hidden] and the L2 normalisation in one kernel
    (kernels.colbert_head). Returns [T, colbert_dim] unit-norm embeddings."""
    pending, x = _encode(ids, cu_seqlens, max_seqlen, w, num_layers)
    return colbert_head(x, proj_weight, proj_bias, w.final_norm, None, w.eps, residual=pending)


def modernbert_forward_positions(input_ids: torch.Tensor, position_ids: torch.Tensor,
                                 w: ModernBertWeights,
                                 num_layers: Optional[int] = None) -> torch.Tensor:
    """The reference's flat vLLM call (models/modernbert/modernbert_encoder.py:430-480:
    input_ids and position_ids of the packed stream): sequence boundaries come
    from the position resets on the device (varlen_from_positions) instead of
    [T, T] masks."""
    cu, max_len = varlen_from_positions(position_ids)
    return modernbert_forward(input_ids.reshape(-1), cu, max_len, w, num_layers)
