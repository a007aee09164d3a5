"""The framework's work as its users have it done: the calls whose time is kept.

listed() names the standing cases, draw() gives further ones of the same
ranges, prepare() makes what a program has in hand before the call, run() is
one pass through the public entry points, work() what such a pass cannot do
without, tolerance() how far another correct implementation may be off, and
exact() the same outputs from plain torch in 64 bits.

Sizes are those of the benchmark configurations in workloads.py (ModernBERT-base,
DeBERTa-v3, mT5-large, GLiNER requests) and the smaller and ragged ones a
server meets between them. The models are encoders: there is a forward
direction only.
"""
import math
import os
import random
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.getcwd(), "vllm-factory_amd"))

import workloads  # noqa: E402
from encoders import modernbert  # noqa: E402
from kernels.flash_attention_rpb import (flash_attention_rpb_final,  # noqa: E402
                                         flash_attention_rpb_varlen)
from kernels.flash_deberta_attention import (flash_deberta_attention,  # noqa: E402
                                             flash_deberta_attention_varlen, rel_chunk_major)
from kernels.fused_glu_mlp import glu_linear  # noqa: E402
from kernels.fused_layernorm import fused_add_layernorm  # noqa: E402
from kernels.gliner_pooler import default_spans, gliner_reps_packed, span_marker_forward  # noqa: E402
from kernels.rms_norm import fused_add_rms_norm  # noqa: E402
from kernels.varlen_attention import varlen_rope_attention  # noqa: E402

DT = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
VOCAB, HIDDEN, HEADS, INTER, LAYERS, COLBERT = 50368, 768, 12, 1152, 22, 128
BUCKETS, MAX_REL = 256, 512          # DeBERTa-v3: position_buckets, max_relative_positions
T5_BUCKETS, T5_DISTANCE = 32, 128
SPAN_WIDTH, ENT = 12, 128001         # GLiNER: span widths, class token


def listed():
    return [
        # one ColBERT query through the whole encoder and head: a search
        # server's smallest call, every launch on the critical path
        {"name": "colbert_query", "op": "encoder", "head": True, "seqs": 1, "lo": 32, "hi": 32},
        # a full indexing batch through the whole encoder, the largest call
        {"name": "encoder_batch", "op": "encoder", "head": False, "seqs": 256, "lo": 512, "hi": 768},
        # one global and one local ModernBERT attention layer over a packed
        # batch (the benchmark's headline step)
        {"name": "attention_pack", "op": "attention", "seqs": 64, "lo": 512, "hi": 768,
         "dtype": "bf16", "masked": False},
        # the same layers for one or two documents of a lightly loaded server,
        # in fp16, with masked keys
        {"name": "attention_request", "op": "attention", "seqs": 2, "lo": 300, "hi": 700,
         "dtype": "fp16", "masked": True},
        # mT5-large attention over a packed batch
        {"name": "rpb_pack", "op": "rpb_pack", "seqs": 32, "lo": 512, "hi": 768, "heads": 16,
         "dtype": "bf16"},
        # mT5-style attention in fp32 on a padded pair with the additive key mask
        {"name": "rpb_fp32", "op": "rpb_padded", "batch": 2, "len": 256, "heads": 8, "dtype": "fp32"},
        # DeBERTa-v3-large attention over a packed batch
        {"name": "deberta_pack", "op": "deberta_pack", "seqs": 32, "lo": 256, "hi": 512, "heads": 16,
         "dtype": "bf16"},
        # the drop-in DeBERTa call as the reference's models make it, with the
        # position projections given, on a padded batch
        {"name": "deberta_dropin", "op": "deberta_dropin", "batch": 8, "len": 371, "heads": 12,
         "dtype": "bf16"},
        # the same call in fp32, the type GLiNER checkpoints come in
        {"name": "deberta_dropin_fp32", "op": "deberta_dropin", "batch": 4, "len": 300, "heads": 12,
         "dtype": "fp32"},
        # the gated MLP projection for one document
        {"name": "mlp_document", "op": "mlp", "rows": 500, "hidden": 768, "inter": 1152,
         "act": "gelu", "dtype": "bf16"},
        # residual add and LayerNorm of a packed batch
        {"name": "add_norm", "op": "norm", "rows": 40265, "hidden": 768, "rms": False, "dtype": "bf16"},
        # GLiNER's span pooler for a batch of requests: prompt and word rows,
        # span marker over every span
        {"name": "gliner_spans", "op": "gliner", "seqs": 16, "lo": 200, "hi": 500, "dtype": "bf16"},
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["encoder", "attention", "attention", "rpb_pack", "rpb_padded", "deberta_pack",
                     "deberta_dropin", "deberta_dropin", "mlp", "mlp", "norm", "gliner"])
    c = {"op": op}
    half = rng.choice(["bf16", "bf16", "fp16"])
    if op in ("encoder", "attention"):
        # a few short queries up to a batch of long documents
        hi = _log(rng, 12, 1500)
        c.update(seqs=_log(rng, 1, max(1, min(64, 40000 // hi))), lo=max(1, int(hi * rng.uniform(0.4, 1))), hi=hi)
        c.update({"head": rng.random() < 0.5} if op == "encoder" else
                 {"dtype": half, "masked": rng.random() < 0.5})
    elif op == "rpb_pack":
        hi = _log(rng, 24, 1024)
        c.update(seqs=_log(rng, 1, max(1, min(32, 24000 // hi))), lo=max(1, int(hi * rng.uniform(0.4, 1))),
                 hi=hi, heads=rng.choice([6, 12, 16]), dtype=half)
    elif op == "rpb_padded":
        c.update(batch=_log(rng, 1, 8), len=_log(rng, 40, 600), heads=rng.choice([6, 8, 12, 16]),
                 dtype=rng.choice(["fp32", "fp32", "bf16"]))
    elif op == "deberta_pack":
        hi = _log(rng, 32, 512)
        c.update(seqs=_log(rng, 1, 32), lo=max(1, int(hi * rng.uniform(0.4, 1))), hi=hi,
                 heads=rng.choice([12, 16]), dtype=half)
    elif op == "deberta_dropin":
        c.update(batch=_log(rng, 1, 16), len=_log(rng, 40, 512), heads=rng.choice([12, 16]),
                 dtype=rng.choice([half, half, "fp32"]))
    elif op == "mlp":
        d, i, act = rng.choice([(768, 1152, "gelu"), (768, 1152, "gelu"), (1024, 2816, "gelu_new")])
        c.update(rows=_log(rng, 12, 40000), hidden=d, inter=i, act=act, dtype=half)
    elif op == "norm":
        c.update(rows=_log(rng, 12, 160000), hidden=rng.choice([768, 1024]), rms=rng.random() < 0.4,
                 dtype=rng.choice(["bf16", "bf16", "fp16", "fp32"]))
    else:
        hi = _log(rng, 60, 700)
        c.update(seqs=_log(rng, 1, 32), lo=int(hi * rng.uniform(0.5, 1)), hi=hi, dtype=half)
    return c


# ---------------------------------------------------------------------------
# shapes and inputs
# ---------------------------------------------------------------------------
def _lengths(c):
    """The sequence lengths of a packed case (part of the case, not of the
    seed); the first has the largest."""
    r = random.Random("%d %d %d" % (c["seqs"], c["lo"], c["hi"]))
    return [c["hi"]] + [r.randint(c["lo"], c["hi"]) for _ in range(c["seqs"] - 1)]


def _valid(c):
    """The valid rows of each sequence of a padded case: right padding, the
    first one full."""
    r = random.Random("%d %d" % (c["batch"], c["len"]))
    return [c["len"]] + [r.randint((c["len"] + 1) // 2, c["len"]) for _ in range(c["batch"] - 1)]


def _requests(c):
    return workloads.gliner_requests(c["seqs"], c["lo"], c["hi"], ent_token_id=ENT, seed=7)


class _Rand:
    def __init__(self, seed, dtype):
        self.g = torch.Generator(device="cuda").manual_seed(seed)
        self.dtype = dtype

    def __call__(self, *shape, std=1.0, mean=0.0):
        return (torch.randn(*shape, generator=self.g, device="cuda") * std + mean).to(self.dtype)


def _cu(lens):
    return torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device="cuda")


def prepare(c, seed):
    op = c["op"]
    rnd = _Rand(seed, DT[c.get("dtype", "bf16")])
    if op == "encoder":
        lens = _lengths(c)
        T = sum(lens)
        ones = lambda: rnd(HIDDEN, std=0.05, mean=1.0)
        layers = [modernbert.ModernBertLayerWeights(
            rnd(3 * HIDDEN, HIDDEN, std=0.02), rnd(HIDDEN, HIDDEN, std=0.02),
            rnd(2 * INTER, HIDDEN, std=0.02), rnd(HIDDEN, INTER, std=0.02),
            None if i == 0 else ones(), ones()) for i in range(LAYERS)]
        w = modernbert.ModernBertWeights(HIDDEN, HEADS, INTER, rnd(VOCAB, HIDDEN, std=0.02), ones(), layers,
                                         ones())
        ids = torch.randint(0, VOCAB, (T,), generator=rnd.g, device="cuda")
        s = {"ids": ids, "cu": _cu(lens), "w": w}
        if c["head"]:
            s["proj"] = rnd(COLBERT, HIDDEN, std=0.02)
    elif op == "attention":
        lens = _lengths(c)
        T = sum(lens)
        s = {"qkv": rnd(T, 3, HEADS, 64, std=1.2), "cu": _cu(lens), "valid": None}
        if c["masked"]:
            s["valid"] = torch.rand(T, generator=rnd.g, device="cuda") > 0.02
    elif op == "rpb_pack":
        lens = _lengths(c)
        s = {"qkv": rnd(sum(lens), 3, c["heads"], 64, std=0.64), "cu": _cu(lens),
             "table": rnd(T5_BUCKETS, c["heads"], std=0.1)}
    elif op == "rpb_padded":
        B, L, H = c["batch"], c["len"], c["heads"]
        keep = torch.arange(L)[None, :] < torch.tensor(_valid(c))[:, None]
        mask = (1.0 - keep.to(rnd.dtype)) * torch.finfo(rnd.dtype).min
        s = {"q": rnd(B, H, L, 64), "k": rnd(B, H, L, 64), "v": rnd(B, H, L, 64),
             "table": rnd(T5_BUCKETS, H, std=0.1), "mask": mask[:, None, None, :].cuda()}
    elif op == "deberta_pack":
        lens = _lengths(c)
        H = c["heads"]
        s = {"qkv": rnd(sum(lens), 3, H, 64, std=0.64), "cu": _cu(lens)}
        s["key_rel"] = rel_chunk_major(rnd(H, 2 * BUCKETS, 64, std=0.64), BUCKETS)
        s["query_rel"] = rel_chunk_major(rnd(H, 2 * BUCKETS, 64, std=0.64), BUCKETS)
    elif op == "deberta_dropin":
        B, L, H = c["batch"], c["len"], c["heads"]
        q, k, v = (rnd(B, L, H, 64, std=0.64).transpose(1, 2).contiguous() for _ in range(3))
        s = {"q": q, "k": k, "v": v, "lens": torch.tensor(_valid(c), dtype=torch.int32, device="cuda"),
             "pos_key": rnd(B, H, L, 2 * BUCKETS, std=3.3), "pos_query": rnd(B, H, L, 2 * BUCKETS, std=3.3)}
    elif op == "mlp":
        s = {"x": rnd(c["rows"], c["hidden"]), "wi": rnd(2 * c["inter"], c["hidden"], std=0.04)}
    elif op == "norm":
        D = c["hidden"]
        s = {"x": rnd(c["rows"], D), "res": rnd(c["rows"], D, std=2.0), "w": rnd(D, std=0.05, mean=1.0)}
    else:
        r = _requests(c)
        D = HIDDEN
        idx, mask, words = [], [], r.text_lengths
        for n in words:
            i, m = default_spans(n, n, SPAN_WIDTH)
            idx.append(i)
            mask.append(m)
        s = {"hidden": rnd(r.ids.numel(), D), "ids": r.ids.cuda(), "words_mask": r.words_mask.cuda(),
             "cu": r.cu_seqlens.cuda(), "words": words, "span_idx": torch.cat(idx).cuda(),
             "span_mask": torch.cat(mask).cuda(), "row_cu": _cu(words),
             "span_cu": _cu([n * SPAN_WIDTH for n in words]),
             "ws": rnd(D, D, std=0.04), "we": rnd(D, D, std=0.04),
             "w1": rnd(4 * D, 2 * D, std=0.03), "b1": rnd(4 * D, std=0.02),
             "w2": rnd(D, 4 * D, std=0.03), "b2": rnd(D, std=0.02)}
    s["c"] = c
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    c = s["c"]
    op = c["op"]
    if op == "encoder":
        if c["head"]:
            return modernbert.modernbert_colbert_forward(s["ids"], s["cu"], c["hi"], s["w"], s["proj"])
        return modernbert.modernbert_forward(s["ids"], s["cu"], c["hi"], s["w"])
    if op == "attention":
        q, k, v = s["qkv"][:, 0], s["qkv"][:, 1], s["qkv"][:, 2]
        return (varlen_rope_attention(q, k, v, s["cu"], c["hi"], -1, 160000.0, 0.125, s["valid"]),
                varlen_rope_attention(q, k, v, s["cu"], c["hi"], 64, 10000.0, 0.125, s["valid"]))
    if op == "rpb_pack":
        return flash_attention_rpb_varlen(s["qkv"][:, 0], s["qkv"][:, 1], s["qkv"][:, 2], s["cu"], c["hi"],
                                          s["table"], T5_BUCKETS, T5_DISTANCE)
    if op == "rpb_padded":
        return flash_attention_rpb_final(s["q"], s["k"], s["v"], s["table"], T5_BUCKETS, T5_DISTANCE, False,
                                         padding_mask=s["mask"], softmax_scale=1.0)
    if op == "deberta_pack":
        return flash_deberta_attention_varlen(s["qkv"][:, 0], s["qkv"][:, 1], s["qkv"][:, 2], s["cu"], c["hi"],
                                              s["key_rel"], s["query_rel"], 1 / math.sqrt(192), BUCKETS,
                                              MAX_REL, True)
    if op == "deberta_dropin":
        return flash_deberta_attention(s["q"], s["k"], s["v"], s["lens"], s["pos_key"], s["pos_query"], False,
                                       1 / math.sqrt(192), BUCKETS, MAX_REL, True)
    if op == "mlp":
        return glu_linear(s["x"], s["wi"], c["act"])
    if op == "norm":
        if c["rms"]:
            return fused_add_rms_norm(s["x"], s["res"], s["w"], 1e-6)
        return fused_add_layernorm(s["x"], s["res"], s["w"], None, 1e-5)
    pe, pe_cu, we, we_cu = gliner_reps_packed(s["hidden"], s["ids"], s["words_mask"], s["cu"], s["words"], ENT)
    spans = span_marker_forward(F.linear(we, s["ws"]), F.linear(we, s["we"]), s["row_cu"], s["span_idx"],
                                s["span_mask"], s["span_cu"], s["w1"], s["b1"], s["w2"], s["b2"])
    return pe, we, spans


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _pairs(lens, window=-1):
    return sum(workloads.window_pairs(n, window) for n in lens)


def work(c):
    op = c["op"]
    e = 4 if c.get("dtype") == "fp32" else 2
    if op == "encoder":
        lens = _lengths(c)
        T = sum(lens)
        n_glob = (LAYERS + 2) // 3
        att = 256 * HEADS * (n_glob * _pairs(lens) + (LAYERS - n_glob) * _pairs(lens, 64))
        per = HIDDEN * (4 * HIDDEN + 3 * INTER)  # weights of a layer
        out = COLBERT if c["head"] else HIDDEN
        head = COLBERT * HIDDEN if c["head"] else 0
        # T embedding rows and every layer weight read once, the output written once
        return {"bytes": 2 * (LAYERS * per + head + T * (HIDDEN + out)) + 8 * T,
                "flops": 2 * T * (LAYERS * per + head) + att}
    if op == "attention":
        lens = _lengths(c)
        T = sum(lens)
        return {"bytes": 2 * 4 * T * HEADS * 64 * e, "flops": 256 * HEADS * (_pairs(lens) + _pairs(lens, 64))}
    if op == "rpb_pack":
        lens = _lengths(c)
        return {"bytes": 4 * sum(lens) * c["heads"] * 64 * e, "flops": 256 * c["heads"] * _pairs(lens)}
    if op == "rpb_padded":
        B, L, H = c["batch"], c["len"], c["heads"]
        return {"bytes": 4 * B * L * H * 64 * e, "flops": 256 * H * L * sum(_valid(c))}
    if op == "deberta_pack":
        lens = _lengths(c)
        T, H = sum(lens), c["heads"]
        # scores, values, and the two projections onto the relative rows in reach
        rel = sum(n * min(2 * n - 1, 2 * BUCKETS) for n in lens)
        return {"bytes": (4 * T * H * 64 + 4 * H * BUCKETS * 64) * e, "flops": H * (256 * _pairs(lens) + 256 * rel)}
    if op == "deberta_dropin":
        B, L, H = c["batch"], c["len"], c["heads"]
        lens = _valid(c)
        # of each position row the columns in reach of its sequence
        pos = sum(n * min(2 * n - 1, 2 * BUCKETS) for n in lens)
        return {"bytes": (H * 64 * (3 * sum(lens) + B * L) + H * pos) * e, "flops": 256 * H * _pairs(lens)}
    if op == "mlp":
        r, d, i = c["rows"], c["hidden"], c["inter"]
        return {"bytes": (r * d + 2 * i * d + r * i) * e, "flops": 4 * r * d * i}
    if op == "norm":
        return {"bytes": 4 * c["rows"] * c["hidden"] * e, "flops": 8 * c["rows"] * c["hidden"]}
    r = _requests(c)
    D, W, T = HIDDEN, sum(r.text_lengths), r.ids.numel()
    C, S = int((r.ids == ENT).sum()), sum(r.text_lengths) * SPAN_WIDTH
    return {"bytes": 2 * D * (2 * C + 2 * W + S) + 2 * 14 * D * D + 16 * T + 24 * S,
            "flops": 2 * W * D * D * (2 + 8) + 2 * S * 4 * D * D}


# ---------------------------------------------------------------------------
# 64 bits
# ---------------------------------------------------------------------------
def _softmax_av(scores, v):
    return torch.softmax(scores, -1) @ v


def _rope64(x, theta):
    """[n, H, 64] rotated by its row number; the angles in fp32, as the model's
    rotary module has them."""
    inv = 1.0 / theta ** (torch.arange(0, 64, 2, device=x.device).float() / 64)
    ang = (torch.arange(x.shape[0], device=x.device).float()[:, None] * inv).double()
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]
    a, b = x[..., :32], x[..., 32:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _modernbert_attention64(qkv, lens, window, theta, valid):
    """qkv [T, 3, H, 64] float64 -> [T, H, 64]."""
    out, at = torch.empty_like(qkv[:, 0]), 0
    for n in lens:
        x = qkv[at:at + n]
        q, k, v = _rope64(x[:, 0], theta), _rope64(x[:, 1], theta), x[:, 2]
        s = q.transpose(0, 1) @ k.permute(1, 2, 0) * 0.125
        i = torch.arange(n, device=s.device)
        hide = torch.zeros(n, n, dtype=torch.bool, device=s.device)
        if window >= 0:
            hide = (i[:, None] - i[None, :]).abs() > window
        if valid is not None:
            hide = hide | ~valid[at:at + n][None, :]
        s = s.masked_fill(hide, float("-inf"))
        p = torch.softmax(s, -1).nan_to_num(0.0)  # a row that sees no key is zero
        out[at:at + n] = (p @ v.transpose(0, 1)).transpose(0, 1)
        at += n
    return out


def _t5_bias64(table, n):
    """[H, n, n]: the bucketed bias of key - query, buckets in fp32 as the model has them."""
    rel = torch.arange(n)[None, :] - torch.arange(n)[:, None]
    half, exact = T5_BUCKETS // 2, T5_BUCKETS // 4
    b = (rel > 0).long() * half
    rel = rel.abs()
    far = exact + (torch.log(rel.float().clamp(min=1) / exact) / math.log(T5_DISTANCE / exact)
                   * (half - exact)).long()
    b = b + torch.where(rel < exact, rel, far.clamp(max=half - 1))
    return table.double()[b.to(table.device)].permute(2, 0, 1)


def _deberta_index(n, device):
    """[n, n] relative row of query - key: log buckets in fp32 as the model has them."""
    rel = torch.arange(n)[:, None] - torch.arange(n)[None, :]
    mid = BUCKETS // 2
    a = torch.where((rel < mid) & (rel > -mid), torch.tensor(mid - 1), rel.abs())
    lg = torch.ceil(torch.log(a / mid) / math.log((MAX_REL - 1) / mid) * (mid - 1)) + mid
    b = torch.where(a <= mid, rel.float(), lg * rel.sign())
    return (b.long() + BUCKETS).clamp(0, 2 * BUCKETS - 1).to(device)


def _deberta64(q, k, v, pos_key, pos_query, n):
    """[H, n, 64] and [H, n, 2S] position rows -> [H, n, 64]."""
    c = _deberta_index(n, q.device)[None].expand(q.shape[0], n, n)
    s = q @ k.transpose(-1, -2) + pos_key.gather(2, c)
    s = s + pos_query.gather(2, c.transpose(1, 2)).transpose(1, 2)
    return _softmax_av(s / math.sqrt(192), v)


def _ln64(x, w, b=None, eps=1e-5):
    return F.layer_norm(x, (x.shape[-1],), w.double(), None if b is None else b.double(), eps)


def exact(c, seed):
    op = c["op"]
    s = prepare(c, seed)
    if op == "encoder":
        lens, w, ids = _lengths(c), s["w"], s["ids"]
        T = sum(lens)
        valid = ids != modernbert.MASK_TOKEN_ID
        x = _ln64(w.emb[ids].double(), w.emb_norm)
        for i, lw in enumerate(w.layers):
            h = x if lw.attn_norm is None else _ln64(x, lw.attn_norm)
            qkv = (h @ lw.wqkv.double().t()).view(T, 3, HEADS, 64)
            glob = i % 3 == 0
            a = _modernbert_attention64(qkv, lens, -1 if glob else 64, 160000.0 if glob else 10000.0, valid)
            x = x + a.reshape(T, HIDDEN) @ lw.wo.double().t()
            y = _ln64(x, lw.mlp_norm) @ lw.wi.double().t()
            x = x + (F.gelu(y[:, :INTER]) * y[:, INTER:]) @ lw.wo_mlp.double().t()
        x = _ln64(x, w.final_norm)
        return F.normalize(x @ s["proj"].double().t(), dim=-1) if c["head"] else x
    if op == "attention":
        x, lens = s["qkv"].double(), _lengths(c)
        return (_modernbert_attention64(x, lens, -1, 160000.0, s["valid"]),
                _modernbert_attention64(x, lens, 64, 10000.0, s["valid"]))
    if op in ("rpb_pack", "deberta_pack"):
        out, at = torch.empty(s["qkv"][:, 0].shape, dtype=torch.float64, device="cuda"), 0
        if op == "deberta_pack":
            kr, qr = (s[n].double().permute(0, 2, 1, 3).reshape(c["heads"], 2 * BUCKETS, 64)
                      for n in ("key_rel", "query_rel"))
        for n in _lengths(c):
            q, k, v = s["qkv"][at:at + n].double().permute(1, 2, 0, 3)
            if op == "rpb_pack":
                o = _softmax_av(q @ k.transpose(-1, -2) + _t5_bias64(s["table"], n), v)
            else:
                o = _deberta64(q, k, v, q @ kr.transpose(-1, -2), k @ qr.transpose(-1, -2), n)
            out[at:at + n] = o.transpose(0, 1)
            at += n
        return out
    if op == "rpb_padded":
        q, k, v = (s[n].double() for n in "qkv")
        return _softmax_av(q @ k.transpose(-1, -2) + _t5_bias64(s["table"], c["len"]) + s["mask"].double(), v)
    if op == "deberta_dropin":
        out = torch.zeros(s["q"].shape, dtype=torch.float64, device="cuda")
        for b, n in enumerate(_valid(c)):
            out[b, :, :n] = _deberta64(*(s[t][b, :, :n].double() for t in ("q", "k", "v", "pos_key", "pos_query")),
                                       n)
        return out
    if op == "mlp":
        y = s["x"].double() @ s["wi"].double().t()
        a = F.gelu(y[:, :c["inter"]], approximate="none" if c["act"] == "gelu" else "tanh")
        return a * y[:, c["inter"]:]
    if op == "norm":
        x = s["x"].double() + s["res"].double()
        if c["rms"]:
            return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * s["w"].double(), x
        return _ln64(x, s["w"]), x
    r = _requests(c)
    D, h = HIDDEN, s["hidden"].double()
    pe, at = h[(s["ids"] == ENT).nonzero()[:, 0]], 0
    wm, starts = r.words_mask.tolist(), set(r.cu_seqlens.tolist())
    first = [t for t, m in enumerate(wm) if m > 0 and (t in starts or m != wm[t - 1])]
    we = h[torch.tensor(first, device="cuda")]
    a = torch.relu(we @ s["ws"].double().t()) @ s["w1"][:, :D].double().t()
    b = torch.relu(we @ s["we"].double().t()) @ s["w1"][:, D:].double().t()
    spans = []
    for n in r.text_lengths:
        i, m = default_spans(n, n, SPAN_WIDTH)
        i = (i * m[:, None]).cuda() + at
        y = torch.relu(a[i[:, 0]] + b[i[:, 1]] + s["b1"].double())
        spans.append(y @ s["w2"].double().t() + s["b2"].double())
        at += n
    return pe, we, torch.cat(spans)


# About four times the largest error against exact() over the ranges of draw():
# (relative, largest over the root mean square) for each path and type.
_TOLERANCE = {
    "attention": {"bf16": (1.6e-2, 0.27), "fp16": (2e-3, 3.5e-2)},
    "rpb": {"bf16": (8e-3, 6.5e-2), "fp16": (1e-3, 5e-3), "fp32": (4e-6, 8e-5)},
    "deberta": {"bf16": (1e-2, 6e-2), "fp16": (1.2e-3, 6e-3), "fp32": (1.4e-6, 1e-5)},
    "mlp": {"bf16": (6.6e-3, 1.6e-2), "fp16": (8.3e-4, 2e-3)},
    "norm": {"bf16": (7e-3, 1.6e-2), "fp16": (8.8e-4, 2e-3), "fp32": (2.7e-7, 1.2e-6)},
    "gliner": {"bf16": (1.4e-2, 7e-2), "fp16": (1.7e-3, 9.2e-3)},
}


def tolerance(c):
    if c["op"] == "encoder":
        # 22 layers with a bf16 residual stream: 1.2e-2 off 64 bits, of which
        # a changed rounding moves a part
        return {"rel": 3e-2, "max": 0.4}
    rel, most = _TOLERANCE[c["op"].split("_")[0]][c["dtype"]]
    return {"rel": rel, "max": most}
