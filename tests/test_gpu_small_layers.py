"""The ModernBERT layers of few tokens (vfk_modernbert_layer_fwd) against the
same layers in 64 bits, at the edges of its tiles: 32 x 32 tiles with the norm
in front (few tokens), 64 x 128 with a separate one, ragged tokens, K slices
that do not divide among the waves, a width that the fused norm does not hold,
hidden keys, a first layer with and without a norm.

Bound: each of a layer's seven 16-bit roundings is off by 2^-9 (bf16) of its
value at most, 2^-9 / sqrt(3) in the mean, so two layers stay within
sqrt(14) * 2^-9 / sqrt(3) = 4.2e-3 of the residual stream's norm; fp16 has
three more bits. Twice that is allowed."""
import pytest
import torch
import torch.nn.functional as F

from encoders import modernbert as mb
from oracle import attention as oa

pytestmark = pytest.mark.gpu
HIDDEN_ID = 7  # the token id that is hidden as a key in these tests


def _weights(D, I, dtype, seed, first_norm=False):
    g = torch.Generator().manual_seed(seed)
    rnd = lambda *s: (torch.randn(*s, generator=g) / s[-1] ** 0.5).to(dtype)
    ones = lambda: (1 + 0.1 * torch.randn(D, generator=g)).to(dtype)
    layers = [mb.ModernBertLayerWeights(rnd(3 * D, D), rnd(D, D), rnd(2 * I, D), rnd(D, I),
                                        None if i == 0 and not first_norm else ones(), ones())
              for i in range(2)]
    return mb.ModernBertWeights(D, D // 64, I, torch.randn(100, D, generator=g).to(dtype), ones(), layers, ones())


def _want(ids, cu, w):
    ln = lambda x, g: F.layer_norm(x, (w.hidden,), g.double(), None, w.eps)
    x = ln(w.emb[ids].double(), w.emb_norm)
    for i, lw in enumerate(w.layers):
        h = x if lw.attn_norm is None else ln(x, lw.attn_norm)
        q, k, v = (h @ lw.wqkv.double().t()).view(-1, 3, w.heads, 64).unbind(1)
        glob = i % w.global_every == 0
        a = oa.varlen_attention(q, k, v, cu, -1 if glob else w.window, w.theta_global if glob else w.theta_local,
                                ids != mb.MASK_TOKEN_ID, 0.125, dtype=torch.float64)
        x = x + a.reshape(-1, w.hidden) @ lw.wo.double().t()
        y = ln(x, lw.mlp_norm) @ lw.wi.double().t()
        x = x + (F.gelu(y[:, :w.inter]) * y[:, w.inter:]) @ lw.wo_mlp.double().t()
    return ln(x, w.final_norm)


def _counted(monkeypatch):
    """A list that grows by one with every call that takes one call a layer."""
    taken, encode_small = [], mb._encode_small
    monkeypatch.setattr(mb, "_encode_small", lambda *a: taken.append(1) or encode_small(*a))
    return taken


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D,I", [(64, 64), (128, 192), (768, 1152), (1024, 320), (1088, 64)])
@pytest.mark.parametrize("lens", [[1], [31], [20, 13], [150, 1, 70], [300, 411], [1000, 30]])
def test_small_layers(dev, dtype, D, I, lens, monkeypatch):
    """Both ways of running the layers, each shown to be the one that ran.
    Calls of more than one sequence have a norm in their first layer, and the
    keys of one whole sequence hidden beside every ninth of the others."""
    print("small layers", dtype, D, I, lens, flush=True)
    monkeypatch.setattr(mb, "MASK_TOKEN_ID", HIDDEN_ID)
    w = _weights(D, I, dtype, D + I + sum(lens), first_norm=len(lens) > 1)
    ids = torch.randint(8, 100, (sum(lens),), generator=torch.Generator().manual_seed(1))
    ids[3::9] = HIDDEN_ID
    if len(lens) > 1:
        ids[lens[0]:lens[0] + lens[1]] = HIDDEN_ID
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32)
    want, wd = _want(ids, cu, w), w.to(dev)
    taken = _counted(monkeypatch)
    small = mb.modernbert_forward(ids.to(dev), cu.to(dev), max(lens), wd).cpu().double()
    assert len(taken) == 1
    monkeypatch.setattr(mb, "_SMALL_TOKENS", 0)
    calls = mb.modernbert_forward(ids.to(dev), cu.to(dev), max(lens), wd).cpu().double()
    assert len(taken) == 1
    bound = 8.4e-3 if dtype == torch.bfloat16 else 1.05e-3
    rel = lambda t: float((t - want).norm() / want.norm())
    assert rel(small) <= bound and rel(calls) <= bound, (rel(small), rel(calls))


@pytest.mark.parametrize("n", [1, 33, 96, 97, 224, 300, 320])
def test_short_sequence_alone_and_packed(dev, n, monkeypatch):
    """A sequence of up to 320 tokens alone agrees with itself in a pack that
    takes the separate kernels to rounding: K and, up to 96 tokens, the keys
    are summed in another order. Four layers round 28 times: 2^-9 / sqrt(3)
    each, sqrt(28) of them and sqrt(2) for the two sides give 8.5e-3 of the
    norm; twice that is allowed."""
    w = mb.random_weights(num_layers=4).to(dev)
    lens = [n] + [512] * 10
    ids = torch.randint(0, 50000, (sum(lens),), generator=torch.Generator().manual_seed(n)).to(dev)
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device=dev)
    taken = _counted(monkeypatch)
    packed = mb.modernbert_forward(ids, cu, 512, w)[:n].double()
    assert not taken
    alone = mb.modernbert_forward(ids[:n], cu[:2], n, w).double()
    assert len(taken) == 1
    assert float((alone - packed).norm() / packed.norm()) <= 1.7e-2


@pytest.mark.parametrize("n", [321, 352, 500])
def test_longer_sequence_alone_and_packed(dev, n, monkeypatch):
    """From 321 tokens on (width 768) every sum runs in the order of the
    separate kernels: the same bits alone and in a pack."""
    w = mb.random_weights(num_layers=4).to(dev)
    lens = [n] + [512] * 10
    ids = torch.randint(0, 50000, (sum(lens),), generator=torch.Generator().manual_seed(n)).to(dev)
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device=dev)
    taken = _counted(monkeypatch)
    packed = mb.modernbert_forward(ids, cu, 512, w)[:n]
    alone = mb.modernbert_forward(ids[:n], cu[:2], n, w)
    assert len(taken) == 1 and torch.equal(alone, packed)


def test_small_layers_refuse(dev):
    """Calls that keep the separate kernels: a weight with its own linear, a
    strided weight, other types, autocast."""
    w = _weights(128, 64, torch.bfloat16, 3).to(dev)
    x = torch.zeros(8, 128, dtype=torch.bfloat16, device=dev)
    cu = torch.tensor([0, 8], dtype=torch.int32, device=dev)
    assert mb._small_layers(x, cu, w, 2)

    class Own(torch.Tensor):
        pass
    keep = w.layers[1].wo
    for bad in (keep.as_subclass(Own), keep.t(), keep.half()):
        w.layers[1].wo = bad
        assert not mb._small_layers(x, cu, w, 2)
    w.layers[1].wo = keep
    with torch.autocast("cuda", torch.float16):
        assert not mb._small_layers(x, cu, w, 2)
    assert not mb._small_layers(x.float(), cu, w, 2)
    # the token limit, and the work limit of wider layers
    wide = _weights(1024, 2624, torch.bfloat16, 5).to(dev)
    for wt, T, want in ((w, 4096, True), (w, 4097, False), (wide, 1600, True), (wide, 1700, False)):
        rows = torch.zeros(T, wt.hidden, dtype=torch.bfloat16, device=dev)
        assert mb._small_layers(rows, cu, wt, 2) is want, (wt.hidden, T)


def test_small_layers_captured(dev):
    """Capture and several replays, with eager work between them."""
    w = _weights(128, 64, torch.bfloat16, 4).to(dev)
    cu = torch.tensor([0, 40, 90], dtype=torch.int32, device=dev)
    ids = torch.randint(0, 100, (90,), device=dev)
    call = lambda: mb.modernbert_forward(ids, cu, 50, w)
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    for seed in range(3):
        ids.copy_(torch.randint(0, 100, (90,), generator=torch.Generator().manual_seed(seed)))
        graph.replay()
        got = out.clone()
        assert torch.equal(got, call())
        torch.cuda.synchronize()


def test_small_layers_without_rotation(dev):
    """theta 0: no rotation in that kind of layer (bound as above)."""
    for field in ("theta_global", "theta_local"):
        w = _weights(128, 192, torch.bfloat16, 6)
        setattr(w, field, 0.0)
        ids = torch.randint(0, 100, (90,), generator=torch.Generator().manual_seed(2))
        cu = torch.tensor([0, 40, 90], dtype=torch.int32)
        want = _want(ids, cu, w)
        got = mb.modernbert_forward(ids.to(dev), cu.to(dev), 50, w.to(dev)).cpu().double()
        assert float((got - want).norm() / want.norm()) <= 8.4e-3


@pytest.mark.parametrize("n", [0, -1])
def test_no_layers(dev, n):
    """No layer runs: the normed embeddings, whatever memory held before."""
    w = _weights(128, 64, torch.bfloat16, 7).to(dev)
    ids = torch.randint(0, 100, (50,), generator=torch.Generator().manual_seed(3)).to(dev)
    cu = torch.tensor([0, 50], dtype=torch.int32, device=dev)
    junk = torch.full((50, 128), float("nan"), dtype=torch.bfloat16, device=dev)
    del junk  # what an uninitialised buffer would show
    got = mb.modernbert_forward(ids, cu, 50, w, num_layers=n)
    x = mb.fused_layernorm(w.emb[ids], 128, w.emb_norm, None, w.eps)
    assert torch.equal(got, mb.fused_layernorm(x, 128, w.final_norm, None, w.eps))
