"""fp32 attention (T5 and DeBERTa) at the edges of its 16-row tiles and 64-key
chunks, against the oracle in 64 bits.

Tolerance 2e-5 absolute: a score is a sum of 64 products of unit-variance
values times a scale of about 0.1, off by at most ~64 * 2^-24 * 8 * 0.1 =
3e-6, which moves a weighted mean of values below 5 by at most twice that
relative error, and the sums over the keys add the same again."""
import math

import pytest
import torch

from oracle import attention as oa

pytestmark = pytest.mark.gpu
ATOL = 2e-5


def _rand(g, *shape):
    return torch.randn(*shape, generator=g)


def _rpb(dev, q, k, v, table, nb, md, causal, mask, scale):
    from kernels.flash_attention_rpb import flash_attention_rpb_final
    d = lambda t: None if t is None else t.to(dev)
    return flash_attention_rpb_final(d(q), d(k), d(v), d(table), nb, md, causal, padding_mask=d(mask),
                                     softmax_scale=scale).cpu().double()


@pytest.mark.parametrize("Lq,Lk", [(1, 1), (15, 63), (16, 64), (17, 65), (40, 257), (300, 129)])
@pytest.mark.parametrize("mask", [None, "key", "full"])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("md", [128, 9000])
def test_rpb(dev, Lq, Lk, mask, causal, md):
    """md = 9000: the bucket changes further out than the LDS table holds."""
    print("rpb fp32", Lq, Lk, mask, causal, md, flush=True)
    g = torch.Generator().manual_seed(Lq + Lk)
    q, k, v = _rand(g, 2, 3, Lq, 64), _rand(g, 2, 3, Lk, 64), _rand(g, 2, 3, Lk, 64)
    table, m = _rand(g, 32, 3), None
    if mask == "key":  # the second row keeps a third of its keys, the lowest value elsewhere
        m = torch.zeros(2, 1, 1, Lk)
        m[1, ..., (Lk + 2) // 3:] = torch.finfo(torch.float32).min
    elif mask == "full":
        m = _rand(g, 2, 1, Lq, Lk)
    want = oa.rpb_attention(q, k, v, table, 32, md, causal, m, 0.125, dtype=torch.float64)
    got = _rpb(dev, q, k, v, table, 32, md, causal, m, 0.125)
    assert (got - want).abs().max() <= ATOL


def test_rpb_every_key_masked(dev):
    """Masks of the type's lowest value on every key: the mean of V, also
    where the keys fill several chunks."""
    g = torch.Generator().manual_seed(1)
    q, k, v = (_rand(g, 1, 2, 200, 64) for _ in range(3))
    m = torch.full((1, 1, 1, 200), torch.finfo(torch.float32).min)
    got = _rpb(dev, q, k, v, None, 32, 128, False, m, 1.0)
    assert (got - v.double().mean(2, keepdim=True)).abs().max() <= ATOL


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
def test_causal_hides_nonfinite_values(dev, bad):
    """A non-finite V reaches the rows that see its key and no other."""
    g = torch.Generator().manual_seed(2)
    L, at = 100, 70
    q, k, v = (_rand(g, 1, 2, L, 64) for _ in range(3))
    clean = oa.rpb_attention(q, k, v, None, 32, 128, True, None, 0.125, dtype=torch.float64)
    v[0, 1, at, 5] = bad
    got = _rpb(dev, q, k, v, None, 32, 128, True, None, 0.125)
    hit = torch.zeros_like(got, dtype=torch.bool)
    hit[0, 1, at:, 5] = True
    assert ((got - clean)[~hit].abs() <= ATOL).all()
    if math.isnan(bad):
        assert got[hit].isnan().all()
    else:
        assert (got[hit] == bad).all()


@pytest.mark.parametrize("M,N", [(1, 1), (16, 16), (47, 47), (130, 130), (20, 90)])
@pytest.mark.parametrize("buckets,maxd,log", [(16, 64, True), (32, 32, True), (0, 24, False), (1, 8, False)])
@pytest.mark.parametrize("pos", ["both", "key", "query"])
def test_deberta(dev, M, N, buckets, maxd, log, pos):
    """Log buckets with unit steps and (32, 32) with larger ones, linear
    buckets, and a span of 1 (no run of four columns)."""
    from kernels.flash_deberta_attention import flash_deberta_attention
    print("deberta fp32", M, N, buckets, maxd, log, pos, flush=True)
    g = torch.Generator().manual_seed(M + N + buckets)
    S = buckets if buckets > 0 else maxd
    q, k, v = _rand(g, 2, 2, M, 64), _rand(g, 2, 2, N, 64), _rand(g, 2, 2, N, 64)
    pk = _rand(g, 2, 2, M, 2 * S) if pos != "query" else None
    # the oracle gathers pos_query over the keys only where M == N
    pq = _rand(g, 2, 2, N, 2 * S) if pos != "key" and M == N else None
    lens = torch.tensor([N, max(1, N // 2)], dtype=torch.int32)
    d = lambda t: None if t is None else t.to(dev)
    got = flash_deberta_attention(d(q), d(k), d(v), d(lens), d(pk), d(pq), False, 0.07, buckets, maxd, log)
    want = oa.deberta_flash_attention(q, k, v, lens, pk, pq, 0.07, buckets, maxd, log, dtype=torch.float64)
    assert (got.cpu().double() - want).abs().max() <= ATOL


def test_deberta_causal(dev):
    from kernels.flash_deberta_attention import flash_deberta_attention
    g = torch.Generator().manual_seed(3)
    q, k, v = (_rand(g, 2, 2, 90, 64) for _ in range(3))
    pk, pq = _rand(g, 2, 2, 90, 64), _rand(g, 2, 2, 90, 64)
    got = flash_deberta_attention(q.to(dev), k.to(dev), v.to(dev), None, pk.to(dev), pq.to(dev), True, 0.07,
                                  32, 64, True)
    want = oa.deberta_flash_attention(q, k, v, None, pk, pq, 0.07, 32, 64, True, True, dtype=torch.float64)
    assert (got.cpu().double() - want).abs().max() <= ATOL


def test_unaligned_rows(dev):
    """fp32 outputs may lie on any 4-byte boundary (inputs are copied)."""
    from kernels.flash_attention_rpb import flash_attention_rpb_final
    g = torch.Generator().manual_seed(4)
    buf = torch.empty(1 * 2 * 50 * 65 + 1, device=dev)
    out = buf[1:].view(1, 2, 50, 65)[..., :64]
    q, k, v = (_rand(g, 1, 2, 50, 65)[..., 1:] for _ in range(3))
    qd, kd, vd = (t.to(dev) for t in (q, k, v))
    flash_attention_rpb_final(qd, kd, vd, None, 32, 128, False, softmax_scale=0.125, out=out)
    want = oa.rpb_attention(q, k, v, None, 32, 128, False, None, 0.125, dtype=torch.float64)
    assert (out.cpu().double() - want).abs().max() <= ATOL


@pytest.mark.parametrize("op", ["rpb", "deberta"])
def test_more_workgroups_than_a_launch_holds(dev, op):
    """2^24 (batch, head) pairs of one row, the largest count that the entry
    points take: 2^32 threads, more than one launch holds. One key each, so
    every row is its batch's V exactly. Inputs are expanded; the output takes
    4 GiB."""
    from kernels.flash_attention_rpb import flash_attention_rpb_final
    from kernels.flash_deberta_attention import flash_deberta_attention
    print("2^24 heads", op, flush=True)
    n = 1 << 12
    q = torch.ones(1, 1, 1, 64, device=dev).expand(n, n, 1, 64)
    rows = torch.arange(n * 64, dtype=torch.float32, device=dev).view(n, 1, 1, 64)
    v = rows.expand(n, n, 1, 64)
    if op == "rpb":
        got = flash_attention_rpb_final(q, q, v, None, 32, 128, False, softmax_scale=0.125)
    else:
        got = flash_deberta_attention(q, q, v, None, None, None, False, 0.125, 16, 64, True)
    assert got.shape == (n, n, 1, 64)
    for b0 in range(0, n, 256):
        assert torch.equal(got[b0:b0 + 256], v[b0:b0 + 256]), b0
