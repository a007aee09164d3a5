"""The attention of few queries (keys rotated where they are used, split over
the waves) against the same call through the pre-pass, and both against the
oracle in 64 bits, at the edges of its 32-row and 64-key tiles.

Bound: P and the output are rounded to 16 bits (2^-9 relative in bf16), the
rotated q and k as well, which moves a score of size |s| by 2^-8 |s| and its
weight as much: for scores of a few units the two forms stay within 2e-2, the
tolerance of this path; against 64 bits the direct form may be no further off
than the other by more than a quarter."""
import pytest
import torch

import kernels.varlen_attention as va
from _tol import assert_attn_close
from kernels import _lib
from oracle import attention as oa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens", [[1], [31, 33], [64, 65, 0, 3], [300], [120] * 7])
@pytest.mark.parametrize("window", [-1, 64, 5])
@pytest.mark.parametrize("masked", [False, True])
def test_direct_matches_prepass(dev, dtype, lens, window, masked, monkeypatch):
    print("direct", dtype, lens, window, masked, flush=True)
    g = torch.Generator().manual_seed(sum(lens) + window)
    T, H = sum(lens), 3
    qkv = torch.randn(T, 3, H, 64, generator=g).to(dtype)
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32)
    valid = torch.rand(T, generator=g) > 0.3 if masked else None
    if masked and len(lens) > 1:
        valid[lens[0]:lens[0] + lens[1]] = False  # rows that see no key are zeros
    d = qkv.to(dev)
    call = lambda: va.varlen_rope_attention(d[:, 0], d[:, 1], d[:, 2], cu.to(dev), max(lens), window, 10000.0,
                                            0.125, None if valid is None else valid.to(dev)).cpu()
    lib = _lib.load()
    assert lib.vfk_varlen_attn_direct(_lib.dtype_code(dtype), H, len(lens), max(lens)) == 1
    direct = call()
    monkeypatch.setattr(lib, "vfk_varlen_attn_direct", lambda *a: 0)
    other = call()
    want = oa.varlen_attention(qkv[:, 0], qkv[:, 1], qkv[:, 2], cu, window, 10000.0, valid, 0.125,
                               dtype=torch.float64)
    assert_attn_close(direct, other, "direct against pre-pass")
    err = lambda t: float((t.double() - want).norm())
    assert err(direct) <= 1.25 * err(other) + 1e-6, (err(direct), err(other))


def test_direct_cuts_at_max_seqlen(dev):
    """Rows past max_seqlen are zeros and hide no key before it."""
    g = torch.Generator().manual_seed(9)
    qkv = torch.randn(90, 3, 2, 64, generator=g).bfloat16().to(dev)
    cu = torch.tensor([0, 50, 90], dtype=torch.int32, device=dev)
    got = va.varlen_rope_attention(qkv[:, 0], qkv[:, 1], qkv[:, 2], cu, 40, -1, 10000.0, 0.125)
    assert (got[40:50] == 0).all()
    cut = torch.cat([qkv[:40], qkv[50:]])
    cu2 = torch.tensor([0, 40, 80], dtype=torch.int32, device=dev)
    want = va.varlen_rope_attention(cut[:, 0], cut[:, 1], cut[:, 2], cu2, 40, -1, 10000.0, 0.125)
    assert torch.equal(torch.cat([got[:40], got[50:]]), want)


@pytest.mark.parametrize("which", [0, 1])
def test_output_in_place(dev, which, monkeypatch):
    """out may be q or k: a short call then gives what it gives through the
    pre-pass, which copies k before anything is written."""
    g = torch.Generator().manual_seed(11)
    qkv = torch.randn(300, 3, 12, 64, generator=g).bfloat16().to(dev)
    cu = torch.tensor([0, 300], dtype=torch.int32, device=dev)
    call = lambda t, out: va.varlen_rope_attention(t[:, 0], t[:, 1], t[:, 2], cu, 300, -1, 10000.0, 0.125, out=out)
    lib = _lib.load()
    assert lib.vfk_varlen_attn_direct(_lib.BF16, 12, 1, 300) == 1
    with monkeypatch.context() as m:
        m.setattr(lib, "vfk_varlen_attn_direct", lambda *a: 0)
        want = call(qkv, None)
    t = qkv.clone()
    assert torch.equal(call(t, t[:, which]), want)
