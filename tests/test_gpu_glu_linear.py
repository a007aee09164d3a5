"""GPU parity of the fused GLU projection (vfk_glu_linear_fwd) against a
float64 reference of the same composition: the projection x W^T followed by
act(input) * gate (oracle.epilogues.glu), i.e. modernbert_encoder.py:157-178
up to Wo. Inputs are scaled so that the projections are O(1); the bound is one
16-bit rounding of the output plus fp32 accumulation, which a missing K slice,
a swapped token or feature block, or a wrong activation exceeds by orders of
magnitude."""
import pytest
import torch

from _tol import assert_elem_close, cosine
from oracle import epilogues as oe

pytestmark = pytest.mark.gpu

ACTS = [("gelu", "gelu_erf"), ("gelu_new", "gelu_tanh"), ("silu", "silu")]


def _inputs(M, K, I, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(M, K, generator=g).to(dtype)
    w = (torch.randn(2 * I, K, generator=g) / K ** 0.5).to(dtype)
    return x, w


def _ref(x, w, act):
    y = x.double() @ w.double().T
    I = w.shape[0] // 2
    return oe.glu(y[:, :I], y[:, I:], act, dtype=torch.float64)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,I", [(1000, 768, 1152), (257, 128, 200), (1, 64, 8),
                                   (300, 1024, 64), (513, 192, 136)])
@pytest.mark.parametrize("act", ACTS, ids=[a[0] for a in ACTS])
def test_glu_linear_matches_reference(dev, dtype, M, K, I, act):
    from kernels.fused_glu_mlp import glu_linear
    x, w = _inputs(M, K, I, dtype, M + K + I)
    got = glu_linear(x.to(dev), w.to(dev), act[0])
    assert got.shape == (M, I) and got.dtype == dtype
    assert_elem_close(got, _ref(x, w, act[1]), dtype, f"glu_linear {M}x{K}x{I} {act[0]}")


def test_glu_linear_strided_rows_and_out(dev):
    """x and out as column slices of wider tensors (row strides K + 64 and
    I + 32), batch dims flattened, and the result written into `out`."""
    from kernels.fused_glu_mlp import glu_linear
    M, K, I = 700, 256, 96
    x, w = _inputs(M, K, I, torch.bfloat16, 5)
    xw = torch.zeros(M, K + 64, dtype=torch.bfloat16)
    xw[:, :K] = x
    xd = xw.to(dev)[:, :K]
    ow = torch.full((M, I + 32), 7.0, dtype=torch.bfloat16, device=dev)
    glu_linear(xd, w.to(dev), "gelu", out=ow[:, :I])
    assert_elem_close(ow[:, :I], _ref(x, w, "gelu_erf"), torch.bfloat16, "strided")
    assert (ow[:, I:] == 7.0).all(), "columns past I were written"
    y3 = glu_linear(x.view(7, 100, K).to(dev), w.to(dev), "gelu")
    assert y3.shape == (7, 100, I)
    assert_elem_close(y3.view(M, I), _ref(x, w, "gelu_erf"), torch.bfloat16, "3-d input")


def test_glu_linear_matches_unfused_path(dev):
    """Against F.linear + fused_gelu_mul_dropout (the layer's unfused path):
    the two differ only by where the projection is rounded to bf16. The
    unfused path rounds twice (projection, then product), which puts a few
    elements past a one-rounding bound, so it is held to the cosine only."""
    import torch.nn.functional as F
    from kernels.fused_glu_mlp import fused_gelu_mul_dropout, glu_linear
    M, K, I = 4096, 768, 1152
    x, w = _inputs(M, K, I, torch.bfloat16, 9)
    xd, wd = x.to(dev), w.to(dev)
    got = glu_linear(xd, wd, "gelu")
    y = F.linear(xd, wd)
    unf = fused_gelu_mul_dropout(y[:, :I], y[:, I:], "gelu")
    want = _ref(x, w, "gelu_erf")
    assert_elem_close(got, want, torch.bfloat16, "fused")
    assert cosine(unf.cpu(), want) >= 0.9999
    # the fused result is at least as close to the float64 reference
    e_f = (got.double().cpu() - want).abs().mean().item()
    e_u = (unf.double().cpu() - want).abs().mean().item()
    assert e_f <= e_u * 1.05, (e_f, e_u)


def test_glu_linear_modernbert_config5_shape(dev):
    """The ModernBERT-base MLP projection of the 256-sequence pack: x
    [163 736, 768], Wi [2304, 768], bf16. Rows checked: 384 sampled rows, the
    first and the last token tile (a partial tile of 152 rows)."""
    from kernels.fused_glu_mlp import glu_linear
    M, K, I = 163736, 768, 1152
    g = torch.Generator().manual_seed(11)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16)
    w = (torch.randn(2 * I, K, generator=g) / K ** 0.5).to(torch.bfloat16)
    got = glu_linear(x.to(dev), w.to(dev), "gelu").cpu()
    rows = torch.cat([torch.arange(256), torch.randint(256, M - 256, (384,), generator=g),
                      torch.arange(M - 256, M)])
    want = _ref(x[rows], w, "gelu_erf")
    assert_elem_close(got[rows], want, torch.bfloat16, "config-5 rows")
    assert torch.isfinite(got.float()).all()
    assert cosine(got[rows], want) >= 0.9999


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tile,M,K,I", [
    # K split unevenly over the four waves
    (32, 1, 64, 8), (32, 31, 192, 40), (32, 33, 320, 1152), (32, 224, 768, 1152),
    (64, 225, 64, 1152), (64, 257, 128, 1160), (64, 500, 768, 1152), (64, 65, 1024, 8200),
    # the line to 256 x 128
    (64, 4600, 128, 1152), (256, 4700, 128, 1152)])
def test_glu_linear_tiles(dev, dtype, tile, M, K, I):
    """Each tile at its edges: K slices that do not divide among the waves,
    fewer slices than stages, ragged tokens and features; x and w with row
    strides above K, whose gaps and tails must not enter (they hold NaN). The
    bound is the one above."""
    from kernels import _lib
    from kernels.fused_glu_mlp import glu_linear
    print("glu tiles", dtype, M, K, I, flush=True)
    assert _lib.load().vfk_glu_linear_tile(M, I) == tile
    x, w = _inputs(M, K, I, dtype, M + K + I)
    xd = torch.full((M, K + 8), float("nan"), dtype=dtype, device=dev)
    wd = torch.full((2 * I, K + 8), float("nan"), dtype=dtype, device=dev)
    xd[:, :K], wd[:, :K] = x.to(dev), w.to(dev)
    out = torch.full((M + 1, I + 8), 7.0, dtype=dtype, device=dev)
    glu_linear(xd[:, :K], wd[:, :K], "gelu", out=out[:M, :I])
    assert (out[M] == 7.0).all() and (out[:, I:] == 7.0).all(), "written past the output"
    y = xd[:, :K].double() @ wd[:, :K].double().t()
    want = torch.nn.functional.gelu(y[:, :I]) * y[:, I:]
    assert_elem_close(out[:M, :I], want, dtype, f"glu_linear {M}x{K}x{I}")


def test_glu_linear_row_alone_and_among_others(dev):
    """A row has the same bits in the 64- and the 256-token tiles, and agrees
    to rounding in the 32-token ones, whose four partial sums are added in
    another order: the fp32 sums differ by 2^-24 times the sum of the terms'
    sizes (11 here) times the square root of their number (28) at most, times a
    gate below 5, 1e-4, and one bf16 step."""
    from kernels import _lib
    from kernels.fused_glu_mlp import glu_linear
    x, w = _inputs(6000, 768, 1152, torch.bfloat16, 3)
    x, w = x.to(dev), w.to(dev)
    tile = _lib.load().vfk_glu_linear_tile
    assert [tile(n, 1152) for n in (6000, 500, 225, 224, 32)] == [256, 64, 64, 32, 32]
    full = glu_linear(x, w, "gelu")
    for n in (225, 500):
        assert torch.equal(glu_linear(x[:n], w, "gelu"), full[:n]), n
    for n in (1, 32, 224):
        got, want = glu_linear(x[:n], w, "gelu").float(), full[:n].float()
        step = torch.maximum(got.abs(), want.abs()) * 2 ** -7  # a bf16 step is at most 2^-7 of the value
        assert ((got - want).abs() <= step + 1e-4).all(), n


@pytest.mark.parametrize("at", [0, 1, 4, 8])
@pytest.mark.parametrize("pad", [1, 3, 8])
def test_glu_linear_single_row_of_any_stride(dev, at, pad):
    """One row cut out of a wider one, at any offset and with any stride to a
    row that is not there: the same bits as the row by itself."""
    from kernels.fused_glu_mlp import glu_linear
    x, w = _inputs(1, 256, 64, torch.bfloat16, 5)
    buf = torch.zeros(1, 256 + at + pad, dtype=torch.bfloat16, device=dev)
    buf[:, at:at + 256] = x.to(dev)
    cut = buf[:, at:at + 256]
    got = glu_linear(cut, w.to(dev), "gelu")
    assert got.shape == (1, 64) and torch.equal(got, glu_linear(x.to(dev), w.to(dev), "gelu"))
