"""Which ModernBERT calls take one entry point a layer (_small_layers): what the
entry point refuses and the separate kernels accept must stay with them. The
rule looks at shapes, types and scalars alone, so it runs without a GPU."""
import torch

from encoders import modernbert as mb


def _weights(D=128, I=64, layers=2, meta=False):
    dev = "meta" if meta else "cpu"
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device=dev)
    ls = [mb.ModernBertLayerWeights(z(3 * D, D), z(D, D), z(2 * I, D), z(D, I), None if i == 0 else z(D), z(D))
          for i in range(layers)]
    return mb.ModernBertWeights(D, D // 64, I, z(8, D), z(D), ls, z(D))


def _rows(w, T=8):
    return torch.zeros(T, w.hidden, dtype=torch.bfloat16, device=w.emb.device)


def _cu(w, *ends):
    return torch.tensor(ends, dtype=torch.int32).to(w.emb.device)


def test_empty_calls_keep_the_separate_kernels(monkeypatch):
    """No sequences or a max_seqlen of 0: the entry point refuses them."""
    w = _weights()
    assert mb._small_layers(_rows(w), _cu(w, 0, 8), w, 2)
    assert not mb._small_layers(_rows(w), _cu(w, 0), w, 2)
    taken = []
    monkeypatch.setattr(mb, "fused_layernorm", lambda x, *a: x)
    monkeypatch.setattr(mb, "_small_layers", lambda *a: True)
    monkeypatch.setattr(mb, "_encode_small", lambda *a: taken.append(a) or (None, a[0]))
    monkeypatch.setattr(mb.F, "linear", lambda *a: (_ for _ in ()).throw(LookupError))
    ids = torch.zeros(8, dtype=torch.int64)
    mb._encode(ids, _cu(w, 0, 8), 8, w, 2)
    assert len(taken) == 1
    try:
        mb._encode(ids, _cu(w, 0, 8), 0, w, 2)
    except LookupError:
        pass
    assert len(taken) == 1


def test_no_rotary_embedding_keeps_the_separate_kernels():
    """theta <= 0 means no rotation, which the entry point does not have."""
    for field in ("theta_global", "theta_local"):
        for theta in (0.0, -1.0):
            w = _weights()
            setattr(w, field, theta)
            assert not mb._small_layers(_rows(w), _cu(w, 0, 8), w, 2)


def test_no_layers_keep_the_separate_kernels():
    """Without a layer (num_layers 0, or below, which runs none either) there
    is no MLP output to add."""
    w = _weights()
    for n in (0, -1, -2):
        assert not mb._small_layers(_rows(w), _cu(w, 0, 8), w, n)


def test_sizes_beyond_the_entry_point_keep_the_separate_kernels():
    """Widths the entry point refuses, few tokens: hidden above 16384,
    intermediate above 65536, a weight of 2 GiB. (Meta tensors: sizes only.)"""
    for D, I, T, want in ((16384, 64, 4, True), (16448, 64, 4, False), (64, 65536, 8, True), (64, 65600, 8, False),
                          (8192, 65472, 2, False), (16384, 32768, 2, False), (16384, 32640, 2, True)):
        w = _weights(D, I, meta=True)
        assert mb._small_layers(_rows(w, T), _cu(w, 0, T), w, 2) is want, (D, I)


def test_the_entry_point_takes_what_the_rule_lets_through():
    """Every weight of a size that the rule accepts lies within the entry
    point's offsets: (rows + 128) rows of it below 2 GiB."""
    for D in range(64, 16385, 64):
        I = min(65536, (mb._MAX_WEIGHT - 1) // (4 * D) // 64 * 64)
        for rows, cols in ((3 * D, D), (D, D), (2 * I, D), (D, I)):
            assert 2 * (rows + 128) * cols < 1 << 31, (D, I)
