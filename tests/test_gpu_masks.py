"""Decode attention under masks: every form and dtype that the hook takes against the same mask as float32 rows of every
query head (which stay with the tile kernels), and the streaming pass with a shared mask at its edges."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tq():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a GPU: torch.cuda.is_available() is False")
    import tqhip
    return tqhip


def _cache(tq, cls, B, n_kv, T, bits=3, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    cache = cls(bits=bits, fused=True)
    mk = lambda *s: torch.randn(s, generator=g, device="cuda", dtype=torch.float16)   # noqa: E731
    cache.update_and_fetch(mk(B, n_kv, T, 128), mk(B, n_kv, T, 128))
    return cache, lambda n_rep: mk(B, n_kv * n_rep, 1, 128)


def _rows(mask, B, n_q, T):
    """The float32 rows of a (B, 1 | n_q, 1, T) mask, one per sequence and head."""
    m = mask.expand(B, mask.shape[1], 1, T).expand(B, n_q, 1, T)[:, :, 0]
    if m.dtype == torch.bool:
        m = torch.zeros(m.shape, device=m.device).masked_fill_(~m, float("-inf"))
    return m.float().contiguous()


# two fp16-operand kernels that sum in another order: a softmax weight rounded to fp16 is off by 2^-11, results of unit size
# by a few of those at most
def _close(a, b):
    a, b = a.float(), b.float()
    assert torch.isfinite(a).all()
    assert (a - b).abs().max().item() <= 1e-3, (a - b).abs().max().item()


# lengths around a wave's 64 and a workgroup's 256 positions; batches that take the tile pass (plan 0) and the streaming
# pass (plan >= 2)
@pytest.mark.parametrize("B,n_kv,n_rep,T,bits", [(2, 2, 4, 63, 3), (2, 2, 4, 1030, 3), (8, 8, 4, 2305, 3), (9, 8, 1, 2111, 3), (8, 8, 4, 6003, 3),
                                                 (6, 8, 4, 4097, 2), (6, 8, 4, 3900, 4), (7, 8, 2, 3840, 1)])
def test_padding_masks(tq, B, n_kv, n_rep, T, bits):
    cache, query = _cache(tq, tq.TurboQuantKVCache, B, n_kv, T, bits)
    q, n_q = query(n_rep), n_kv * n_rep
    pos = torch.arange(T, device="cuda").view(1, 1, 1, -1)
    pad = torch.tensor([(i * T) // B for i in range(B)], device="cuda").view(B, 1, 1, 1)
    pad[-1] = T - 1
    boolean = pos >= pad
    holes = boolean.clone()
    holes[..., 40:min(700, T - 1)] = False                                 # whole steps excluded in the middle of a row
    for b in (boolean, holes):
        rows = _rows(b, B, n_q, T)
        want = tq.scaled_dot_product_attention(q, None, None, cache, 0.09, rows[:, :, None])
        add = torch.zeros(b.shape, device="cuda").masked_fill_(~b, float("-inf"))
        for m in (b, add, add.half(), add.bfloat16(), b.expand(B, 1, 3, T), b[:, 0], b.transpose(0, 1).contiguous().transpose(0, 1)):
            _close(tq.scaled_dot_product_attention(q, None, None, cache, 0.09, m), want)
    # finite biases, and a mask of the type's lowest value instead of -inf
    bias = torch.randn(1, 1, 1, T, device="cuda")
    low = torch.zeros(boolean.shape, device="cuda").masked_fill_(~boolean, torch.finfo(torch.float32).min) + bias.clamp(max=0)
    for m in (bias, low, bias[0, 0, 0], bias[0, 0]):
        full = (m if m.dim() == 4 else m.reshape(1, 1, 1, T))
        _close(tq.scaled_dot_product_attention(q, None, None, cache, 0.09, m),
               tq.scaled_dot_product_attention(q, None, None, cache, 0.09, _rows(full, B, n_q, T)[:, :, None]))
    # one sequence without any visible position
    none = boolean.clone()
    none[0] = False
    got = tq.scaled_dot_product_attention(q, None, None, cache, 0.09, none)
    want = tq.scaled_dot_product_attention(q, None, None, cache, 0.09, _rows(none, B, n_q, T)[:, :, None])
    assert torch.equal(got[0], want[0]) and not got[0].any()
    _close(got, want)


def test_mask_excludes_rows_of_odd_norms(tq):
    """Rows with NaN or infinite norms behind a mask behave as the tile pass has them."""
    cache, query = _cache(tq, tq.TurboQuantKVCache, 8, 8, 3000)
    q = query(4)
    b = torch.arange(3000, device="cuda").view(1, 1, 1, -1) >= 1100
    for value in (float("nan"), float("inf")):
        cache.v_norms[3, 2, 500] = value
        got = tq.scaled_dot_product_attention(q, None, None, cache, 0.09, b)
        want = tq.scaled_dot_product_attention(q, None, None, cache, 0.09, _rows(b, 8, 32, 3000)[:, :, None])
        assert torch.equal(got.isnan(), want.isnan())
        cache.v_norms[3, 2, 500] = 1.0


def test_vonly_and_thresholded_masks(tq):
    B, n_kv, T = 3, 2, 1501
    pad = torch.tensor([0, 700, 1500], device="cuda").view(B, 1, 1, 1)
    b = torch.arange(T, device="cuda").view(1, 1, 1, -1) >= pad
    for cls in (tq.VOnlyTurboQuantCache, tq.TurboQuantKVCache):
        cache, query = _cache(tq, cls, B, n_kv, T)
        q = query(4)
        for thr in (None, 1e-4):
            cache.sparse_v_threshold = thr
            want = tq.scaled_dot_product_attention(q, None, None, cache, 0.09, _rows(b, B, 8, T)[:, :, None])
            for m in (b, b.expand(B, 8, 1, T), torch.zeros(b.shape, device="cuda", dtype=torch.bfloat16).masked_fill_(~b, float("-inf"))):
                _close(tq.scaled_dot_product_attention(q, None, None, cache, 0.09, m), want)
    with pytest.raises((RuntimeError, ValueError)):
        tq.scaled_dot_product_attention(q, None, None, cache, 0.09, b[..., :-1])
