"""The composed decode step in three launches against its operations one by one (scores, softmax, thresholded value sum) and
against the oracle: lengths at the edges of a wave's 64 and a tile's 512 positions, head groupings, masks, odd values."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import polarquant_oracle as o  # noqa: E402

pytestmark = pytest.mark.gpu

D = 128


@pytest.fixture(scope="module")
def tq():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a GPU: torch.cuda.is_available() is False")
    import tqhip
    return tqhip


def _cache(tq, B, n_kv, T, bits, seed=0, dtype=torch.float16):
    g = torch.Generator(device="cuda").manual_seed(seed)
    cache = tq.TurboQuantKVCache(bits=bits, fused=True)
    mk = lambda *s: torch.randn(s, generator=g, device="cuda", dtype=dtype)   # noqa: E731
    cache.update_and_fetch(mk(B, n_kv, T, D), mk(B, n_kv, T, D))
    return cache, mk


def _one_by_one(tq, q, cache, scale, rows, thr):
    outs = []
    kq, vq, T = cache._k_q, cache._v_q, cache.offset
    n_rep = q.shape[1] // cache.k_packed.shape[1]
    for b in range(q.shape[0]):
        qr = tq.prerotate_query(q[b, :, 0], kq.signs)
        s = tq.prerot_fused_qk_scores(qr, cache.k_packed[b, :, :T], cache.k_norms[b, :, :T], kq.centroids, D, cache.quant_bits, n_rep=n_rep)
        w = tq.softmax_rows(s, scale, None if rows is None else rows[b])
        outs.append(tq.sparse_v_matvec(w, cache.v_packed[b, :, :T], cache.v_norms[b, :, :T], vq.centroids, vq.signs, D, cache.quant_bits,
                                       threshold=thr, n_rep=n_rep))
    return torch.stack(outs)[:, :, None]


@pytest.mark.parametrize("B,n_kv,n_rep,T,bits", [(1, 1, 1, 1, 3), (2, 2, 3, 63, 3), (1, 2, 7, 512, 3), (3, 2, 4, 513, 2), (2, 1, 16, 1029, 4),
                                                 (2, 3, 8, 2047, 1), (1, 4, 7, 20001, 3)])
def test_composed_step(tq, B, n_kv, n_rep, T, bits):
    cache, mk = _cache(tq, B, n_kv, T, bits)
    n_q = n_kv * n_rep
    q = mk(B, n_q, 1, D).float()
    scale = D ** -0.5
    pad = torch.tensor([(b * T) // (2 * B) for b in range(B)], device="cuda").view(B, 1, 1, 1)
    keep = torch.arange(T, device="cuda").view(1, 1, 1, -1) >= pad
    for mask, rows in ((None, None), (keep, torch.zeros(B, 1, T, device="cuda").masked_fill_(~keep[:, 0], float("-inf"))),
                       (torch.randn(n_q, T, device="cuda"), None)):
        if rows is None and mask is not None:
            rows = mask[None].expand(B, n_q, T)
        for thr in (0.0, 1e-5):
            got = tq.turboquant_attention(q, cache, scale, mask, sparse_v_threshold=thr)
            want = _one_by_one(tq, q, cache, scale, rows, thr)
            # float32 throughout: sums in another order (2^-24 a step), weights at the threshold may fall on either side (1e-5 of
            # a value of a few units each, one or two of them)
            bound = 3e-6 * want.abs().max().item() + (1.5e-4 if thr else 0.0)
            assert (got - want).abs().max().item() <= bound, ((got - want).abs().max().item(), bound)
    for dt in (torch.float16, torch.bfloat16):
        got = tq.turboquant_attention(q.to(dt), cache, scale)
        want = _one_by_one(tq, q.to(dt), cache, scale, None, 0.0)
        assert got.dtype == dt and torch.allclose(got.float(), want, rtol=2e-3 if dt == torch.float16 else 1e-2, atol=1e-6)


def test_composed_odd_values(tq):
    """Rows without a visible position, NaN and infinite norms give NaN where the single operations do."""
    cache, mk = _cache(tq, 2, 2, 1200, 3)
    q = mk(2, 8, 1, D).float()
    rows = torch.zeros(2, 8, 1200, device="cuda")
    rows[0, 3] = float("-inf")
    rows[1, 1] = torch.finfo(torch.float32).min
    for which, value in ((None, 0.0), ("k_norms", float("nan")), ("k_norms", float("inf")), ("v_norms", float("nan"))):
        if which:
            getattr(cache, which)[1, 0, 700] = value
        got = tq.turboquant_attention(q, cache, 0.09, rows[:, :, None])
        want = _one_by_one(tq, q, cache, 0.09, rows, 0.0)
        assert torch.equal(got.isnan(), want.isnan()), which
        if which:
            getattr(cache, which)[1, 0, 700] = 1.0


def test_composed_in_several_calls(tq, monkeypatch):
    cache, mk = _cache(tq, 5, 2, 700, 3)
    q = mk(5, 6, 1, D)
    mask = torch.arange(700, device="cuda").view(1, 1, 1, -1) >= torch.arange(5, device="cuda").view(5, 1, 1, 1) * 50
    whole = tq.turboquant_attention(q, cache, 0.09, mask)
    monkeypatch.setattr(tq.ops, "_COMPOSED_WORKSPACE", 100_000)
    assert torch.equal(whole, tq.turboquant_attention(q, cache, 0.09, mask))


@pytest.mark.parametrize("B,most", [(4, 1 << 20), (1, 17 << 20)])
def test_composed_scores_are_not_kept(tq, monkeypatch, B, most):
    """The scores of a large call (37 MB here) are free again after it; a small one (9 MB) may leave them in the workspace of
    its stream."""
    cache, mk = _cache(tq, B, 4, 65536, 3)
    q = mk(B, 28, 1, D)
    monkeypatch.setattr(tq.ops, "_workspaces", {})
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    out = tq.turboquant_attention(q, cache, 0.09)
    kept = torch.cuda.memory_allocated() - before - out.numel() * out.element_size()
    assert kept < most, kept


@pytest.mark.parametrize("T", [5, 700])
def test_queries_of_the_first_sequences(tq, T):
    """Fewer queries than the cache holds sequences: those of the first ones, for a decode step and for a chunk."""
    cache, mk = _cache(tq, 3, 2, T, 3)
    q, rows = mk(3, 6, 1, D), mk(3, 6, 4, D)
    whole, chunk = tq.turboquant_attention(q, cache, 0.09), tq.turboquant_prefill_attention(rows, cache, 0.09)
    for n in (1, 2):
        assert torch.equal(tq.turboquant_attention(q[:n], cache, 0.09), whole[:n])
        got = tq.turboquant_prefill_attention(rows[:n], cache, 0.09)
        assert (got - chunk[:n]).abs().max() <= 4e-3 * chunk.abs().max()        # fp16 results, another split of the positions
