"""Infinite and NaN norms where the scores of few query heads share register groups: the same heads in a group of sixteen, whose
scores share nothing, give the same infinities and NaN, and the other kv heads keep their bits."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

D = 128


@pytest.fixture(scope="module")
def tq():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a GPU: torch.cuda.is_available() is False")
    import tqhip
    return tqhip


def _sixteen(q, n_rep):
    """The heads of each kv head, repeated up to sixteen."""
    n_seq, n_q, d = q.shape
    at = torch.arange(16, device=q.device) % n_rep
    return q.view(n_seq, -1, n_rep, d)[:, :, at].reshape(n_seq, -1, d).contiguous()


def _call(tq, path, q, n_rep, ks, vs, cb, sides, lens, mask):
    bits, sc = 3, D ** -0.5
    if path == "composed":
        return tq.ops.composed_decode(q, ks, *sides, cb, cb, vs, D, bits, sc, n_rep=n_rep, seq_len=lens[0])
    kw = dict(n_rep=n_rep)
    if path == "ragged":
        kw.update(seq_offsets=torch.tensor([0] + lens, device="cuda").cumsum(0).to(torch.int32), max_seq_len=max(lens))
    if path == "masked":
        kw.update(mask=mask)
    if path == "threshold":
        kw.update(sparse_v_threshold=1e-6)
    return tq.ops.flash_from_query(q, ks, *sides, cb, cb, vs, D, bits, sc, **kw)


# path, sequences, kv heads, positions: tiles of four waves and of eight, the streaming pass plain, masked, shared out and thresholded
@pytest.mark.parametrize("n_rep", [1, 3, 4, 5, 8])
@pytest.mark.parametrize("path,n_seq,n_kv,T", [("tiles", 1, 2, 700), ("tiles", 2, 8, 5001), ("stream", 2, 8, 10001), ("masked", 3, 8, 6003),
                                               ("ragged", 70, 8, 2320), ("threshold", 2, 8, 17001), ("composed", 1, 2, 1300)])
def test_odd_norms_stay_in_their_head(tq, path, n_seq, n_kv, T, n_rep):
    g = torch.Generator(device="cuda").manual_seed(100 * T + n_rep)
    lib = tq._lib.load()
    plan = lib.tq_flash_decode_plan(n_seq, n_kv, T, int(path == "ragged"), 0)
    assert (plan >= 2) == (path in ("stream", "masked", "ragged", "threshold"))
    if path == "ragged":
        assert lib.tq_flash_decode_groups(n_seq, n_kv, T) > 0
    cb = tq.quantizer.gaussian_codebook(3)
    ks, vs = (tq.random_diagonal_sign(D, seed=s, device="cuda") for s in (42, 43))
    lens = [T - 900 * (i % 3) for i in range(n_seq)] if path == "ragged" else [T] * n_seq
    lead = (n_kv, sum(lens)) if path == "ragged" else (n_seq, n_kv, T)
    sides = []
    for s in (ks, vs):
        x = torch.randn((*lead, D), generator=g, device="cuda")
        p, n = tq.fused_quantize(x.view(-1, D), s, tq.quantizer.gaussian_boundaries(cb), D, 3)
        sides += [p.view(*lead, -1), n.view(lead)]
    q = torch.randn((n_seq, n_kv * n_rep, D), generator=g, device="cuda")
    mask = None
    if path == "masked":
        mask = torch.zeros((n_seq, 1, T), device="cuda")
        mask[0, :, :T // 3] = float("-inf")
    clean = _call(tq, path, q, n_rep, ks, vs, cb, sides, lens, mask)
    assert clean.isfinite().all()
    at = T // 2 + 37                                                        # of the first sequence: it is visible
    for which in (1, 3):                                                    # norms of keys, of values
        norms = sides[which]
        cell = norms[1] if path == "ragged" else norms[0, 1]
        kept = cell[at].clone()
        for value in (float("nan"), float("inf")):
            cell[at] = value
            got = _call(tq, path, q, n_rep, ks, vs, cb, sides, lens, mask).view(n_seq, n_kv, n_rep, D)
            want = _call(tq, path, _sixteen(q, n_rep), 16, ks, vs, cb, sides, lens, mask).view(n_seq, n_kv, 16, D)[:, :, :n_rep]
            assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isposinf(), want.isposinf())
            assert torch.equal(got.isneginf(), want.isneginf())
            other = torch.ones((n_seq, n_kv), dtype=torch.bool, device="cuda")
            other[0, 1] = False
            assert torch.equal(got[other], clean.view(got.shape)[other])
            both = got.isfinite()
            # the weights are the same numbers; their sum is taken in another order, of at most T terms in tiles: 200 * 2^-24 of it
            assert ((got - want)[both].abs() <= 200 * 2.0 ** -24 * want[both].abs().amax()).all()
        cell[at] = kept
