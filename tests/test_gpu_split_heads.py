"""The passes over operands of two fp16 numbers at the head counts where their register groups change, against the float32 kernels."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tq():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a GPU: torch.cuda.is_available() is False")
    import tqhip
    return tqhip


# heads per kv head on both sides of the lines at 4 and 8; a last tile of one row, of part of a wave's 64, of all but one row
@pytest.mark.parametrize("bits", [3, 4, 2, 1])
@pytest.mark.parametrize("n_rep,T", [(1, 513), (3, 577), (4, 1023), (5, 1), (8, 63), (9, 1100), (16, 2047)])
def test_split_passes_at_every_head_count(tq, bits, n_rep, T):
    n_kv, D, thr = 2, 128, 1e-4
    g = torch.Generator(device="cuda").manual_seed(100 * T + n_rep)
    cache = tq.TurboQuantKVCache(bits=bits, fused=True)
    k, v = (torch.randn((1, n_kv, T, D), generator=g, device="cuda") for _ in range(2))
    cache.update_and_fetch(k, v)
    kq, vq = cache._k_q, cache._v_q
    q = torch.randn((1, n_kv * n_rep, 1, D), generator=g, device="cuda")
    keys = (tq.prerotate_query(q[0, :, 0], kq.signs), cache.k_packed[0, :, :T], cache.k_norms[0, :, :T], kq.centroids, D, bits)
    s = tq.prerot_fused_qk_scores(*keys, n_rep=n_rep)
    want_s = tq.prerot_fused_qk_scores(*keys, n_rep=n_rep, precision="fp32")
    # 128 float32 additions in two orders and operands of 22 bits: 130 * 2^-24 of the sum of magnitudes, which is |q| |k| at most
    bound = 130 * 2.0 ** -24 * (q[0, :, 0].norm(dim=-1)[:, None] * k[0].norm(dim=-1).repeat_interleave(n_rep, 0))
    assert s.shape == want_s.shape and ((s - want_s).abs() <= bound).all()
    w = tq.softmax_rows(want_s, D ** -0.5)
    values = (cache.v_packed[0, :, :T], cache.v_norms[0, :, :T], vq.centroids, vq.signs, D, bits)
    out = tq.sparse_v_matvec(w, *values, threshold=thr, n_rep=n_rep)
    want = tq.sparse_v_matvec(w, *values, threshold=thr, n_rep=n_rep, precision="fp32")
    # as many float32 additions as positions, though in a tree of 512: 700 * 2^-24 of sum w |v|
    bound = 700 * 2.0 ** -24 * (w * v[0].norm(dim=-1).repeat_interleave(n_rep, 0)).sum(-1, keepdim=True)
    assert ((out - want).abs() <= bound).all()
    got = tq.turboquant_attention(q, cache, D ** -0.5, sparse_v_threshold=0.0)[0, :, 0]
    full = tq.sparse_v_matvec(w, *values, threshold=0.0, n_rep=n_rep, precision="fp32")
    # weights change by the bound on the scores, twice (numerator and sum): 2 * 130 * 2^-24 * 11 * 11 / 11.3 = 1.7e-4 = 4 * 700 * 2^-24
    assert ((got - full).abs() <= 4 * bound).all()
