"""The streaming pass over given softmax statistics at the head counts where its register groups change, against the composition of
scores, softmax and float32 value sums."""
import math

import pytest

torch = pytest.importorskip("torch")

import edge_rows  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tq():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a GPU: torch.cuda.is_available() is False")
    import tqhip
    return tqhip


# heads per kv head on both sides of the lines at 4 and 8; more than 1 024 steps of 256 positions (there the pass streams), with a
# last block of one row, of a part of a tile, and whole; half of the weight lies on rows at the edges of blocks and ranges
@pytest.mark.parametrize("bits", [3, 4, 2, 1])
@pytest.mark.parametrize("n_rep,T", [(1, 16641), (4, 16700), (5, 17152), (8, 16641), (9, 16800), (16, 16403)])
def test_threshold_streams_at_every_head_count(tq, bits, n_rep, T):
    n_seq, n_kv, D, thr = 2, 8, 128, 1e-4
    g = torch.Generator(device="cuda")
    g.manual_seed(T + n_rep)
    cache = tq.VOnlyTurboQuantCache(bits=bits, fused=True)
    k, v = (torch.randn((n_seq, n_kv, T, D), generator=g, device="cuda", dtype=torch.float16) for _ in range(2))
    q = torch.randn((n_seq, n_kv * n_rep, 1, D), generator=g, device="cuda", dtype=torch.float16)
    steps = tq._lib.load().tq_flash_decode_plan(n_seq, n_kv, T, 0, 0)
    assert steps >= 2
    edges = edge_rows.edge_positions(T, (64, 256, 256 * steps))
    for b in range(n_seq):
        edge_rows.plant(k[b], v[b], q[b, :, 0], edges)
    cache.update_and_fetch(k, v)
    sc = 1 / math.sqrt(D)
    got = tq.vonly_decode_attention(q, cache, sc, sparse_v_threshold=thr)
    kv, vq = cache._v_tq, cache._v_tq._v_q
    for b in range(n_seq):
        w = tq.softmax_rows(tq.dense_qk_scores(q[b, :, 0], k[b], 1.0, n_rep=n_rep), sc)
        assert (w < thr).any() and (w >= thr).any()
        vp, vn = kv.v_packed[b, :, :T], kv.v_norms[b, :, :T]
        want = tq.sparse_v_matvec(w, vp, vn, vq.centroids, vq.signs, D, bits, threshold=thr, n_rep=n_rep, precision="fp32")
        values = tq.packed_dequantize(vp.reshape(n_kv * T, -1), vn.reshape(-1), vq.centroids, vq.signs, D, bits).view(n_kv, T, D)
        close = edge_rows.fp16_weights_bound(values, bits)
        # and two weights at the threshold may round to its other side (rows between the edges have values of one to five)
        edge_rows.check(got[b, :, 0], want, q[b, :, 0], k[b], values, sc, edges, lambda w, terms: close(w, terms) + 2 * thr * 5)
