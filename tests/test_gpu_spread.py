"""Ragged decode batches whose steps are cut into equal ranges over the workgroups, against the float32 kernels, which take
one sequence after the other."""
import math

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tq():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a GPU: torch.cuda.is_available() is False")
    import tqhip
    return tqhip


# lengths at the edges of a step (256 positions) and of a workgroup's share, empty sequences first, last and in a row, more
# sequences than a wavefront has lanes, kv heads that do not divide the launch, one long sequence, a bound on the lengths far
# above them, a launch cut down to what the workspace holds (three sequences of one kv head)
CASES = [
    ([0, 0, 5000, 256, 0, 1, 4097, 20000, 255, 0], 8, 4, 0),
    ([(i * 97) % 700 for i in range(70)] + [0, 6000], 4, 2, 0),
    ([70001], 8, 1, 0),
    ([16384, 8192, 512, 8191, 8193], 6, 7, 0),
    ([43777, 3, 30000], 1, 16, 0),
    ([300, 40, 1, 3100, 2900, 3000], 8, 4, 9341),
]


@pytest.mark.parametrize("bits", [3, 1, 2, 4])
@pytest.mark.parametrize("lens,n_kv,n_rep,bound", CASES)
def test_spread_ranges(tq, bits, lens, n_kv, n_rep, bound):
    D, n_seq, rows = 128, len(lens), sum(lens)
    longest = bound or max(lens)
    assert tq._lib.load().tq_flash_decode_plan(n_seq, n_kv, longest, 1, 0) >= 2          # a streaming launch
    g = torch.Generator(device="cuda")
    g.manual_seed(rows + bits)
    cb = tq.quantizer.gaussian_codebook(bits)
    bd = tq.quantizer.gaussian_boundaries(cb)
    ks, vs = (tq.random_diagonal_sign(D, seed=s, device="cuda") for s in (42, 43))
    sides = []
    for s in (ks, vs):
        p, n = tq.fused_quantize(torch.randn((n_kv * rows, D), generator=g, device="cuda"), s, bd, D, bits)
        sides += [p.view(n_kv, rows, -1), n.view(n_kv, rows)]
    kp, kn, vp, vn = sides
    q = torch.randn((n_seq, n_kv * n_rep, D), generator=g, device="cuda")
    q[:, 0] *= 8                                                                          # a head whose maximum moves late
    offs = torch.tensor([0] + lens, device="cuda").cumsum(0).to(torch.int32)
    sc = 1 / math.sqrt(D)
    q_rot = tq.prerotate_query(q.view(-1, D), ks).view(n_seq, -1, D)
    for other in (1.0, 1.25):                                                             # one table for keys and values, or two
        kw = dict(n_rep=n_rep, seq_offsets=offs, max_seq_len=longest)
        got = tq.flash_decode(q_rot, kp, kn, vp, vn, cb, cb * other, vs, D, bits, sc, **kw)
        again = tq.flash_decode_from_q(q, ks, kp, kn, vp, vn, cb, cb * other, vs, D, bits, sc, **kw)
        assert torch.equal(got, again)
        for i, n in enumerate(lens):
            if n == 0:
                assert not got[i].any()
                continue
            a = sum(lens[:i])
            want = tq.flash_decode(q_rot[i:i + 1], kp[:, a:a + n], kn[:, a:a + n], vp[:, a:a + n], vn[:, a:a + n], cb, cb * other, vs,
                                   D, bits, sc, n_rep=n_rep, seq_offsets=torch.tensor([0, n], device="cuda", dtype=torch.int32),
                                   max_seq_len=n, precision="fp32")
            # weights enter the products as fp16, 2^-11 of the sum of |weight x value|, and the peaked head's sum is a few values, as
            # large as the row's largest result: the bar of 1e-3 + 2e-3 of the row's magnitude is four times that
            assert ((got[i] - want[0]).abs() <= 1e-3 + 2e-3 * want[0].abs().amax(-1, keepdim=True)).all(), (i, n)
