"""Ragged decode batches on the streaming pass, with a workgroup per partial and with the partials shared out in equal ranges of
steps, against the float32 kernels, which take one sequence after the other."""
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


# lengths at the edges of a step (256 positions) and of a workgroup's share, empty sequences first, last and in a row, more
# sequences than a wavefront has lanes, kv heads that do not divide the launch, one long sequence, a bound on the lengths far
# above them, fewer steps than workgroups; partials of two, three and four steps; last: the partials are shared out
CASES = [
    ([0, 0, 5000, 256, 0, 1, 4097, 20000, 255, 0], 8, 4, 0, True),
    ([(i * 97) % 700 for i in range(70)] + [0, 6000], 4, 2, 0, True),
    ([70001], 8, 1, 0, False),
    ([16384, 8192, 512, 8191, 8193], 6, 7, 0, False),
    ([43777, 3, 30000], 1, 16, 0, False),
    ([300, 40, 1, 3100, 2900, 3000], 8, 4, 9341, False),
    ([100001], 16, 1, 0, True),
    ([max(0, 1024 * (i % 7) + i % 3 - 1) for i in range(39)] + [6259], 6, 7, 0, True),
    ([66000, 3, 30000] + [0] * 20 + [257], 1, 16, 0, True),
    ([4138, 768, 0, 1537, 3000, 4138, 2304, 1, 767, 769], 32, 4, 0, True),
    ([2320] + [33 * i for i in range(69)], 8, 5, 0, True),
]


@pytest.mark.parametrize("bits", [3, 1, 2, 4])
@pytest.mark.parametrize("lens,n_kv,n_rep,bound,shared", CASES)
def test_spread_ranges(tq, bits, lens, n_kv, n_rep, bound, shared):
    D, n_seq, rows = 128, len(lens), sum(lens)
    longest = bound or max(lens)
    assert tq._lib.load().tq_flash_decode_plan(n_seq, n_kv, longest, 1, 0) >= 2          # a streaming launch
    assert (tq._lib.load().tq_flash_decode_groups(n_seq, n_kv, longest) > 0) == shared
    g = torch.Generator(device="cuda")
    g.manual_seed(rows + bits)
    cb = tq.quantizer.gaussian_codebook(bits)
    bd = tq.quantizer.gaussian_boundaries(cb)
    ks, vs = (tq.random_diagonal_sign(D, seed=s, device="cuda") for s in (42, 43))
    steps = tq._lib.load().tq_flash_decode_plan(n_seq, n_kv, longest, 1, 0)
    x = [torch.randn((n_kv, rows, D), generator=g, device="cuda") for _ in range(2)]
    q = torch.randn((n_seq, n_kv * n_rep, D), generator=g, device="cuda")
    first = [sum(lens[:i]) for i in range(n_seq)]
    edges = [edge_rows.edge_positions(n, (64, 256, 256 * steps)) if n else [] for n in lens]
    for i, n in enumerate(lens):                                                          # weight on the rows at the edges of blocks and partials
        if n:
            edge_rows.plant(*(t[:, first[i]:first[i] + n] for t in x), q[i], edges[i], kappa={1: 0.8, 2: 0.94}.get(bits, 1.0))
    q[:, 0] *= 8                                                                          # a head whose maximum moves late
    sides = []
    for s, t in zip((ks, vs), x):
        p, n = tq.fused_quantize(t.view(-1, D), s, bd, D, bits)
        sides += [p.view(n_kv, rows, -1), n.view(n_kv, rows)]
    kp, kn, vp, vn = sides
    del x
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
            mine = [t[:, first[i]:first[i] + n] for t in (kp, kn, vp, vn)]
            want = tq.flash_decode(q_rot[i:i + 1], *mine, cb, cb * other, vs, D, bits, sc, n_rep=n_rep,
                                   seq_offsets=torch.tensor([0, n], device="cuda", dtype=torch.int32), max_seq_len=n, precision="fp32")
            k, v = (tq.packed_dequantize(p.reshape(n_kv * n, -1), m.reshape(-1), c, sign, D, bits).view(n_kv, n, D)
                    for p, m, c, sign in ((mine[0], mine[1], cb, ks), (mine[2], mine[3], cb * other, vs)))
            edge_rows.check(got[i], want[0], q[i], k, v, sc, edges[i], edge_rows.fp16_weights_bound(v, bits))


# partials of two, three and four steps, in shared-out ranges and a workgroup each; the bound on the lengths and the number of
# sequences stay, the lengths beside one sequence change: its partials then fall to other workgroups, alone or behind others
@pytest.mark.parametrize("n_seq,n_kv,n_rep,bound,steps,shared", [(3, 8, 4, 9000, 2, False), (70, 8, 4, 2320, 2, True),
                                                                 (10, 32, 8, 4138, 3, True), (4, 16, 1, 40000, 4, True)])
def test_neighbours_change_no_bit(tq, n_seq, n_kv, n_rep, bound, steps, shared):
    D, bits = 128, 3
    lib = tq._lib.load()
    assert lib.tq_flash_decode_plan(n_seq, n_kv, bound, 1, 0) == steps
    assert (lib.tq_flash_decode_groups(n_seq, n_kv, bound) > 0) == shared
    cb = tq.quantizer.gaussian_codebook(bits)
    bd = tq.quantizer.gaussian_boundaries(cb)
    ks, vs = (tq.random_diagonal_sign(D, seed=s, device="cuda") for s in (42, 43))
    own = bound - 500                                                                     # a last step of part of its rows
    g = torch.Generator(device="cuda").manual_seed(bound)
    x = [torch.randn((n_kv, own, D), generator=g, device="cuda") for _ in range(2)]
    q = torch.randn((n_seq, n_kv * n_rep, D), generator=g, device="cuda")
    first = None
    for at, others in ((0, [bound] * (n_seq - 1)), (0, [700] * (n_seq - 1)), (n_seq - 1, [bound // 2 + 77 * i for i in range(n_seq - 1)]),
                       (1, [0] * (n_seq - 2) + [700]), (0, [500])):
        lens = others[:at] + [own] + others[at:]
        if lib.tq_flash_decode_plan(len(lens), n_kv, bound, 1, 0) != steps:
            continue                                                                      # the last one: fewer sequences, the same partials
        sides, a = [], sum(lens[:at])
        for s, mine in zip((ks, vs), x):
            rows = torch.randn((n_kv, sum(lens), D), generator=g, device="cuda")
            rows[:, a:a + own] = mine
            p, n = tq.fused_quantize(rows.view(-1, D), s, bd, D, bits)
            sides += [p.view(n_kv, sum(lens), -1), n.view(n_kv, sum(lens))]
        offs = torch.tensor([0] + lens, device="cuda").cumsum(0).to(torch.int32)
        queries = q.roll(at, 0)[:len(lens)]
        out = tq.flash_decode_from_q(queries, ks, *sides, cb, cb, vs, D, bits, D ** -0.5, n_rep=n_rep, seq_offsets=offs, max_seq_len=bound)
        first = out[at] if first is None else first
        assert torch.equal(out[at], first), lens
