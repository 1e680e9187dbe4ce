"""The streaming codec at row counts that are no multiple of its pass and at head dimensions 64 and 256: bit-exact
against the oracle, destination rows of strided groups included."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import polarquant_oracle as o  # noqa: E402

pytestmark = pytest.mark.gpu

_DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


@pytest.fixture(scope="module")
def tq():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a GPU: torch.cuda.is_available() is False")
    import tqhip
    return tqhip


def _rows(rng, n, dim):
    """Random scales, a zero row, one-hot rows, and rows along a Hadamard vector (one butterfly output of sqrt(dim))."""
    x = (rng.standard_normal((n, dim)) * rng.choice([1e-3, 1.0, 300.0], size=(n, 1))).astype(np.float32)
    x[1] = 0.0
    x[2] = 0.0
    x[2, dim - 1] = -2.5
    for r in range(3, 11):
        k = int(rng.integers(0, dim))
        x[r] = [(-1.0) ** bin(j & k).count("1") for j in range(dim)]
    return x


# groups of one row, of odd counts below, around and above the 32 / 16 / 8 vectors of a pass; totals at the lower
# edges of the streaming forms and above the size from which a wavefront makes four passes
@pytest.mark.parametrize("dim,bits,dtype,groups,rows,alloc", [
    (64, 4, "f16", 12288, 1, 3), (64, 3, "bf16", 401, 31, 40), (64, 2, "f32", 373, 33, 33), (64, 1, "f16", 12, 1037, 1040),
    (128, 3, "bf16", 9, 1001, 1024), (128, 3, "f16", 8193, 1, 1), (128, 4, "f32", 547, 15, 16), (128, 2, "f16", 47, 177, 256),
    (128, 1, "bf16", 483, 17, 20), (128, 3, "f16", 3, 100003, 100096),
    (256, 3, "f16", 878, 7, 9), (256, 4, "bf16", 683, 9, 9), (256, 2, "f32", 1, 6151, 6151), (256, 1, "f16", 2, 4097, 4100),
    (64, 3, "f16", 1, 6143, 6144), (128, 3, "f16", 1, 5121, 5121), (256, 3, "f16", 3, 1027, 1027),
])
def test_codec_rows(tq, dim, bits, dtype, groups, rows, alloc):
    rng = np.random.default_rng(dim + bits + rows)
    c = o.gaussian_codebook(bits)
    b = o.gaussian_boundaries(c)
    s = o.random_diagonal_sign(dim, 42)
    n = groups * rows
    small = min(n, 6000)                               # the oracle's share of a large case: its first and last rows
    x = torch.from_numpy(_rows(rng, small, dim)).to(_DT[dtype])
    x = x.repeat(-(-n // small), 1)[:n]
    x[n - 1] = x[3]
    x = x.cuda()
    sg = torch.from_numpy(s).cuda()
    pd = tq.packed_dim(dim, bits)
    packed = torch.full((groups, alloc, pd), -1, dtype=torch.int32, device="cuda").view(torch.uint32)
    norms = torch.full((groups, alloc), -1.0, dtype=torch.float32, device="cuda")
    off = alloc - rows
    for variant in ("metal", "mlx"):
        tq.encode_into(x, sg, b, packed, norms, n_groups=groups, rows_per_group=rows, packed_group_stride=alloc,
                       norms_group_stride=alloc, dim=dim, bits=bits, variant=variant, packed_row_offset=off, norms_row_offset=off)
        p = packed.view(torch.int32)
        got_p, got_n = p[:, off:].reshape(n, pd), norms[:, off:].reshape(n)
        assert bool((p[:, :off] == -1).all()) and bool((norms[:, :off] == -1.0).all())
        for lo, hi in ((0, small), (n - min(n, 300), n)):
            wp, wn = o.fused_quantize(x[lo:hi].float().cpu().numpy(), s, b, dim, bits, variant)
            assert np.array_equal(got_p[lo:hi].cpu().numpy().view(np.uint32), wp)
            assert np.array_equal(got_n[lo:hi].cpu().numpy(), wn)
    for dt in (torch.float16, torch.bfloat16, torch.float32):
        out = torch.full((groups, alloc + 1, dim), 7.0, dtype=dt, device="cuda")
        tq.dequant_into(packed, norms, c, sg, out, n_groups=groups, rows_per_group=rows, packed_group_stride=alloc,
                        norms_group_stride=alloc, out_group_stride=alloc + 1, dim=dim, bits=bits, packed_row_offset=off,
                        norms_row_offset=off, out_row_offset=1)
        assert bool((out[:, :1] == 7.0).all()) and bool((out[:, 1 + rows:] == 7.0).all())
        got = out[:, 1:1 + rows].reshape(n, dim)
        for lo, hi in ((0, small), (n - min(n, 300), n)):
            w = o.packed_dequantize(got_p[lo:hi].cpu().numpy().view(np.uint32), got_n[lo:hi].cpu().numpy(), c, s, dim, bits)
            assert torch.equal(got[lo:hi].cpu(), torch.from_numpy(w).to(dt))


@pytest.mark.parametrize("dim", [64, 128, 256])
def test_codec_rows_nan(tq, dim):
    """A row with a NaN gets index 0 everywhere (comparisons with NaN are false) and leaves its neighbours alone."""
    rng = np.random.default_rng(9)
    c = o.gaussian_codebook(3)
    b = o.gaussian_boundaries(c)
    s = o.random_diagonal_sign(dim, 43)
    x = rng.standard_normal((7777, dim)).astype(np.float16)
    bad = [0, 300, 7776]
    x[bad, 3] = np.nan
    ok = np.setdiff1d(np.arange(7777), bad)
    gp, gn = tq.fused_quantize(torch.from_numpy(x).cuda(), torch.from_numpy(s).cuda(), b, dim, 3)
    gp, gn = gp.cpu().numpy(), gn.cpu().numpy()
    wp, wn = o.fused_quantize(x[ok], s, b, dim, 3)
    assert np.array_equal(gp[ok], wp) and np.array_equal(gn[ok], wn)
    assert (gp[bad] == 0).all() and np.isnan(gn[bad]).all()


# decision boundaries far out, where only rows along a Hadamard vector (one butterfly output of sqrt(dim)) reach them: the level
# table of the streaming encoder has 64 cells (128 at four bits), and at d = 256 outputs beyond it are clamped into the last
@pytest.mark.parametrize("dim,bounds", [
    (256, [14.0]), (256, [-14.0]), (256, [11.4]), (256, [15.9]), (256, [-13.0, 0.0, 13.0]), (256, [10.0, 12.5, 15.0]),
    (256, [-15.0, -14.0, -13.0, 0.0, 13.0, 14.0, 15.0]), (256, [float(i) * 2.1 for i in range(-7, 8)]),
    (256, [-15.5] + [0.3 * i for i in range(-6, 7)] + [15.5]), (128, [11.0]), (128, [-11.2, 0.0, 11.2]), (128, [30.0]), (64, [7.9]),
])
def test_boundaries_near_the_largest_output(tq, dim, bounds):
    bits = {1: 1, 3: 2, 7: 3, 15: 4}[len(bounds)]
    rng = np.random.default_rng(dim)
    n = 6151
    x = _rows(rng, n, dim)
    s = o.random_diagonal_sign(dim, 42)
    for r in range(100, 1600):                          # along +- a Hadamard vector of the signed rows, with and without noise
        k = int(rng.integers(0, dim))
        h = np.array([(-1.0) ** bin(j & k).count("1") for j in range(dim)])
        x[r] = (rng.choice([-1.0, 1.0]) * h + rng.choice([0.0, 0.1, 0.5]) * rng.standard_normal(dim)) * s
    b = np.asarray(bounds, dtype=np.float32)
    gp, gn = tq.fused_quantize(torch.from_numpy(x).cuda(), torch.from_numpy(s).cuda(), b, dim, bits)
    wp, wn = o.fused_quantize(x, s, b, dim, bits)
    idx = o.unpack_indices(wp, bits, dim)
    assert idx.max() > 0 or max(bounds) > dim ** 0.5
    assert np.array_equal(gp.cpu().numpy(), wp) and np.array_equal(gn.cpu().numpy(), wn)


@pytest.mark.parametrize("call", ["append", "encode"])
def test_small_calls_do_not_wait_for_the_level_search(tq, call):
    """The search for the streaming encoder's level line (13 ms at four bits) is no part of a call that does not take it: a
    token's append, a few rows.  Each call has boundaries that no call has had before."""
    import time
    dim, bits, n = 64, 4, 8
    s = torch.from_numpy(o.random_diagonal_sign(dim, 42)).cuda()
    base = np.asarray(o.gaussian_boundaries(o.gaussian_codebook(bits)), dtype=np.float32)
    x = torch.randn(1, 1, n, dim, device="cuda").half()
    k, v = (torch.zeros(1, 1, n, dim, dtype=torch.float16, device="cuda") for _ in range(2))
    vp = torch.zeros(1, 1, n, tq.packed_dim(dim, bits), dtype=torch.int32, device="cuda").view(torch.uint32)
    vn = torch.zeros(1, 1, n, device="cuda")
    took = []
    for i in range(12):
        b = base * np.float32(1.0 + 0.01 * i + (0.003 if call == "encode" else 0.0))
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        if call == "append":
            tq.ops.vonly_append_into(x, x, s, b, k, v, vp, vn, position=0, bits=bits)
        else:
            tq.fused_quantize(x[0, 0], s, b, dim, bits)
        took.append(time.perf_counter() - t0)
    assert sorted(took)[len(took) // 2] < 2e-3, took


@pytest.mark.parametrize("dim", [64, 128, 256])
@pytest.mark.parametrize("bounds", [[-30.0], [-60.0, -40.0, 0.5], [0.3]])
def test_infinities_under_boundaries_that_no_output_reaches(tq, dim, bounds):
    """A row with an infinity has an infinite norm and outputs that are no numbers: every index 0."""
    rng = np.random.default_rng(dim)
    x = _rows(rng, 6151, dim)
    x[20:40, 3] = np.inf
    x[40:60, dim - 1] = -np.inf
    s = o.random_diagonal_sign(dim, 42)
    b = np.asarray(bounds, dtype=np.float32)
    bits = {1: 1, 3: 2}[len(bounds)]
    with np.errstate(invalid="ignore"):
        wp, wn = o.fused_quantize(x, s, b, dim, bits)
    assert not wp[20:60].any()
    gp, gn = tq.fused_quantize(torch.from_numpy(x).cuda(), torch.from_numpy(s).cuda(), b, dim, bits)
    assert np.array_equal(gp.cpu().numpy(), wp) and np.array_equal(gn.cpu().numpy(), wn)
