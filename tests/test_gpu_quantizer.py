"""PolarQuantizer's one-launch forms against the packed words in between (which other tests hold to the oracle): equal bytes,
norms and float32 rows, bit for bit."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tq():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a GPU: torch.cuda.is_available() is False")
    import tqhip
    return tqhip


def _rows(n, dim, dtype, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    x = torch.randn((n, dim), generator=g, device="cuda") * torch.logspace(-3, 3, n, device="cuda")[:, None]
    for at, value in ((1, 0.0), (3, float("nan")), (6, float("inf"))):   # a zero row, rows with one NaN or infinity
        if at < n:
            x[at] = value if value == 0.0 else x[at].index_fill(0, torch.tensor([dim // 3], device="cuda"), value)
    return x.to(dtype)


def _bits_of(t):
    return torch.where(t.isnan(), torch.full_like(t, 7e9), t).view(torch.int32)   # the sign of a NaN means nothing


# rows below, at and past a pass of each head dimension (32, 16, 8 vectors) and a workgroup of four; the last ones past the
# line from which words are streamed (12 288, 8 192, 6 144)
@pytest.mark.parametrize("bits", [1, 2, 3, 4])
@pytest.mark.parametrize("n,dim", [(1, 64), (33, 64), (129, 64), (12289, 64), (7, 128), (16, 128), (65, 128), (8193, 128),
                                   (9, 256), (31, 256), (6145, 256), (65, 32)])
def test_round_trip_is_the_two_step_one(tq, bits, n, dim):
    pq = tq.PolarQuantizer(dim, bits=bits)
    for dtype in (torch.float16, torch.bfloat16, torch.float32):
        x = _rows(n, dim, dtype, 100 * dim + n)
        packed, norms = tq.fused_quantize(x, pq.signs, pq.boundaries, dim, bits)
        idx, got_norms = pq.quantize(x)
        assert idx.dtype == torch.uint8 and torch.equal(idx, tq.unpack_indices(packed, bits, dim))
        assert torch.equal(_bits_of(got_norms), _bits_of(norms))
        want = tq.packed_dequantize(packed, norms, pq.centroids, pq.signs, dim, bits)
        for levels in (idx, idx.int()):
            assert torch.equal(_bits_of(pq.dequantize(levels, norms)), _bits_of(want))
    # rows that start off a 16-byte boundary, rows apart, leading axes
    x = _rows(n + 1, dim, torch.float16, 5).view(-1)[1:1 + n * dim].view(n, dim)
    idx, norms = pq.quantize(x)
    assert torch.equal(idx, pq.quantize(x.clone())[0])
    off = torch.empty(n * dim + 1, dtype=torch.uint8, device="cuda")[1:].view(n, dim).copy_(idx)
    want = _bits_of(pq.dequantize(idx, norms))
    assert torch.equal(_bits_of(pq.dequantize(off, norms)), want)
    apart = torch.stack([x, x], dim=1)[:, 0]
    assert torch.equal(pq.quantize(apart)[0], idx)
    assert torch.equal(_bits_of(pq.dequantize(idx[None], norms[None].double())[0]), want)


@pytest.mark.parametrize("bits", [1, 2, 3, 4])
@pytest.mark.parametrize("n,dim", [(50, 64), (12300, 64), (50, 128), (48, 128), (8200, 128), (50, 256), (6200, 256)])
def test_bytes_past_the_width_mean_what_packing_makes_of_them(tq, bits, n, dim):
    g = torch.Generator().manual_seed(n + bits)
    pq = tq.PolarQuantizer(dim, bits=bits)
    idx = torch.randint(0, 1 << bits, (n, dim), generator=g, dtype=torch.uint8)
    at = torch.randint(0, n * dim, (n,), generator=g)
    idx.view(-1)[at] = torch.randint(0, 256, (n,), generator=g, dtype=torch.uint8)
    idx[:20] = torch.randint(0, 1 << bits, (20, dim), generator=g, dtype=torch.uint8)   # passes without one beside passes with
    idx, norms = idx.cuda(), torch.rand(n, generator=g).cuda()
    want = tq.packed_dequantize(tq.pack_indices(idx, bits), norms, pq.centroids, pq.signs, dim, bits)
    assert torch.equal(pq.dequantize(idx, norms), want)


def test_boundaries_without_a_level_line_and_empty_calls(tq):
    pq = tq.PolarQuantizer(128, bits=3)
    x = _rows(100, 128, torch.float16, 1)
    pq.boundaries = torch.tensor([-9.0, -8.9, -0.1, 0.0, 0.001, 0.0011, 30.0])     # no line gives each its own cell
    idx, norms = pq.quantize(x)
    packed, _ = tq.fused_quantize(x, pq.signs, pq.boundaries, 128, 3)
    assert torch.equal(idx, tq.unpack_indices(packed, 3, 128))
    idx, norms = pq.quantize(x[:0])
    assert idx.shape == (0, 128) and norms.shape == (0,)
    with pytest.raises(RuntimeError):
        pq.quantize(x.cpu())


@pytest.mark.parametrize("bits", [1, 2, 3, 4])
@pytest.mark.parametrize("n,dim", [(1, 64), (100, 64), (7, 128), (100, 128), (8200, 128), (31, 256)])
def test_levels_of_the_other_variant(tq, bits, n, dim):
    """Thresholds of the variant without a half-step at the boundaries: another level line, also below the row count from which
    words come from the streaming encoder."""
    pq = tq.PolarQuantizer(dim, bits=bits)
    for dtype in (torch.float16, torch.float32):
        x = _rows(n, dim, dtype, 7 * dim + n)
        packed, norms = tq.fused_quantize(x, pq.signs, pq.boundaries, dim, bits, variant="metal")
        idx, got_norms = tq.ops.quantize_indices(x, pq.signs, pq.boundaries, dim, bits, variant="metal")
        assert torch.equal(idx, tq.unpack_indices(packed, bits, dim))
        assert torch.equal(_bits_of(got_norms), _bits_of(norms))


def test_rows_of_another_width_are_refused(tq):
    pq = tq.PolarQuantizer(128, bits=3)
    for shape in ((100, 64), (100, 2, 128)):
        with pytest.raises((RuntimeError, ValueError)):
            tq.ops.quantize_indices(torch.zeros(shape, device="cuda"), pq.signs, pq.boundaries, 128, 3)
