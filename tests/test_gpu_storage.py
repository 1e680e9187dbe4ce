"""Cache storage set-up on the GPU: prefix copies and zeros in one launch, sign vectors, and the launches that take the
keys and the values together."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import polarquant_oracle as o  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tq():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a GPU: torch.cuda.is_available() is False")
    import tqhip
    return tqhip


# inner 13 words: 52-byte rows, 16-byte accesses only where the bounds allow them; 1: norms; 128 halfs: buffers
@pytest.mark.parametrize("groups,rows,inner,dtype,old_rows,copy,keep", [
    (3, 512, 13, torch.int32, 256, 255, 1), (5, 256, 1, torch.float32, 256, 0, 7), (2, 1024, 13, torch.int32, 1000, 512, 4),
    (1500, 256, 1, torch.float32, 3, 3, 0), (4, 768, 128, torch.float16, 511, 511, 2), (1, 8, 1, torch.bfloat16, 1, 0, 0),
])
def test_storage_fill(tq, groups, rows, inner, dtype, old_rows, copy, keep):
    from tqhip.ops import StorageFill
    tail = (inner,) if inner > 1 else ()
    dst = torch.full((1, groups, rows) + tail, 5, dtype=dtype, device="cuda")
    old = torch.arange(groups * old_rows * inner, device="cuda").remainder(251).to(dtype).reshape((1, groups, old_rows) + tail)
    fill = StorageFill()
    fill.add(dst, inner, copy + keep, rows, src=old if copy else None, src_stride=old_rows, copy=copy)
    fill.add(torch.empty(16, device="cuda"), 1, 4, 4)                   # nothing to do
    fill.run()
    assert torch.equal(dst[:, :, :copy], old[:, :, :copy])
    assert bool((dst[:, :, copy:copy + keep] == 5).all()) and bool((dst[:, :, copy + keep:] == 0).all())


@pytest.mark.parametrize("seeds,dim", [([42, 43], 128), ([0], 1), ([2 ** 63 + 5, 1, 7], 257)])
def test_random_signs(tq, seeds, dim):
    from tqhip.rotation import sign_pattern
    got = tq.ops.random_signs(seeds, dim, torch.device("cuda")).cpu()
    assert got.tolist() == [sign_pattern(dim, s) for s in seeds]


@pytest.mark.parametrize("seeds,dim,segments", [([42, 43], 128, 0), ([7], 64, 3), ([1, 2 ** 64 - 1, 3, 4], 257, 8), ([5, 6], 128, 11)])
def test_signs_join_the_fill(tq, seeds, dim, segments):
    """One launch for both; more segments than a launch takes; signs alone."""
    from tqhip.rotation import sign_pattern
    fill = tq.ops.StorageFill()
    dst = [torch.full((2, 20 + i, 13), 5, dtype=torch.int32, device="cuda") for i in range(segments)]
    for i, t in enumerate(dst):
        fill.add(t, 13, i, 20 + i)
    got = fill.signs(seeds, dim, torch.device("cuda"))
    fill.run()
    assert got.tolist() == [sign_pattern(dim, s) for s in seeds]
    for i, t in enumerate(dst):
        assert bool((t[:, :i] == 5).all()) and not t[:, i:].any()


def test_an_insert_that_fails_leaves_no_sign_vectors_behind(tq, monkeypatch):
    cache = tq.TurboQuantKVCache(bits=3)
    k = torch.randn(1, 2, 30, 128, device="cuda")
    monkeypatch.setattr(cache, "_fetch_buffers", lambda *a: (_ for _ in ()).throw(MemoryError()))
    with pytest.raises(MemoryError):
        cache.update_and_fetch(k, k)
    assert cache._k_q is None and cache._v_q is None and cache.offset == 0 and cache.k_packed is None
    monkeypatch.undo()
    other = tq.TurboQuantKVCache(bits=3)
    for got, want in zip(cache.update_and_fetch(k, k), other.update_and_fetch(k, k)):
        assert torch.equal(got, want)


@pytest.mark.parametrize("dim,bits,rows,alloc,off", [(128, 3, 1, 256, 9), (128, 3, 48, 64, 16), (128, 4, 1001, 1024, 3),
                                                     (64, 2, 2001, 2048, 0), (256, 3, 700, 768, 1), (32, 1, 77, 80, 2)])
def test_keys_and_values_in_one_launch(tq, dim, bits, rows, alloc, off):
    """Same bits as one call per tensor; the oracle holds those (tests of the codec)."""
    rng = np.random.default_rng(bits)
    G = 5
    c = o.gaussian_codebook(bits)
    b = o.gaussian_boundaries(c)
    pd = tq.packed_dim(dim, bits)
    x = [torch.from_numpy(rng.standard_normal((G * rows, dim)).astype(np.float16)).cuda() for _ in range(2)]
    s = [torch.from_numpy(o.random_diagonal_sign(dim, k)).cuda() for k in (42, 43)]
    p, n, want_p, want_n = ([torch.zeros((G, alloc) + t, dtype=d, device="cuda") for _ in range(2)]
                            for t, d in (((pd,), torch.int32), ((), torch.float32)) * 2)
    tq.ops.encode_kv_into(x[0], s[0], p[0], n[0], x[1], s[1], p[1], n[1], b, n_groups=G, rows_per_group=rows,
                          group_stride=alloc, dim=dim, bits=bits, row_offset=off)
    outs, want = ([torch.zeros((G, alloc, dim), dtype=torch.bfloat16, device="cuda") for _ in range(2)] for _ in range(2))
    tq.ops.dequant_kv_into(p[0], n[0], s[0], outs[0], p[1], n[1], s[1], outs[1], c, n_groups=G, rows_per_group=rows,
                           group_stride=alloc, out_group_stride=alloc, dim=dim, bits=bits, row_offset=off, out_row_offset=off)
    for i in range(2):
        tq.encode_into(x[i], s[i], b, want_p[i], want_n[i], n_groups=G, rows_per_group=rows, packed_group_stride=alloc,
                       norms_group_stride=alloc, dim=dim, bits=bits, packed_row_offset=off, norms_row_offset=off)
        tq.dequant_into(want_p[i], want_n[i], c, s[i], want[i], n_groups=G, rows_per_group=rows, packed_group_stride=alloc,
                        norms_group_stride=alloc, out_group_stride=alloc, dim=dim, bits=bits, packed_row_offset=off,
                        norms_row_offset=off, out_row_offset=off)
        assert torch.equal(p[i], want_p[i]) and torch.equal(n[i], want_n[i]) and torch.equal(outs[i], want[i])


def test_table_of_a_gpu_tensor_is_not_kept_by_address(tq):
    """A codebook tensor on the GPU is read anew when another one takes its place in memory, or its values change."""
    s = torch.from_numpy(o.random_diagonal_sign(128, 42)).cuda()
    p, n = tq.fused_quantize(torch.randn(16, 128, device="cuda"), s, o.gaussian_boundaries(o.gaussian_codebook(3)), 128, 3)
    base = torch.tensor(o.gaussian_codebook(3).tolist())
    for k in (1.0, 2.0, 3.0):
        cb = (base * k).cuda()
        got = tq.packed_dequantize(p, n, cb, s, 128, 3)
        assert torch.equal(got, tq.packed_dequantize(p, n, (base * k).tolist(), s, 128, 3))
        cb.mul_(0.5)
        assert torch.equal(tq.packed_dequantize(p, n, cb, s, 128, 3), tq.packed_dequantize(p, n, (base * k * 0.5).tolist(), s, 128, 3))
        del cb
