"""Growth of cache storage without a GPU: what the storage fill is asked to copy and to zero, on CPU tensors."""
import pytest

torch = pytest.importorskip("torch")

import tqhip  # noqa: E402
from tqhip import ops  # noqa: E402

B, H = 2, 3


def _grown(cache, dim, n):
    """A cache of n positions on the CPU whose stored words and norms are numbered."""
    cache._ensure_quantizer(dim, dim, torch.device("cpu"))
    cache._ensure_storage(B, H, n, torch.device("cpu"))
    for t in _stored(cache):
        t[:, :, :n] = torch.arange(1, t[:, :, :n].numel() + 1, dtype=torch.int32).reshape(t[:, :, :n].shape).to(t.dtype)
    cache.offset = n
    return cache


def _stored(cache):
    ts = [cache.v_packed, cache.v_norms] + ([] if cache.v_only else [cache.k_packed, cache.k_norms])
    return [t.view(torch.int32) if t.dtype == torch.uint32 else t for t in ts]


@pytest.mark.parametrize("v_only", [False, True])
@pytest.mark.parametrize("dim,bits", [(d, b) for d in (32, 64, 128, 256) for b in (1, 2, 3, 4)])
def test_growth_keeps_the_stored_prefix(dim, bits, v_only):
    """(32, 1) packs a vector into one word: storage [B, H, T, 1], whose last axis is not the positions."""
    cache = _grown(tqhip.TurboQuantKVCache(bits=bits, v_only=v_only), dim, 250)
    before = [t[:, :, :250].clone() for t in _stored(cache)]
    assert all(not t[:, :, 250:].any() for t in _stored(cache))
    cache._ensure_storage(B, H, 10, torch.device("cpu"))
    for t, want in zip(_stored(cache), before):
        assert t.shape[2] == 512 and torch.equal(t[:, :, :250], want) and not t[:, :, 250:].any()


@pytest.mark.parametrize("dim,bits", [(d, b) for d in (32, 64, 128, 256) for b in (1, 2, 3, 4)])
def test_fill_segments_stay_inside_the_tensors(monkeypatch, dim, bits):
    """The byte ranges that a GPU launch would get for the same growth."""
    segments = []

    def add(self, dst, inner, zero_from, zero_to, src=None, src_stride=0, copy=0, axis=None):
        groups, rows = dst.shape[:axis].numel(), dst.shape[axis]
        assert dst.is_contiguous() and groups * rows * inner == dst.numel() and groups == B * H
        s = ops.StorageFill.segment(dst, src, groups, rows, inner, zero_from, zero_to, src_stride, copy)
        _, _, dst_stride, src_stride, copy_bytes, z0, z1, n = s
        assert (n - 1) * dst_stride + max(copy_bytes, z1) <= dst.nbytes and copy_bytes <= z0 <= z1 <= dst_stride
        if copy_bytes:
            assert src.dtype == dst.dtype and (n - 1) * src_stride + copy_bytes <= src.nbytes
        segments.append(s)

    cache = _grown(tqhip.TurboQuantKVCache(bits=bits), dim, 250)
    monkeypatch.setattr(ops.StorageFill, "add", add)
    cache._ensure_storage(B, H, 10, torch.device("cpu"), incoming=10)
    assert len(segments) == 4


def test_fill_refuses_rows_outside_the_tensor():
    fill = ops.StorageFill()
    with pytest.raises(ValueError):
        fill.add(torch.zeros(1, 2, 8, 1), 1, 4, 8)                 # the trailing axis taken for the rows
    with pytest.raises(ValueError):
        fill.segment(torch.zeros(2, 8, 4), torch.zeros(2, 4, 4), 2, 8, 4, 4, 8, 5, 4)


@pytest.mark.parametrize("v_only", [False, True])
@pytest.mark.parametrize("was,now", [(a, b) for a in (torch.float16, torch.bfloat16, torch.float32)
                                     for b in (torch.float16, torch.bfloat16, torch.float32)])
def test_buffer_growth_casts_rows_of_another_dtype(monkeypatch, was, now, v_only):
    """Dequantised buffers that grow under rows of another dtype: the prefix is cast, never copied byte by byte."""
    cache = _grown(tqhip.TurboQuantKVCache(bits=3, v_only=v_only), 128, 256)
    sides = 1 if v_only else 2
    old = [torch.randn(B, H, 256, 128).to(was) for _ in range(sides)]
    cache._deq_offset = 256
    raw = []
    add = ops.StorageFill.add

    def checked(self, dst, inner, zero_from, zero_to, src=None, src_stride=0, copy=0, axis=None):
        if copy:
            raw.append(src.dtype)
            assert src.dtype == dst.dtype
            ops.StorageFill.segment(dst, src, B * H, dst.shape[axis], inner, zero_from, zero_to, src_stride, copy)
        return add(self, dst, inner, zero_from, zero_to, src=src, src_stride=src_stride, copy=copy, axis=axis)

    monkeypatch.setattr(ops.StorageFill, "add", checked)
    monkeypatch.setattr(tqhip.TurboQuantKVCache, "_dequant_rows", lambda self, outs, *a: [o.zero_() for o in outs if o is not None and o.shape[2] == 1])
    grown = cache._incremental(list(old), B, H, 256, 257, [now] * sides)
    assert len(raw) == (sides if was == now else 0)
    for new, o in zip(grown, old):
        assert new.dtype == now and new.shape[2] == 512
        assert torch.equal(new[:, :, :256], o.to(now)) and not new[:, :, 257:].any()


class _LateFill(ops.StorageFill):
    """A storage fill that does its work in run(), as on the GPU."""

    def __init__(self):
        super().__init__()
        self.asked = []

    def add(self, *args, **kw):
        self.asked.append((args, kw))

    def run(self):
        for args, kw in self.asked:
            super().add(*args, **kw)
        self.asked = []


def _words(cache, n):
    return [t[:, :, :n].clone() for t in _stored(cache)]


@pytest.mark.parametrize("mode", [dict(), dict(fused=True), dict(v_only=True)])
@pytest.mark.parametrize("at", range(8))
def test_a_failed_allocation_leaves_the_cache_as_it_was(monkeypatch, mode, at):
    """Allocation number `at` of an insert that grows the storage fails; the caller makes room and tries again."""
    monkeypatch.setattr(ops, "StorageFill", _LateFill)
    for name in ("encode_into", "encode_kv_into", "dequant_into", "dequant_kv_into"):
        monkeypatch.setattr(ops, name, lambda *a, **kw: None)
    cache = _grown(tqhip.TurboQuantKVCache(bits=3, **mode), 128, 250)
    want = _words(cache, 250)
    kept = _stored(cache)
    x = torch.randn(B, H, 10, 128).half()
    left = [at]

    def failing(real):
        def alloc(*args, **kw):
            left[0] -= 1
            if left[0] < 0:
                raise torch.OutOfMemoryError("no room")
            return real(*args, **kw)
        return alloc
    with monkeypatch.context() as m:
        m.setattr(torch, "empty", failing(torch.empty))
        m.setattr(torch.Tensor, "new_empty", failing(torch.Tensor.new_empty))
        try:
            cache.update_and_fetch(x, x)
            failed = False
        except torch.OutOfMemoryError:
            failed = True
    assert failed == (left[0] < 0)
    if failed:
        assert cache.offset == 250 and all(a.data_ptr() == b.data_ptr() for a, b in zip(_stored(cache), kept))
        out = cache.update_and_fetch(x, x)
        if cache.fused:
            assert not any(t.any() for t in out)
    assert cache.offset == 260
    for got, w in zip(_words(cache, 250), want):
        assert torch.equal(got, w)


def test_rows_that_one_side_never_held_are_zero(monkeypatch):
    """A cache restored from the state of a v_only one has values and no keys: its first insert makes key storage whose rows
    before the insert are zeros, not what memory held."""
    cache = _grown(tqhip.TurboQuantKVCache(bits=3, v_only=True), 128, 250)
    cache.v_only = False
    cache._ensure_quantizer(128, 128, torch.device("cpu"))
    real = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, **kw: real(*a, **kw).view(torch.uint8).fill_(7).view(kw["dtype"]))
    cache._ensure_storage(B, H, 10, torch.device("cpu"), incoming=10)
    for t in (cache.k_packed.view(torch.int32), cache.k_norms):
        assert t.shape[2] == 512 and not t[:, :, :250].any() and not t[:, :, 260:].any()
