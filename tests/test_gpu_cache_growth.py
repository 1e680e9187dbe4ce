"""Caches whose storage grows while they are filled, against a cache filled by one insert."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tq():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a GPU: torch.cuda.is_available() is False")
    import tqhip
    return tqhip


def _rows(dim, n, seed=0, B=2, H=4):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn((B, H, n, dim), generator=g, device="cuda").half() for _ in range(2)]


def _same(a, b):
    for x, y in zip(a, b):
        x, y = (t.view(torch.int32) if t.dtype == torch.uint32 else t for t in (x, y))
        assert torch.equal(x, y)


@pytest.mark.parametrize("dim,bits", [(32, 1), (32, 2), (64, 1), (128, 3)])      # (32, 1): one word a row
@pytest.mark.parametrize("kind", ["default", "fused", "vonly", "vonly_nobuf"])
def test_storage_grows_with_its_contents(tq, dim, bits, kind):
    k, v = _rows(dim, 530)

    def make():
        if kind.startswith("vonly"):
            return tq.VOnlyTurboQuantCache(bits=bits, no_v_buffer=kind == "vonly_nobuf")
        return tq.TurboQuantKVCache(bits=bits, fused=kind == "fused")
    whole, parts = make(), make()
    want = whole.update_and_fetch(k, v)
    got = None
    for lo, hi in ((0, 100), (100, 255), (255, 258), (258, 500), (500, 530)):
        got = parts.update_and_fetch(k[:, :, lo:hi], v[:, :, lo:hi])
    _same(parts.state, whole.state)
    _same(got, want)
    store = parts._v_tq if kind.startswith("vonly") else parts
    for t in (store.v_packed, store.v_norms):
        assert not (t.view(torch.int32) if t.dtype == torch.uint32 else t)[:, :, 530:].any()


@pytest.mark.parametrize("kind", ["default", "vonly"])
@pytest.mark.parametrize("was,now", [(torch.float16, torch.float16), (torch.float16, torch.bfloat16), (torch.bfloat16, torch.float16),
                                     (torch.float16, torch.float32), (torch.float32, torch.float16), (torch.bfloat16, torch.float32)])
def test_buffer_grows_under_tokens_of_another_dtype(tq, was, now, kind):
    """A prompt in one dtype, tokens in another, over a boundary of 256 positions, where the dequantised buffers grow: every
    position is what a full dequantisation in its own dtype gives, cast to the buffer's."""
    B, H, n, dim = 2, 4, 254, 128
    k, v = _rows(dim, n + 4)
    cls = tq.VOnlyTurboQuantCache if kind == "vonly" else tq.TurboQuantKVCache
    cache = cls(bits=3)
    cache.update_and_fetch(k[:, :, :n].to(was), v[:, :, :n].to(was))
    prompt = cache._v_tq._v_deq_buf[:, :, :n].clone() if kind == "vonly" else cache._v_deq_buf[:, :, :n].clone()
    for i in range(n, n + 4):
        _, got = cache.update_and_fetch(k[:, :, i:i + 1].to(now), v[:, :, i:i + 1].to(now))
    store = cache._v_tq if kind == "vonly" else cache
    full = store._full_dequant(store.v_packed, store.v_norms, store._v_q, dim, B, H, n + 4, torch.float16)
    assert got.dtype == now and torch.equal(got[:, :, :n], prompt.to(now))
    assert torch.equal(got[:, :, n + 2:], full[:, :, n + 2:].to(now))       # the tokens after the growth


@pytest.mark.parametrize("kind", ["default", "fused", "vonly"])
def test_inserts_without_a_sequence(tq, kind):
    x = torch.randn(0, 4, 20, 128, device="cuda").half()
    cache = tq.VOnlyTurboQuantCache(bits=3) if kind == "vonly" else tq.TurboQuantKVCache(bits=3, fused=kind == "fused")
    for n in (20, 40):
        k, v = cache.update_and_fetch(x, x)
        assert k.shape == v.shape == (0, 4, n, 128) and cache.offset == n


@pytest.mark.parametrize("nobuf", [False, True])
@pytest.mark.parametrize("dtype", [torch.float64, torch.int32])
def test_vonly_insert_of_keys_that_are_no_kernel_dtype(tq, dtype, nobuf):
    """Cast to float16, as any other key, whatever the number of new rows."""
    k, v = _rows(128, 40)
    k = (k * 8).round()
    want, got = (tq.VOnlyTurboQuantCache(bits=3, no_v_buffer=nobuf) for _ in range(2))
    for lo, hi in ((0, 30), (30, 39), (39, 40)):
        a = want.update_and_fetch(k[:, :, lo:hi], v[:, :, lo:hi])
        b = got.update_and_fetch(k[:, :, lo:hi].to(dtype), v[:, :, lo:hi])
        _same(a, b)
    _same(want.state, got.state)


def test_vonly_insert_of_no_rows(tq):
    x = torch.randn(2, 4, 0, 128, device="cuda").half()
    cache = tq.VOnlyTurboQuantCache(bits=3)
    for _ in range(2):
        k, v = cache.update_and_fetch(x, x)
        assert k.shape == v.shape == (2, 4, 0, 128) and cache.offset == 0
    k, v = _rows(128, 5)
    cache.update_and_fetch(k, v)
    assert cache.update_and_fetch(x, x)[1].shape == (2, 4, 5, 128)


def test_insert_into_a_restored_v_only_cache(tq):
    """Restored without its mode, it keeps keys from then on; the rows before are zeros."""
    k, v = _rows(128, 5)
    junk = torch.full((1 << 22,), 3, dtype=torch.int32, device="cuda")       # what the allocator hands out next
    del junk
    cache = tq.TurboQuantKVCache(bits=3, v_only=True)
    cache.update_and_fetch(k[:, :, :3], v[:, :, :3])
    back = tq.TurboQuantKVCache.from_state(cache.state, cache.meta_state)
    back.update_and_fetch(k[:, :, 3:], v[:, :, 3:])
    kp, kn, _, _ = back.state
    assert not kp.view(torch.int32)[:, :, :3].any() and not kn[:, :, :3].any() and bool(kn[:, :, 3:].all())


def test_fused_vonly_insert_refuses_other_key_dtypes(tq):
    """As ever: a fused cache's small inserts go through the one-launch append, which takes kernel dtypes."""
    k, v = _rows(128, 4)
    with pytest.raises(ValueError, match="unsupported dtype"):
        tq.VOnlyTurboQuantCache(bits=3, fused=True).update_and_fetch(k.double(), v)


_CASTS = [(a, b, c) for a in (torch.float16, torch.float32) for b in (torch.float16, torch.bfloat16, torch.float32)
          for c in (torch.float16, torch.bfloat16)]


@pytest.mark.parametrize("was,now_k,now_v", _CASTS)
def test_tokens_of_another_dtype_than_the_buffer(tq, was, now_k, now_v):
    """A token's dequantised rows: in half precision, cast to the token's dtype, then to the buffer's; float16 tokens go into the
    buffer as its dtype takes them."""
    B, H, n, dim = 2, 4, 40, 128
    k, v = _rows(dim, n + 1)
    cache = tq.TurboQuantKVCache(bits=3)
    cache.update_and_fetch(k[:, :, :n].to(was), v[:, :, :n].to(was))
    got = cache.update_and_fetch(k[:, :, n:].to(now_k), v[:, :, n:].to(now_v))
    sides = ((cache.k_packed, cache.k_norms, cache._k_q, now_k), (cache.v_packed, cache.v_norms, cache._v_q, now_v))
    for out, (p, nr, q, now) in zip(got, sides):
        half = now == torch.float16
        full = cache._full_dequant(p, nr, q, dim, B, H, n + 1, was if half else torch.float16)[:, :, n:]
        assert out.dtype == was and torch.equal(out[:, :, n:], full if half else full.to(now).to(was))
