"""Decode attention at head dimensions 64 and 256 on the matrix cores against the float32 vector kernels (precision="fp32") and,
on small cases, the float64 arithmetic of the oracle: tile and wave edges, more heads than a workgroup serves, masks, ragged
batches, magnitudes outside fp16."""
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


def _case(tq, B, n_kv, n_rep, T, D, bits, seed=1):
    g = torch.Generator(device="cuda").manual_seed(seed)
    mk = lambda *s: torch.randn(s, generator=g, device="cuda")   # noqa: E731
    pack = lambda: tq.pack_indices(torch.randint(0, 1 << bits, (B, n_kv, T, D), generator=g, device="cuda", dtype=torch.uint8), bits)  # noqa: E731
    return mk(B, n_kv * n_rep, D), pack(), mk(B, n_kv, T).abs() * 8 + 0.1, pack(), mk(B, n_kv, T).abs() * 8 + 0.1, mk(B, n_kv, T, D).half()


# float32 arithmetic on both sides, sums in another order and operands of 22 bits.  A score that is off by a few 2^-24 of its
# magnitude, up to 30 here, moves its weight by that much: 30 x 4 x 6e-8, half of it to either side.
_REL = 4e-6


@pytest.mark.parametrize("bits", [1, 2, 3, 4])
@pytest.mark.parametrize("B,n_kv,n_rep,T", [(1, 1, 1, 1), (2, 2, 3, 63), (1, 2, 8, 257), (2, 1, 17, 511), (3, 2, 4, 1300), (1, 1, 33, 320)])
def test_split_dims(tq, bits, B, n_kv, n_rep, T):
    c = o.gaussian_codebook(bits)
    n_q = n_kv * n_rep
    mask = torch.randn(B, n_q, T, device="cuda")
    mask[:, :, : T // 3] = float("-inf")
    for D, packed in ((64, True), (64, False), (256, False)):
        q, kp, kn, vp, vn, kd = _case(tq, B, n_kv, n_rep, T, D, bits)
        signs = torch.from_numpy(o.random_diagonal_sign(D, 43)).cuda()
        sc = 1.0 / (8.0 * D ** 0.5) if packed else D ** -0.5
        for m in (None, mask):
            def run(**kw):
                if packed:
                    return tq.flash_decode(q, kp, kn, vp, vn, c, c, signs, D, bits, sc, n_rep=n_rep, mask=m, **kw)
                return tq.vonly_decode(q, kd, vp, vn, c, signs, D, bits, sc, n_rep=n_rep, mask=m, **kw)
            got, want = run(), run(precision="fp32")
            assert (got - want).abs().max() <= _REL * want.abs().max(), (D, packed, m is None)
        if not packed:
            for dt in (torch.float16, torch.bfloat16):
                args = (kd, vp, vn, c, signs, D, bits, sc)
                got = tq.vonly_decode(q.to(dt), *args, n_rep=n_rep)
                want = tq.vonly_decode(q.to(dt).float(), *args, n_rep=n_rep, precision="fp32")
                assert (got - want).abs().max() <= _REL * want.abs().max()


def test_split_dims_ragged_and_scales(tq):
    D, bits, n_kv, n_rep = 64, 3, 2, 4
    c = o.gaussian_codebook(bits)
    lens = [1, 700, 64, 255, 257]
    q, kp, kn, vp, vn, _ = _case(tq, 1, n_kv, n_rep, sum(lens), D, bits)
    q = torch.randn(len(lens), n_kv * n_rep, D, device="cuda")
    signs = torch.from_numpy(o.random_diagonal_sign(D, 43)).cuda()
    off = torch.tensor([0] + lens, device="cuda").cumsum(0).to(torch.int32)
    for qs, vs in ((1.0, 1.0), (1e7, 1e-6), (1e-9, 3e8)):                 # queries and value norms outside fp16
        def run(**kw):
            return tq.flash_decode(q * qs, kp[0], kn[0], vp[0], vn[0] * vs, c, c, signs, D, bits, 0.02 / qs, n_rep=n_rep,
                                   seq_offsets=off, max_seq_len=max(lens), **kw)
        got, want = run(), run(precision="fp32")
        assert (got - want).abs().max() <= _REL * want.abs().max(), (qs, vs)


def test_split_dims_against_float64(tq):
    """No further from 64-bit arithmetic than a few times what the float32 kernels are."""
    B, n_kv, n_rep, T, D, bits = 1, 2, 4, 900, 64, 4
    c = o.gaussian_codebook(bits)
    q, kp, kn, vp, vn, _ = _case(tq, B, n_kv, n_rep, T, D, bits)
    signs = o.random_diagonal_sign(D, 43)
    ki, vi = (o.unpack_indices(x[0].cpu().numpy().reshape(-1, x.shape[-1]), bits, D).reshape(n_kv, T, D) for x in (kp, vp))
    cc = np.asarray(c, dtype=np.float64)
    had = np.array([[(-1.0) ** bin(i & j).count("1") for j in range(D)] for i in range(D)])
    want = np.zeros((n_kv * n_rep, D))
    for h in range(n_kv * n_rep):
        kv = h // n_rep
        s = (cc[ki[kv]] @ q[0, h].double().cpu().numpy()) * kn[0, kv].double().cpu().numpy() / D * 0.02
        p = np.exp(s - s.max())
        want[h] = (had @ ((p / p.sum() * vn[0, kv].double().cpu().numpy()) @ cc[vi[kv]])) * np.asarray(signs, dtype=np.float64) / D
    sg = torch.from_numpy(signs).cuda()
    err = [np.linalg.norm(tq.flash_decode(q, kp, kn, vp, vn, c, c, sg, D, bits, 0.02, n_rep=n_rep, precision=pr)[0].double().cpu().numpy() - want)
           / np.linalg.norm(want) for pr in ("fp16", "fp32")]
    print("relative error, split / float32 kernels:", err)
    assert err[0] <= max(4 * err[1], 1e-6), err


def _had(D):
    i = np.arange(D)
    return np.array([[(-1.0) ** bin(a & b).count("1") for b in i] for a in i])


def _float64(tq, q, kp, kn, kd, vp, vn, c, signs, D, bits, sc, n_rep, mask):
    """The step in 64 bits: kp / kn packed keys in the rotated domain, or kd fp16 keys."""
    cc = torch.from_numpy(np.asarray(c, dtype=np.float64))
    B, n_kv, T = vn.shape
    vals = cc[tq.unpack_indices(vp, bits, D).cpu().long()] * vn.cpu().double()[..., None]
    keys = kd.cpu().double() if kp is None else cc[tq.unpack_indices(kp, bits, D).cpu().long()] * (kn.cpu().double() / D)[..., None]
    rep = lambda t: t.repeat_interleave(n_rep, dim=1)   # noqa: E731
    s = (rep(keys) * q.cpu().double()[:, :, None, :]).sum(-1) * sc + (0 if mask is None else mask.cpu().double())
    s = torch.nan_to_num(s, neginf=-np.inf)
    w = torch.softmax(s, dim=-1)
    rot = (rep(vals) * torch.where(w > 0, w, 0.0)[..., None]).sum(2)
    return (rot @ torch.from_numpy(_had(D)) * signs.cpu().double() / D).numpy()


@pytest.mark.parametrize("D,packed", [(64, True), (64, False), (256, False)])
@pytest.mark.parametrize("octaves", [0, 3, 13])
def test_split_dims_heads_of_different_magnitude(tq, D, packed, octaves):
    """Heads of one wave that attend rows whose value norms lie far apart: head h sees the positions h, h + 8, ... only, whose
    norms are 2^(-octaves h).  Per head, no further from 64-bit arithmetic than the float32 kernel, a few units of float32
    (2^-24 = 6e-8) allowed for sums in another order."""
    B, n_kv, n_rep, T, bits = 2, 2, 8, 700, 3
    c = o.gaussian_codebook(bits)
    q, kp, kn, vp, vn, kd = _case(tq, B, n_kv, n_rep, T, D, bits)
    signs = torch.from_numpy(o.random_diagonal_sign(D, 43)).cuda()
    pos = torch.arange(T, device="cuda") % n_rep
    vn = (vn * torch.exp2(-octaves * pos.float())).contiguous()
    head = torch.arange(n_kv * n_rep, device="cuda") % n_rep
    mask = torch.where(pos[None, :] == head[:, None], 0.0, float("-inf")).float()[None].expand(B, -1, -1).contiguous()
    sc = 1.0 / (8.0 * D ** 0.5) if packed else D ** -0.5

    def run(precision):
        if packed:
            return tq.flash_decode(q, kp, kn, vp, vn, c, c, signs, D, bits, sc, n_rep=n_rep, mask=mask, precision=precision)
        return tq.vonly_decode(q, kd, vp, vn, c, signs, D, bits, sc, n_rep=n_rep, mask=mask, precision=precision)
    want = _float64(tq, q, kp if packed else None, kn, kd, vp, vn, c, signs, D, bits, sc, n_rep, mask)
    err = [np.linalg.norm(run(p).cpu().double().numpy() - want, axis=-1) / np.linalg.norm(want, axis=-1) for p in ("fp16", "fp32")]
    print(D, packed, octaves, "largest relative error of a head, split / float32:", err[0].max(), err[1].max())
    assert err[0].max() <= 1.5 * err[1].max() + 1.2e-7, (err[0].max(), err[1].max())


@pytest.mark.parametrize("D", [64, 256])
def test_split_dims_infinite_keys(tq, D):
    """Keys that overflowed float16: a head whose score of such a position is -inf leaves it out, as the float32 kernel does."""
    B, n_kv, n_rep, T, bits = 1, 2, 4, 300, 3
    c = o.gaussian_codebook(bits)
    q, _, _, vp, vn, kd = _case(tq, B, n_kv, n_rep, T, D, bits)
    signs = torch.from_numpy(o.random_diagonal_sign(D, 43)).cuda()
    q[..., 7] = q[..., 7].abs() + 0.25
    q[0, 3] = torch.randint(-8, 9, (D,), device="cuda").float()              # no remainder: exact in fp16
    q[0, 3, 7] = 2.0
    for at, value in ((5, float("-inf")), (70, float("-inf")), (299, float("-inf")), (130, 65504.0)):
        kd[:, :, at, 7] = value
    args = (q, kd, vp, vn, c, signs, D, bits, D ** -0.5)
    got, want = tq.vonly_decode(*args, n_rep=n_rep), tq.vonly_decode(*args, n_rep=n_rep, precision="fp32")
    assert bool(torch.isfinite(want).all()) and bool(torch.isfinite(got).all())
    assert (got - want).abs().max() <= _REL * want.abs().max()


@pytest.mark.parametrize("scale", [1e35, 1e-35])
def test_split_dims_extreme_norms(tq, scale):
    """Value norms near the ends of float32."""
    D, bits, n_rep = 64, 3, 4
    c = o.gaussian_codebook(bits)
    q, kp, kn, vp, vn, _ = _case(tq, 1, 2, n_rep, 200, D, bits)
    signs = torch.from_numpy(o.random_diagonal_sign(D, 43)).cuda()
    args = (q, kp, kn, vp, vn * scale, c, c, signs, D, bits, 0.02)
    got, want = tq.flash_decode(*args, n_rep=n_rep), tq.flash_decode(*args, n_rep=n_rep, precision="fp32")
    assert bool(torch.isfinite(want).all()) and (got.double() - want.double()).abs().max() <= _REL * want.double().abs().max()


@pytest.mark.parametrize("D,packed", [(64, True), (64, False), (256, False)])
@pytest.mark.parametrize("scale", [1e4, 100.0, 1e-6])
def test_split_dims_codebooks_of_another_scale(tq, D, packed, scale):
    """A given codebook need not be that of a unit Gaussian."""
    bits, n_rep = 3, 4
    c = (np.asarray(o.gaussian_codebook(bits)) * scale).astype(np.float32)
    q, kp, kn, vp, vn, kd = _case(tq, 1, 2, n_rep, 700, D, bits)
    signs = torch.from_numpy(o.random_diagonal_sign(D, 43)).cuda()

    def run(**kw):
        if packed:
            return tq.flash_decode(q, kp, kn, vp, vn, c, c, signs, D, bits, 0.02 / scale, n_rep=n_rep, **kw)
        return tq.vonly_decode(q, kd, vp, vn, c, signs, D, bits, D ** -0.5, n_rep=n_rep, **kw)
    got, want = run(), run(precision="fp32")
    assert (got - want).abs().max() <= _REL * want.abs().max()


@pytest.mark.parametrize("D,packed", [(64, True), (64, False), (256, False)])
def test_split_dims_infinite_value_norms(tq, D, packed):
    """One position, whose value norm is infinite: the infinities and the no-numbers of the float32 kernel."""
    bits, n_rep = 3, 4
    c = o.gaussian_codebook(bits)
    q, kp, kn, vp, vn, kd = _case(tq, 2, 2, n_rep, 1, D, bits)
    vn[1] = float("inf")
    signs = torch.from_numpy(o.random_diagonal_sign(D, 43)).cuda()
    vp[1, 0] = tq.pack_indices(torch.full((1, D), 6, device="cuda", dtype=torch.uint8), bits)     # one sign: one output is infinite

    def run(**kw):
        if packed:
            return tq.flash_decode(q, kp, kn, vp, vn, c, c, signs, D, bits, 0.02, n_rep=n_rep, **kw)
        return tq.vonly_decode(q, kd, vp, vn, c, signs, D, bits, D ** -0.5, n_rep=n_rep, **kw)
    got, want = run(), run(precision="fp32")
    assert int(torch.isinf(want).sum()) == n_rep and bool(torch.isfinite(want[0]).all())
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    assert torch.equal(got[torch.isinf(got)], want[torch.isinf(want)])
