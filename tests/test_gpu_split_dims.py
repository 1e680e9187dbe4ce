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


# float32 arithmetic on both sides, sums in another order and operands of 22 bits: a few 2^-22 of the magnitudes summed,
# which scores of up to 30 in the exponent multiply
_REL = 3e-5


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
