"""The batched prefill: rows at the edges of a wavefront's 32 and a workgroup's eight row tiles, head groupings that divide
them or not, one split and several, lengths around the 64 positions of a block, against the oracle sequence by sequence."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import polarquant_oracle as o  # noqa: E402

pytestmark = pytest.mark.gpu

D = 128


@pytest.fixture(scope="module")
def tq():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a GPU: torch.cuda.is_available() is False")
    import tqhip
    return tqhip


def _case(B, n_kv, n_rep, T, S, bits, dtype, spare=5):
    rng = np.random.default_rng(B * 1000 + T + S)
    kp, vp = (o.pack_indices(rng.integers(0, 1 << bits, size=(B, n_kv, T + spare, D)).astype(np.uint8), bits) for _ in range(2))
    kn, vn = (np.abs(rng.standard_normal((B, n_kv, T + spare))).astype(np.float32) * 10 + 0.1 for _ in range(2))
    q = torch.from_numpy(rng.standard_normal((B, n_kv * n_rep, S, D)).astype(np.float32)).to(dtype)
    return kp, kn, vp, vn, q


# (batch, kv heads, heads per kv head, cached positions, query rows, width, dtype)
@pytest.mark.parametrize("B,n_kv,n_rep,T,S,bits,dtype", [
    (1, 1, 1, 1, 1, 3, torch.float16), (3, 2, 3, 33, 33, 3, torch.bfloat16), (2, 1, 4, 64, 64, 3, torch.float32),
    (2, 2, 7, 65, 31, 2, torch.float16), (2, 3, 1, 300, 257, 4, torch.bfloat16), (4, 1, 8, 129, 128, 1, torch.float16),
    (2, 2, 4, 1111, 95, 3, torch.float16), (1, 2, 16, 700, 40, 3, torch.bfloat16), (2, 1, 2, 3001, 2, 3, torch.float16),
])
@pytest.mark.parametrize("causal", [True, False])
def test_prefill_batch(tq, B, n_kv, n_rep, T, S, bits, dtype, causal):
    kp, kn, vp, vn, q = _case(B, n_kv, n_rep, T, S, bits, dtype)
    c = o.gaussian_codebook(bits)
    ks, vs = o.random_diagonal_sign(D, 42), o.random_diagonal_sign(D, 43)
    dev = [torch.from_numpy(x).cuda() for x in (kp.view(np.int32), kn, vp.view(np.int32), vn)]
    signs = torch.from_numpy(np.concatenate([[1.0], ks, [1.0], vs]).astype(np.float32)).cuda()
    got = tq.ops.prefill_attention_batch(q.cuda(), *dev, c, c, signs[1:129], signs[130:], D, bits, 0.05, n_rep=n_rep, kv_len=T,
                                         q_pos0=T - S, causal=causal)
    # the same rows from an odd address: element-wise loads
    odd = torch.empty(q.numel() + 1, dtype=dtype, device="cuda")[1:].view(q.shape)
    odd.copy_(q)
    assert torch.equal(got, tq.ops.prefill_attention_batch(odd, *dev, c, c, signs[1:129], signs[130:], D, bits, 0.05, n_rep=n_rep,
                                                           kv_len=T, q_pos0=T - S, causal=causal))
    for b in range(B):
        want = o.prefill_attention(q[b].float().numpy(), kp[b, :, :T], kn[b, :, :T], vp[b, :, :T], vn[b, :, :T], c, c, ks, vs, D, bits,
                                   0.05, T - S, n_rep, causal=causal)
        out = got[b].float().cpu().numpy()
        # operands of the matrix instructions rounded to fp16 (2^-11), the result rounded to bfloat16 (2^-9) where q is
        tol = (1e-3 + 2e-3 * np.abs(want)) + (2.0 ** -8 * np.abs(want) if dtype == torch.bfloat16 else 0.0)
        assert np.all(np.abs(out - want) <= tol * np.maximum(1.0, np.abs(want).max())), np.abs(out - want).max()
        one = tq.prefill_attention(q[b].cuda(), *(x[b] for x in dev), c, c, signs[1:129], signs[130:], D, bits, 0.05, n_rep=n_rep,
                                   kv_len=T, q_pos0=T - S, causal=causal)
        assert torch.allclose(one.float(), got[b].float(), rtol=2e-3 if dtype != torch.bfloat16 else 8e-3, atol=2e-3 * np.abs(want).max())
