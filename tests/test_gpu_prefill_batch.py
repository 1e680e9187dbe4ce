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


@pytest.mark.parametrize("n_kv,n_rep,n_rows,T,causal", [(8, 4, 1, 5262, True), (8, 4, 1, 5262, False), (4, 7, 3, 9001, True), (2, 6, 100, 2500, True),
                                                        (1, 1, 1, 700, True), (8, 1, 33, 20000, True), (1, 8, 40, 16500, False)])
def test_the_split_does_not_depend_on_the_bytes_at_hand(tq, n_kv, n_rep, n_rows, T, causal):
    """Equal calls give equal bits, whatever workspace earlier calls left behind: through the package and through both C entries
    with the workspace asked for and with a larger one."""
    from tqhip import _lib
    lib = _lib.load()
    D, bits, n_q = 128, 3, n_kv * n_rep
    g = torch.Generator(device="cuda").manual_seed(T)
    q = torch.randn(n_q, n_rows, D, generator=g, device="cuda")
    kp, vp = (tq.pack_indices(torch.randint(0, 8, (n_kv, T, D), generator=g, device="cuda", dtype=torch.uint8), bits) for _ in range(2))
    kn, vn = (torch.rand(n_kv, T, generator=g, device="cuda") * 8 + 1 for _ in range(2))
    ks, vs = (torch.from_numpy(o.random_diagonal_sign(D, s)).cuda() for s in (42, 43))
    c = torch.tensor(np.asarray(o.gaussian_codebook(bits), dtype=np.float32))
    stream = torch.cuda.current_stream().cuda_stream

    def entry(batch, extra):
        flags, pos0 = int(causal), T - n_rows
        need = (lib.tq_prefill_batch_workspace_bytes(1, n_kv, n_rep, n_rows, T, pos0, D, flags) if batch
                else lib.tq_prefill_workspace_bytes(n_q, n_rows, T, D))
        ws = torch.empty(need + extra, dtype=torch.uint8, device="cuda")
        out = torch.empty(n_q, n_rows, D, device="cuda")
        p = [t.data_ptr() for t in (q, kp, kn, vp, vn, c, c, ks, vs, out, ws)]
        head = (p[0], 0, *p[1:10], 0, p[10], ws.numel())
        tail = (T, T, T, T, D, bits, 0.02, flags, stream)
        rc = (lib.tq_prefill_attn_batch(*head, 1, n_kv, n_rep, n_rows, T, pos0, 0, 0, 0, 0, *tail) if batch
              else lib.tq_prefill_attn(*head, n_kv, n_rep, n_rows, T, pos0, *tail))
        assert rc == 0, lib.tq_last_error()
        torch.cuda.synchronize()
        return out
    for batch in (False, True):
        assert torch.equal(entry(batch, 0), entry(batch, 64 << 20))

    def package():
        return tq.prefill_attention(q, kp, kn, vp, vn, c, c, ks, vs, D, bits, 0.02, n_rep=n_rep, causal=causal)
    tq.ops._workspaces.clear()
    before = package()
    tq.ops._workspace(q.device, stream, 64 << 20)
    assert torch.equal(before, package()) and torch.equal(before, entry(True, 0))
    tq.ops._workspaces.clear()


@pytest.mark.parametrize("T", [70, 6000])                                 # one split, several
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_rows_whose_query_is_no_number(tq, T, bad):
    """A row none of whose scores is a number comes out as zeros, whatever the number of splits; other rows do not notice."""
    kp, kn, vp, vn, q = _case(1, 2, 3, T, 40, 3, torch.float32)
    c = o.gaussian_codebook(3)
    ks, vs = (torch.from_numpy(o.random_diagonal_sign(D, s)).cuda() for s in (42, 43))
    dev = [torch.from_numpy(x).cuda() for x in (kp.view(np.int32), kn, vp.view(np.int32), vn)]

    def run(x):
        return tq.ops.prefill_attention_batch(x.cuda(), *dev, c, c, ks, vs, D, 3, 0.05, n_rep=3, kv_len=T, q_pos0=T - 40)
    want = run(q)
    hurt = q.clone()
    hurt[0, 1, 7, 5] = bad
    hurt[0, 4, 39, 127] = bad
    got = run(hurt)
    for h, r in ((1, 7), (4, 39)):
        assert not got[0, h, r].any()
        got[0, h, r] = want[0, h, r]
    assert torch.equal(got, want)
