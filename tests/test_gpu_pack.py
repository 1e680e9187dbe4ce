"""pack_indices / unpack_indices on the GPU against the oracle and against the tensor operations that the CPU runs."""
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


# row lengths at the edges of the 16-index and 4-index forms, of a packed word (8, 10, 16, 32 indices) and below them
@pytest.mark.parametrize("bits", [1, 2, 3, 4])
@pytest.mark.parametrize("lead,dim", [((1,), 1), ((7,), 9), ((3, 5), 10), ((257,), 31), ((33,), 33), ((5,), 16), ((63,), 48),
                                      ((2, 129), 64), ((1031,), 128), ((300,), 100), ((19,), 256), ((4,), 1000)])
def test_pack_unpack(tq, bits, lead, dim):
    rng = np.random.default_rng(dim * 8 + bits)
    idx = rng.integers(0, 1 << bits, size=lead + (dim,)).astype(np.uint8)
    want = o.pack_indices(idx.reshape(-1, dim), bits).reshape(*lead, -1)
    for dtype in (torch.uint8, torch.int32, torch.int64, torch.int16):
        got = tq.pack_indices(torch.from_numpy(idx).to(dtype).cuda(), bits)
        assert got.dtype == torch.uint32 and np.array_equal(got.cpu().numpy(), want), dtype
    back = tq.unpack_indices(got, bits, dim)
    assert back.dtype == torch.uint8 and np.array_equal(back.cpu().numpy(), idx)
    wide = tq.unpack_indices(got, bits, dim + 1000)                      # cut at what the words hold
    cpu = tq.unpack_indices(got.cpu(), bits, dim + 1000)
    assert torch.equal(wide.cpu(), cpu)
    if dim > 1:                                                          # rows of a view, off a 4- or 16-byte boundary
        view = torch.from_numpy(idx).cuda()[..., 1:]
        assert torch.equal(tq.pack_indices(view, bits).cpu(), tq.pack_indices(view.cpu(), bits))
        assert torch.equal(tq.unpack_indices(got, bits, dim - 1).cpu(), torch.from_numpy(idx[..., :-1]))


def test_pack_out_of_range_and_empty(tq):
    g = torch.Generator().manual_seed(3)
    idx = torch.randint(-300, 5000, (37, 25), generator=g)
    words = torch.randint(-2 ** 31, 2 ** 31, (41, 13), generator=g).to(torch.int32)
    for bits in (1, 2, 3, 4):
        assert torch.equal(tq.pack_indices(idx.cuda(), bits).cpu(), tq.pack_indices(idx, bits))
        assert torch.equal(tq.pack_indices(idx.to(torch.uint8).cuda(), bits).cpu(), tq.pack_indices(idx.to(torch.uint8), bits))
        assert torch.equal(tq.unpack_indices(words.cuda(), bits, 96).cpu(), tq.unpack_indices(words, bits, 96))
        assert tq.pack_indices(idx[:0].cuda(), bits).shape == tq.pack_indices(idx[:0], bits).shape
        assert tq.unpack_indices(words[:0].cuda(), bits, 96).shape == (0, 96)
        assert tq.unpack_indices(words.cuda(), bits, 0).shape == (41, 0)


@pytest.mark.parametrize("bits", [1, 2, 3, 4])
def test_packing_can_be_traced(tq, bits):
    """A graph recorded from real tensors gives the words of the tensors that it is run on, not of those it was made with."""
    from torch.fx.experimental.proxy_tensor import make_fx
    dim = 40
    a, b = (torch.randint(0, 1 << bits, (6, dim), device="cuda", dtype=torch.uint8) for _ in range(2))

    def both(x):
        p = tq.pack_indices(x, bits).view(torch.int32)
        return p, tq.unpack_indices(p, bits, dim)
    want = both(b)
    got = make_fx(both)(a)(b)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], b)
