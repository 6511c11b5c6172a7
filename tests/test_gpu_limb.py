"""Integer products on the 8-bit matrix cores (signed-byte digits), against torch's wrapping CPU
products: every value pattern of the digits' carries, tile and K-step edges, K slices, and a sum
long enough to wrap the 32-bit partial sums of the 64-bit products."""
import pytest
import torch

import metalblas_amd as mb

pytestmark = pytest.mark.gpu

TYPES = [torch.int8, torch.uint8, torch.int16, torch.int32, torch.int64]


def _values(shape, dtype, g):
    """Full-range values, one in four a pattern at a byte's sign edge (0x7f, 0x80, all ones, the
    extremes)."""
    i = torch.iinfo(dtype)
    t = torch.randint(i.min, i.max, shape, generator=g, dtype=torch.int64)
    edge = torch.tensor([0x7f, 0x80, 0x7f80, 0x8080807f, 0x7f7f7f7f, -1, 0, i.min, i.max, 0x80808080 << 8])
    pick = edge[torch.randint(0, len(edge), shape, generator=g)]
    return torch.where(torch.rand(shape, generator=g) < 0.25, pick, t).to(dtype)


def _operand(rows, cols, layout, dtype, g):
    t = _values((rows, cols) if layout == "r" else (cols, rows), dtype, g)
    return t if layout == "r" else t.t()


@pytest.mark.parametrize("dtype", TYPES, ids=str)
@pytest.mark.parametrize("layout", ["rr", "rc", "cr", "cc"])
def test_edges(dev, dtype, layout):
    g = torch.Generator().manual_seed(1)
    for M, N, K in ((33, 17, 1), (17, 33, 64), (40, 70, 65), (16, 48, 128), (130, 67, 200), (256, 250, 256),
                    (513, 520, 129), (64, 96, 1025), (200, 72, 2100)):
        a, b = _operand(M, K, layout[0], dtype, g), _operand(K, N, layout[1], dtype, g)
        da, db = (t.cuda() if t.is_contiguous() else t.t().cuda().t() for t in (a, b))
        assert torch.equal(mb.matmul(da, db, backend="generic").cpu(), a @ b), (M, N, K)
        assert torch.equal(mb.matmul(da, db).cpu(), a @ b), (M, N, K)


@pytest.mark.parametrize("dtype", TYPES, ids=str)
def test_strided_views_epilogue_and_batches(dev, dtype):
    g = torch.Generator().manual_seed(2)
    a, b = _values((70, 201), dtype, g), _values((200, 90), dtype, g)
    view = a.cuda()[:, 1:]                                 # rows at an odd element offset
    assert torch.equal(mb.matmul(view, b.cuda()).cpu(), a[:, 1:] @ b)
    bias = _values((90,), dtype, g)
    got = mb.addmm(bias.cuda(), view, b.cuda(), beta=3, alpha=5).cpu()
    assert torch.equal(got, (3 * bias + 5 * (a[:, 1:] @ b)).to(dtype))
    x, y = _values((5, 40, 130), dtype, g), _values((5, 130, 60), dtype, g)
    assert torch.equal(mb.bmm(x.cuda(), y.cuda()).cpu(), torch.stack([x[i] @ y[i] for i in range(5)]))


@pytest.mark.parametrize("K", [8191, 8192, 8200, 33000])
def test_long_sums_of_the_extremes(dev, K):
    """Every digit product of int64's smallest values has the same sign: the 32-bit partial sums
    would wrap past 2^31 / (8 2^14) terms if they were not added up on the way."""
    for v in (-(2 ** 63), 2 ** 63 - 1, 0x7f7f7f7f7f7f7f7f, -0x7f7f7f7f7f7f7f80):
        a = torch.full((40, K), v, dtype=torch.int64)
        b = torch.full((K, 24), v, dtype=torch.int64)
        got = mb.matmul(a.cuda(), b.cuda()).cpu()
        want = (v * v * K + 2 ** 63) % 2 ** 64 - 2 ** 63
        assert bool((got == want).all()), (K, v)
