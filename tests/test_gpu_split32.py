"""fp32 and complex64 products on the fp16 matrix cores (split into high and low parts): accuracy
against float64, every operand form, and the values that are left to the fp32 kernels.

The limit is that of a K-term fp32 sum, |got - exact| <= K 2^-24 (|A| @ |B|) elementwise (for
complex: K' = 2K real terms per part, on the parts' magnitudes), doubled where alpha, beta and a
bias add two more roundings."""
import pytest
import torch

import metalblas_amd as mb

pytestmark = pytest.mark.gpu

F32_TILE = (64, 64, 32, 2, 2, 1)   # a tile request runs the fp32 kernels


def _operand(rows, cols, layout, dtype, g, batch=None):
    shape = (rows, cols) if layout == "r" else (cols, rows)
    t = torch.randn(((batch,) if batch else ()) + shape, generator=g, dtype=dtype).cuda()
    return t if layout == "r" else t.transpose(-1, -2)


def _wide(t):
    return t.to(torch.complex128 if t.is_complex() else torch.float64).resolve_conj().contiguous()


def _check(got, a, b, alpha=1.0, beta=0.0, bias=None):
    A, B = _wide(a), _wide(b)
    exact = alpha * torch.matmul(A, B)
    mag = (lambda t: t.real.abs() + t.imag.abs()) if got.is_complex() else (lambda t: t.abs())
    k = A.shape[-1] * (2 if got.is_complex() else 1)
    limit = abs(alpha) * k * 2.0 ** -24 * torch.matmul(mag(A), mag(B))
    if bias is not None:
        exact = exact + beta * _wide(bias)
        limit = 2 * limit + 2.0 ** -22 * mag(beta * _wide(bias))
    assert bool((mag(_wide(got) - exact) <= limit).all()), ((mag(_wide(got) - exact)) / limit).max().item()
    return float(torch.linalg.vector_norm(_wide(got) - exact) / torch.linalg.vector_norm(exact))


def _takes_split(a, b):
    return mb.kernels.plan(a, b)["tile"][:6] == (128, 128, 32, 2, 4, 4)


@pytest.mark.parametrize("layout", ["rr", "rc", "cr", "cc"])
@pytest.mark.parametrize("shape", [(1280, 1280, 1280), (1025, 1300, 1543), (520, 4100, 1111), (2100, 3000, 417),
                                   (1031, 717, 4099)], ids=str)
def test_fp32(dev, shape, layout):
    M, N, K = shape
    g = torch.Generator().manual_seed(K)
    a, b = _operand(M, K, layout[0], torch.float32, g), _operand(K, N, layout[1], torch.float32, g)
    assert _takes_split(a, b)
    err = _check(mb.matmul(a, b), a, b)
    fp32 = _check(mb.matmul(a, b, backend="mpp_tensor", tile=F32_TILE), a, b)
    assert err <= fp32, (err, fp32)
    bias = torch.randn(N, generator=g).cuda()
    _check(mb.addmm(bias, a, b, beta=0.5, alpha=-2.0), a, b, -2.0, 0.5, bias)
    out = torch.randn(N, M, generator=g).cuda().t()      # column-major, and its own bias
    was = out.clone()
    _check(mb.addmm(out, a, b, out=out), a, b, 1.0, 1.0, was)


@pytest.mark.parametrize("conj", ["", "a", "b", "ab"])
@pytest.mark.parametrize("layout", ["rr", "rc", "cr", "cc"])
def test_complex64(dev, layout, conj):
    g = torch.Generator().manual_seed(5)
    for M, N, K in ((768, 768, 768), (701, 1027, 900), (2100, 520, 333)):
        a, b = _operand(M, K, layout[0], torch.complex64, g), _operand(K, N, layout[1], torch.complex64, g)
        assert _takes_split(a, b)
        a, b = (a.conj() if "a" in conj else a), (b.conj() if "b" in conj else b)
        _check(mb.matmul(a, b), a, b)
        bias = _operand(M, N, "r", torch.complex64, g)
        _check(mb.addmm(bias, a, b, beta=0.5 - 1j, alpha=2j), a, b, 2j, 0.5 - 1j, bias)


@pytest.mark.parametrize("dtype", [torch.float32, torch.complex64], ids=str)
def test_batches(dev, dtype):
    g = torch.Generator().manual_seed(6)
    for layout in ("rr", "rc", "cr"):
        a, b = _operand(800, 800, layout[0], dtype, g, 7), _operand(800, 1000, layout[1], dtype, g, 7)
        assert _takes_split(a, b)
        _check(mb.bmm(a, b), a, b)
        shared = b[:1].expand(7, 800, 1000)
        _check(mb.bmm(a, shared), a, shared)
        _check(mb.bmm(a[:1].expand(7, 800, 800), b), a[:1].expand(7, 800, 800), b)


def _same_bits(x, y):
    return torch.equal(torch.nan_to_num(x, 3.0, 5.0, 7.0), torch.nan_to_num(y, 3.0, 5.0, 7.0)) and \
        torch.equal(torch.isfinite(x), torch.isfinite(y))


@pytest.mark.parametrize("value", ["inf", "-inf", "nan", "lowest", "tiny", "wide"])
def test_values_left_to_the_fp32_kernels(dev, value):
    """An infinity, a NaN, or an element too small beside its row's largest: the result is bit for
    bit that of the fp32 kernels, whichever operand and layout holds it."""
    g = torch.Generator().manual_seed(7)
    for layout in ("rr", "cc"):
        for side in (0, 1):
            ops = [_operand(1300, 1408, layout[0], torch.float32, g), _operand(1408, 1200, layout[1], torch.float32, g)]
            t = ops[side]
            if value == "wide":
                t[37] *= torch.logspace(-25, 10, t.shape[1], device=dev)
            else:
                t[37, 41] = {"inf": float("inf"), "-inf": -float("inf"), "nan": float("nan"),
                             "lowest": torch.finfo(torch.float32).min, "tiny": 1e-30}[value]
            a, b = ops
            assert _takes_split(a, b)
            tile = mb.kernels.plan(a, b, backend="mpp_tensor")["tile"]   # the fp32 plan behind the split
            assert _same_bits(mb.matmul(a, b), mb.matmul(a, b, backend="mpp_tensor")), (layout, side, tile)


def test_scaled_rows_zeros_and_denormals_stay_on_the_split(dev):
    """Row and column scales of any size, zero rows and columns, denormal rows."""
    g = torch.Generator().manual_seed(8)
    a, b = _operand(1300, 1408, "r", torch.float32, g), _operand(1408, 1200, "r", torch.float32, g)
    s = torch.logspace(-20, 15, 1300, device=dev)[:, None]
    t = torch.logspace(-15, 15, 1200, device=dev)[None]
    _check(mb.matmul(a * s, b * t), a * s, b * t)
    z = a.clone()
    z[:200] = 0
    z[:, 1000:] = 0
    got = mb.matmul(z, b)
    assert bool((got[:200] == 0).all())
    _check(got, z, b)
    d, big = a * 1e-41, b * 1e30     # denormal operands, normal results
    _check(mb.matmul(d, big), d, big)


@pytest.mark.parametrize("dtype", [torch.float32, torch.complex64], ids=str)
def test_graph_replays_choose_the_kernels_by_the_values(dev, dtype):
    """A captured product decides at each replay: finite values run split, an infinity the fp32
    kernels, and finite ones again after it."""
    g = torch.Generator().manual_seed(9)
    a, b = _operand(1024, 1500, "r", dtype, g), _operand(1500, 1400, "r", dtype, g)
    mb.matmul(a, b)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        c = mb.matmul(a, b)
    view = torch.view_as_real if dtype.is_complex else (lambda t: t)
    for i in range(4):
        a.copy_(_operand(1024, 1500, "r", dtype, g))
        if i == 1:
            a[3, 5] = float("inf")
        graph.replay()
        eager = mb.matmul(a, b)
        torch.cuda.synchronize()
        assert _same_bits(view(c), view(eager)), i
        assert bool(torch.isfinite(view(c)).all()) == (i != 1)
