"""The 64 x 64 ring against float64: unsplit and over K slices, 1 to 9 stages (the ring holds 4) with
and without a K edge, tile edges, misaligned output rows, batches and the fused epilogue.

Limit: |got - exact| <= u |exact| + K 2^-24 (|A| @ |B|), u the unit roundoff of the output type."""
import pytest
import torch

import metalblas_amd as mb

pytestmark = pytest.mark.gpu

RING = (64, 64, 64, 2, 2, 3)


def _check(got, a, b, tag, alpha=1.0, add=None):
    A, B = a.double().contiguous(), b.double().contiguous()
    exact = alpha * torch.matmul(A, B)
    u = 2.0 ** -8 if got.dtype == torch.bfloat16 else 2.0 ** -11
    limit = abs(alpha) * a.shape[-1] * 2.0 ** -24 * torch.matmul(A.abs(), B.abs()) + 2.0 ** -25
    if add is not None:
        exact = exact + add.double()
    limit = limit + u * exact.abs() + (0 if add is None else 2.0 ** -22 * add.double().abs())
    assert bool(((got.double() - exact).abs() <= limit).all()), tag


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("layout", ["rr", "rc", "cr", "cc"])
def test_stages_and_edges(dev, dtype, layout):
    g = torch.Generator().manual_seed(4)

    def operand(rows, cols, o):
        t = torch.randn((rows, cols) if o == "r" else (cols, rows), generator=g).to(dtype).cuda()
        return t if o == "r" else t.t()
    for K in (8, 64, 72, 128, 200, 256, 264, 576, 2056):
        for M, N in ((8, 64), (72, 136), (200, 120)):
            a, b = operand(M, K, layout[0]), operand(K, N, layout[1])
            _check(mb.matmul(a, b, backend="mpp_tensor", tile=RING), a, b, (M, N, K))
            out = torch.empty(M, N + 1, dtype=dtype, device=dev)[:, 1:]     # odd rows
            mb.matmul(a, b, backend="mpp_tensor", tile=RING, out=out)
            _check(out, a, b, (M, N, K, "odd rows"))


def test_static_plans_batches_and_slices(dev):
    """Plans below K = 2048, batched, with an epilogue; and K slices on request."""
    import ctypes
    from metalblas_amd import _lib
    g = torch.Generator().manual_seed(5)
    M, N, K = 500, 516, 1000
    a, b = (torch.randn(s, generator=g).to(torch.bfloat16).cuda() for s in ((M, K), (K, N)))
    assert mb.kernels.plan(a, b)["tile"][:6] == RING
    _check(mb.matmul(a, b), a, b, "plain")
    bias = torch.randn(N, generator=g).to(torch.bfloat16).cuda()
    _check(mb.addmm(bias, a, b, beta=0.5, alpha=-2), a, b, "addmm", -2.0, 0.5 * bias)
    for batch in (3, 11):
        x = torch.randn(batch, 130, 520, generator=g).to(torch.bfloat16).cuda()
        y = torch.randn(batch, 520, 72, generator=g).to(torch.bfloat16).cuda()
        _check(mb.bmm(x, y), x, y, batch)
    for split in (2, 3, 7):
        c = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
        d = _lib.make_desc(torch.bfloat16, 1, M, N, K, (a, K, 1, 0), (b, N, 1, 0), (c, N, 1, 0), tile=RING)
        d.split_k = split
        need = _lib.workspace_bytes(d)
        ws = torch.empty(need, dtype=torch.uint8, device=dev)
        d.workspace, d.workspace_bytes = ws.data_ptr(), need
        _lib.check(_lib.load().mb_gemm(ctypes.byref(d), torch._C._cuda_getCurrentRawStream(0)))
        _check(c, a, b, split)
