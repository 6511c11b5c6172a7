"""Outputs whose rows are not 16-byte aligned (odd N, offset and padded views): the values against
float64, and the gaps of the buffer, which unaligned wide stores must leave alone."""
import pytest
import torch

import metalblas_amd as mb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.int8, torch.float32, torch.complex64], ids=str)
@pytest.mark.parametrize("offset,pad", [(0, 0), (1, 0), (3, 5)])
def test_values_and_gaps(dev, dtype, offset, pad):
    g = torch.Generator().manual_seed(offset)
    for M, N, K in ((257, 263, 512), (97, 1000, 640), (130, 129, 64), (2050, 2047, 1024)):
        if dtype is torch.int8:
            a, b = (torch.randint(-8, 9, s, generator=g, dtype=dtype).cuda() for s in ((M, K), (K, N)))
        else:
            wide = dtype if dtype.is_complex else torch.float32
            a, b = (torch.randn(s, generator=g, dtype=wide).to(dtype).cuda() for s in ((M, K), (K, N)))
        base = torch.full((offset + M * (N + pad) + 9,), 7, dtype=dtype, device=dev)
        view = base[offset:offset + M * (N + pad)].view(M, N + pad)
        mb.matmul(a, b, out=view[:, :N])
        w = torch.complex128 if dtype.is_complex else torch.float64
        A, B = a.to(w), b.to(w)
        exact = A @ B
        if dtype is torch.int8:
            assert torch.equal(view[:, :N], exact.to(torch.int64).to(dtype)), (M, N, K)
        else:
            # one rounding to the type and that of a K-term fp32 sum (complex: 2 K real terms)
            u = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}.get(dtype, 2.0 ** -24)
            limit = u * exact.abs() + 4 * K * 2.0 ** -24 * (A.abs() @ B.abs())
            assert bool(((view[:, :N].to(w) - exact).abs() <= limit).all()), (M, N, K)
        assert bool((view[:, N:] == 7).all() and (base[:offset] == 7).all() and (base[offset + M * (N + pad):] == 7).all())
