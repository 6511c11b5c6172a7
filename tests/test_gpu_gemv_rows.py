"""W @ x with K-contiguous rows: the row lengths where the streaming kernel or its loads in flight
change (256 and 1024 16-byte chunks), their neighbours and ragged row counts, against float64.

Limit: one rounding to the output type (u = 2^-8 bf16, 2^-11 fp16, 2^-24 fp32) plus that of a K-term
fp32 sum, K 2^-24 (|W| @ |x|)."""
import pytest
import torch

import metalblas_amd as mb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,u", [(torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -11),
                                     (torch.float32, 2.0 ** -24)], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("rows", [1, 7, 1030, 20000])
def test_row_lengths(dev, dtype, u, rows):
    g = torch.Generator().manual_seed(rows)
    per = 16 // torch.empty((), dtype=dtype).element_size()   # elements per chunk
    for chunks in (1, 64, 255, 256, 257, 512, 1023, 1024, 1025):
        K = chunks * per
        w = torch.randn(rows, K, generator=g).to(dtype).cuda()
        x = torch.randn(K, generator=g).to(dtype).cuda()
        exact = w.double() @ x.double()
        limit = u * exact.abs() + K * 2.0 ** -24 * (w.double().abs() @ x.double().abs()) + 2.0 ** -25
        assert bool(((mb.mv(w, x).double() - exact).abs() <= limit).all()), (rows, K)
        y = torch.randn(rows, generator=g).to(dtype).cuda()
        got = mb.addmm(y[:, None], w, x[:, None], beta=0.5, alpha=2).double()[:, 0]
        want = 2 * exact + 0.5 * y.double()
        assert bool(((got - want).abs() <= 2 * limit + u * (want.abs() + y.double().abs())).all()), (rows, K)
