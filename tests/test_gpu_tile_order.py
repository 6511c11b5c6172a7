"""The XCD-contiguous order of (batch entry, tile) indices (csrc/tile_order.hpp)."""
import pytest
import torch

import metalblas_amd as mb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 2, 3, 7, 8, 9, 16, 17, 31])
def test_every_batch_entry_holds_its_product(dev, batch):
    """The order is a bijection for any count of tiles and batch entries.  Integer-valued operands
    with sums below 2^8: the products are exact, so the outputs are compared for equality."""
    g = torch.Generator().manual_seed(batch)
    for M, N, K in ((200, 136, 72), (72, 520, 64), (328, 328, 40)):
        a = torch.randint(-1, 2, (batch, M, K), generator=g).to(torch.bfloat16).cuda()
        b = torch.randint(-1, 2, (batch, K, N), generator=g).to(torch.bfloat16).cuda()
        want = torch.stack([a[i].float() @ b[i].float() for i in range(batch)])
        for dtype in (torch.bfloat16, torch.float32):
            assert torch.equal(mb.bmm(a.to(dtype), b.to(dtype)).float(), want), (M, N, K, dtype)
