"""The K ping-pong tiles (128 x 128 and 256 x 128) against a float64 product, at the sizes where the
stage ring, the phase split between the wave groups and the tile edges change.

The limit is derived: one rounding to the output type plus the rounding of a K-term fp32 sum,
|got - exact| <= u |exact| + K 2^-24 (|A| @ |B|), u the unit roundoff of an 8-bit (bf16: 2^-8) or
11-bit significand (fp16: 2^-11, and half of its smallest subnormal, 2^-25)."""
import pytest
import torch

import metalblas_amd as mb

pytestmark = pytest.mark.gpu


def _operand(rows, cols, layout, dtype, g, batch=None):
    shape = (rows, cols) if layout == "r" else (cols, rows)
    t = torch.randn(((batch,) if batch else ()) + shape, generator=g).to(dtype).cuda()
    return t if layout == "r" else t.transpose(-1, -2)


def _check(got, a, b, tag):
    exact = torch.matmul(a.double().contiguous(), b.double().contiguous())
    terms = torch.matmul(a.double().abs().contiguous(), b.double().abs().contiguous())
    u, tiny = (2.0 ** -8, 0.0) if got.dtype == torch.bfloat16 else (2.0 ** -11, 2.0 ** -25)
    limit = u * exact.abs() + a.shape[-1] * 2.0 ** -24 * terms + tiny
    over = ((got.double() - exact).abs() / limit).max().item()
    assert over <= 1.0, (tag, over)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("layout", ["rr", "rc", "cr", "cc"])
@pytest.mark.parametrize("bm", [128, 256])
def test_stage_counts_and_edges(dev, dtype, layout, bm):
    """1 to 9 stages of 64 (whole, and with a K edge), tiles cut at the row and column edges."""
    g = torch.Generator().manual_seed(bm)
    for K in (8, 64, 72, 128, 192, 200, 256, 264, 328, 384, 520, 576):
        for M, N in ((8, 128), (256, 136), (264, 120), (520, 264)):
            a, b = _operand(M, K, layout[0], dtype, g), _operand(K, N, layout[1], dtype, g)
            got = mb.matmul(a, b, backend="mpp_tensor", tile=(bm, 128, 64, 2, 4, 4))
            _check(got, a, b, (M, N, K))


@pytest.mark.parametrize("split", [2, 3])
def test_k_slices_and_epilogue(dev, split):
    """The tiles under an explicit K-slice request (fp32 planes and their reduction) and with the
    fused epilogue into a column-major output."""
    from metalblas_amd import _lib
    import ctypes
    g = torch.Generator().manual_seed(split)
    M, N, K = 264, 392, 1096
    a, b = _operand(M, K, "r", torch.bfloat16, g), _operand(K, N, "r", torch.bfloat16, g)
    for bm in (128, 256):
        c = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
        d = _lib.make_desc(torch.bfloat16, 1, M, N, K, (a, K, 1, 0), (b, N, 1, 0), (c, N, 1, 0),
                           tile=(bm, 128, 64, 2, 4, 4))
        d.split_k = split
        info = _lib.plan(d)
        assert info.tile[5] == 4 and info.split_k == split
        need = _lib.workspace_bytes(d)
        ws = torch.empty(need, dtype=torch.uint8, device=dev)
        d.workspace, d.workspace_bytes = ws.data_ptr(), need
        _lib.check(_lib.load().mb_gemm(ctypes.byref(d), torch._C._cuda_getCurrentRawStream(0)))
        _check(c, a, b, (bm, split))


def test_plans_take_the_tiles(dev):
    """One round of 128 x 128 tiles, and of 256 x 128 where those need two."""
    def tile(M, N, K):
        a, b = (torch.empty(s, dtype=torch.bfloat16, device=dev) for s in ((M, K), (K, N)))
        return mb.kernels.plan(a, b)["tile"][:6]
    assert tile(2048, 2048, 4096) == (128, 128, 64, 2, 4, 4)
    assert tile(1536, 1536, 4096) == (128, 128, 64, 2, 4, 4)
    assert tile(2048, 4096, 2048) == (256, 128, 64, 2, 4, 4)
    assert tile(4096, 4096, 4096)[:2] == (256, 256)
