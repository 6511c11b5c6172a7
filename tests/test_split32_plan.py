"""Which fp32 / complex64 products take the fp16 split (planned on the CPU; nothing is queued)."""
import ctypes

import pytest
import torch

from metalblas_amd import _lib

SPLIT = (128, 128, 32, 2, 4, 4)


class _Ptr:   # stands in for a tensor: only data_ptr() is read
    def __init__(self, p):
        self.p = p

    def data_ptr(self):
        return self.p


def _desc(dtype, M, N, K, batch=1, b_stride=None, **kw):
    ops = [(_Ptr(0x7f0000000000 + (i << 40)), c, 1, 0 if batch == 1 else r * c)
           for i, (r, c) in enumerate(((M, K), (K, N), (M, N)))]
    if b_stride is not None:
        ops[1] = ops[1][:3] + (b_stride,)
    return _lib.make_desc(dtype, batch, M, N, K, *ops, flags=_lib.FLAG_DRY_RUN, **kw)


def _split(d):
    return tuple(_lib.plan(d).tile[:6]) == SPLIT


f32, c64 = torch.float32, torch.complex64


@pytest.mark.parametrize("dtype,shape,batch,taken", [
    (f32, (2048, 2048, 2048), 1, True), (f32, (1280, 1280, 1280), 1, True), (f32, (1024, 1024, 1024), 1, False),
    (f32, (4096, 4096, 64), 1, False), (f32, (16, 8192, 65536), 1, False), (f32, (128, 512, 512), 64, False),
    (f32, (1024, 1024, 1024), 8, True), (c64, (2048, 2048, 2048), 1, True), (c64, (512, 512, 512), 1, False),
    (c64, (768, 768, 768), 1, True), (torch.bfloat16, (2048, 2048, 2048), 1, False)], ids=str)
def test_rule(dtype, shape, batch, taken):
    assert _split(_desc(dtype, *shape, batch=batch)) == taken


def test_requests_keep_the_fp32_kernels():
    assert not _split(_desc(f32, 2048, 2048, 2048, backend=_lib.BACKEND_MATRIX))
    assert not _split(_desc(f32, 2048, 2048, 2048, backend=_lib.BACKEND_GENERIC))
    assert not _split(_desc(f32, 2048, 2048, 2048, tile=(128, 128, 32)))
    cands = _lib.tile_candidates(_desc(f32, 2048, 2048, 2048), 24)
    assert tuple(cands[0][:2]) == (128, 128) and cands[0][5] == 4
    assert any(c[5] == 1 for c in cands[1:])   # the fp32 tiles are its rivals


@pytest.mark.parametrize("dtype", [f32, c64], ids=str)
def test_scratch_limits(dtype):
    """With the workspace that the library asks for the split runs; with less, or none, the plan
    falls back to what ran before it (nothing is refused that needed less)."""
    lib = _lib.load()
    d = _desc(dtype, 2048, 2048, 2048)
    need = _lib.workspace_bytes(d)
    n = 2048 * 2048
    # split planes, 4 bytes per real element: A and B, or (complex: panels of A rows, so that the
    # product still fits the scratch of the allocation-free entry point) B and a part of A
    assert (8 * n if dtype is f32 else 8 * n + 4 * n) <= need <= lib.mb_gemm_noalloc_scratch_bytes()
    for have in (need, need - 1, 1 << 20, 0):
        d.workspace, d.workspace_bytes = (0x7e0000000000 if have else None), have
        assert lib.mb_gemm(ctypes.byref(d), None) == _lib.OK, have
    if torch.cuda.is_available():
        return
    d = _desc(f32, 2048, 2048, 2048)
    assert lib.mb_gemm_noalloc(ctypes.byref(d), None) in (_lib.OK, _lib.ERR_NO_DEVICE)
