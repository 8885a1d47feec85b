"""Blocks up from and down to column-major host memory: every dtype, sizes
around the layout tile and the 2 MB pieces of the pinned pipeline, host leading
dimensions past n, part of the columns (the others untouched)."""
import ctypes as C

import numpy as np
import pytest

from rayleighchebyshevgpgpu_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32, np.complex128])
@pytest.mark.parametrize("n,cols,part,pad", [
    (1, 1, 1, 0), (31, 33, 33, 0), (33, 7, 5, 3), (4097, 65, 64, 0), (65280, 5, 5, 1),
    (131072, 4, 4, 0), (262145, 3, 2, 7)])
def test_upload_download(n, cols, part, pad, dtype):
    from rayleighchebyshevgpgpu_amd import solver as rcg
    g = np.random.default_rng(n)

    def draw(rows, c):
        x = g.standard_normal((c, rows))
        if dtype == np.complex128:
            x = x + 1j * g.standard_normal((c, rows))
        return np.ascontiguousarray(x.astype(dtype)).T

    full, host = draw(n, cols), draw(n + pad, part)
    b = rcg.Block.from_host(full)
    assert np.array_equal(b.download(), full)
    capi.check(capi.lib().rcg_block_upload(b.h, host.ctypes.data_as(C.c_void_p), n + pad, part))
    want = full.copy(order="F")
    want[:, :part] = host[:n]
    assert np.array_equal(b.download(), want)
    back = np.full((n + pad, cols), 7, dtype=dtype, order="F")
    capi.check(capi.lib().rcg_block_download(b.h, back.ctypes.data_as(C.c_void_p), n + pad, part))
    assert np.array_equal(back[:n, :part], want[:, :part])
    assert np.all(back[n:] == 7) and np.all(back[:, part:] == 7)


def test_refused():
    from rayleighchebyshevgpgpu_amd import solver as rcg
    b = rcg.Block(8, 2)
    x = np.zeros((8, 3), order="F")
    for ld, cols in ((7, 2), (8, 3), (8, -1)):
        assert capi.lib().rcg_block_upload(b.h, x.ctypes.data_as(C.c_void_p), ld, cols) != capi.RCG_OK
    assert capi.lib().rcg_block_download(b.h, x.ctypes.data_as(C.c_void_p), 8, 0) == capi.RCG_OK
