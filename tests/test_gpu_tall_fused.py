"""Products that also form column norms or the next Gram matrix, through the
piecewise entry points, at the edges of their tiles: 16-column subtiles, the
64-column limit of the fused Gram products, 64-row tiles, real and complex.

Tolerance: columns of unit norm from FP64 products over n <= 5000 rows; the
error of each entry is a few eps times the condition of the block (below 10
here), so 1e-12 leaves three digits.
"""
import ctypes as C

import numpy as np
import pytest

from rayleighchebyshevgpgpu_amd import capi

pytestmark = pytest.mark.gpu


def draw(g, n, c, cplx):
    x = g.standard_normal((n, c))
    return x + 1j * g.standard_normal((n, c)) if cplx else x


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("n,cols,found", [
    (70, 1, 1), (200, 15, 17), (257, 16, 33), (1000, 33, 16), (4097, 64, 64), (333, 65, 5),
    (640, 31, 65), (5000, 48, 32), (129, 32, 32)])
def test_deflate_orthonormalize_rotate(n, cols, found, cplx):
    from rayleighchebyshevgpgpu_amd import solver as rcg
    g = np.random.default_rng(n + cols)
    L = capi.lib()
    X = draw(g, n, cols, cplx)
    Y = np.linalg.qr(draw(g, n, found, cplx))[0] if found <= n else None
    bx, bt, by = rcg.Block.from_host(X), rcg.Block(n, cols, dtype=X.dtype), rcg.Block.from_host(Y)
    capi.check(L.rcg_deflate(bx.h, cols, by.h, found))
    D = X - Y @ (Y.conj().T @ X)
    D -= Y @ (Y.conj().T @ D)
    D /= np.linalg.norm(D, axis=0)
    assert np.max(np.abs(bx.download() - D)) < 1e-12
    if cols + found > n:
        return
    capi.check(L.rcg_orthonormalize(bx.h, bt.h, cols))
    Q = bx.download()
    assert np.max(np.abs(Q.conj().T @ Q - np.eye(cols))) < 1e-12
    R = Q.conj().T @ D
    assert np.max(np.abs(np.tril(R, -1))) < 1e-12 and np.all(np.real(np.diag(R)) > 0)
    Z = np.asfortranarray(draw(g, cols, cols, cplx) + 3 * np.eye(cols))
    capi.check(L.rcg_rotate(bx.h, bt.h, cols, Z.ctypes.data_as(C.c_void_p)))
    V = Q @ Z
    V /= np.linalg.norm(V, axis=0)
    assert np.max(np.abs(bx.download() - V)) < 1e-12
