"""Gram products, in one tile (up to 64 columns, passes of 32 or 64 rows per wave) and in 64x64 tiles
through LDS (chunks of 32 rows), at the edges of both, through deflation (Y^T X) and
orthonormalisation (X^T X).

Tolerances: with unit columns an entry of a Gram product is off by at most (n + 32) u.  Deflation
twice leaves Y^T X off by f times that; CholQR twice leaves X^T X off by b times that (the second
pass's matrix is the identity up to cond^2 u) and X = Q R with R upper triangular.
"""
import numpy as np
import pytest

from rayleighchebyshevgpgpu_amd import capi

pytestmark = pytest.mark.gpu

U = 2.0**-53


def unit(g, n, cols):
    X = g.standard_normal((n, cols))
    return X / np.linalg.norm(X, axis=0)


@pytest.mark.parametrize("n,b", [(300, 65), (383, 128), (512, 127), (1000, 97), (2053, 193),
                                 (4128, 130), (40001, 66),
                                 (1, 1), (63, 2), (300, 15), (259, 17), (4099, 33), (4101, 47),
                                 (30011, 49), (9999, 63), (50000, 64)])
def test_orthonormalize(n, b):
    from rayleighchebyshevgpgpu_amd import solver as rcg
    print(f"case: orthonormalize n={n} b={b}", flush=True)
    X = unit(np.random.default_rng(n), n, b)
    bx, bt = rcg.Block.from_host(X), rcg.Block(n, b)
    capi.check(capi.lib().rcg_orthonormalize(bx.h, bt.h, b))
    Q = bx.download()
    tol = 4 * b * (n + 32) * U
    assert np.max(np.abs(Q.T @ Q - np.eye(b))) <= tol
    R = Q.T @ X
    assert np.max(np.abs(Q @ R - X)) <= tol
    assert np.max(np.abs(np.tril(R, -1))) <= tol


@pytest.mark.parametrize("n,b,f", [(200, 1, 65), (257, 65, 1), (1000, 2, 129), (999, 129, 3),
                                   (2047, 66, 65), (4100, 67, 127), (40003, 96, 33),
                                   (70, 1, 1), (300, 1, 64), (4097, 17, 1), (5000, 33, 48),
                                   (9999, 63, 64), (30001, 16, 31)])
def test_deflate(n, b, f):
    from rayleighchebyshevgpgpu_amd import solver as rcg
    print(f"case: deflate n={n} b={b} f={f}", flush=True)
    g = np.random.default_rng(n)
    Y = np.linalg.qr(unit(g, n, f))[0]
    X = unit(g, n, b)
    bx, by = rcg.Block.from_host(X), rcg.Block.from_host(Y)
    capi.check(capi.lib().rcg_deflate(bx.h, b, by.h, f))
    D = bx.download()
    ref = X - Y @ (Y.T @ X)
    ref -= Y @ (Y.T @ ref)
    ref /= np.linalg.norm(ref, axis=0) / np.linalg.norm(D, axis=0)
    assert np.max(np.abs(D - ref)) <= 4 * f * (n + 32) * U * max(1.0, np.abs(D).max())


@pytest.mark.parametrize("n,b,f", [(257, 65, 1), (4097, 17, 1), (4097, 1, 24), (4100, 1, 96),
                                   (9999, 96, 1), (2050, 31, 45)])
def test_deflate_beside_nan(n, b, f):
    """Columns of either block past the ones in use hold NaN, which reaches no result."""
    from rayleighchebyshevgpgpu_amd import solver as rcg
    print(f"case: deflate beside NaN n={n} b={b} f={f}", flush=True)
    g = np.random.default_rng(n)
    Y, X = np.full((n, f + 3), np.nan), np.full((n, b + 3), np.nan)
    Y[:, :f] = np.linalg.qr(unit(g, n, f))[0]
    X[:, :b] = unit(g, n, b)
    bx, by = rcg.Block.from_host(X), rcg.Block.from_host(Y)
    capi.check(capi.lib().rcg_deflate(bx.h, b, by.h, f))
    D = bx.download()
    assert np.isnan(D[:, b:]).all() and np.isfinite(D[:, :b]).all()
    D, Y, X = D[:, :b], Y[:, :f], X[:, :b]
    ref = X - Y @ (Y.T @ X)
    ref -= Y @ (Y.T @ ref)
    ref /= np.linalg.norm(ref, axis=0) / np.linalg.norm(D, axis=0)
    assert np.max(np.abs(D - ref)) <= 4 * f * (n + 32) * U * max(1.0, np.abs(D).max())
