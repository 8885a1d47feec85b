"""The CSR step over LDS tiles (schedule "lds-tiles") against the row-block step.

Both sum a row's nonzeros in the same order with the same fused operations: the
results must be the same bits.  Grids that tiles do not divide, both boundary
kinds, 2-D and 3-D, column counts around the 64-element panel, the FP64, mixed
and complex filters, and operators that tiles must refuse (rows too long, rows
that reach everywhere) although the hint names a grid.
"""
import ctypes as C
import os

import numpy as np
import pytest

from rayleighchebyshevgpgpu_amd import capi
from rayleighchebyshevgpgpu_amd import operators as ops

pytestmark = pytest.mark.gpu


def filtered(rcg, A, grid, X, cols, m, mixed, sched):
    old = os.environ.get("RCG_FILTER_SCHED")
    os.environ["RCG_FILTER_SCHED"] = sched
    try:
        op = rcg.CsrOperator(A, grid=grid)
        bx, bt = rcg.Block.from_host(X), rcg.Block(X.shape[0], X.shape[1], dtype=X.dtype)
        if mixed:
            th = np.linspace(0.0, 1.0, cols)
            rz = (np.arange(cols) % 3 != 2).astype(np.int32)
            capi.check(capi.lib().rcg_cheb_filter_mixed(
                op.h, bx.h, bt.h, cols, m, 1, 14.0, 1.0, th.ctypes.data_as(C.c_void_p),
                rz.ctypes.data_as(C.c_void_p)))
        else:
            capi.check(capi.lib().rcg_cheb_filter(op.h, bx.h, bt.h, cols, m, 1, 14.0, 1.0))
    finally:
        if old is None:
            del os.environ["RCG_FILTER_SCHED"]
        else:
            os.environ["RCG_FILTER_SCHED"] = old
    return bx.download()


def same(a, b):
    x = np.ascontiguousarray(a).view(np.float64)
    y = np.ascontiguousarray(b).view(np.float64)
    ok = ~np.isnan(x)
    return np.array_equal(np.isnan(x), np.isnan(y)) and np.array_equal(x[ok], y[ok])


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("grid,bc,cols,m", [
    ((4, 4, 4), "dirichlet", 1, 2), ((5, 7, 9), "periodic", 64, 3), ((16, 8, 12), "periodic", 65, 2),
    ((17, 6, 5), "dirichlet", 33, 5), ((9, 30, 21), "dirichlet", 128, 3), ((37, 41), "dirichlet", 45, 4),
    ((64, 24), "periodic", 96, 2), ((8, 8), "periodic", 63, 3), ((33, 34, 35), "periodic", 48, 4)])
def test_tiles_equal_rows(grid, bc, cols, m, mixed):
    from rayleighchebyshevgpgpu_amd import solver as rcg
    n = int(np.prod(grid))
    pot = ops.anderson_potential(n, 3.0, n)
    A = ops.laplacian_2d(*grid, bc, pot) if len(grid) == 2 else ops.laplacian_3d(*grid, bc, pot)
    X = np.random.default_rng(n).standard_normal((n, cols + 1))
    X[n // 2, 0], X[n // 3, cols // 2] = np.inf, np.nan
    a = filtered(rcg, A, grid, X, cols, m, mixed, "lds-tiles")
    assert same(a, filtered(rcg, A, grid, X, cols, m, mixed, "rows"))
    assert np.array_equal(a[:, cols:], X[:, cols:])


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("L,cols", [(64, 96), (64, 33), (128, 5)])
def test_tiles_equal_rows_complex(L, cols, mixed):
    from rayleighchebyshevgpgpu_amd import solver as rcg
    A = ops.hofstadter_2d(L, W=2.0)
    g = np.random.default_rng(L)
    X = g.standard_normal((A.n, cols)) + 1j * g.standard_normal((A.n, cols))
    a = filtered(rcg, A, (L, L), X, cols, 3, mixed, "lds-tiles")
    assert same(a, filtered(rcg, A, (L, L), X, cols, 3, mixed, "rows"))


@pytest.mark.parametrize("kind", ["long rows", "scattered"])
def test_operators_tiles_refuse(kind):
    from rayleighchebyshevgpgpu_amd import solver as rcg
    n = 12 * 12 * 12
    g = np.random.default_rng(1)
    q = 9 if kind == "long rows" else 7
    col = np.concatenate([np.sort(g.choice(n, q, replace=False)) for _ in range(n)])
    A = ops.Csr(n, np.arange(n + 1) * q, col, g.standard_normal(n * q))
    X = g.standard_normal((n, 8))
    with pytest.raises(capi.RcgError):
        filtered(rcg, A, (12, 12, 12), X, 8, 2, False, "lds-tiles")
    a = filtered(rcg, A, (12, 12, 12), X, 8, 2, False, "rows")
    assert same(a, filtered(rcg, A, None, X, 8, 2, False, "rows"))
