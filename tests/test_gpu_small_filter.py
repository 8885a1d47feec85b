"""The one-launch filter of small CSR operators against the general step kernel.

The rule takes n <= 4096 (complex128: 2048) with rows of at most 7 nonzeros on
average and 12 at most; RCG_FILTER_PANEL forces the general kernel.  Both sum
a row's nonzeros in the same order with the same fused operations, so the
results must be the same bits, columns past `cols` untouched.
"""
import ctypes as C
import os

import numpy as np
import pytest

from rayleighchebyshevgpgpu_amd import capi
from rayleighchebyshevgpgpu_amd import operators as ops

pytestmark = pytest.mark.gpu


def operator(n, longest, cplx, seed):
    """Rows of uneven length, some of them empty; not Hermitian, which the filter's
    arithmetic does not need."""
    g = np.random.default_rng(seed)
    length = np.minimum(g.integers(0, 6, n), n)
    length[g.integers(0, n, max(1, n // 50))] = min(longest, n)
    rowptr = np.concatenate([[0], np.cumsum(length)])
    col = np.concatenate([np.sort(g.choice(n, q, replace=False)) for q in length] or [[]])
    val = g.standard_normal(rowptr[-1])
    if cplx:
        val = val + 1j * g.standard_normal(rowptr[-1])
    return ops.Csr(n, rowptr, col, val if cplx else val.astype(np.float64))


def filtered(rcg, A, X, cols, m, rep, mixed, general):
    op = rcg.CsrOperator(A)
    bx, bt = rcg.Block.from_host(X), rcg.Block(X.shape[0], X.shape[1], dtype=X.dtype)
    old = os.environ.get("RCG_FILTER_PANEL")
    if general:
        os.environ["RCG_FILTER_PANEL"] = str(X.shape[1] * 2)
    try:
        if mixed:
            th = np.linspace(-1.0, 1.0, cols)
            rz = (np.arange(cols) % 3 != 2).astype(np.int32)
            capi.check(capi.lib().rcg_cheb_filter_mixed(
                op.h, bx.h, bt.h, cols, m, rep, 9.0, 5.0, th.ctypes.data_as(C.c_void_p),
                rz.ctypes.data_as(C.c_void_p)))
        else:
            capi.check(capi.lib().rcg_cheb_filter(op.h, bx.h, bt.h, cols, m, rep, 9.0, 5.0))
    finally:
        if general:
            if old is None:
                del os.environ["RCG_FILTER_PANEL"]
            else:
                os.environ["RCG_FILTER_PANEL"] = old
    return bx.download()


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("n,cols,m,rep,longest", [
    (1, 1, 2, 1, 1), (63, 3, 2, 2, 5), (63, 2, 1, 1, 5), (1024, 5, 3, 1, 7), (1025, 12, 8, 1, 12),
    (2048, 7, 5, 1, 8), (2049, 2, 4, 1, 5), (4095, 3, 5, 1, 12), (4096, 16, 7, 1, 7),
    (4097, 3, 3, 1, 7), (1500, 4, 3, 1, 40)])
def test_one_launch_equals_general_step(n, cols, m, rep, longest, mixed, cplx):
    from rayleighchebyshevgpgpu_amd import solver as rcg
    A = operator(n, longest, cplx, 7 * n + m)
    g = np.random.default_rng(n)
    X = g.standard_normal((n, cols + 2))
    if cplx:
        X = X + 1j * g.standard_normal((n, cols + 2))
    if n > 100:  # not-finite entries spread as in the general kernel
        X[n // 2, 0], X[n // 3, 1] = np.inf, np.nan
    a = filtered(rcg, A, X, cols, m, rep, mixed, False)
    b = filtered(rcg, A, X, cols, m, rep, mixed, True)
    view = np.float64
    x, y = np.ascontiguousarray(a).view(view), np.ascontiguousarray(b).view(view)
    assert np.array_equal(np.isnan(x), np.isnan(y))
    ok = ~np.isnan(x)
    assert np.array_equal(x[ok], y[ok]) and np.array_equal(np.signbit(x[ok]), np.signbit(y[ok]))
    assert np.array_equal(a[:, cols:], X[:, cols:])
