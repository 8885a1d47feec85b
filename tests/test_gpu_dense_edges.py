"""Dense steps at the edges of their tiles (128 / 64 rows, 64 columns, K chunks of 16 / 32), of the
loop without guards and of the K splits, against the FP64 oracle filter.

Tolerance: with ||A||_inf <= 1 a product is off by at most (n + 32) u max|X|, and the recurrence
passes each of the m products' errors on with a factor of at most m + 1 before its final
division by m + 1; u is 2^-53, 2^-24 for the mixed filter's FP32 steps.
"""
import ctypes as C

import numpy as np
import pytest

from rayleighchebyshevgpgpu_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,cols", [(1, 1), (15, 3), (63, 64), (65, 65), (127, 5), (129, 66),
                                    (255, 1), (256, 64), (383, 63), (511, 130), (1025, 31),
                                    (2047, 64), (2048, 129), (4099, 9)])
@pytest.mark.parametrize("mixed", [False, True])
def test_filter_at_tile_edges(orc, n, cols, mixed):
    from rayleighchebyshevgpgpu_amd import solver as rcg
    print(f"case: dense filter n={n} cols={cols} mixed={mixed}", flush=True)
    m = 4
    g = np.random.default_rng(n)
    A = g.uniform(-1, 1, (n, n))
    A += A.T
    A = np.asfortranarray(A / np.abs(A).sum(axis=0).max())
    X = g.uniform(-1, 1, (n, cols))
    ref = orc.filter_dense(A, X, m, 2.0, 1.0)
    op = rcg.DenseOperator(A)
    bx, bt = rcg.Block.from_host(X), rcg.Block(n, cols)
    if mixed:
        th = np.array([X[:, j] @ (A @ X[:, j]) / (X[:, j] @ X[:, j]) for j in range(cols)])
        rz = np.ones(cols, dtype=np.int32)
        capi.check(capi.lib().rcg_cheb_filter_mixed(op.h, bx.h, bt.h, cols, m, 1, 2.0, 1.0,
                                                    th.ctypes.data_as(C.c_void_p),
                                                    rz.ctypes.data_as(C.c_void_p)))
    else:
        capi.check(capi.lib().rcg_cheb_filter(op.h, bx.h, bt.h, cols, m, 1, 2.0, 1.0))
    u = 2.0 ** (-24 if mixed else -53)
    assert np.max(np.abs(bx.download() - ref)) <= m * (n + 32) * u * np.max(np.abs(X))


@pytest.mark.parametrize("n,lda,cols", [(200, 204, 7), (1029, 1036, 66), (2050, 2052, 64)])
def test_padded_rows(n, lda, cols):
    """A matrix on the device whose rows are lda apart, with NaN between them."""
    from rayleighchebyshevgpgpu_amd import solver as rcg
    print(f"case: dense n={n} lda={lda} cols={cols}", flush=True)
    g = np.random.default_rng(n)
    A = np.full((n, lda), np.nan)
    A[:, :n] = g.uniform(-1, 1, (n, n))
    A[:, :n] += A[:, :n].T.copy()
    mem = rcg.Block.from_host(A)  # rows of lda entries: lda is a multiple of 4
    ptr = C.c_void_p()
    capi.check(capi.lib().rcg_block_info(mem.h, None, None, None, None, C.byref(ptr)))
    assert mem.ld == lda
    h = C.c_void_p()
    capi.check(capi.lib().rcg_operator_dense_create(rcg.default_context().h, n, ptr, lda,
                                                    capi.MEM_DEVICE, C.byref(h)))
    X = g.uniform(-1, 1, (n, cols))
    bx, bt = rcg.Block.from_host(X), rcg.Block(n, cols)
    capi.check(capi.lib().rcg_operator_apply(h, bx.h, bt.h, 1.0, 0.0, cols))
    ref = A[:, :n] @ X
    scale = np.max(np.abs(A[:, :n]).sum(axis=1))
    assert np.max(np.abs(bt.download() - ref)) <= 2 * (n + 32) * 2.0**-53 * scale
    capi.check(capi.lib().rcg_cheb_filter(h, bx.h, bt.h, cols, 1, 1, 4.0 * n, 0.0))
    assert np.isfinite(bx.download()).all()
    capi.check(capi.lib().rcg_operator_destroy(h))


def dense_products(rcg, A, X):
    """A X by every entry point that forms it, as their W or out block."""
    n, cols = X.shape
    op = rcg.DenseOperator(A)
    bv = rcg.Block.from_host(X)
    th, res = np.zeros(cols), np.zeros(cols)
    H = np.zeros((cols, cols), order="F")
    out = {}
    for name in ("residuals", "noalloc", "project", "apply"):
        bw = rcg.Block(n, cols)
        p = [a.ctypes.data_as(C.c_void_p) for a in (th, res, H)]
        L = capi.lib()
        capi.check({"residuals": lambda: L.rcg_residuals(op.h, bv.h, bw.h, cols, p[0], p[1]),
                    "noalloc": lambda: L.rcg_residuals_noalloc(op.h, bv.h, bw.h, cols, p[0], p[1]),
                    "project": lambda: L.rcg_project(op.h, bv.h, bw.h, cols, p[2]),
                    "apply": lambda: L.rcg_operator_apply(op.h, bv.h, bw.h, 1.0, 0.0, cols)}[name]())
        out[name] = (bw.download(), res.copy() if name in ("residuals", "noalloc") else None)
    return out


@pytest.mark.parametrize("n,cols", [(255, 5), (700, 48), (1500, 130), (2900, 64), (4099, 130)])
def test_one_product_everywhere(n, cols):
    """A dense FP64 product has the same bits from every entry point, also where the fixed
    workspace of the no-allocation residuals holds the partial sums of some columns only,
    and the no-allocation residuals are those of the others."""
    from rayleighchebyshevgpgpu_amd import solver as rcg
    print(f"case: dense products n={n} cols={cols}", flush=True)
    g = np.random.default_rng(n)
    A = g.uniform(-1, 1, (n, n))
    A = np.asfortranarray((A + A.T) / n)
    X = g.uniform(-1, 1, (n, cols))
    got = dense_products(rcg, A, X)
    W, res = got["residuals"]
    scale = np.max(np.abs(A).sum(axis=1))
    assert np.max(np.abs(W - A @ X)) <= 2 * (n + 32) * 2.0**-53 * scale
    for name, (w, r) in got.items():
        assert np.array_equal(w, W), name
        assert r is None or np.max(np.abs(r - res) / res) <= 1e-14


@pytest.mark.parametrize("n,cols,pad", [(3000, 64, 4), (2049, 64, 4)])
def test_products_do_not_depend_on_earlier_calls(n, cols, pad):
    """The same call before and after one that needs more workspace: the same bits."""
    from rayleighchebyshevgpgpu_amd import solver as rcg
    print(f"case: dense history n={n} cols={cols}", flush=True)
    g = np.random.default_rng(n)
    A = g.uniform(-1, 1, (n, n))
    A = np.asfortranarray((A + A.T) / n)
    X = np.zeros((n, cols + pad))
    X[:, :cols] = g.uniform(-1, 1, (n, cols))
    ctx = rcg.Context(0)
    op = rcg.DenseOperator(A, ctx=ctx)

    def filtered():
        bx, bt = rcg.Block.from_host(X, ctx), rcg.Block(n, cols + pad, ctx=ctx)
        capi.check(capi.lib().rcg_cheb_filter(op.h, bx.h, bt.h, cols, 3, 1, 2.0, 1.0))
        return bx.download(cols)

    first = filtered()
    wide, tmp = rcg.Block(100000, 200, ctx=ctx), rcg.Block(100000, 200, ctx=ctx)
    wide.randomize(0, 200, 1, 0)
    capi.check(capi.lib().rcg_orthonormalize(wide.h, tmp.h, 200))
    assert np.array_equal(filtered(), first)
