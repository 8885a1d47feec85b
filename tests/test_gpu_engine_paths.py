"""Branches of the solve's engine that a whole solve reaches only with unusual
blocks, driven piece by piece through tests/cpp/engine_paths.cpp.

An iteration's orthonormalisation takes one CholQR pass where the block is known to
be nearly orthonormal, else two, and three after a shift; the first factor is made
on the device for real blocks of at most 32 columns.  Whatever the way, the basis
must be orthonormal and span the block, H = Q^H A Q, and the residuals those of Q;
the numbers of launches say which way was taken.

Tolerance: an entry of a Gram product of unit columns is summed in chains of fewer
than 256 terms (a lane's rows of a row block, then the partials), so it is off by at
most 256 u, and a basis of b columns by b times that.
"""
import ctypes as C
import gc
import os

import numpy as np
import pytest

from rayleighchebyshevgpgpu_amd import capi
from rayleighchebyshevgpgpu_amd import operators as ops

pytestmark = pytest.mark.gpu

U = 2.0**-53
LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "libengine_paths.so")


@pytest.fixture(scope="module")
def eng():
    """The Python classes over the test library."""
    from rayleighchebyshevgpgpu_amd import solver
    old = capi._lib, capi.LIB_PATH, solver._default_ctx
    capi._lib, capi.LIB_PATH, solver._default_ctx = None, LIB, None
    L = capi.lib()
    vp, i64 = C.c_void_p, C.c_int64
    L.test_ortho_project.argtypes = [vp, vp, vp, vp, vp, i64, vp, vp, vp]
    L.test_alloc_limit.argtypes = [i64]
    L.test_apply_tiles.argtypes = [vp, i64, vp]
    L.test_filter_route.argtypes = [vp, vp, vp, i64, i64, vp, i64, vp, vp]
    yield L
    gc.collect()
    if solver._default_ctx is not None:
        solver._default_ctx.close()
    capi._lib, capi.LIB_PATH, solver._default_ctx = old


def operator(shape, cx):
    if cx:
        return ops.hofstadter_2d(shape[0], phi=1.0 / 8, W=1.0)
    n = int(np.prod(shape))
    return ops.laplacian_3d(*shape, "dirichlet", ops.anderson_potential(n, 3.0, n))


def block(kind, n, b, cx, seed):
    g = np.random.default_rng(seed)

    def draw(r, c):
        x = g.standard_normal((r, c))
        return x + 1j * g.standard_normal((r, c)) if cx else x

    Q = np.linalg.qr(draw(n, b))[0]
    if kind == "near":  # as a filter leaves Ritz vectors
        return Q + 1e-3 / np.sqrt(n) * draw(n, b)
    if kind == "random":
        return Q @ (np.diag(np.logspace(0, -4, b)) @ np.linalg.qr(draw(b, b))[0])
    if kind == "pivots":  # every pivot above 1/2, and yet a condition of thousands
        R = np.zeros((b, b))
        for j in range(b):
            k = min(4, j)
            R[j, j] = np.sqrt(0.51) if k else 1.0
            R[j - k:j, j] = -np.sqrt(0.49 / k) if k else 0.0
        assert np.linalg.cond(R) > 1e3
        return Q @ R
    if kind == "rank":  # half of the directions below the Gram matrix's roundoff
        return Q @ (np.diag(np.where(np.arange(b) % 2, 1e-9, 1.0)) @ np.linalg.qr(draw(b, b))[0])
    assert kind == "zero"
    Q[:, b // 2] = 0.0
    return Q


def ortho_project(L, A, V, prime):
    from rayleighchebyshevgpgpu_amd import solver as rcg
    n, b = V.shape
    op = rcg.CsrOperator(A)
    bp = None if prime is None else rcg.Block.from_host(prime)
    bv = rcg.Block.from_host(V)
    bt, bw = rcg.Block(n, b, dtype=V.dtype), rcg.Block(n, b, dtype=V.dtype)
    H, res = np.zeros((b, b), dtype=V.dtype, order="F"), np.zeros(b)
    counts = np.full(3, -1, dtype=np.int32)
    capi.check(L.test_ortho_project(op.h, bp and bp.h, bv.h, bt.h, bw.h, b,
                                    H.ctypes.data_as(C.c_void_p), res.ctypes.data_as(C.c_void_p),
                                    counts.ctypes.data_as(C.c_void_p)))
    return bv.download(), H, res, counts.tolist()


# launches (device factors, paired, single Gram products) of the block by kind, and
# of the same after a nearly orthonormal block, where one pass is tried first
SMALL = {"near": ([1, 1, 0], [0, 1, 0]), "random": ([1, 1, 0], [1, 2, 0]),
         "pivots": ([1, 1, 0], [1, 2, 0]), "rank": ([1, 1, 4], [1, 2, 4])}
HOST = {"near": ([0, 1, 1], [0, 1, 0]), "random": ([0, 1, 1], [0, 2, 1]),
        "pivots": ([0, 1, 1], [0, 2, 1]), "rank": ([0, 0, 4], [0, 1, 4])}
LARGE = {"near": ([0, 0, 2], [0, 0, 2]), "random": ([0, 0, 2], [0, 0, 4]),
         "pivots": ([0, 0, 2], [0, 0, 4]), "rank": ([0, 0, 3], [0, 0, 5])}


@pytest.mark.parametrize("primed", [False, True])
@pytest.mark.parametrize("kind", ["near", "random", "pivots", "rank"])
@pytest.mark.parametrize("shape,b,cx,want", [
    ((12, 12, 12), 24, False, SMALL), ((11, 12, 13), 32, False, SMALL), ((10, 9, 11), 40, False, HOST),
    ((24, 24), 24, True, HOST), ((64, 64, 64), 24, False, LARGE)])
def test_ortho_project(eng, shape, b, cx, want, kind, primed):
    print(f"case: {shape} b={b} cx={cx} {kind} primed={primed}", flush=True)
    A = operator(shape, cx)
    V = block(kind, A.n, b, cx, 1)
    prime = block("near", A.n, b, cx, 2) if primed else None
    Q, H, res, counts = ortho_project(eng, A, V, prime)
    tol = 256 * b * U
    S = A.to_scipy()
    AQ = S @ Q
    norm = np.abs(S).sum(axis=1).max()
    assert np.max(np.abs(Q.conj().T @ Q - np.eye(b))) <= tol
    assert np.max(np.abs(Q @ (Q.conj().T @ V) - V)) <= 2 * tol
    assert np.max(np.abs(Q.conj().T @ AQ - H)) <= 2 * norm * tol
    ref = np.linalg.norm(Q * np.real(np.diag(H)) - AQ, axis=0)
    assert np.max(np.abs(res - ref)) <= 2 * norm * tol
    assert counts == want[kind][primed]


@pytest.mark.parametrize("primed", [False, True])
@pytest.mark.parametrize("shape,b,cx", [((12, 12, 12), 24, False), ((24, 24), 24, True)])
def test_zero_column_is_refused(eng, shape, b, cx, primed):
    """A block with a zero column has no orthonormal basis: the shifted passes end with
    an error whichever way they are reached."""
    A = operator(shape, cx)
    with pytest.raises(capi.RcgError, match="CholQR breakdown after a shifted pass"):
        ortho_project(eng, A, block("zero", A.n, b, cx, 1),
                      block("near", A.n, b, cx, 2) if primed else None)


def filter_route(L, A, grid, cols, m, op=None):
    from rayleighchebyshevgpgpu_amd import solver as rcg
    op = op or rcg.CsrOperator(A, grid=grid)
    bx, bt = rcg.Block(A.n, cols), rcg.Block(A.n, cols)
    bx.randomize(0, cols, 1, 0)
    name, panel, launches = C.create_string_buffer(64), C.c_int64(), C.c_int64()
    capi.check(L.test_filter_route(op.h, bx.h, bt.h, cols, m, name, 64, C.byref(panel),
                                   C.byref(launches)))
    return name.value.decode(), panel.value, launches.value


@pytest.mark.parametrize("grid,cols,tiles", [
    ((300, 300, 3), 32, True), ((45, 45, 45), 48, True), ((12, 10000, 1), 32, True),
    ((256, 256, 2), 32, False), ((5, 5, 8000), 32, False), ((5, 40000, 1), 32, False),
    ((9, 9, 1500), 32, False)])
def test_thin_grids_keep_row_blocks(eng, grid, cols, tiles):
    """FP64 steps go over LDS tiles where the grid fills them by two thirds."""
    print(f"case: route on {grid} x {cols}", flush=True)
    n = int(np.prod(grid))
    pot = ops.anderson_potential(n, 3.0, n)
    A = ops.laplacian_2d(*grid[:2], "dirichlet", pot) if grid[2] == 1 else \
        ops.laplacian_3d(*grid, "dirichlet", pot)
    name, _, _ = filter_route(eng, A, grid, cols, 3)
    assert (name == "lds-tiles") == tiles, name


@pytest.mark.parametrize("env,want", [
    ({}, ("lds-tiles", 96, 6)),  # 64 columns and 32 more, a launch each
    ({"RCG_FILTER_PANEL": "32"}, (None, 32, 9)),
    ({"RCG_FILTER_PANEL": "96"}, (None, 96, 3)),
    ({"RCG_FILTER_PANEL": "0"}, ("lds-tiles", 96, 6)),
    ({"RCG_FILTER_SCHED": "lds-tiles", "RCG_FILTER_PANEL": "32"}, ("lds-tiles", 96, 6)),
    ({"RCG_FILTER_SCHED": "rows", "RCG_FILTER_PANEL": "16"}, ("rows", 16, 18))])
def test_forced_panel(eng, monkeypatch, env, want):
    """RCG_FILTER_PANEL forces the column panel of the row orders, also where tiles (which
    have no panels) would be taken, and the launches are counted as they are made."""
    for k in ("RCG_FILTER_SCHED", "RCG_FILTER_PANEL"):
        monkeypatch.delenv(k, raising=False)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    grid = (40, 40, 44)
    n = int(np.prod(grid))
    A = ops.laplacian_3d(*grid, "periodic", ops.anderson_potential(n, 3.0, n))
    name, panel, launches = filter_route(eng, A, grid, 96, 3)
    assert name == want[0] if want[0] else name != "lds-tiles"
    assert (panel, launches) == want[1:]


@pytest.fixture
def scarce(eng):
    """limit(bytes): device allocations above that fail until the test ends."""
    def limit(nbytes):
        capi.check(eng.rcg_memory_trim())
        eng.test_alloc_limit(nbytes)
    yield limit
    eng.test_alloc_limit(-1)


def test_calls_after_a_failed_allocation(eng, scarce):
    """A context whose workspace could not be had is as good as new once there is memory."""
    from rayleighchebyshevgpgpu_amd import solver as rcg
    ctx = rcg.Context(0)
    g = np.random.default_rng(3)
    X = g.standard_normal((5000, 24))
    bx, bt = rcg.Block.from_host(X, ctx), rcg.Block(5000, 24, ctx=ctx)
    scarce(0)
    for _ in range(2):
        assert eng.rcg_orthonormalize(bx.h, bt.h, 24) == 3  # RCG_ERR_ALLOC
    eng.test_alloc_limit(-1)
    capi.check(eng.rcg_orthonormalize(bx.h, bt.h, 24))
    Q = bx.download()
    assert np.max(np.abs(Q.T @ Q - np.eye(24))) <= 256 * 24 * U
    assert np.max(np.abs(Q @ (Q.T @ X) - X)) <= 2 * 256 * 24 * U * np.linalg.norm(X, axis=0).max()


@pytest.mark.parametrize("dtype", [np.float64, np.float32, np.complex128])
@pytest.mark.parametrize("n,cols,part,pad,limit", [
    (70001, 9, 7, 3, 0), (300007, 5, 4, 1, 1 << 20), (70001, 9, 9, 0, 1 << 20),
    (300007, 3, 3, 5, 5 << 20), (33, 2, 1, 1, 0)])
def test_transfers_with_little_memory(scarce, n, cols, part, pad, limit, dtype):
    """Blocks go up and down whatever device memory is left: through a small buffer, by
    columns and by rows, or with none through the host."""
    from rayleighchebyshevgpgpu_amd import solver as rcg
    print(f"case: transfer n={n} cols={cols} limit={limit}", flush=True)
    g = np.random.default_rng(n)

    def draw(rows, c):
        x = g.standard_normal((c, rows))
        return np.ascontiguousarray((x + 1j * x[::-1] if dtype == np.complex128 else x).astype(dtype)).T

    full, host = draw(n, cols), draw(n + pad, part)
    b = rcg.Block.from_host(full)
    scarce(limit)
    capi.check(capi.lib().rcg_block_upload(b.h, host.ctypes.data_as(C.c_void_p), n + pad, part))
    want = full.copy(order="F")
    want[:, :part] = host[:n]
    back = np.full((n + pad, cols), 7, dtype=dtype, order="F")
    capi.check(capi.lib().rcg_block_download(b.h, back.ctypes.data_as(C.c_void_p), n + pad, cols))
    assert np.array_equal(back[:n], want) and np.all(back[n:] == 7)


@pytest.mark.parametrize("kind", ["grid", "dense"])
def test_products_with_little_memory(eng, scarce, kind):
    """rcg_operator_apply needs no device memory of its own: with none left it takes the
    default row order, or the unsplit dense product."""
    from rayleighchebyshevgpgpu_amd import solver as rcg
    print(f"case: apply with no memory, {kind}", flush=True)
    g = np.random.default_rng(5)
    if kind == "grid":
        grid = (64, 64, 64)
        A = ops.laplacian_3d(*grid, "periodic", ops.anderson_potential(64**3, 3.0, 1))
        op, S, cols, n = rcg.CsrOperator(A, grid=grid), A.to_scipy(), 20, 64**3
    else:
        n, cols = 900, 24
        S = g.uniform(-1, 1, (n, n))
        S = (S + S.T) / n
        op = rcg.DenseOperator(S)
    X = g.uniform(-1, 1, (n, cols))
    bx, by = rcg.Block.from_host(X), rcg.Block(n, cols)
    scarce(0)
    capi.check(eng.rcg_operator_apply(op.h, bx.h, by.h, 1.0, 0.0, cols))
    eng.test_alloc_limit(-1)
    scale = np.max(np.abs(S).sum(axis=1))
    assert np.max(np.abs(by.download() - S @ X)) <= 2 * (min(n, 1000) + 32) * U * scale


def test_operators_of_one_pattern_share_their_tiles(eng, scarce):
    """The tile plan holds the pattern only: operators that share a pattern and a grid share
    it, whichever of them made it."""
    from rayleighchebyshevgpgpu_amd import solver as rcg
    grid = (40, 40, 44)
    n = int(np.prod(grid))
    A = ops.laplacian_3d(*grid, "periodic", ops.anderson_potential(n, 3.0, n))
    base = rcg.CsrOperator(A, grid=grid)
    first, second = base.share(2.0 * A.val), base.share(A.val)
    assert filter_route(eng, A, None, 96, 3, first)[0] == "lds-tiles"
    bx, bt = rcg.Block(n, 96), rcg.Block(n, 96)
    bx.randomize(0, 96, 1, 0)
    X = bx.download()
    scarce(0)
    name = C.create_string_buffer(64)
    k, m = C.c_int64(), C.c_int64()
    for op in (second, base):
        capi.check(eng.test_filter_route(op.h, bx.h, bt.h, 96, 2, name, 64, C.byref(k), C.byref(m)))
        assert name.value == b"lds-tiles"
    eng.test_alloc_limit(-1)
    # a grid of its own ends it
    capi.check(eng.rcg_operator_set_grid(second.h, n, 1, 1))
    assert filter_route(eng, A, None, 96, 2, second)[0] != "lds-tiles"
    assert filter_route(eng, A, None, 96, 2, first)[0] == "lds-tiles"
    # the filter is the operator's own: the second and the base have one value array's content
    os.environ["RCG_FILTER_SCHED"] = "rows"
    try:
        by = rcg.Block.from_host(X)
        for op in (second, base):
            capi.check(eng.test_filter_route(op.h, by.h, bt.h, 96, 2, name, 64, C.byref(k), C.byref(m)))
    finally:
        del os.environ["RCG_FILTER_SCHED"]
    assert np.array_equal(bx.download(), by.download())


@pytest.mark.parametrize("kind,cols", [("tiles", 520), ("small", 520), ("small complex", 260)])
def test_width_limit_on_every_route(eng, kind, cols):
    """CSR operators take at most 256 16-byte column vectors (512 FP64 columns) whichever
    kernel would run, and refuse more without touching the block."""
    from rayleighchebyshevgpgpu_amd import solver as rcg
    print(f"case: width limit, {kind}", flush=True)
    grid = (20, 20, 20) if kind == "tiles" else (10, 10, 10)
    A = ops.hofstadter_2d(32, phi=1.0 / 8, W=1.0) if "complex" in kind else \
        ops.laplacian_3d(*grid, "dirichlet", ops.anderson_potential(int(np.prod(grid)), 3.0, 1))
    op = rcg.CsrOperator(A)
    dt = np.complex128 if A.is_complex else np.float64
    bx, bt = rcg.Block(A.n, cols, dtype=dt), rcg.Block(A.n, cols, dtype=dt)
    bx.randomize(0, cols, 1, 0)
    X = bx.download()
    th, rz = np.zeros(cols), np.ones(cols, dtype=np.int32)
    assert eng.rcg_cheb_filter(op.h, bx.h, bt.h, cols, 8, 1, 14.0, 1.0) == 6
    assert eng.rcg_cheb_filter_mixed(op.h, bx.h, bt.h, cols, 8, 1, 14.0, 1.0,
                                     th.ctypes.data_as(C.c_void_p), rz.ctypes.data_as(C.c_void_p)) == 6
    assert eng.rcg_operator_apply(op.h, bx.h, bt.h, 1.0, 0.0, cols) == 6
    assert np.array_equal(bx.download(), X)
    most = 256 if A.is_complex else 512
    capi.check(eng.rcg_cheb_filter(op.h, bx.h, bt.h, most, 8, 1, 14.0, 1.0))
    assert np.array_equal(bx.download()[:, most:], X[:, most:])


@pytest.mark.parametrize("grid,cx,cases", [
    ((512, 512, 1), False, {24: 0, 64: 0, 72: 1}), ((1024, 1024, 1), False, {24: 0, 36: 1, 64: 1}),
    ((64, 64, 64), False, {24: 0, 64: 0, 72: 1}), ((100, 100, 100), False, {24: 1, 36: 0, 48: 1}),
    ((512, 512, 1), True, {48: 0, 64: 0, 80: 1})])
def test_products_over_tiles_where_faster(eng, grid, cx, cases):
    """A product takes tiles at fewer sizes than the filter's steps do, and has the same
    bits either way."""
    from rayleighchebyshevgpgpu_amd import solver as rcg
    print(f"case: products on {grid}", flush=True)
    n = int(np.prod(grid))
    A = operator(grid, True) if cx else ops.laplacian_2d(*grid[:2]) if grid[2] == 1 else \
        ops.laplacian_3d(*grid)
    op, rows = rcg.CsrOperator(A, grid=grid), rcg.CsrOperator(A, grid=(n, 1, 1))
    for cols, want in cases.items():
        got = C.c_int32(-1)
        capi.check(eng.test_apply_tiles(op.h, C.c_int64(cols), C.byref(got)))
        assert got.value == want, cols
    dt = np.complex128 if cx else np.float64
    bx, by, bz = (rcg.Block(n, cols, dtype=dt) for _ in range(3))
    bx.randomize(0, cols, 1, 0)
    op.apply(bx, by)
    rows.apply(bx, bz)
    assert np.array_equal(by.download(), bz.download())
