"""A caller's apply that itself calls this library on the same context, with blocks of
its own (a projector or a preconditioner beside the product): the solve keeps nothing
in the context's scratch over the call, so it gives the same bits as with an apply
that does not."""
import ctypes as C

import numpy as np
import pytest

from rayleighchebyshevgpgpu_amd import capi
from tests.test_gpu_callback import rcg, stencils  # noqa: F401 (fixtures)
from rayleighchebyshevgpgpu_amd import operators as ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,k,inc,buf", [(10, 8, 8, 8), (12, 20, 20, 20), (64, 8, 8, 8)])
def test_library_calls_inside_apply(rcg, stencils, L, k, inc, buf):  # noqa: F811
    """Blocks whose first factor is made on the device, on the host, and by the product
    that leaves the next Gram matrix (2^22 entries)."""
    print(f"case: reentrant apply, {L}^3, k={k} inc={inc} buf={buf}", flush=True)
    n = L ** 3
    diag = np.ascontiguousarray(6.0 + ops.anderson_potential(n, 4.0, 1))
    user = stencils.anderson3d_create(L, diag.ctypes.data)
    assert user
    mine, tmp = rcg.Block(4096, inc + buf), rcg.Block(4096, inc + buf)
    calls = [0]
    mat = np.asfortranarray(np.full((inc + buf, inc + buf), 0.5) + np.eye(inc + buf))
    turn = mat.ctypes.data_as(C.c_void_p)

    def solve(inner):
        def apply(pin, pout, n, cols, ld, alpha, beta, stream):
            if inner:
                calls[0] += 1
                mine.randomize(0, inc + buf, calls[0], 0)
                capi.check(capi.lib().rcg_rotate(mine.h, tmp.h, inc + buf, turn))
                capi.check(capi.lib().rcg_orthonormalize(mine.h, tmp.h, inc + buf))
            if stencils.anderson3d_apply(user, pin, pout, n, cols, ld, alpha, beta, stream) != 0:
                raise RuntimeError("stencil apply failed")

        op = rcg.CallbackOperator(n, apply)
        rc = rcg.RayleighChebyshevLM()
        rc.setStopCondition("RESIDUAL_ONLY")
        V, ev = rcg.Block(n, max(k, inc + buf)), []
        found = rc.getMinEigenSystem(k, 1e-7, inc, buf, None, op, rcg.RandomizeOp(0), ev, V)
        return found, np.array(ev), V.download(found)

    plain, nested = solve(False), solve(True)
    stencils.anderson3d_destroy(user)
    assert calls[0] > 0
    assert plain[0] == nested[0] >= k
    assert np.array_equal(plain[1], nested[1]) and np.array_equal(plain[2], nested[2])
