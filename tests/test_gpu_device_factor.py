"""Solves whose first CholQR pass factors on the device (real blocks of at most 32
columns): every width class against the oracle, and blocks whose Gram matrix does
not factor, which must fall back to the shifted host passes.

Tolerances as for every solve: eigenvalues within 1e-10 with the reference's
floor, orthonormal vectors to 1e-9 (residual tolerance over the gaps).
"""
import numpy as np
import pytest

from rayleighchebyshevgpgpu_amd import operators as ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("inc,buf,side", [(1, 1, 9), (8, 8, 11), (9, 8, 12), (16, 8, 13),
                                          (17, 8, 14), (24, 8, 16), (24, 9, 15)])
def test_widths(orc, inc, buf, side):
    from rayleighchebyshevgpgpu_amd import solver as rcg
    n = side ** 3
    A = ops.laplacian_3d(side, bc="dirichlet", potential=ops.anderson_potential(n, 4.0, side))
    rc = rcg.RayleighChebyshevLM()
    rc.setStopCondition("RESIDUAL_ONLY")
    V, ev = rcg.Block(n, inc + buf), []
    f = rc.getMinEigenSystem(inc, 1e-10, inc, buf, None, rcg.CsrOperator(A), rcg.RandomizeOp(0), ev, V)
    ref = orc.solve(A, inc, 1e-10, inc, buf, seed=0, stop="RESIDUAL_ONLY")
    assert f == ref["found"]
    ev, want = np.array(ev), ref["eigenvalues"]
    assert np.max(np.abs(ev - want) / np.maximum(np.abs(want), 0.1)) < 1e-10
    X = V.download(f)
    assert np.max(np.abs(X.T @ X - np.eye(f))) < 1e-9


def test_dependent_start_columns():
    """A start block with repeated columns: its Gram matrix is singular."""
    from rayleighchebyshevgpgpu_amd import solver as rcg
    n = 12 ** 3
    A = ops.laplacian_3d(12, bc="dirichlet", potential=ops.anderson_potential(n, 4.0, 3))
    want = np.linalg.eigvalsh(A.to_scipy().toarray())[:6]
    x = np.random.default_rng(0).standard_normal((n, 1))
    rc = rcg.RayleighChebyshevLM()
    rc.setStopCondition("RESIDUAL_ONLY")
    rc.setNonRandomStartFlag(True)
    V = rcg.Block(n, 12)
    V.upload(np.repeat(x, 12, axis=1) * (1 + 1e-13 * np.arange(12)))
    V.valid_cols = 12
    ev = []
    try:
        f = rc.getMinEigenSystem(6, 1e-8, 6, 6, None, rcg.CsrOperator(A), rcg.RandomizeOp(0), ev, V)
    except rcg.capi.RcgError as e:  # a block of rank one may be refused, with the reason
        assert "rank" in str(e) or "CholQR" in str(e)
        return
    assert f == 6 and np.max(np.abs(np.array(ev) - want)) < 1e-6
