"""The unrefined FP32 solve on meshes whose triangles differ much in size (poles
of a latitude-longitude surface): its residual is that of the same
solve in numpy, single precision, with block inverses by substitution, within
a small factor."""
import numpy as np
import pytest
import scipy.linalg as sla

import test_precond_blocks_gpu as blocks

pytestmark = pytest.mark.gpu


def _block_inverse_solve(Z, B, nb=256):
    """LU, the nb x nb diagonal blocks inverted by substitution, all in complex64."""
    n = len(Z)
    lu, piv = sla.lu_factor(Z.astype(np.complex64))
    x = B.astype(np.complex64)
    for i, p in enumerate(piv):
        x[[i, p]] = x[[p, i]]
    starts = range(0, n, nb)
    for lower in (True, False):
        for s in starts if lower else reversed(starts):
            e = min(s + nb, n)
            inv = sla.solve_triangular(lu[s:e, s:e], np.eye(e - s, dtype=np.complex64), lower=lower, unit_diagonal=lower)
            x[s:e] = inv @ x[s:e]
            rest = slice(e, n) if lower else slice(0, s)
            x[rest] -= lu[rest, s:e] @ x[s:e]
    return x.astype(complex)


@pytest.mark.parametrize("nlat,nlon", [(12, 11), (14, 37), (24, 30)])
def test_first_residual(bem, nlat, nlon):
    v, t = blocks._cylinder(nlat, nlon)
    with bem.Context(0) as ctx:
        N = ctx.set_mesh(v, t, 4)
        n = 2 * N
        print(f"FP32 solve of {n} unknowns", flush=True)
        ctx.assemble(2.0 + 0j, 3.0 + 0.01j, 1.0, 1 / 1.5)
        Z = ctx.get_Z()
        rs = np.random.RandomState(n)
        B = Z @ (rs.randn(n, 4) + 1j * rs.randn(n, 4))
        assert ctx.factor("fp32") == 0
        X, _ = ctx.solve(B, ir_tol=1.0, ir_max=0)
    ref = _block_inverse_solve(Z, B)
    res = lambda x: (np.linalg.norm(B - Z @ x, axis=0) / np.linalg.norm(B, axis=0)).max()
    # rounding of 3M products (a factor 2 on real ones) and tournament instead of partial pivoting (2)
    assert res(X) <= 4 * res(ref), (res(X), res(ref))
