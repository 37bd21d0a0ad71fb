"""The unrefined FP32 solve on meshes whose triangles differ much in size (poles
of a latitude-longitude surface): its residual is that of single-precision
LAPACK within a small factor, so the block inverses lose nothing."""
import numpy as np
import pytest
import scipy.linalg as sla

import test_precond_blocks_gpu as blocks

pytestmark = pytest.mark.gpu


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
    ref = sla.lu_solve(sla.lu_factor(Z.astype(np.complex64)), B.astype(np.complex64)).astype(complex)
    res = lambda x: (np.linalg.norm(B - Z @ x, axis=0) / np.linalg.norm(B, axis=0)).max()
    # rounding of 3M products (a factor 2 on real ones) and tournament instead of partial pivoting (2)
    assert res(X) <= 4 * res(ref), (res(X), res(ref))
