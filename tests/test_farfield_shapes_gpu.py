"""Far field at the edges of its direction groups (64 per wave), odd numbers of
coefficient sets, odd point counts, absorbing media and phases on both sides
of the general reduction."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ndir,n_calls,order,k", [
    (1, 1, 7, 2.0 + 0j), (63, 2, 4, 3.0 + 0j), (64, 3, 7, 1.5 + 0.2j), (65, 5, 13, 2.0 + 0j), (128, 2, 7, 2.5 + 0j),
    (129, 1, 13, 40.0 + 0j), (181, 4, 7, 2.0 + 0.05j), (33, 2, 7, 3.0e5 + 0j), (5, 2, 7, 1.0e14 + 0j)])
def test_farfield_shapes(oracle, bem, ndir, n_calls, order, k):
    print(f"far field ndir={ndir} calls={n_calls} quadrature={order} k={k}", flush=True)
    p = oracle.Problem.from_shape("sphere", 1, quad_order=order)
    rs = np.random.RandomState(ndir)
    no = (n_calls + 1) // 2
    cJ, cM = (rs.randn(n_calls, p.N) + 1j * rs.randn(n_calls, p.N) for _ in range(2))
    rh = rs.randn(no, ndir, 3)
    rh /= np.linalg.norm(rh, axis=2, keepdims=True)
    with bem.Context(0) as ctx:
        ctx.set_mesh(p.verts, p.tris, order)
        F = ctx.farfield(cJ, cM, rh, k, 1.0, n_calls=n_calls, n_orient=no)
        F1 = ctx.farfield(cJ, cM, rh, k, 1.0, n_calls=n_calls, n_orient=no, noalloc=True)
    # each phase k rhat.x carries (a few) eps |k|; the terms add up in absolute
    # value to at most |k| / 2 pi * sum |coef| * (area of a half ~ 4 pi / N)
    eps = 2.2e-16
    scale = abs(k) / 2 * 4 / p.N * max(np.abs(cJ).sum(1).max(), np.abs(cM).sum(1).max()) * np.exp(k.imag)
    tol = 8 * eps * (10 + abs(k)) * scale
    for c in range(n_calls):
        Fo = p.farfield_vec(cJ[c], cM[c], k, 1.0, rh[c // 2])
        assert np.abs(F[c] - Fo).max() <= tol
        assert np.abs(F1[c] - Fo).max() <= tol
