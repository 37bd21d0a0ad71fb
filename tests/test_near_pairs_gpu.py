"""Touching triangle pairs, one lane per test point and wavenumber: every quadrature
rule (4, 7 and 13 of 4, 8 and 16 lanes) in the matrix and in its derivatives."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("quad", [4, 7, 13])
@pytest.mark.parametrize("m", [1.3116 + 0.0j, 1.33 + 0.05j])
def test_touching_pairs(oracle, bem, quad, m):
    # the icosahedron: 20 triangles, all but the 20 x 2 farthest pairs touch
    print(f"near pairs quad={quad} m={m}", flush=True)
    prob = oracle.Problem.from_shape("sphere", 0, quad_order=quad)
    args = (1.5 + 0j, 1.5 * m, 1.0, 1.0 / abs(m))
    with bem.Context(0) as ctx:
        ctx.set_mesh(prob.verts, prob.tris, quad)
        ctx.assemble(*args)
        Z = ctx.get_Z()
    Zo = prob.assemble_pmchwt(*args)
    # FP64 pairs exactly, the far ones to the FP32 trigonometry (a few 6e-8 of the entry)
    assert np.abs(Z - Zo).max() <= 1e-6 * np.abs(Zo).max()


@pytest.mark.parametrize("quad", [4, 13])
def test_derivative_records(oracle, bem, quad):
    print(f"derivatives quad={quad}", flush=True)
    ka, m, nth = 1.5, 1.33 + 0.02j, 9
    prob = oracle.Problem.from_shape("sphere", 0, quad_order=quad)
    Gw = np.random.RandomState(quad).randn(16, nth)

    def loss(ka, m):
        return float(np.sum(Gw * prob.dense_orient(ka, m, 2, 1, 1, mirror=False, ntheta=nth)[1].reshape(16, nth)))

    h = 1e-5
    fd = np.array([(loss(ka + c, m + a + 1j * b) - loss(ka - c, m - a - 1j * b)) / (2 * h)
                   for a, b, c in [(h, 0, 0), (0, h, 0), (0, 0, h)]])
    with bem.Context(0) as ctx:
        ctx.set_mesh(prob.verts, prob.tris, quad)
        ctx.assemble(complex(ka), ka * m, 1.0, 1.0 / abs(m))
        RT, w = bem.orientations(2, 1, 1, mirror=False)
        kh, e0 = bem.planewave_orient_rhs(RT)
        ctx.rhs_planewave(ka, 1.0, kh, e0)
        assert ctx.factor("fp64") == 0
        ctx.solve(None, ir_tol=1e-12, ir_max=30, return_X=False, nrhs=len(kh))
        ctx.orient_mueller(ka, 1.0, RT, w, np.linspace(0, np.pi, nth), gamma_mirror=False)
        grad = ctx.mueller_grad(Gw.reshape(4, 4, nth))
    # central differences of step 1e-5: truncation h^2 and rounding 1e-13 / h are far below
    # the FP32 trigonometry of the far pairs
    assert np.abs(grad - fd).max() <= 1e-5 * np.abs(fd).max()
