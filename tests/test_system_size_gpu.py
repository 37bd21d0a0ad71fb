"""A caller's own matrix (no mesh, or another size than the mesh's): the Python
front end sizes its buffers by the system on the device."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mesh", [False, True])
def test_buffers_fit_the_matrix(bem, mesh):
    n = 37
    print(f"own matrix of {n}, mesh {mesh}", flush=True)
    rs = np.random.RandomState(8)
    Z = rs.randn(n, n) + 1j * rs.randn(n, n)
    B = rs.randn(n, 3) + 1j * rs.randn(n, 3)
    with bem.Context(0) as ctx:
        if mesh:
            ctx.set_mesh(*bem.make_mesh("sphere", 0))
            ctx.assemble(1.0 + 0j, 1.3 + 0j, 1.0, 1 / 1.3)
            assert ctx.get_Z().shape == (60, 60)
        ctx.set_Z(Z)
        for bad in (B[:-1], np.vstack([B, B])):
            with pytest.raises(ValueError):
                ctx.solve_gmres(bad, precond="none")
        with pytest.raises(ValueError):
            ctx.set_Z(Z[:-1])
        assert np.array_equal(ctx.get_Z(), Z)
        assert ctx.factor("fp64") == 0
        X, _ = ctx.solve(B, ir_max=0)
        Y, _ = ctx.solve(None, ir_max=0, nrhs=3)  # the same columns from the device
        with pytest.raises(ValueError):
            ctx.solve(B[:-1])
    assert np.array_equal(X, Y) and np.linalg.norm(Z @ X - B) <= 1e-12 * np.linalg.norm(B)
