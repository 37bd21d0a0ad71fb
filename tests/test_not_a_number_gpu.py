"""A solution that is not finite is never reported as converged: NaN in the
caller's right-hand sides or matrix, direct solves and GMRES.  Right-hand sides
whose squared norms overflow are still solved and measured."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 300


def _system(seed):
    rs = np.random.RandomState(seed)
    Z = rs.randn(N, N) + 1j * rs.randn(N, N) + 40 * np.eye(N)
    return Z, rs.randn(N, 3) + 1j * rs.randn(N, 3)


@pytest.mark.parametrize("column", [0, 2])
@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("how", ["fp32", "fp64", "gmres"])
def test_right_hand_side(bem, how, value, column):
    print(f"{value} in column {column}, {how}", flush=True)
    Z, B = _system(1)
    B[17, column] = value
    with bem.Context(0) as ctx:
        ctx.set_Z(Z)
        assert ctx.factor("fp64" if how == "fp64" else "fp32") == 0
        if how == "gmres":
            X, st = ctx.solve_gmres(B, tol=1e-10, restart=20, max_iter=40, allow_noconv=True)
        else:
            X, st = ctx.solve(B, ir_tol=1e-10, ir_max=10, allow_noconv=True)
        assert st["converged"] == 0 and not st["residual"] <= 1e-10, st
        with pytest.raises(bem.BemError):
            ctx.solve(B, ir_tol=1e-10, ir_max=10)
    if how == "gmres":  # the other columns are their own processes
        keep = [j for j in range(3) if j != column]
        assert (np.linalg.norm(B[:, keep] - Z @ X[:, keep], axis=0)
                <= 1.1e-10 * np.linalg.norm(B[:, keep], axis=0)).all()


@pytest.mark.parametrize("how", ["fp32", "fp64", "gmres"])
def test_matrix(bem, how):
    print(f"NaN in the matrix, {how}", flush=True)
    Z, B = _system(2)
    Z[200, 100] = np.nan
    with bem.Context(0) as ctx:
        ctx.set_Z(Z)
        ctx.factor("fp64" if how == "fp64" else "fp32")
        if how == "gmres":
            _, st = ctx.solve_gmres(B, tol=1e-10, restart=5, max_iter=10, allow_noconv=True, precond="none")
        else:
            _, st = ctx.solve(B, ir_tol=1e-10, ir_max=10, allow_noconv=True)
    assert st["converged"] == 0 and not st["residual"] <= 1e-10, st


@pytest.mark.parametrize("middle", [1.0, 2.0**600])
def test_squares_beyond_the_range(bem, middle):
    print(f"right-hand sides of 1e198, {middle:.0e} and 1e198, FP64", flush=True)
    Z, B = _system(3)
    with bem.Context(0) as ctx:
        ctx.set_Z(Z)
        assert ctx.factor("fp64") == 0
        ref, _ = ctx.solve(B, ir_tol=1e-13, ir_max=5)
        s = np.array([2.0**660, middle, 2.0**660])
        X, st = ctx.solve(B * s, ir_tol=1e-13, ir_max=5)
    # powers of two: the same solutions, bit for bit
    assert st["converged"] == 1 and 0.0 < st["residual"] <= 1e-13
    assert np.array_equal(X, ref * s)
