"""The panel steps of the LU at the sizes where they change: tournament sets of
256 and 512 rows, one to three levels, remainders of every blocking, and pivot
orders whose swaps chain through the top rows."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = 2.2e-16


def _matrix(n, kind):
    rs = np.random.RandomState(n)
    if kind == "random":
        return rs.randn(n, n) + 1j * rs.randn(n, n)
    Z = 0.01 * (rs.randn(n, n) + 1j * rs.randn(n, n)) / np.sqrt(n)
    p = np.arange(n)
    if kind == "reversed":  # every pivot far below, top rows displaced once
        p = p[::-1]
    elif kind == "cycle":   # the pivots of a step are top rows of the same step
        b = n // 32 * 32
        p[:b] = np.concatenate([np.roll(np.arange(s, s + 32), 5) for s in range(0, b, 32)])
    elif kind == "shuffle":
        p = rs.permutation(n)
    Z[np.arange(n), p] += 1.0
    return Z


@pytest.mark.parametrize("n,kind", [(31, "random"), (250, "cycle"), (257, "reversed"), (480, "shuffle"), (513, "random"),
                                    (545, "cycle"), (800, "reversed"), (2049, "shuffle"), (2305, "random")])
def test_fp64_factors(bem, n, kind):
    print(f"FP64 factors n={n} {kind}", flush=True)
    Z = _matrix(n, kind)
    with bem.Context(0) as ctx:
        ctx.set_Z(Z)
        assert ctx.factor("fp64") == 0
        LU, ip = ctx.get_lu(n), ctx.get_pivots(n)
    perm = np.arange(n)
    for i, q in enumerate(ip - 1):
        perm[[i, q]] = perm[[q, i]]
    L, U = np.tril(LU, -1) + np.eye(n), np.triu(LU)
    # Gaussian elimination: |PZ - LU| <= n eps |L||U| elementwise (Higham, Theorem 9.3, gamma_n)
    err = np.abs(Z[perm] - L @ U)
    assert (err <= 2 * n * EPS * (np.abs(L) @ np.abs(U))).all()
    # a tournament's multipliers are bounded by those of partial pivoting over a few levels
    assert np.abs(L).max() < 8


@pytest.mark.parametrize("n,kind", [(250, "cycle"), (513, "reversed"), (1056, "shuffle"), (2080, "random"),
                                    (4100, "shuffle"), (4400, "reversed")])
def test_fp32_refined(bem, n, kind):
    print(f"FP32 + refinement n={n} {kind}", flush=True)
    Z = _matrix(n, kind)
    rs = np.random.RandomState(1)
    B = rs.randn(n, 3) + 1j * rs.randn(n, 3)
    with bem.Context(0) as ctx:
        ctx.set_Z(Z)
        assert ctx.factor("fp32") == 0
        assert sorted(np.unique(ctx.get_pivots(n))) and ctx.get_pivots(n).min() >= 1
        X, st = ctx.solve(B, ir_tol=1e-11, ir_max=30)
    assert st["converged"] == 1
    assert (np.linalg.norm(Z @ X - B, axis=0) <= 1.5e-11 * np.linalg.norm(B, axis=0)).all()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n,col", [(40, 7), (300, 7), (300, 280), (2100, 40), (2305, 2300)])
def test_zero_column(bem, n, col, precision):
    """A zero column takes the lowest open row: info names it and no pivot
    leaves the matrix (its padding has rows of zeros there too)."""
    print(f"zero column {col} of {n}, {precision}", flush=True)
    Z = _matrix(n, "random")
    Z[:, col] = 0
    with bem.Context(0) as ctx:
        ctx.set_Z(Z)
        assert ctx.factor(precision) == col + 1
        ip = ctx.get_pivots(n)
    assert (ip >= np.arange(1, n + 1)).all() and ip.max() <= n
