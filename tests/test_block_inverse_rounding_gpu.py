"""Rounding of the FP32 block inverses, seen through an unrefined solve of an
upper triangular system with the identity on the right: X is the inverse.
Its 32 x 32 diagonal triangles are powers of two, inverted without rounding,
so all error comes from joining them, level by level."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U32 = 2.0**-24


def _upper(n, size, rs):
    U = np.triu(rs.randn(n, n) + 1j * rs.randn(n, n)) * size
    for d in range(0, n, 32):
        U[d:d + 32, d:d + 32] = 0
    U[np.arange(n), np.arange(n)] = 2.0 ** rs.randint(-1, 2, size=n) * 1j ** rs.randint(4, size=n)
    return U.astype(np.complex64).astype(complex)


def _inverse(U):
    """U^-1 by substitution in extended precision."""
    n, A = len(U), U.astype(np.clongdouble)
    X = np.zeros((n, n), np.clongdouble)
    for i in range(n - 1, -1, -1):
        X[i] = -(A[i, i + 1:] @ X[i + 1:])
        X[i, i] += 1
        X[i] /= A[i, i]
    return X.astype(complex)


def _join_error(U, X):
    """Bound of the joins' errors: X12 = -U11^-1 U12 X22 carries its own rounding
    and |U11^-1 U12| times the error of X22."""
    E = np.zeros(U.shape)
    h = 32
    while h < len(U):
        for d in range(0, len(U), 2 * h):
            a, b = slice(d, d + h), slice(d + h, d + 2 * h)
            E[a, b] = U32 * np.abs(X[a, b]) + np.abs(X[a, a] @ U[a, b]) @ E[b, b]
        h *= 2
    return E


@pytest.mark.parametrize("nblk", [1, 3])
@pytest.mark.parametrize("size", [0.05, 0.1, 0.3])
def test_joined_inverse_is_good_to_its_rounding(bem, size, nblk):
    n = 256 * nblk
    print(f"upper triangles, n={n}, entries of {size}", flush=True)
    rs = np.random.RandomState(int(100 * size) + nblk)
    blocks = [_upper(256, size, rs) for _ in range(nblk)]
    Z = np.zeros((n, n), complex)
    for p, U in enumerate(blocks):
        Z[256 * p:256 * (p + 1), 256 * p:256 * (p + 1)] = U
    with bem.Context(0) as ctx:
        ctx.set_Z(Z)
        assert ctx.factor("fp32") == 0
        assert np.array_equal(ctx.get_pivots(n), np.arange(1, n + 1))
        X, _ = ctx.solve(np.eye(n, dtype=complex), ir_tol=1.0, ir_max=0)
    for p, U in enumerate(blocks):
        s = slice(256 * p, 256 * (p + 1))
        exact = _inverse(U)
        # second-order terms a quarter; 3M products with the identity: X + X' - X, rounded to 3 u |X| at most
        assert (np.abs(X[s, s] - exact) <= 1.25 * _join_error(U, exact) + 4 * U32 * np.abs(exact)).all()
