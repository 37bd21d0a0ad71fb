"""Host matrices into the padded device planes and back: both orders, edges of the
32 x 32 tiles, and matrices of more than one staging chunk.  Copies: bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _values(shape):
    rs = np.random.RandomState(shape[0])
    Z = rs.randn(*shape) + 1j * rs.randn(*shape)
    Z.flat[:: 7] *= 1e-310  # denormals
    Z.flat[0] = complex(-0.0, np.inf)
    return Z


@pytest.mark.parametrize("n", [1, 31, 33, 255, 257, 1500])
def test_matrix_round_trip(bem, n):
    print(f"matrix n={n}", flush=True)
    Z = _values((n, n))
    with bem.Context(0) as ctx:
        for order_in in (1, 0):
            ctx._check(ctx._L.bem_set_Z(ctx._h, bem._p(Z), n, order_in), "set_Z")
            for order_out in (1, 0):
                got = np.full((n, n), 7.0 + 7.0j)
                ctx._check(ctx._L.bem_get_Z(ctx._h, bem._p(got), order_out), "get_Z")
                np.testing.assert_array_equal(got, Z if order_in == order_out else Z.T)
        ip = np.arange(1, n + 1, dtype=np.int32)
        ctx.set_lu(Z, ip)
        np.testing.assert_array_equal(ctx.get_lu(n), Z)


@pytest.mark.parametrize("n,nrhs", [(1, 1), (33, 31), (257, 17), (1500, 1500)])
def test_identity_solve_returns_the_right_hand_sides(bem, n, nrhs):
    print(f"right-hand sides {n} x {nrhs}", flush=True)
    rs = np.random.RandomState(n)
    B = rs.randn(n, nrhs) + 1j * rs.randn(n, nrhs)
    with bem.Context(0) as ctx:
        ctx.set_Z(np.eye(n, dtype=np.complex128))  # the padding has to be the identity, too
        assert ctx.factor("fp64") == 0
        X, _ = ctx.solve(B, ir_tol=0.0, ir_max=0)
    np.testing.assert_array_equal(X, B)
