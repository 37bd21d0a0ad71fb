"""The unrefined FP32 solve at the sizes where the tournament's sets and levels
change: its residual is that of the same solve in numpy, single precision, with
block inverses by substitution, within the factor of its products and pivots."""
import numpy as np
import pytest

import test_fp32_inverses_gpu as inverses

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [33, 256, 257, 513, 800, 2060, 3840])
def test_residual(bem, n):
    print(f"unrefined FP32 solve n={n}", flush=True)
    rs = np.random.RandomState(n)
    Z = rs.randn(n, n) + 1j * rs.randn(n, n)
    B = rs.randn(n, 8) + 1j * rs.randn(n, 8)
    with bem.Context(0) as ctx:
        ctx.set_Z(Z)
        assert ctx.factor("fp32") == 0
        X, _ = ctx.solve(B, ir_tol=1.0, ir_max=0)
    ref = inverses._block_inverse_solve(Z, B)
    res = lambda x: np.linalg.norm(B - Z @ x) / np.linalg.norm(B)
    # rounding of 3M products (a factor 2 on real ones) and tournament instead of partial pivoting (2)
    assert res(X) <= 4 * res(ref), (res(X), res(ref))
    print(f"n={n}: {res(X) / res(ref):.2f} times numpy's residual")
