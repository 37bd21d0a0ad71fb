"""The FP32 solves and the FP64 residual of the refinement at the edges of their kernels:
one to several groups of one to five column tiles, one- and two-level solves, split and
unsplit sums, rows and columns of padding."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = 2.3e-16


@pytest.mark.parametrize("n,nrhs", [(1, 1), (250, 1), (257, 17), (300, 48), (700, 64), (513, 65), (1030, 129),
                                    (260, 209), (770, 1100), (8200, 17)])
def test_refinement_residual(bem, n, nrhs):
    print(f"residual n={n} nrhs={nrhs}", flush=True)
    rs = np.random.RandomState(n + nrhs)
    Z = rs.randn(n, n) + 1j * rs.randn(n, n) + 3 * np.sqrt(n) * np.eye(n)
    B = (rs.randn(n, nrhs) + 1j * rs.randn(n, nrhs)) * 10.0 ** rs.randint(-3, 4, nrhs)
    with bem.Context(0) as ctx:
        ctx.set_Z(Z)
        assert ctx.factor("fp32") == 0
        X0, st0 = ctx.solve(B, ir_tol=1.0, ir_max=0)
        X, st = ctx.solve(B, ir_tol=1e-13, ir_max=20)
    rel = lambda x: np.linalg.norm(B - Z @ x, axis=0) / np.linalg.norm(B, axis=0)
    # rounding of a residual of n-term sums in the 3M form: |Z||X| <= 4 sqrt(2) n / (3 sqrt(n)) |B| / sqrt(n) roughly
    noise = 8 * np.sqrt(n) * EPS
    assert abs(st0["residual"] - rel(X0).max()) <= noise
    assert st["converged"] and rel(X).max() <= 1e-13 + noise
