"""FP32 tournaments with sets of 512 rows (8 waves): one set, several sets with
a merge of few rows, and the sizes around where they take over.  Block inverses
whose last panel has 2 mod 4 columns, for each number of rows per thread.  GMRES
whose transfer of an iteration is larger than the staging area."""
import numpy as np
import pytest

import test_precond_blocks_gpu as blocks

pytestmark = pytest.mark.gpu

U32 = 6e-8


@pytest.mark.parametrize("n", [256, 257, 300, 512, 513, 2048, 2060, 2500, 3840, 4096, 4100])
def test_fp32_factors(bem, n):
    print(f"FP32 factors n={n}", flush=True)
    rs = np.random.RandomState(n)
    Z = rs.randn(n, n) + 1j * rs.randn(n, n)
    B = rs.randn(n, 5) + 1j * rs.randn(n, 5)
    with bem.Context(0) as ctx:
        ctx.set_Z(Z)
        assert ctx.factor("fp32") == 0
        piv = ctx.get_pivots(n)
        X, _ = ctx.solve(B, ir_tol=1.0, ir_max=0)
    assert (piv >= np.arange(1, n + 1)).all() and piv.max() <= n
    # backward error of Gaussian elimination with partial pivoting: gamma_n |L||U| / |Z|, rounding errors of
    # random sign (sqrt n of them) times the growth of |L||U| (sqrt n) at most
    be = np.linalg.norm(B - Z @ X, axis=0) / (np.linalg.norm(Z) * np.linalg.norm(X, axis=0))
    assert (be <= n * U32).all()


@pytest.mark.parametrize("nlat,nlon,cols", [(4, 3, 3), (10, 13, 17), (14, 17, 16), (16, 19, 5)])
def test_block_inverse_partial_window(bem, nlat, nlon, cols):
    blocks.test_one_block_is_the_inverse(bem, nlat, nlon, cols)


@pytest.mark.parametrize("nrhs", [3, 600, 800])
def test_gmres_many_columns(bem, nrhs):
    n = 300
    print(f"GMRES n={n}, {nrhs} columns", flush=True)
    rs = np.random.RandomState(3)
    Z = (rs.randn(n, n) + 1j * rs.randn(n, n)) / np.sqrt(2 * n) + 1.5 * np.eye(n)
    B = rs.randn(n, nrhs) + 1j * rs.randn(n, nrhs)
    with bem.Context(0) as ctx:
        ctx.set_Z(Z)
        X, st = ctx.solve_gmres(B, tol=1e-10, restart=100, max_iter=200, precond="none")
    # 4 k + 1 rows of products and norms come back in iteration k, 8 bytes a column: beyond 1 MiB from k = 41 on
    # for 800 columns
    assert st["converged"] == 1 and st["iterations"] > 41
    assert (np.linalg.norm(B - Z @ X, axis=0) <= 1.1e-10 * np.linalg.norm(B, axis=0)).all()
