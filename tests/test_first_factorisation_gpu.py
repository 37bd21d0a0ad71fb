"""The first FP32 factorisation of a size times no GEMM tiles: neither it nor the
solves take them.  The first FP64 one does and keeps the plan."""
import json

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_fp32_times_no_tiles(bem, tmp_path, monkeypatch):
    path = tmp_path / "plans.json"
    monkeypatch.setenv("BEM_TUNE_CACHE", str(path))
    monkeypatch.delenv("BEM_AUTOTUNE", raising=False)
    n, nrhs = 700, 361  # a size and column count that no other test has: no plan of this process fits
    rs = np.random.RandomState(6)
    Z = rs.randn(n, n) + 1j * rs.randn(n, n)
    B = rs.randn(n, nrhs) + 1j * rs.randn(n, nrhs)
    timed = {}
    for prec in ("fp32", "fp64"):
        print(f"first {prec} factorisation of n={n}, {nrhs} columns", flush=True)
        with bem.Context(0) as ctx:
            ctx.set_Z(Z)
            ctx.solve_gmres(B, tol=1e-1, max_iter=1, precond="none", allow_noconv=True)  # the columns
            assert ctx.factor(prec) == 0
            X, st = ctx.solve(B, ir_tol=1e-11, ir_max=10)
            assert st["converged"] == 1
        timed[prec] = path.exists() and [p["prec"] for p in json.loads(path.read_text())["plans"]]
    assert not timed["fp32"] and timed["fp64"] == [8]
