"""Block inverses of the block-Jacobi preconditioner at the sizes where the
elimination's panels change shape: one block of the whole system (2N unknowns)
below and at one inner panel, within one outer panel, at the edges of the
panel kernel's rows per thread and beyond what its registers hold."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _cylinder(nlat, nlon):
    """Closed latitude-longitude surface with N = 3 nlon (nlat - 1) edges."""
    th = np.pi * np.arange(1, nlat) / nlat
    ph = 2 * np.pi * np.arange(nlon) / nlon
    s, z = np.sin(th)[:, None], np.cos(th)[:, None]
    v = np.concatenate([[(0, 0, 1.0)], np.stack([s * np.cos(ph), s * np.sin(ph), z + 0 * ph], 2).reshape(-1, 3),
                        [(0, 0, -1.0)]])
    f, last = [], len(v) - 1
    for j in range(nlon):
        k = (j + 1) % nlon
        f += [(0, 1 + j, 1 + k), (last, 1 + (nlat - 2) * nlon + k, 1 + (nlat - 2) * nlon + j)]
        for i in range(nlat - 2):
            p, q = 1 + i * nlon, 1 + (i + 1) * nlon
            f += [(p + j, q + j, q + k), (p + j, q + k, p + k)]
    return v, np.array(f, np.int32)


# (nlat, nlon): 2N = 6 nlon (nlat - 1)
@pytest.mark.parametrize("nlat,nlon,cols", [(3, 3, 1), (3, 5, 17), (5, 3, 33), (9, 10, 5), (9, 11, 70), (12, 16, 2),
                                            (14, 17, 2), (16, 18, 3)])
def test_one_block_is_the_inverse(bem, nlat, nlon, cols):
    v, t = _cylinder(nlat, nlon)
    with bem.Context(0) as ctx:
        N = ctx.set_mesh(v, t, 4)
        n = 2 * N
        print(f"block of {n} unknowns, {cols} columns", flush=True)
        ctx.assemble(1.0 + 0j, 1.3 + 0.1j, 1.0, 0.75, z32=False)
        rs = np.random.RandomState(n)
        # a random matrix whose large entries are off the diagonal: every step needs its pivot
        Z = (rs.randn(n, n) + 1j * rs.randn(n, n)) / np.sqrt(n)
        Z[np.arange(n), rs.permutation(n)] += 2.0
        ctx.set_Z(Z)
        nb, _ = ctx.block_jacobi(1e3, N, 0)
        assert nb == 1
        R = rs.randn(n, cols) + 1j * rs.randn(n, cols)
        X = ctx.precond_apply(R, "block")
    # numpy's relative residual bound for a stable inverse: n eps cond, cond < 20 here
    err = np.linalg.norm(X - np.linalg.solve(Z, R)) / np.linalg.norm(X)
    assert err < n * 2.2e-16 * 20 * 10
