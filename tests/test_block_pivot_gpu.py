"""The block-Jacobi inverse takes the largest entry of a column as its pivot, to
the last bits: pairs of unknowns are coupled by [[s, 1], [b, 0]] with s just
below and b just above 1e-30, the modulus below which a pivot is replaced
(precond.cu:842-859)."""
import numpy as np
import pytest

import test_precond_blocks_gpu as blocks

pytestmark = pytest.mark.gpu


# 2N = 36 .. 1620: panels of one, two and three rows per thread and from memory
@pytest.mark.parametrize("nlat,nlon", [(3, 3), (5, 6), (9, 11), (14, 17), (16, 18)])
@pytest.mark.parametrize("gap", [2.0**-12, 2.0**-24, 2.0**-35, 2.0**-45])
def test_largest_entry(bem, nlat, nlon, gap):
    v, t = blocks._cylinder(nlat, nlon)
    with bem.Context(0) as ctx:
        N = ctx.set_mesh(v, t, 4)
        n = 2 * N
        print(f"block of {n} unknowns, gap {gap:.0e}", flush=True)
        ctx.assemble(1.0 + 0j, 1.3 + 0.1j, 1.0, 0.75, z32=False)
        rs = np.random.RandomState(n)
        Z, inv = np.eye(n, dtype=complex), np.eye(n, dtype=complex)
        s, b = 1e-30 * (1 - gap), 1e-30 * (1 + gap)
        pairs = rs.permutation(n)[:n // 2 * 2].reshape(-1, 2)
        for pq in pairs:
            f = 1j ** rs.randint(4, size=2)  # the rows turned by multiples of 90 degrees
            Z[np.ix_(pq, pq)] = np.array([[s, 1], [b, 0]]) * f[:, None]
            inv[np.ix_(pq, pq)] = np.array([[0, 1 / b], [1, -s / b]]) / f
        ctx.set_Z(Z)
        nb, _ = ctx.block_jacobi(1e3, N, 0)
        assert nb == 1
        cols = pairs[:20].ravel()
        X = ctx.precond_apply(np.eye(n, dtype=complex)[:, cols], "block")
    # a reciprocal by 1 / |b|^2 and a product: under 8 roundings; the zeros are exact
    assert np.allclose(X, inv[:, cols], rtol=8 * 2.2e-16, atol=0)
