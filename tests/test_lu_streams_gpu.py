"""The factorisation's panel stream when a process holds several contexts: whichever
hardware queues their streams share, the factors are the same."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("before", [1, 3])
def test_factors_beside_other_contexts(bem, before):
    rs = np.random.RandomState(before)
    n = 2100  # the streams are looked at from 2048 padded unknowns on
    Z = rs.randn(n, n) + 1j * rs.randn(n, n)
    others = [bem.Context(0) for _ in range(before)]
    got = []
    try:
        for o in others:
            o.set_Z(Z[:40, :40])
            assert o.factor("fp32") == 0
        for _ in range(2):
            with bem.Context(0) as ctx:
                for _ in range(2):
                    ctx.set_Z(Z)
                    assert ctx.factor("fp64") == 0
                    got.append((ctx.get_lu(n), ctx.get_pivots(n)))
    finally:
        for o in others:
            o.close()
    for lu, ip in got[1:]:
        np.testing.assert_array_equal(ip, got[0][1])
        np.testing.assert_allclose(lu, got[0][0], rtol=0, atol=1e-12 * np.abs(got[0][0]).max())
