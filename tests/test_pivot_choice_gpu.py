"""The rows that the pivot tournament chooses: in the first 32 columns the rows
are shared out so that no column changes another's, with magnitudes that
differ by little, and the largest of each column has to be its pivot."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _shared_out(n, gap, seed):
    """Column j < 32 has the values 1 - gap * rank, turned by multiples of 90
    degrees, in the rows r = j mod 32; the other columns are random."""
    rs = np.random.RandomState(seed)
    Z = rs.randn(n, n) + 1j * rs.randn(n, n)
    Z[:, :32] = 0
    want = []
    for j in range(32):
        rows = np.arange(j, n, 32)
        rank = rs.permutation(len(rows))
        Z[rows, j] = (1 - gap * rank) * 1j ** rs.randint(4, size=len(rows))
        want.append(rows[rank == 0][0])
    return Z, np.array(want)


def _first_rows(ip, k):
    perm = np.arange(len(ip))
    for i, q in enumerate(ip - 1):
        perm[[i, q]] = perm[[q, i]]
    return perm[:k]


# sets of 256 and 512 rows, one to three levels, partial sets
@pytest.mark.parametrize("n", [64, 256, 300, 513, 1100, 2100, 4100])
# gaps the keys can tell: |x|^2 to 23 bits in FP32 (2 ulp of |x|^2 at least), to 20 in FP64
@pytest.mark.parametrize("precision,gap", [("fp32", 2.0**-21), ("fp64", 2.0**-19)])
def test_largest_of_near_ties(bem, n, precision, gap):
    print(f"near ties n={n} {precision}", flush=True)
    Z, want = _shared_out(n, gap, n)
    with bem.Context(0) as ctx:
        ctx.set_Z(Z)
        assert ctx.factor(precision) == 0
        ip = ctx.get_pivots(n)
    assert (ip >= np.arange(1, n + 1)).all() and ip.max() <= n
    assert (_first_rows(ip, 32) == want).all()
