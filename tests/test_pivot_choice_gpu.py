"""The rows that the pivot tournament chooses.  Near ties: in the first 32 columns the rows
are shared out so that no column changes another's, with magnitudes that
differ by little, and the largest of each column has to be its pivot.  FP32
entries whose squares leave the range: chosen and divided by as any others."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _shared_out(n, gap, seed):
    """Column j < 32 has the values 1.5 + gap * (8 - rank), turned by multiples of 90
    degrees, in the rows r = j mod 32; the other columns are random."""
    rs = np.random.RandomState(seed)
    Z = rs.randn(n, n) + 1j * rs.randn(n, n)
    Z[:, :32] = 0
    want = []
    for j in range(32):
        rows = np.arange(j, n, 32)
        rank = rs.permutation(len(rows))
        Z[rows, j] = (1.5 + gap * (8 - rank)) * 1j ** rs.randint(4, size=len(rows))
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


@pytest.mark.parametrize("n", [40, 300, 1100, 4100])
@pytest.mark.parametrize("scale", ["small", "large", "mixed"])
def test_fp32_columns_of_any_scale(bem, n, scale):
    """Columns times powers of two, squares of the entries beyond the FP32
    range: the same pivots, and the solution divided by them to the last bit.
    (Beyond 2^90 the corrections of the block inverses, 2^-24 of 2^-90 / |u|,
    leave the range themselves.)"""
    print(f"scaled columns n={n} {scale}", flush=True)
    rs = np.random.RandomState(n)
    Z = rs.randn(n, n) + 1j * rs.randn(n, n)
    B = rs.randn(n, 3) + 1j * rs.randn(n, 3)
    e = {"small": np.full(n, -90), "large": np.full(n, 90), "mixed": rs.randint(-90, 91, size=n)}[scale]
    d = 2.0 ** e.astype(float)
    with bem.Context(0) as ctx:
        ctx.set_Z(Z)
        assert ctx.factor("fp32") == 0
        ip = ctx.get_pivots(n)
        X, _ = ctx.solve(B, ir_tol=1.0, ir_max=0)
        ctx.set_Z(Z * d)
        assert ctx.factor("fp32") == 0
        ip2 = ctx.get_pivots(n)
        X2, _ = ctx.solve(B, ir_tol=1.0, ir_max=0)
    assert np.array_equal(ip, ip2)
    assert np.array_equal(X, X2 * d[:, None])


def test_fp32_small_entries_are_no_zeros(bem):
    """A column of zeros and one small entry takes the entry as its pivot."""
    n = 300
    print("small pivots, FP32", flush=True)
    rs = np.random.RandomState(4)
    Z = np.zeros((n, n), complex)
    p = rs.permutation(n)
    Z[p, np.arange(n)] = 1e-30 * (1 + 1j)
    B = rs.randn(n, 2) + 1j * rs.randn(n, 2)
    with bem.Context(0) as ctx:
        ctx.set_Z(Z)
        assert ctx.factor("fp32") == 0
        X, st = ctx.solve(1e-30 * B, ir_tol=1e-12, ir_max=10)
    assert st["converged"] == 1
    assert np.allclose(X, B[p] / (1 + 1j), rtol=1e-11, atol=0)
