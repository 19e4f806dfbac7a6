"""The neighbour search over cells against the oracle's exhaustive search, bit
for bit: clustered points at the edges of the search's operand widths, group
and cell sizes, with rare clusters, duplicates and points far off."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _points(n, d, groups, seed, spread=8.0, dup=0):
    rng = np.random.default_rng(seed)
    centre = rng.normal(0, spread, (groups, d))
    lab = np.minimum(rng.geometric(2.0 / groups, n) - 1, groups - 1)  # uneven, some rare
    X = (centre[lab] + rng.normal(0, 1.0, (n, d))).astype(np.float32)
    if dup:
        X[rng.integers(0, n, dup)] = X[rng.integers(0, n, dup)]
    return np.asfortranarray(X)


@pytest.mark.parametrize("include_self", [True, False])
@pytest.mark.parametrize("n,d,k,groups,dup",
                         [(4096, 20, 10, 12, 0), (4097, 21, 5, 7, 200), (6001, 31, 24, 20, 0),
                          (9000, 41, 30, 9, 0), (5000, 52, 20, 30, 500), (4999, 63, 1, 5, 0),
                          (12345, 50, 20, 40, 0), (7000, 3, 15, 6, 0)])
def test_cells_bit_exact(sev, orc, n, d, k, groups, dup, include_self):
    X = _points(n, d, groups, seed=n + d, dup=dup)
    ridx, rdist = orc.knn(X, k, include_self=include_self)
    for precision in ("fp32", "bf16"):
        idx, dist = sev.ann(X, k, include_self=include_self, precision=precision)
        assert np.array_equal(idx, ridx), precision
        assert np.array_equal(dist, rdist), precision


@pytest.mark.parametrize("include_self", [True, False])
@pytest.mark.parametrize("n,d,k,spread", [(18001, 4, 10, 8.0), (12000, 51, 15, 1e-3),
                                          (12100, 50, 30, 1e6)])
def test_cells_fp64_bit_exact(sev, orc, n, d, k, spread, include_self):
    """FP64 points, among them clusters so tight or so far from the origin
    that their FP32 roundings coincide (those rows are searched exhaustively)."""
    rng = np.random.default_rng(n)
    X = np.asfortranarray(_points(n, d, 15, seed=k, spread=spread).astype(np.float64) +
                          rng.normal(0, 1e-3, (n, d)))
    idx, dist = sev.ann(X, k, include_self=include_self)
    ridx, rdist = orc.knn(X, k, include_self=include_self)
    assert np.array_equal(idx, ridx) and np.array_equal(dist, rdist)


def test_cells_degenerate(sev, orc):
    """Identical points, one point far from all others, all-zero columns."""
    X = _points(5000, 12, 4, seed=3)
    X[:3000] = X[0]
    X[4999] = 1e4
    X[:, 5] = 0.0
    idx, dist = sev.ann(X, 15, precision="fp32")
    ridx, rdist = orc.knn(X, 15)
    assert np.array_equal(idx, ridx) and np.array_equal(dist, rdist)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n,d,k", [(70, 5, 63), (65, 2, 64), (255, 7, 20), (257, 50, 1),
                                   (4095, 9, 30), (4400, 17, 12)])
def test_exhaustive_head_bound(sev, orc, dtype, n, d, k):
    """The exhaustive search at the edges of its tiles and of the head sweep
    that bounds the k-th neighbour, with many equal distances."""
    X = _points(n, d, 3, seed=n + k, dup=n // 3).astype(dtype)
    X[: n // 4] = np.round(X[: n // 4])
    for include_self in (True, False):
        kk = min(k, n if include_self else n - 1)
        idx, dist = sev.ann(np.asfortranarray(X), kk, include_self=include_self,
                            precision="exact")
        ridx, rdist = orc.knn(np.asfortranarray(X), kk, include_self=include_self)
        assert np.array_equal(idx, ridx) and np.array_equal(dist, rdist)


@pytest.mark.parametrize("scale", [1e-18, 3e-19])
@pytest.mark.parametrize("precision", ["fp32", "bf16"])
def test_cells_tiny_values(sev, orc, precision, scale):
    """Coordinates so small that the operands' scale stops at 2^60: the parts of
    the norms that are taken as zero then weigh as much as the gaps between
    neighbours, and rows must not be certified on them."""
    rng = np.random.default_rng(17)
    n, d = 12500, 20
    X = rng.normal(0, 0.3, (12, d))[rng.integers(0, 12, n)] + rng.normal(0, 0.02, (n, d))
    X = np.asfortranarray((X * scale).astype(np.float32))
    idx, dist = sev.ann(X, 10, precision=precision)
    ridx, rdist = orc.knn(X, 10)
    assert np.array_equal(idx, ridx) and np.array_equal(dist, rdist)


def test_cells_wide_rows_left(sev, orc):
    """FP32, 52 <= d <= 63 and k > 24: no matrix-core lists exist for the rows
    that the cells leave without a certificate (among them a block of points
    with more equal distances than a list holds), and only those rows are
    searched exhaustively."""
    n, d, k = 12500, 55, 30
    X = _points(n, d, 20, seed=55)
    X[100:200] = X[100]
    idx, dist, left = sev.ann(X, k, return_fallback=True)
    ridx, rdist = orc.knn(X, k)
    assert np.array_equal(idx, ridx) and np.array_equal(dist, rdist)
    assert 100 <= left < n // 2
