"""The neighbour search over cells against the oracle's exhaustive search, bit
for bit: clustered points at the edges of the search's operand widths, group
and cell sizes, with rare clusters, duplicates and points far off.  And which
search a shape takes, from the names of the regions that ran: the tests of one
search say that they reached it."""
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


def _search(sev, X, k, include_self=True, precision="fp32"):
    """Lists, rows searched exhaustively, and the regions of the search."""
    p = sev.Pipeline()
    p.set_embedding(X)
    p.profile(True)
    left = p.neighbours(k, include_self=include_self, precision=precision)
    idx, dist = p.get_neighbours(len(X))
    ran = {r for r in p.profile_read() if r.startswith("knn_")}
    p.close()
    return idx, dist, left, ran


# one operand width of each form: 3 d + 3 columns in two parts (64, 96, 128, 160,
# 192), d + 3 in one (32, 64, 96)
@pytest.mark.parametrize("include_self", [True, False])
@pytest.mark.parametrize("n,d,k,groups,dup",
                         [(18000, 20, 10, 12, 0), (18001, 21, 5, 7, 200), (15200, 31, 20, 20, 0),
                          (19500, 32, 24, 9, 0), (17600, 41, 30, 9, 0), (13500, 42, 21, 12, 0),
                          (12345, 50, 20, 40, 0), (12200, 52, 20, 30, 500), (11300, 63, 1, 5, 0),
                          (13001, 62, 20, 10, 0), (29000, 3, 15, 6, 0)])
def test_cells_bit_exact(sev, orc, n, d, k, groups, dup, include_self):
    X = _points(n, d, groups, seed=n + d, dup=dup)
    ridx, rdist = orc.knn(X, k, include_self=include_self)
    for precision in ("fp32", "bf16"):
        idx, dist, _, ran = _search(sev, X, k, include_self, precision)
        assert "knn_cell" in ran
        assert np.array_equal(idx, ridx), precision
        assert np.array_equal(dist, rdist), precision


@pytest.mark.parametrize("include_self", [True, False])
@pytest.mark.parametrize("n,d,k,spread", [(26700, 4, 10, 8.0), (12100, 51, 15, 8.0),
                                          (12100, 51, 15, 1e-3), (15300, 50, 30, 1e6)])
def test_cells_fp64_bit_exact(sev, orc, n, d, k, spread, include_self):
    """FP64 points, among them clusters so tight or so far from the origin
    that their FP32 roundings coincide (those rows are searched exhaustively)."""
    rng = np.random.default_rng(n)
    X = np.asfortranarray(_points(n, d, 15, seed=k, spread=spread).astype(np.float64) +
                          rng.normal(0, 1e-3, (n, d)))
    idx, dist, left = sev.ann(X, k, include_self=include_self, return_fallback=True)
    ridx, rdist = orc.knn(X, k, include_self=include_self)
    assert np.array_equal(idx, ridx) and np.array_equal(dist, rdist)
    if spread == 8.0:
        assert left < n // 10  # by cells


@pytest.mark.parametrize("precision", ["fp32", "bf16"])
def test_cells_degenerate(sev, orc, precision):
    """Identical points, one point far from all others, all-zero columns."""
    n = 21100
    X = _points(n, 12, 4, seed=3)
    X[:3000] = X[0]
    X[n - 1] = 1e4
    X[:, 5] = 0.0
    idx, dist, left, ran = _search(sev, X, 15, precision=precision)
    ridx, rdist = orc.knn(X, 15)
    assert np.array_equal(idx, ridx) and np.array_equal(dist, rdist)
    assert "knn_cell" in ran and left >= 3000


@pytest.mark.parametrize("include_self", [True, False])
@pytest.mark.parametrize("n,d,k", [(13500, 42, 15), (19500, 32, 24), (18000, 40, 28),
                                   (11900, 60, 10)])
def test_cells_rows_left(sev, orc, n, d, k, include_self):
    """Rows that the cells leave without a certificate (blocks of 50 points with
    equal distances, which shorter lists than the cells' cannot hold either, and
    of 200, which none can) go on through the lists over all points for those
    rows, then the exhaustive search."""
    X = _points(n, d, 12, seed=n)
    X[100:150] = X[100]
    X[400:600] = X[400]
    ridx, rdist = orc.knn(X, k, include_self=include_self)
    for precision in ("fp32", "bf16"):
        idx, dist, left, ran = _search(sev, X, k, include_self, precision)
        assert np.array_equal(idx, ridx) and np.array_equal(dist, rdist)
        assert {"knn_cell", "knn_cand_fp32", "knn_exact"} <= ran
        assert precision == "fp32" or any(r.startswith("knn_cand_bf16") for r in ran)
        assert 200 <= left < n // 4


@pytest.mark.parametrize("precision,offset", [("fp32", 300.0), ("bf16", 3000.0), ("fp32", -2e4),
                                              ("fp64", 1e6)])
def test_cells_far_from_the_origin(sev, orc, precision, offset):
    """Points far from the origin compared with their distances: the operands
    are taken around their centre, so rows keep their certificates."""
    n, d, k = 13000, 48, 15
    X = _points(n, d, 12, seed=48).astype(np.float64 if precision == "fp64" else np.float32)
    X[:, ::2] += X.dtype.type(offset)
    if precision == "fp64":
        idx, dist, left = sev.ann(X, k, return_fallback=True)
    else:
        idx, dist, left, ran = _search(sev, X, k, precision=precision)
        assert "knn_cell" in ran
    ridx, rdist = orc.knn(X, k)
    assert np.array_equal(idx, ridx) and np.array_equal(dist, rdist)
    assert left < n // 100


# both sides of the lines between the searches, for points in groups and without
@pytest.mark.parametrize("n,d,k,precision,grouped,want",
                         [(12300, 50, 20, "fp32", True, "exhaustive"),
                          (12400, 50, 20, "fp32", True, "cells"),
                          (12400, 50, 20, "fp32", False, "cells"),
                          (12300, 50, 20, "bf16", True, "exhaustive"),
                          (12400, 50, 20, "bf16", True, "cells"),
                          (12400, 50, 20, "bf16", False, "lists"),
                          (16000, 50, 24, "fp32", True, "exhaustive"),
                          (16200, 50, 24, "fp32", True, "cells"),
                          (16200, 60, 30, "fp32", True, "exhaustive"),
                          (16400, 60, 30, "fp32", True, "cells"),
                          (30000, 51, 40, "fp32", False, "exhaustive"),
                          (30001, 51, 40, "fp32", False, "lists"),
                          (30001, 51, 40, "bf16", True, "lists"),
                          (25000, 51, 45, "bf16", False, "lists"),
                          (25000, 40, 45, "bf16", False, "exhaustive"),
                          (25000, 51, 60, "bf16", False, "exhaustive"),
                          (19900, 100, 15, "fp32", False, "exhaustive"),
                          (20100, 100, 15, "fp32", False, "lists"),
                          (11000, 126, 15, "bf16", False, "exhaustive"),
                          (11200, 126, 15, "bf16", True, "lists"),
                          (40000, 70, 30, "fp32", True, "exhaustive")])
def test_search_of_a_shape(sev, n, d, k, precision, grouped, want):
    rng = np.random.default_rng(n)
    X = _points(n, d, 9, seed=1) if grouped else rng.standard_normal((n, d)).astype(np.float32)
    _, _, left, ran = _search(sev, np.asfortranarray(X), k, precision=precision)
    if want == "exhaustive":
        assert ran == {"knn_exact"} and left == n
    elif want == "cells":
        assert "knn_cell" in ran and left < n
    else:
        assert "knn_cell" not in ran and any(r.startswith("knn_cand") for r in ran)


@pytest.mark.parametrize("n,d,k,cells", [(18000, 15, 15, False), (20011, 15, 15, True),
                                         (12100, 50, 20, False), (12200, 50, 20, True),
                                         (15200, 50, 24, False), (15300, 50, 24, True)])
def test_search_of_a_shape_fp64(sev, n, d, k, cells):
    X = np.asfortranarray(_points(n, d, 9, seed=2).astype(np.float64))
    assert (sev.ann(X, k, return_fallback=True)[2] < n) == cells


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
    n, d = 18000, 20
    X = rng.normal(0, 0.3, (12, d))[rng.integers(0, 12, n)] + rng.normal(0, 0.02, (n, d))
    X = np.asfortranarray((X * scale).astype(np.float32))
    idx, dist, _, ran = _search(sev, X, 10, precision=precision)
    ridx, rdist = orc.knn(X, 10)
    assert np.array_equal(idx, ridx) and np.array_equal(dist, rdist)
    assert "knn_cell" in ran


def test_cells_wide_rows_left(sev, orc):
    """FP32, 52 <= d <= 63 and k > 24: no matrix-core lists exist for the rows
    that the cells leave without a certificate (among them a block of points
    with more equal distances than a list holds), and only those rows are
    searched exhaustively."""
    n, d, k = 17500, 55, 30
    X = _points(n, d, 20, seed=55)
    X[100:200] = X[100]
    idx, dist, left, ran = _search(sev, X, k)
    ridx, rdist = orc.knn(X, k)
    assert np.array_equal(idx, ridx) and np.array_equal(dist, rdist)
    assert {"knn_cell", "knn_exact"} <= ran and 100 <= left < n // 2
