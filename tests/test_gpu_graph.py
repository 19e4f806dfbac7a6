"""GPU parity: exact kNN and the Jaccard SNN graph against the oracle
(bit-exact indices, distances and weights)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("include_self", [True, False])
@pytest.mark.parametrize("n,d,k", [(1000, 10, 7), (3000, 50, 20), (257, 3, 64)])
def test_ann_exact(sev, orc, dtype, include_self, n, d, k):
    rng = np.random.default_rng(n + d)
    X = rng.standard_normal((n, d)).astype(dtype)
    idx, dist = sev.ann(X, k, include_self=include_self)
    ridx, rdist = orc.knn(X, k, include_self=include_self)
    assert np.array_equal(idx, ridx)
    assert np.array_equal(dist, rdist)


def test_ann_ties_and_duplicates(sev, orc):
    rng = np.random.default_rng(5)
    base = rng.random((300, 5)).astype(np.float32)
    X = np.concatenate([base, base, base[:100], np.zeros((5, 5), np.float32)])
    idx, dist = sev.ann(X, 6)
    ridx, rdist = orc.knn(X, 6)
    assert np.array_equal(idx, ridx) and np.array_equal(dist, rdist)


def test_find_neighbours_abi_strided(sev, orc):
    """FindNeighboursEuclidean32 with ld > n (a view of the leading rows)."""
    import ctypes
    rng = np.random.default_rng(6)
    full = np.asfortranarray(rng.standard_normal((700, 12)).astype(np.float32))
    n, d, k = 500, 12, 9
    idx = np.zeros((n, k), np.int32, order="F")
    dist = np.zeros((n, k), np.float32, order="F")
    L = sev.load()
    L.FindNeighboursEuclidean32(full.ctypes.data, n, d, 700, k, 24, 1, 123, idx.ctypes.data,
                                dist.ctypes.data)
    ridx, rdist = orc.knn(np.asfortranarray(full[:n]), k)
    assert np.array_equal(idx, ridx) and np.array_equal(dist, rdist)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("include_self", [True, False])
@pytest.mark.parametrize("precision", ["fp32", "bf16", "exact"])
def test_ann_cosine_exact(sev, orc, dtype, include_self, precision):
    """Cosine form (unit rows, D / 2) bit for bit against the oracle, with
    scaled copies of rows (distance 0 ties) and an all-zero row."""
    if dtype == np.float64 and precision == "bf16":
        pytest.skip("the BF16 candidate form is for Float32 points")
    rng = np.random.default_rng(21)
    base = rng.standard_normal((2500, 30)).astype(dtype)
    X = np.concatenate([base, 3.0 * base[:200], np.zeros((1, 30), dtype)])
    idx, dist = sev.ann(X, 12, include_self=include_self, precision=precision, metric="cosine")
    ridx, rdist = orc.knn_cosine(X, 12, include_self=include_self)
    assert np.array_equal(idx, ridx)
    assert np.array_equal(dist, rdist)


def test_find_neighbours_cosine_abi(sev, orc):
    """FindNeighboursCosine32/64 with ld > n (libcell's signature)."""
    rng = np.random.default_rng(22)
    for dt, name in ((np.float32, "FindNeighboursCosine32"), (np.float64, "FindNeighboursCosine64")):
        full = np.asfortranarray(rng.standard_normal((900, 16)).astype(dt))
        n, d, k = 700, 16, 10
        idx = np.zeros((n, k), np.int32, order="F")
        dist = np.zeros((n, k), dt, order="F")
        getattr(sev.load(), name)(full.ctypes.data, n, d, 900, k, 32, 0, 7, idx.ctypes.data,
                                  dist.ctypes.data)
        ridx, rdist = orc.knn_cosine(np.asfortranarray(full[:n]), k, include_self=False)
        assert np.array_equal(idx, ridx) and np.array_equal(dist, rdist), name


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("k,prune", [(20, 1 / 15), (15, 1 / 15), (30, 1 / 15), (10, 0.0)])
def test_snn_vs_oracle(sev, orc, dt, k, prune):
    rng = np.random.default_rng(k)
    X = rng.standard_normal((4000, 10)).astype(np.float32)
    idx, _ = orc.knn(X, k)
    S = sev.api._snn_from_index(idx, k, prune, dt)
    cp, rv, nz = orc.snn(idx, k, prune, dt)
    assert np.array_equal(S.indptr, cp - 1) and np.array_equal(S.indices, rv - 1)
    assert S.data.dtype == dt and np.array_equal(S.data, nz)


def test_snn_hub_columns(sev, orc):
    """A few hubs that many cells list force the block and global-table
    paths (candidate unions above the wavefront table)."""
    rng = np.random.default_rng(9)
    n, k = 6000, 20
    idx = np.zeros((n, k), np.int32)
    for i in range(n):
        hubs = [1, 2, 3, 4] if i % 2 == 0 else [5, 6]
        others = rng.choice(np.arange(7, n + 1), size=k - len(hubs), replace=False)
        idx[i] = np.array(hubs + others.tolist(), np.int32)
    idx = np.asfortranarray(idx)
    S = sev.api._snn_from_index(idx, k, 1 / 15, np.float64)
    cp, rv, nz = orc.snn(idx, k, 1 / 15, np.float64)
    assert np.array_equal(S.indptr, cp - 1) and np.array_equal(S.indices, rv - 1)
    assert np.array_equal(S.data, nz)


def test_jaccard_index_from_nn_matrix(sev, orc):
    rng = np.random.default_rng(2)
    X = rng.standard_normal((1500, 8))
    nn = sev.nearest_neighbours(X, 12)
    assert nn.shape == (1500, 1500) and nn.nnz == 1500 * 12
    S = sev.jaccard_index(nn, prune=1 / 15)
    ridx, _ = orc.knn(X, 12)
    cp, rv, nz = orc.snn(ridx, 12, 1 / 15, np.float64)
    assert np.array_equal(S.indptr, cp - 1) and np.array_equal(S.data, nz)


def test_pipeline_graph_end_to_end(sev, orc):
    """Config-1 shaped path at reduced size: every stage checked against the
    oracle given the previous stage's device output."""
    t = sev.nb_tables(4000, seed=0, density=0.05)
    C = 4000
    p = sev.Pipeline()
    p.synth_counts(C, t)
    p.normalize("lognormalize", 1e4)
    feats = sev.top_mean_features(t, 800)
    p.select_scale(feats, 10.0)
    p.pca(20, init=np.random.default_rng(0).standard_normal(800))
    s, U, V, Z = p.get_pca()
    p.neighbours(20)
    idx, dist = p.get_neighbours(C)
    ridx, rdist = orc.knn(Z, 20)
    assert np.array_equal(idx, ridx) and np.array_equal(dist, rdist)
    nnz = p.snn(1 / 15, np.float32)
    S = p.get_snn(C)
    cp, rv, nz = orc.snn(ridx, 20, 1 / 15, np.float32)
    assert nnz == len(rv)
    assert np.array_equal(S.indptr, cp - 1) and np.array_equal(S.indices, rv - 1)
    assert np.array_equal(S.data, nz)


@pytest.mark.parametrize("what", [0, 1, 2, 4])
def test_mfma_lane_layout_selftest(sev, what):
    import ctypes
    r = ctypes.c_double(-1.0)
    sev._lib.check(sev.load().sev_selftest(what, ctypes.byref(r)))
    assert r.value == 0.0


@pytest.mark.parametrize("precision", ["fp32", "bf16", "fp8", "exact"])
@pytest.mark.parametrize("include_self", [True, False])
@pytest.mark.parametrize("n,d,k", [(5000, 50, 20), (3000, 30, 30), (6000, 20, 40), (700, 10, 5),
                                   (130, 3, 64)])
def test_ann_precision_forms_bit_exact(sev, orc, precision, include_self, n, d, k):
    rng = np.random.default_rng(n * 7 + d)
    # clustered data: neighbours much closer than the norms
    centers = rng.standard_normal((max(n // 200, 2), d)) * 5.0
    X = (centers[rng.integers(0, len(centers), n)] + rng.standard_normal((n, d))).astype(np.float32)
    idx, dist, nfb = sev.ann(X, k, include_self=include_self, precision=precision,
                             return_fallback=True)
    ridx, rdist = orc.knn(X, k, include_self=include_self)
    assert np.array_equal(idx, ridx)
    assert np.array_equal(dist, rdist)
    print(f"{precision} n={n} d={d} k={k}: {nfb} fallback rows")


def test_ann_mfma_duplicates(sev, orc):
    rng = np.random.default_rng(8)
    base = rng.standard_normal((1000, 20)).astype(np.float32)
    X = np.concatenate([base, base, base[:300]])
    for prec in ("fp32", "bf16", "fp8"):
        idx, dist = sev.ann(X, 10, precision=prec)
        ridx, rdist = orc.knn(X, 10)
        assert np.array_equal(idx, ridx) and np.array_equal(dist, rdist)


@pytest.mark.parametrize("precision", ["fp32", "bf16"])
@pytest.mark.parametrize("include_self", [True, False])
def test_ann_norm_order_ties(sev, orc, precision, include_self):
    """Exact duplicates, copies with the coordinates reversed (equal norms,
    other points) and a block of zero vectors.  (Few points: searched
    exhaustively; the lists in norm order meet the same ties in
    test_lists_over_all_points.)"""
    rng = np.random.default_rng(31)
    base = rng.standard_normal((3000, 16)).astype(np.float32)
    X = np.concatenate([base, base[:, ::-1], base[:2000], np.zeros((50, 16), np.float32)])
    idx, dist, nfb = sev.ann(X, 20, include_self=include_self, precision=precision,
                             return_fallback=True)
    ridx, rdist = orc.knn(X, 20, include_self=include_self)
    assert np.array_equal(idx, ridx)
    assert np.array_equal(dist, rdist)
    print(f"{precision} include_self={include_self}: {nfb} fallback rows")


@pytest.mark.parametrize("precision", ["fp32", "bf16", "fp8"])
def test_pipeline_neighbours_forms(sev, orc, precision):
    t = sev.nb_tables(3000, seed=1, density=0.05)
    C = 6000
    p = sev.Pipeline()
    p.synth_counts(C, t)
    p.normalize("lognormalize", 1e4)
    p.select_scale(sev.top_mean_features(t, 600), 10.0)
    p.pca(30, init=np.random.default_rng(0).standard_normal(600))
    _, _, _, Z = p.get_pca()
    nfb = p.neighbours(20, precision=precision)
    idx, dist = p.get_neighbours(C)
    ridx, rdist = orc.knn(Z, 20)
    assert np.array_equal(idx, ridx) and np.array_equal(dist, rdist)
    print(f"pipeline {precision}: {nfb} of {C} rows fell back")
    if precision == "fp8":
        left = p.knn_passes()
        assert left[0] >= left[1] >= left[2] == nfb
        print(f"fp8 passes: rows left after FP8 / BF16 / FP32 candidates: {left.tolist()}")


@pytest.mark.parametrize("precision", ["fp32", "bf16", "exact", "fp8"])
def test_pipeline_neighbours_cosine(sev, orc, precision):
    """The device-resident pipeline's cosine form (metric=CosineDist() of
    nearest_neighbours) equals the oracle's on the embedding's first ndims
    columns, and its SNN is built from those lists."""
    rng = np.random.default_rng(23)
    Z = np.asfortranarray(rng.standard_normal((3000, 40)).astype(np.float32))
    Z[:, :5] *= 4.0
    p = sev.Pipeline()
    p.set_embedding(Z)
    p.neighbours(15, include_self=True, ndims=30, precision=precision, metric="cosine")
    idx, dist = p.get_neighbours(3000)
    ridx, rdist = orc.knn_cosine(np.asfortranarray(Z[:, :30]), 15)
    assert np.array_equal(idx, ridx) and np.array_equal(dist, rdist)
    p.snn(1 / 15, np.float32)
    S = p.get_snn(3000)
    cp, rv, nz = orc.snn(ridx, 15, 1 / 15, np.float32)
    assert np.array_equal(S.indptr, cp - 1) and np.array_equal(S.data, nz)
    p.close()


def test_large_results_in_slots(sev):
    """Results large enough to come through the pinned slots (from 32 MiB; sizes
    that are no multiple of a slot) equal the one-shot calls', which copy
    directly."""
    rng = np.random.default_rng(5)
    m, k = 420_011, 20
    Z = np.asfortranarray(rng.standard_normal((m, 3)).astype(np.float32))
    p = sev.Pipeline()
    p.set_embedding(Z)
    p.neighbours(k, include_self=True)
    idx, dist = p.get_neighbours(m)
    ridx, rdist = sev.ann(Z, k)
    assert np.array_equal(idx, ridx) and np.array_equal(dist, rdist)
    p.snn(1 / 15, np.float32)
    S = p.get_snn(m)
    assert S.nnz * 4 >= 32 << 20
    R = sev.shared_nearest_neighbours(Z, k)
    assert np.array_equal(S.indptr, R.indptr) and np.array_equal(S.indices, R.indices)
    assert np.array_equal(S.data, R.data)
    p.close()


def test_large_result_to_null_is_refused(sev):
    """A result above the size that comes through the pinned slots, asked for
    without an array to put it in, is an error as a small one is."""
    import scipy.sparse as sp
    m, n = 500_000, 18
    rng = np.random.default_rng(2)
    X = sp.csc_matrix((rng.integers(1, 9, m * n).astype(np.int32), np.tile(np.arange(m), n),
                       np.arange(n + 1) * m), shape=(m, n))
    p = sev.Pipeline()
    p.load_counts(X)
    p.normalize("lognormalize", 1e4)
    assert m * n * 4 >= 32 << 20
    L = sev.load()
    assert L.sev_pipeline_get_normalized(p._h, None) == -1
    assert b"NULL" in L.sev_last_error()
    assert len(p.get_normalized()) == m * n
    p.close()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_fallback_counts_rows_searched_exhaustively(sev, dtype):
    """n_fallback is n wherever the whole search is exhaustive (few points, the
    exact form), and the rows left without a certificate (here few or none)
    where candidates are proposed."""
    rng = np.random.default_rng(3)
    def points(n, d):
        return np.asfortranarray((rng.normal(0, 6, (9, d))[rng.integers(0, 9, n)] +
                                  rng.normal(0, 1, (n, d))).astype(dtype))
    for n, d, precision in ((900, 8, "fp32"), (900, 8, "bf16"), (5000, 50, "fp32"),
                            (20000, 20, "exact")):
        assert sev.ann(points(n, d), 10, precision=precision, return_fallback=True)[2] == n
    for precision in ("fp32", "bf16"):
        assert sev.ann(points(20000, 20), 10, precision=precision, return_fallback=True)[2] < 200
    if dtype == np.float32:
        p = sev.Pipeline()
        p.set_embedding(points(900, 8))
        assert p.neighbours(10) == 900
        p.set_embedding(points(20000, 20))
        assert p.neighbours(10) < 200
        p.close()


@pytest.mark.parametrize("include_self", [True, False])
@pytest.mark.parametrize("n,d,k,precision",
                         [(30100, 16, 40, "fp32"), (30100, 16, 40, "bf16"),
                          (30100, 51, 31, "fp32"), (30100, 51, 31, "bf16"),
                          (30100, 20, 45, "fp32"), (30100, 20, 45, "bf16"),
                          (15900, 126, 20, "fp32"), (11300, 126, 20, "bf16"),
                          (15900, 70, 40, "bf16"), (30500, 16, 20, "bf16"),
                          (16800, 52, 12, "bf16")])
def test_lists_over_all_points(sev, orc, n, d, k, precision, include_self):
    """The candidate lists over all points (sizes beyond the exhaustive search
    that the cells do not take, or points without clusters in the BF16 form),
    in ascending norm with seeded thresholds: exact duplicates, copies with the
    coordinates reversed (equal norms, other points) and a block of zero
    vectors at the head of the order.  The lists depend on the order only
    through ties, and the certified result must not.  All rows against the
    exhaustive form, 1,500 of them against the oracle."""
    rng = np.random.default_rng(n + d)
    u = n // 3
    z = 40 if d < 60 else 10  # in many dimensions they are near every point
    base = rng.standard_normal((u, d)).astype(np.float32)
    X = np.concatenate([base, base[:, ::-1], base[:n - 2 * u - z],
                        np.zeros((z, d), np.float32)])
    X = np.asfortranarray(X)
    p = sev.Pipeline()
    p.set_embedding(X)
    p.profile(True)
    left = p.neighbours(k, include_self=include_self, precision=precision)
    idx, dist = p.get_neighbours(n)
    ran = set(p.profile_read())
    assert "knn_cell" not in ran and left < n
    assert any(r.startswith("knn_cand_" + precision) for r in ran)
    p.neighbours(k, include_self=include_self, precision="exact")
    xidx, xdist = p.get_neighbours(n)
    p.close()
    assert np.array_equal(idx, xidx) and np.array_equal(dist, xdist)
    q = np.sort(np.concatenate([rng.choice(n - 40, 1460, replace=False), np.arange(n - 40, n)]))
    ridx, rdist = orc.knn(X, k, include_self=include_self, qidx=q)
    assert np.array_equal(idx[q], ridx) and np.array_equal(dist[q], rdist)
