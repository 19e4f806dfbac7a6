"""The work that the framework is timed on.

A single-cell program normalises its counts, scales the selected genes, embeds
the cells by PCA, searches neighbours, builds the Jaccard graph and clusters
it.  Each case is one of these blocks, called as such a program calls it: on a
resident ``Pipeline``, or through the one-shot functions on host arrays.

Blocks rather than whole paths, since neighbours and graph are compared value
by value: the embedding a graph is built from is an input here, and the PCA
returns all of its factors.

Counts come from the library's seeded negative-binomial generator.  A data set
is a stack of cell types (each type with its own gene means, types of uneven
size), so that its spectrum has the leading components and the noise bulk that
real counts have.  Embeddings are Gaussian groups with decaying scales.
"""
import ctypes
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    if "severo_jl_amd" not in sys.modules:
        d = os.path.join(ROOT, "severo.jl_amd")
        spec = importlib.util.spec_from_file_location(
            "severo_jl_amd", os.path.join(d, "__init__.py"), submodule_search_locations=[d])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["severo_jl_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["severo_jl_amd"]


sev = _package()

PRUNE, SCALE_FACTOR, SCALE_MAX, TOL = 1.0 / 15, 1e4, 10.0, 1e-5
GRAPH_ROOM = 16
PRECISION = {"fp32": 0, "bf16": 1}
GENE_LOG_MEAN, GENE_LOG_SD, DISPERSION = -1.0, 1.5, 0.3


def listed():
    return [
        # the smallest call: neighbours of a subset of cells in few components
        dict(name="ann_2k", kind="ann", cells=2003, dims=15, k=10, dtype="float32",
             metric="euclidean", include_self=True, precision="fp32"),
        # the one-shot functions on a tutorial-sized data set, host arrays in and out
        dict(name="calls_3k", kind="calls", cells=2700, genes=13714, density=0.06, types=8,
             nfeat=2000, npcs=50, work=0),
        # the reference's own small workload, resident, with its default basis
        dict(name="embed_5k_fp32", kind="embed", cells=5000, genes=20000, density=0.05, boost=0.0,
             types=12, nfeat=2000, npcs=50, work=0, precision="fp32"),
        # one ordinary data set, 5% of the cells with three times the library size
        dict(name="embed_100k_fp32", kind="embed", cells=100_000, genes=33538, density=0.04,
             boost=0.05, types=24, nfeat=2000, npcs=50, work=112, precision="fp32"),
        # an atlas, in the precision form
        dict(name="embed_1m_bf16", kind="embed", cells=1_000_000, genes=27998, density=0.03,
             boost=0.0, types=40, nfeat=2000, npcs=50, work=112, precision="bf16"),
        # many uneven samples at once
        dict(name="embed_batch64", kind="batch", samples=64, lo=500, hi=50_000, genes=20000,
             types=6, nfeat=2000, npcs=30, work=64),
        # neighbours and graph of the three single data sets
        dict(name="graph_5k_fp32", kind="graph", cells=5000, dims=50, k=20, groups=12,
             precision="fp32"),
        dict(name="graph_100k_fp32", kind="graph", cells=100_000, dims=50, k=20, groups=24,
             precision="fp32"),
        dict(name="graph_1m_bf16", kind="graph", cells=1_000_000, dims=50, k=20, groups=40,
             precision="bf16"),
        # neighbours of a host embedding in double precision, as an embedding's coordinates
        # are, an odd number of cells
        dict(name="ann_20k_fp64", kind="ann", cells=20_011, dims=50, k=15, dtype="float64",
             metric="euclidean", include_self=True, precision="fp32"),
        # the variable genes of the atlas
        dict(name="hvg_1m", kind="hvg", cells=1_000_000, genes=27998, density=0.03, boost=0.0,
             types=40, nfeat=2000),
        # Louvain clusters of an ordinary graph, ten random starts
        dict(name="cluster_50k", kind="cluster", cells=50_000, dims=50, k=20, groups=24,
             starts=10),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["ann", "calls", "embed", "embed", "embed", "batch", "graph", "graph",
                       "graph", "ann", "hvg", "cluster"])
    if kind == "ann":
        return dict(kind=kind, cells=_log_int(rng, 1000, 40_000), dims=rng.randint(5, 60),
                    k=rng.randint(5, 40), dtype=rng.choice(["float32", "float64"]),
                    metric=rng.choice(["euclidean", "euclidean", "cosine"]),
                    include_self=rng.random() < 0.75, precision=rng.choice(["fp32", "bf16"]))
    if kind == "calls":
        return dict(kind=kind, cells=_log_int(rng, 1000, 8000), genes=_log_int(rng, 5000, 20_000),
                    density=rng.uniform(0.03, 0.08), types=rng.randint(5, 12),
                    nfeat=rng.randint(700, 2200), npcs=rng.choice([20, 30, 50]), work=0)
    if kind == "embed":
        cells = _log_int(rng, 2000, 500_000)
        return dict(kind=kind, cells=cells, genes=_log_int(rng, 12_000, 34_000),
                    density=rng.uniform(0.02, 0.05), boost=rng.choice([0.0, 0.05]),
                    types=rng.randint(8, 40), nfeat=rng.randint(900, 3000),
                    npcs=rng.choice([20, 30, 50]), work=rng.choice([96, 112, 128]),
                    precision=rng.choice(["fp32", "bf16"]) if cells <= 250_000 else "bf16")
    if kind == "batch":
        return dict(kind=kind, samples=rng.randint(3, 64), lo=_log_int(rng, 300, 1000),
                    hi=_log_int(rng, 5000, 50_000), genes=_log_int(rng, 8000, 20_000),
                    types=rng.randint(3, 8), nfeat=rng.randint(800, 2200),
                    npcs=rng.choice([15, 20, 30]), work=64)
    if kind == "graph":
        precision = rng.choice(["fp32", "bf16"])
        return dict(kind=kind, cells=_log_int(rng, 1000, 250_000 if precision == "fp32"
                                              else 800_000),
                    dims=rng.randint(10, 60), k=rng.randint(10, 30), groups=rng.randint(5, 40),
                    precision=precision)
    if kind == "hvg":
        return dict(kind=kind, cells=_log_int(rng, 3000, 900_000),
                    genes=_log_int(rng, 12_000, 28_000), density=rng.uniform(0.02, 0.04),
                    boost=rng.choice([0.0, 0.05]), types=rng.randint(8, 40),
                    nfeat=rng.randint(500, 3000))
    return dict(kind=kind, cells=_log_int(rng, 2000, 60_000), dims=rng.randint(10, 55),
                k=rng.randint(10, 30), groups=rng.randint(5, 30), starts=rng.choice([1, 3, 10]))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _type_tables(genes, density, boost, types, seed):
    """One generator table per cell type: the base means of a data set, each
    type with a share of its genes shifted (log-normal) and types of graded
    strength."""
    rng = np.random.default_rng([seed, 1])
    base = sev.nb_tables(genes, seed=seed % (1 << 31), density=density, log_mean=GENE_LOG_MEAN,
                         log_sd=GENE_LOG_SD, dispersion=DISPERSION, boost_frac=boost)
    out = []
    for t in range(types):
        shifted = rng.random(genes) < rng.uniform(0.05, 0.4)
        m = base.gene_mean * np.where(shifted, np.exp(rng.normal(0.0, 0.8, genes)), 1.0)
        out.append(_table(base, m, base.size_factor, int(rng.integers(1 << 31))))
    return out, rng


def _table(base, mean, size, seed):
    p0, q = np.empty(2 * len(mean)), np.empty(2 * len(mean))
    for c, f in ((0, 1.0), (1, base.boost)):
        mu = size * f * mean
        p0[c::2] = np.power(base.r / (base.r + mu), base.r)
        q[c::2] = mu / (base.r + mu)
    return sev.NBTables(base.n_genes, seed, base.r, size, base.boost_frac, base.boost, mean, p0, q)


def _split(rng, total, parts, least):
    """total cells in uneven parts of at least `least` each."""
    w = rng.uniform(0.3, 1.7, parts)
    n = least + np.floor((total - least * parts) * w / w.sum()).astype(np.int64)
    n[0] += total - n.sum()
    return n


def _counts(case, seed):
    """A pipeline holding the counts of one data set (its types stacked)."""
    tables, rng = _type_tables(case["genes"], case["density"], case.get("boost", 0.0),
                               case["types"], seed)
    p = sev.Pipeline()
    p.synth_batch(_split(rng, case["cells"], case["types"], 20), tables)
    p.set_batch(None)
    return p, rng


def _sample_tables(case, seed):
    """Cells per sample (part of the case), and from the seed `types` generator
    tables per sample, densities of 2-8%."""
    rng = np.random.default_rng([case["samples"], case["lo"], case["hi"]])
    cells = np.exp(rng.uniform(np.log(case["lo"]), np.log(case["hi"]),
                               case["samples"])).astype(np.int64)
    cells[0], cells[-1] = case["lo"], case["hi"]
    rng = np.random.default_rng([seed, 2])
    lo, hi = (sev.nb_tables(case["genes"], seed=seed % (1 << 31), density=d,
                            log_mean=GENE_LOG_MEAN, log_sd=GENE_LOG_SD, dispersion=DISPERSION)
              for d in (0.02, 0.08))
    tabs, parts, feats = [], [], []
    for s in range(case["samples"]):
        size = math.exp(rng.uniform(math.log(lo.size_factor), math.log(hi.size_factor)))
        own = lo.gene_mean * np.exp(rng.normal(0.0, 0.3, case["genes"]))
        for t in range(case["types"]):
            shifted = rng.random(case["genes"]) < rng.uniform(0.05, 0.4)
            m = own * np.where(shifted, np.exp(rng.normal(0.0, 0.8, case["genes"])), 1.0)
            tabs.append(_table(lo, m, size, int(rng.integers(1 << 31))))
        parts.append(_split(rng, int(cells[s]), case["types"], 8))
        feats.append(np.argsort(-own, kind="stable")[:case["nfeat"]])
    return cells, tabs, np.concatenate(parts), np.stack(feats), rng


def _embedding(cells, dims, groups, seed, dtype):
    """Host embedding (cells x dims, column-major): groups of uneven size,
    scales decaying over the components as those of a PCA do."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    kw = dict(device="cuda", dtype=torch.float64, generator=g)
    scale = 8.0 * torch.arange(1, dims + 1, device="cuda", dtype=torch.float64) ** -0.6
    centre = torch.randn(groups, dims, **kw) * scale
    share = torch.rand(groups, **kw) + 0.2
    label = torch.multinomial(share, cells, replacement=True, generator=g)
    Z = torch.empty(dims, cells, device="cuda", dtype=getattr(torch, dtype))
    for t in range(dims):
        Z[t] = centre[label, t] + torch.randn(cells, **kw) * (0.5 + 0.15 * scale[t])
    return Z.cpu().numpy().T


class _Graph:
    """A handle of the C interface holding an embedding, and the host program's
    own arrays that the graph is copied to: sized for GRAPH_ROOM entries per
    cell and neighbour (the graph's own number of entries follows from the
    data)."""

    def __init__(self, case, seed):
        self.case, self.lib, self.handle = case, sev.load(), ctypes.c_void_p()
        n, d, k = case["cells"], case["dims"], case["k"]
        Z = np.asfortranarray(_embedding(n, d, case["groups"], seed, "float32"))
        self.check(self.lib.sev_pipeline_create(ctypes.byref(self.handle)))
        self.check(self.lib.sev_pipeline_set_embedding(self.handle, n, d, Z.ctypes.data, n))
        self.colptr = np.zeros(n + 1, np.int64)
        self.rows = np.zeros(GRAPH_ROOM * n * k, np.int64)
        self.weights = np.zeros(GRAPH_ROOM * n * k, np.float32)

    def check(self, status):
        if status:
            raise RuntimeError(self.lib.sev_last_error().decode())

    def __del__(self):
        self.lib.sev_pipeline_destroy(self.handle)

    def build(self):
        passes, nnz = ctypes.c_int64(), ctypes.c_int64()
        self.check(self.lib.sev_pipeline_neighbours(self.handle, self.case["k"], 1, 0,
                                                    PRECISION[self.case["precision"]],
                                                    ctypes.byref(passes)))
        self.check(self.lib.sev_pipeline_snn(self.handle, PRUNE, 0, ctypes.byref(nnz)))
        if nnz.value > self.rows.size:
            raise RuntimeError("the graph has more entries than the program's arrays")
        self.check(self.lib.sev_pipeline_get_snn(self.handle, self.colptr.ctypes.data,
                                                 self.rows.ctypes.data,
                                                 self.weights.ctypes.data))
        return dict(colptr=self.colptr, rows=self.rows, weights=self.weights)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "ann":
        X = _embedding(case["cells"], case["dims"], 10, seed, case["dtype"])
        return dict(case=case, X=X)
    if kind == "graph":
        return _Graph(case, seed)
    if kind == "cluster":
        p = sev.Pipeline()
        p.set_embedding(_embedding(case["cells"], case["dims"], case["groups"], seed, "float32"))
        p.neighbours(case["k"])
        p.snn(PRUNE, np.float32)
        return dict(case=case, p=p, seed=seed)
    if kind == "batch":
        cells, tabs, parts, feats, rng = _sample_tables(case, seed)
        p = sev.Pipeline()
        p.synth_batch(parts, tabs)
        p.set_batch(cells)
        init = rng.standard_normal((case["samples"], case["nfeat"]))
        return dict(case=case, p=p, feats=feats, init=init)
    p, rng = _counts(case, seed)
    if kind == "hvg":
        return dict(case=case, p=p)
    feats = p.find_variable_features(case["nfeat"])
    init = rng.standard_normal(case["nfeat"])
    if kind == "calls":
        X = p.get_counts()
        p.close()
        return dict(case=case, X=X, feats=feats, init=init)
    return dict(case=case, p=p, feats=feats, init=init)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    if isinstance(state, _Graph):
        return state.build()
    case = state["case"]
    kind = case["kind"]
    if kind == "ann":
        idx, dist = sev.ann(state["X"], case["k"], include_self=case["include_self"],
                            precision=case["precision"], metric=case["metric"])
        return dict(index=idx, distance=dist)
    if kind == "calls":
        Y = sev.normalize_cells(state["X"], scale_factor=SCALE_FACTOR)
        A = sev.scale_features(Y, scale_max=SCALE_MAX, features=state["feats"])
        em = sev.embedding(A, case["npcs"], init=state["init"])
        return dict(coordinates=em.coordinates, stdev=em.stdev, basis=em.basis)
    p = state["p"]
    if kind == "cluster":
        labels, q = p.cluster(case["cells"], nrandomstarts=case["starts"], seed=state["seed"],
                              return_modularity=True)
        return dict(labels=labels, modularity=q)
    if kind == "hvg":
        sel, metric = p.find_variable_features(case["nfeat"], return_metric=True)
        return dict(selected=sel, metric=metric)
    p.normalize("lognormalize", SCALE_FACTOR)
    if kind == "batch":
        p.select_scale_batch(state["feats"], SCALE_MAX)
        p.pca_batch(case["npcs"], init=state["init"], tol=TOL, work=case["work"])
        s, U, V, Z = p.get_pca_batch()
    else:
        p.select_scale(state["feats"], SCALE_MAX)
        p.pca(case["npcs"], init=state["init"], tol=TOL, precision=case["precision"],
              work=case["work"])
        s, U, V, Z = p.get_pca()
    return dict(s=s, U=U, V=V, Z=Z)


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how far two correct results may differ
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind in ("ann", "graph"):
        n, d, k = case["cells"], case["dims"], case["k"]
        size = 8 if case.get("dtype") == "float64" else 4
        out = n * k * (4 + size) if kind == "ann" else 8 * n + 2 * n * k * (8 + size)
        return dict(bytes=n * d * size + out, flops=2.0 * n * n * d)
    if kind == "cluster":
        edges = 2 * case["cells"] * case["k"]
        return dict(bytes=case["starts"] * (8 * edges + 8 * case["cells"]),
                    flops=2.0 * case["starts"] * edges)
    if kind == "batch":
        # cells log-uniform between lo and hi, densities log-uniform in 2-8%
        cells = case["samples"] * (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
        density, share = 0.043, 0.35
    else:
        cells, density, share = case["cells"], case["density"], 0.1
    nnz = cells * case["genes"] * density
    if kind == "hvg":
        return dict(bytes=8 * nnz + 16 * case["genes"], flops=6.0 * nnz)
    # normalised and scaled once, then (at least) one product pair per Lanczos vector
    sel = cells * case["nfeat"] * share
    vectors = case["work"] or case["npcs"] + 7
    return dict(bytes=12 * nnz + 16 * sel + 12.0 * cells * case["npcs"],
                flops=10.0 * nnz + 4.0 * sel * vectors)


def tolerance(case):
    kind = case["kind"]
    if kind in ("ann", "graph"):
        return "exact"
    if kind == "cluster":
        return dict(rel=1e-9, differ=0.0)
    if kind == "hvg":
        return dict(rel=1e-9, differ=1e-3)
    # a PCA stops when its 50 triplets have converged to tol = 1e-5: bases of 108 and 112
    # vectors, or tol = 1e-7, move the factors by up to 1.2e-3 in the 2-norm and 0.04 root
    # mean squares in one entry (components in the noise bulk, 1e-4 apart)
    return dict(rel=5e-3, max=0.2)


# ---------------------------------------------------------------------------
# the same in 64 bits, without the framework's kernels
# ---------------------------------------------------------------------------
def _counts_host(p):
    _, _, cp, rv, val = p.get_counts_julia()
    return (torch.from_numpy(cp).cuda() - 1, torch.from_numpy(rv).cuda() - 1,
            torch.from_numpy(val).cuda())


def _stdevs(m, cp, row, val, feats, npcs):
    """Singular values of the scaled, centred, clipped selection (FP64 Gram
    matrix of dense row blocks)."""
    total = torch.zeros(m, dtype=torch.float64, device="cuda")
    total.index_add_(0, row, val.double())
    cols, F = [], len(feats)
    cp_h = cp.cpu()
    for g in feats:
        b, e = int(cp_h[g]), int(cp_h[g + 1])
        cols.append((row[b:e], torch.log1p(SCALE_FACTOR * val[b:e].double() / total[row[b:e]])))
    D = torch.zeros(F, m, dtype=torch.float64, device="cuda")
    for j, (r, v) in enumerate(cols):
        D[j, r] = v
    mu = D.mean(1, keepdim=True)
    D -= mu
    sd = torch.sqrt((D * D).sum(1, keepdim=True) / (m - 1))
    D = torch.clamp(D / torch.where(sd > 0, sd, torch.ones_like(sd)), max=SCALE_MAX)
    G = D @ D.T
    w = torch.linalg.eigvalsh(G).flip(0)[:npcs]
    return torch.sqrt(torch.clamp(w, min=0.0)).cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "ann":
        X = torch.from_numpy(np.ascontiguousarray(prepare(case, seed)["X"])).cuda().double()
        if case["metric"] == "cosine" or case["cells"] > 60_000:
            return None
        out, cols = [], X.T.contiguous()
        for b in range(0, len(X), 1024):
            q = cols[:, b:b + 1024]
            d = torch.zeros(q.shape[1], len(X), dtype=torch.float64, device="cuda")
            for t in range(len(cols)):
                d += (q[t][:, None] - cols[t][None, :]) ** 2
            if not case["include_self"]:
                at = torch.arange(q.shape[1], device="cuda")
                d[at, b + at] = torch.inf
            out.append(d.topk(case["k"], largest=False, sorted=True).values.sqrt())
        return dict(index=None, distance=torch.cat(out).cpu().numpy())
    if kind == "embed" and case["cells"] <= 120_000:
        state = prepare(case, seed)
        p = state["p"]
        cp, row, val = _counts_host(p)
        p.close()
        s = _stdevs(case["cells"], cp, row, val, state["feats"], case["npcs"])
        return dict(s=s, U=None, V=None, Z=None)
    return None
