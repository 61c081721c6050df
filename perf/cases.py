"""The work that a user has this framework do, as cases that can be timed and compared.

The operations are the stages of a graph build and of mapping onto a finished reference:

* ``query``    new cells (already reduced) against a reference index kept in HBM, the call
               behind scarf's ``transform_ann`` and every chunk of the mapping service;
* ``selfknn``  the index of an embedding and the k neighbours of each of its own cells, as
               ``make_graph`` does it: FP32 (certified exact), BF16 and FP8 screens;
* ``stats``    library sizes and feature means / deviations of resident CSR counts;
* ``pca``      the incremental PCA fit in scarf's block order;
* ``project``  the sparse projection of counts onto stored loadings;
* ``smooth``   the fuzzy edge weights of a kNN table;
* ``graph``    the whole ``build_graph`` call with a stored reduction (a second graph of a
               dataset, with other parameters or another k).

Embeddings follow what PCA of log-normalised negative-binomial counts looks like in this
repository's workloads: a wide library-size axis, one axis per latent group beyond the
first, and near-isotropic noise whose scale grows with the library size.
"""
import functools
import math

import numpy as np
import torch

from scarf_amd.device import DeviceCSR
from scarf_amd.graph import GraphParams, build_graph
from scarf_amd.knn import GpuIndex
from scarf_amd.normalize import NormParams, chunk_bounds, feature_stats
from scarf_amd.pca import Projector, fit_pca
from scarf_amd.smooth import smooth_knn
from scarf_amd.synth import generate_csr_gpu, make_gene_model

DEV = "cuda"


def listed():
    return [
        # one cell against the serving reference (500k cells): latency and launches
        dict(name="query_1_of_500k", op="query", nq=1, nr=500_000, D=50, k=11, pool=64,
             screen="bf16", groups=20),
        # the median request of the mapping service
        dict(name="query_1k_of_500k", op="query", nq=1000, nr=500_000, D=50, k=11, pool=64,
             screen="bf16", groups=20),
        # a full chunk of a large mapping request
        dict(name="query_16k_of_500k", op="query", nq=16_384, nr=500_000, D=50, k=11, pool=64,
             screen="bf16", groups=20),
        # certified exact self query of a small experiment (ragged size)
        dict(name="self_fp32_19k", op="selfknn", n=19_001, D=50, k=11, pool=64, screen="fp32",
             groups=5),
        # the 100,000-cell workload
        dict(name="self_bf16_100k", op="selfknn", n=100_000, D=50, k=11, pool=64, screen="bf16",
             groups=8),
        # the million-cell workload (the headline benchmark's kNN)
        dict(name="self_bf16_1m", op="selfknn", n=1_000_000, D=50, k=21, pool=64,
             screen="bf16", groups=20),
        # an atlas: the 4-million-cell workload's dimensions and screen at 1.5 million cells
        dict(name="self_fp8_1500k", op="selfknn", n=1_500_000, D=100, k=11, pool=128,
             screen="fp8", groups=40),
        # first pass over the counts of half a million cells
        dict(name="stats_500k", op="stats", n=500_000, d=2000, groups=20, density=0.08,
             chunk=50_000),
        # the 100,000-cell workload's incremental fit: five partial fits of 20,000 cells
        dict(name="pca_100k", op="pca", n=100_000, d=2000, groups=8, density=0.10,
             chunk=20_000, dims=50),
        # reduction of half a million cells
        dict(name="project_500k", op="project", n=500_000, d=2000, groups=20, density=0.08,
             dims=50),
        # edge weights of the million-cell graph
        dict(name="smooth_1m", op="smooth", n=1_000_000, k=21, chunk=50_000),
        # a whole small build with scarf's default chunk of 1000 cells and a stored reduction
        dict(name="graph_5k", op="graph", n=5_000, d=2000, groups=4, density=0.10, chunk=1000,
             dims=50, k=11, pool=64, screen="fp32"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["query"] * 5 + ["selfknn"] * 5 + ["stats", "pca", "project", "smooth",
                                                       "graph"])
    if op == "query":
        return dict(op=op, nq=_log(rng, 1, 50_000), nr=_log(rng, 4_000, 500_000),
                    D=rng.randint(8, 60), k=rng.randint(3, 40), pool=rng.choice([64, 64, 100]),
                    screen=rng.choice(["bf16", "bf16", "fp32"]), groups=rng.randint(1, 30))
    if op == "selfknn":
        screen = rng.choice(["fp32", "bf16", "bf16", "fp8"])
        n = {"fp32": _log(rng, 2_000, 60_000), "bf16": _log(rng, 10_000, 700_000),
             "fp8": _log(rng, 60_000, 800_000)}[screen]
        return dict(op=op, n=n, D=rng.randint(64, 110) if screen == "fp8" else
                    rng.randint(10, 100), k=rng.randint(5, 30),
                    pool=128 if screen == "fp8" else rng.choice([64, 64, 128]), screen=screen,
                    groups=rng.randint(1, 40))
    if op == "smooth":
        return dict(op=op, n=_log(rng, 1_000, 1_000_000), k=rng.randint(5, 40),
                    chunk=rng.choice([1000, 20_000, 50_000]))
    case = dict(op=op, n=_log(rng, 3_000, {"graph": 20_000, "pca": 60_000}.get(op, 500_000)),
                d=rng.randint(600, 3000), groups=rng.randint(1, 20),
                density=round(rng.uniform(0.04, 0.12), 3))
    if op in ("stats", "graph"):
        case.update(chunk=rng.choice([1000, 5000, 20_000]))
    if op in ("pca", "project", "graph"):
        case.update(dims=rng.randint(11, 60))
    if op == "pca":
        case.update(chunk=max(1000, case["n"] // rng.randint(1, 5)))
    if op == "graph":
        case.update(k=rng.randint(5, 21), pool=64, screen=rng.choice(["fp32", "bf16"]))
    return case


# -- inputs -----------------------------------------------------------------------------------

def _gen(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed(1_000_003 * int(seed) + salt)
    return g


def _embedding(n, D, groups, seed, salt=1):
    """FP32 [n, D] PCA-like embedding; the group centres depend on the seed alone."""
    gc, g = _gen(seed, 0), _gen(seed, salt)
    amp = 1.7 if groups <= 8 else 1.0
    centers = torch.randn(groups, D, generator=gc, device=DEV) * amp
    centers[:, min(max(groups, 1), D):] = 0.0
    size = torch.randn(n, generator=g, device=DEV)
    E = torch.randn(n, D, generator=g, device=DEV) * 1.03
    E += centers[torch.randint(0, groups, (n,), generator=g, device=DEV)]
    E *= torch.exp(0.14 * size)[:, None]
    E[:, 0] = 3.9 * size + 0.35 * (size * size - 1.0)
    return E


@functools.lru_cache(maxsize=8)
def _model(d, groups, density):
    return make_gene_model(d, groups, density, seed=17)


def _counts(case, seed):
    v, c, r = generate_csr_gpu(case["n"], _model(case["d"], case["groups"], case["density"]),
                               seed=int(seed))
    return DeviceCSR(v, c, r, case["d"])


def _loadings(d, dims, seed):
    """Orthonormal FP64 loadings [d, dims], as a stored reduction holds them."""
    g = _gen(seed, 5)
    return torch.linalg.qr(torch.randn(d, dims, generator=g, device=DEV,
                                       dtype=torch.float64))[0].cpu().numpy()


NORM = NormParams(size_factor=1e4, clip=10.0)


def _params(case):
    return GraphParams(dims=case["dims"], k=case["k"], batch_size=case["chunk"],
                       size_factor=1e4, clip=10.0, screen=case["screen"], pool=case["pool"])


def prepare(case, seed):
    op = case["op"]
    s = dict(case=case)
    if op == "query":
        index = GpuIndex("l2", case["D"], screen=case["screen"], pool=case["pool"])
        index.init_index(case["nr"])
        index.add_items(_embedding(case["nr"], case["D"], case["groups"], seed))
        index.packed()
        s.update(index=index, Q=_embedding(case["nq"], case["D"], case["groups"], seed, 2))
    elif op == "selfknn":
        s.update(E=_embedding(case["n"], case["D"], case["groups"], seed))
    elif op == "smooth":
        g = _gen(seed, 3)
        n, k = case["n"], case["k"]
        gap = torch.rand(n, k, generator=g, device=DEV) + 0.02
        base = 20.0 + 30.0 * torch.rand(n, 1, generator=g, device=DEV)
        s.update(dist=base + 2.0 * torch.cumsum(gap / torch.arange(
                     1, k + 1, device=DEV).sqrt(), 1),
                 idx=torch.randint(0, n, (n, k), generator=g, device=DEV))
    else:
        s.update(csr=_counts(case, seed))
        if op == "pca":
            s.update(stats=feature_stats(s["csr"], case["chunk"], NORM))
        if op == "project":
            st = feature_stats(s["csr"], 50_000, NORM)
            s.update(stats=st, proj=Projector.build(
                _loadings(case["d"], case["dims"], seed), st.mu.cpu().numpy(),
                st.sigma.cpu().numpy(), clip=NORM.clip))
        if op == "graph":
            s.update(loadings=_loadings(case["d"], case["dims"], seed))
    return s


# -- one pass ---------------------------------------------------------------------------------

def run(state):
    case = state["case"]
    op = case["op"]
    if op == "query":
        return state["index"].knn_query_tensor(state["Q"], case["k"])
    if op == "selfknn":
        index = GpuIndex("l2", case["D"], screen=case["screen"], pool=case["pool"])
        index.init_index(case["n"])
        index.add_items(state["E"])
        return index.knn_query_tensor(index.embedding(), case["k"], self_offset=0)
    if op == "stats":
        st = feature_stats(state["csr"], case["chunk"], NORM)
        return dict(mu=st.mu, sigma=st.sigma, libsize=st.libsize, sums=st.chunk_sums,
                    sumsq=st.chunk_sumsq, mean=st.chunk_mean)
    if op == "pca":
        fit = fit_pca(state["csr"], state["stats"], NORM, case["dims"], case["chunk"])
        return dict(loadings=fit.loadings, var=fit.state.explained_variance_,
                    mean=fit.state.mean_)
    if op == "project":
        return state["proj"].project(state["csr"], NORM, libsize=state["stats"].libsize)
    if op == "smooth":
        return smooth_knn(state["dist"], state["idx"], case["chunk"])
    g = build_graph(state["csr"], _params(case), loadings=state["loadings"])
    return dict(mu=g.mu, sigma=g.sigma, embedding=g.embedding, indices=g.indices,
                distances=g.distances, weights=g.weights)


# -- what a pass cannot do without --------------------------------------------------------------

def _nnz(case):
    return case["n"] * case["d"] * case["density"]


def work(case):
    op = case["op"]
    if op in ("query", "selfknn"):
        nq, nr = (case["nq"], case["nr"]) if op == "query" else (case["n"], case["n"])
        rows = nr + (nq if op == "query" else 0)
        return dict(bytes=4 * rows * case["D"] + nq * (12 * case["k"] + 4),
                    flops=2 * nq * nr * case["D"])
    if op == "smooth":
        return dict(bytes=case["n"] * (16 * case["k"] + 8), flops=case["n"] * case["k"] * 20)
    csr = 8 * _nnz(case) + 8 * case["n"]
    if op == "stats":
        chunks = -(-case["n"] // case["chunk"])
        return dict(bytes=csr + 8 * case["n"] + 24 * chunks * case["d"], flops=4 * _nnz(case))
    if op == "pca":
        per_row = case["d"] * case["density"]
        return dict(bytes=csr + 8 * case["d"] * case["dims"],
                    flops=case["n"] * per_row * per_row + 10 * case["d"] ** 2 * case["dims"])
    if op == "project":
        return dict(bytes=csr + 8 * case["n"] + 4 * case["dims"] * (case["n"] + case["d"]),
                    flops=2 * _nnz(case) * case["dims"])
    return dict(bytes=csr + case["n"] * (8 + 4 * case["dims"] + 16 * case["k"]),
                flops=2 * _nnz(case) * case["dims"] + 2 * case["n"] ** 2 * case["dims"])


# -- the same in 64 bits ------------------------------------------------------------------------

def _exact_knn(Q, R, k, drop_self):
    """FP64 [nq, k] squared distances of the nearest rows, each query's own row left out."""
    Q, R = Q.double(), R.double()
    out = torch.empty(Q.shape[0], k, dtype=torch.float64, device=DEV)
    step = max(1, int(2e8 // R.shape[0]))
    rn = (R * R).sum(1)
    for a in range(0, Q.shape[0], step):
        q = Q[a:a + step]
        d = rn[None, :] - 2.0 * (q @ R.T)
        if drop_self:
            i = torch.arange(q.shape[0], device=DEV)
            d[i, a + i] = math.inf
        near = torch.topk(d, k, dim=1, largest=False).indices
        d = ((q[:, None, :] - R[near]) ** 2).sum(2)
        out[a:a + step] = torch.sort(d, 1).values
    return out


def _blocks(csr, step=20_000):
    """(first row, dense FP64 counts) of the matrix, ``step`` rows at a time."""
    for a in range(0, csr.n_rows, step):
        rp = csr.rowptr[a:min(csr.n_rows, a + step) + 1]
        e0, e1 = int(rp[0]), int(rp[-1])
        rows = torch.repeat_interleave(torch.arange(rp.numel() - 1, device=DEV), rp[1:] - rp[:-1])
        x = torch.zeros(rp.numel() - 1, csr.n_cols, dtype=torch.float64, device=DEV)
        x[rows, csr.cols[e0:e1].long()] = csr.vals[e0:e1].double()
        yield a, x


def _normed(x):
    lib = x.sum(1)
    lib = torch.where(lib == 0, torch.ones_like(lib), lib)
    return torch.log1p(NORM.size_factor * x / lib[:, None]), lib


def _exact_stats(csr, chunk):
    sums, sqs, libs, n = [], [], [], csr.n_rows
    for a, b in chunk_bounds(n, chunk):
        s = q = 0.0
        sub = DeviceCSR(csr.vals, csr.cols, csr.rowptr[a:b + 1], csr.n_cols)
        for _, x in _blocks(sub):
            x, lib = _normed(x)
            s, q = s + x.sum(0), q + (x * x).sum(0)
            libs.append(lib)
        sums.append(s)
        sqs.append(q)
    sums, sqs = torch.stack(sums), torch.stack(sqs)
    counts = torch.tensor([b - a for a, b in chunk_bounds(n, chunk)], device=DEV)
    mu = sums.sum(0) / n
    m2 = torch.zeros_like(mu)
    for _, x in _blocks(csr):
        m2 += ((_normed(x)[0] - mu) ** 2).sum(0)
    sd = (m2 / n).sqrt()
    sd = torch.where(sd == 0, torch.ones_like(sd), sd)
    return dict(mu=mu, sigma=sd, libsize=torch.cat(libs), sums=sums, sumsq=sqs,
                mean=sums / counts[:, None])


def _exact_z(csr, mu, sd):
    for a, x in _blocks(csr):
        z = (_normed(x)[0] - mu) / sd
        yield a, z.clamp(-NORM.clip, NORM.clip)


def _exact_pca(csr, chunk, dims):
    st = _exact_stats(csr, chunk)
    bounds = chunk_bounds(csr.n_rows, chunk)
    order = [b for b in bounds[1:]] + [bounds[0]]
    if any(b - a < dims + 1 for a, b in order):
        return None
    V = S2 = mean = None
    seen = 0
    for a, b in order:
        sub = DeviceCSR(csr.vals, csr.cols, csr.rowptr[a:b + 1], csr.n_cols)
        n, G, s = b - a, 0.0, 0.0
        for _, z in _exact_z(sub, st["mu"], st["sigma"]):
            G, s = G + z.T @ z, s + z.sum(0)
        bm = s / n
        M = G - n * torch.outer(bm, bm)
        if seen:
            mc = math.sqrt(seen * n / (seen + n)) * (mean - bm)
            M = M + (V.T * S2) @ V + torch.outer(mc, mc)
        w, U = np.linalg.eigh(M.cpu().numpy())
        S2 = torch.from_numpy(w[::-1][:dims + 1].copy()).to(DEV)
        V = torch.from_numpy(U[:, ::-1][:, :dims + 1].T.copy()).to(DEV)
        at = V.abs().argmax(1)
        V = V * torch.sign(V[torch.arange(dims + 1, device=DEV), at])[:, None]
        mean = bm if not seen else (mean * seen + s) / (seen + n)
        seen += n
    return dict(loadings=V[:-1].T, var=S2 / (seen - 1), mean=mean)


def _exact_project(csr, W, mu, sd):
    W = torch.from_numpy(W).to(DEV) if isinstance(W, np.ndarray) else W
    return torch.cat([z @ W for _, z in _exact_z(csr, mu, sd)])


def _exact_smooth(dist, idx, chunk):
    d = dist.double()
    n, k = d.shape
    first = torch.where(d > 0, d, torch.full_like(d, math.inf)).min(1).values
    rho = torch.where(torch.isinf(first), torch.zeros_like(first), first)
    gap = d[:, 1:] - rho[:, None]
    target = math.log2(k) * 1.5
    lo = torch.zeros(n, dtype=torch.float64, device=DEV)
    hi = torch.full_like(lo, math.inf)
    mid = torch.ones_like(lo)
    done = torch.zeros(n, dtype=torch.bool, device=DEV)
    for _ in range(64):
        psum = torch.where(gap > 0, torch.exp(-gap / mid[:, None]), torch.ones_like(gap)).sum(1)
        done |= (psum - target).abs() < 1e-5
        up = (psum > target) & ~done
        down = ~up & ~done
        hi, lo = torch.where(up, mid, hi), torch.where(down, mid, lo)
        new = torch.where(torch.isinf(hi), mid * 2, (lo + hi) / 2)
        mid = torch.where(done, mid, new)
    chunks = torch.arange(n, device=DEV) // chunk
    total = torch.zeros(int(chunks[-1]) + 1, dtype=torch.float64, device=DEV)
    cmean = total.index_add(0, chunks, d.mean(1)) / torch.bincount(chunks)
    floor = 1e-3 * torch.where(rho > 0, d.mean(1), cmean[chunks])
    sigma = torch.maximum(mid, floor)
    g = d - rho[:, None]
    w = torch.where(g <= 0, torch.ones_like(g), torch.exp(-g / sigma[:, None]))
    w[idx == (torch.arange(n, device=DEV) - chunks * chunk)[:, None]] = 0.0
    least = 1.0
    for c in range(int(chunks[-1]) + 1):
        wc = w[c * chunk:(c + 1) * chunk]
        if bool((wc == 0).any()) and bool((wc > 0).any()):
            least = min(least, float(wc[wc > 0].min()))
    return sigma, rho, torch.where(w == 0, torch.full_like(w, least), w).reshape(-1)


def exact(case, seed):
    op = case["op"]
    if op in ("query", "selfknn"):
        nq, nr = (case["nq"], case["nr"]) if op == "query" else (case["n"], case["n"])
        # the FP8 screen is approximate by choice, and the largest take too long
        if case["screen"] == "fp8" or nq * nr > 1.5e10:
            return None
        R = _embedding(nr, case["D"], case["groups"], seed)
        Q = R if op == "selfknn" else _embedding(nq, case["D"], case["groups"], seed, 2)
        return None, _exact_knn(Q, R, case["k"], op == "selfknn"), None
    if op == "smooth":
        s = prepare(case, seed)
        return _exact_smooth(s["dist"], s["idx"], case["chunk"])
    csr = _counts(case, seed)
    if op == "stats":
        return _exact_stats(csr, case["chunk"])
    if op == "pca":
        return _exact_pca(csr, case["chunk"], case["dims"])
    st = _exact_stats(csr, 50_000)
    W = _loadings(case["d"], case["dims"], seed)
    E = _exact_project(csr, W, st["mu"], st["sigma"])
    if op == "project":
        return E
    dist = _exact_knn(E, E, case["k"], True)
    return dict(mu=st["mu"], sigma=st["sigma"], embedding=E, indices=None, distances=dist,
                weights=None)
