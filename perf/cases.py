"""The work that programs built on this framework have it do, as cases that can be timed.

Every case goes through the public entry points of the package: the sparse product on a kept operator
(``AccelSpMM.run`` and its strided and epilogue forms), the GCN layer around it (``GcnLayer.forward``), an operator
for a graph that has just arrived (create, preprocess, one product), new edge weights in front of a product
(``update_values_async``), and the partition stage on host arrays (``accel_partition_gpu``, called through ctypes the
way the reference's script would call it).  All of them compute in fp32 with int32 indices, the only types the
operator has; there is no backward path.

Graphs are synthetic with self-loops, made on the GPU from the seed.  Shapes follow the framework's own benchmark
workloads (10 k to 2.45 M nodes, 200 k to 125 M non-zeros, 2 to 500 non-zeros per row) and the reference's sweep over
every column count from 16 to 128.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import __graft_entry__

pkg = __graft_entry__.load_package()

# ---------------------------------------------------------------------------------------------------------------
# what is measured
# ---------------------------------------------------------------------------------------------------------------
# The kinds of graph, each from one of the framework's workloads.
CITATION = {"graph": "powerlaw", "nodes": 170_000, "nnz": 2_450_000, "gamma": 2.3, "max_degree": 15_000}
COPURCHASE = {"graph": "powerlaw", "nodes": 2_450_000, "nnz": 125_000_000, "gamma": 2.1, "max_degree": 17_000}

MAX_NNZ = COPURCHASE["nnz"]
MAX_GATHERED = 100 * MAX_NNZ          # non-zeros times columns of the largest listed product
MAX_FLOPS = 2.0 * 1_000_000 * 602 * 128   # the dense half of the largest listed layer


def listed():
    return [
        # A teaching-size graph: one launch of some ten microseconds, so launches and the host path count.
        {"name": "product small", "call": "product", "graph": "powerlaw", "nodes": 10_000, "nnz": 208_000,
         "gamma": 2.5, "max_degree": 400, "N": 32},
        # A citation network at an odd column count, rows packed: one step of the reference's sweep over 16..128.
        {"name": "product citation odd", "call": "product", **CITATION, "N": 99},
        # A social network with dense neighbourhoods: 490 non-zeros per row, lognormal degrees.
        {"name": "product social", "call": "product", "graph": "lognormal", "nodes": 233_000, "nnz": 114_000_000,
         "sigma": 1.2, "max_degree": 21_000, "N": 64},
        # A co-purchase network, the benchmark's default workload.
        {"name": "product copurchase", "call": "product", **COPURCHASE, "N": 64},
        # The same with rows that do not end on a cache line (100 features).
        {"name": "product copurchase 100", "call": "product", **COPURCHASE, "N": 100},
        # Extreme skew: 64 hub rows hold a third of the non-zeros, most other rows hold one or two; wide rows of X.
        {"name": "product hub", "call": "product", "graph": "hub", "nodes": 1_000_000, "nnz": 30_000_000,
         "gamma": 1.8, "N": 256},
        # A batch of molecules: two non-zeros per row, next to the diagonal.
        {"name": "product molecules", "call": "product", "graph": "local", "nodes": 1_890_000, "nnz": 4_000_000,
         "spread": 16, "N": 64},
        # A GCN layer on wide input features (602 of them), bias and ReLU included.
        {"name": "layer features", "call": "layer", "graph": "powerlaw", "nodes": 1_000_000, "nnz": 10_000_000,
         "gamma": 2.3, "max_degree": 15_000, "K": 602, "N": 128},
        # A graph that is used once (a sampled subgraph, a mini-batch): operator, preprocessing, one product.
        {"name": "new graph citation", "call": "new graph", **CITATION, "N": 64},
        # The same on the large graph: what a program pays before its first product.
        {"name": "new graph copurchase", "call": "new graph", **COPURCHASE, "N": 64},
        # Edge weights that change on every step of a training loop (attention, dropped edges), narrow features.
        {"name": "new values citation", "call": "new values", **CITATION, "N": 16},
        # The partition stage by itself, on the row pointers of a degree-sorted graph in host memory.
        {"name": "partition copurchase", "call": "partition", **COPURCHASE},
    ]


def _between(rng, lo, hi):
    """A whole number, spread over the logarithm of its range."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    call = rng.choice(["product"] * 6 + ["layer"] * 2 + ["new graph"] * 2 + ["new values", "partition"])
    kind = rng.choice(["powerlaw", "powerlaw", "powerlaw", "lognormal", "hub", "local"])
    if call == "partition":
        kind = "powerlaw"
    nodes = _between(rng, 10_000, 2_450_000)
    mean = {"powerlaw": (3, 60), "lognormal": (50, 500), "hub": (8, 40), "local": (2, 8)}[kind]
    nnz = min(int(nodes * math.exp(rng.uniform(math.log(mean[0]), math.log(mean[1])))), MAX_NNZ, nodes * nodes // 16)
    nnz = max(nnz, 2 * nodes)
    case = {"call": call, "graph": kind, "nodes": nodes, "nnz": nnz}
    if kind == "powerlaw":
        case["gamma"] = round(rng.uniform(2.1, 2.5), 3)
        case["max_degree"] = min(int(nnz / nodes * math.exp(rng.uniform(math.log(20), math.log(1000)))), nodes // 10)
    elif kind == "lognormal":
        case["sigma"], case["max_degree"] = 1.2, min(45 * nnz // nodes, nodes // 10)
    elif kind == "hub":
        case["gamma"] = round(rng.uniform(1.6, 2.0), 3)
    else:
        case["spread"] = _between(rng, 8, 2_000)        # how far from the diagonal the columns lie
    if call == "partition":
        return case
    N = _between(rng, 8, 256)
    while nnz * N > MAX_GATHERED:
        N = _between(rng, 8, 256)
    case["N"] = N
    if call == "layer":
        case["K"] = min(_between(rng, 16, 700), max(16, int(MAX_FLOPS / (2.0 * nodes * N))))
    elif call == "product":
        case["epilogue"] = rng.random() < 0.25          # bias and ReLU in the product's store
        case["padded"] = rng.random() < 0.2             # rows of X and Y padded to whole cache lines
    return case


# ---------------------------------------------------------------------------------------------------------------
# graphs
# ---------------------------------------------------------------------------------------------------------------
def _powerlaw_offset(n, total, w_max, alpha):
    """i0 such that total * (i + i0) ** -alpha / sum_j (j + i0) ** -alpha is w_max at i = 0."""
    lo, hi, e = 1e-3, float(n), 1.0 - alpha
    for _ in range(100):
        mid = math.sqrt(lo * hi)
        peak = total * e / ((n + mid) ** e - mid ** e) * mid ** -alpha
        lo, hi = (mid, hi) if peak > w_max else (lo, mid)
    return math.sqrt(lo * hi)


def _weights(case, gen):
    """Expected row degrees and column popularities (up to a factor), fp64 on the GPU."""
    n, edges = case["nodes"], case["nnz"] - case["nodes"]
    relabel = torch.randperm(n, generator=gen, device="cuda")
    if case["graph"] == "powerlaw":
        alpha = 1.0 / (case["gamma"] - 1.0)
        i0 = _powerlaw_offset(n, edges, case["max_degree"], alpha)
        w = (torch.arange(n, dtype=torch.float64, device="cuda") + i0) ** -alpha
        return w[relabel], w[relabel]
    if case["graph"] == "lognormal":
        w = torch.exp(torch.randn(n, generator=gen, device="cuda", dtype=torch.float64) * case["sigma"])
        w = torch.clamp(w * (edges / w.sum()), max=float(case["max_degree"]))
        return w, w
    # hub: 64 rows share a third of the edges, the others follow a truncated Zipf law; popular columns (rank ** -0.8)
    # with the hubs as the most popular
    u = torch.rand(n, generator=gen, device="cuda", dtype=torch.float64).clamp_min(1e-6)
    tail = torch.clamp(u ** (-1.0 / (case["gamma"] - 1.0)), max=n / 40)
    tail[relabel[:64]] = 0
    rows = tail * (edges * 2 / 3 / tail.sum())
    hubs = 0.25 + torch.rand(64, generator=gen, device="cuda", dtype=torch.float64)
    rows[relabel[:64]] = hubs * (edges / 3 / hubs.sum())
    cols = torch.empty_like(rows)
    cols[relabel] = torch.arange(1, n + 1, dtype=torch.float64, device="cuda") ** -0.8
    return rows, cols


def _csr(case, gen):
    """A square matrix with exactly case["nnz"] non-zeros: every diagonal entry, and distinct off-diagonal ones drawn
    at random.  int32 row pointers and columns (ascending within a row), fp32 values, on the GPU."""
    n, edges = case["nodes"], case["nnz"] - case["nodes"]
    if case["graph"] == "local":
        def ends(count):
            src = torch.randint(n, (count,), generator=gen, device="cuda")
            off = torch.randn(count, generator=gen, device="cuda") * case["spread"]
            return src, (src + off.round().long()).clamp_(0, n - 1)
    else:
        cdfs = [w.cumsum(0).div_(w.sum()) for w in _weights(case, gen)]

        def ends(count):
            return [torch.searchsorted(c, torch.rand(count, generator=gen, device="cuda", dtype=torch.float64),
                                       right=True).clamp_(max=n - 1) for c in cdfs]
    key = torch.empty(0, dtype=torch.int64, device="cuda")
    while key.numel() < edges:
        src, dst = ends(int((edges - key.numel()) * 1.15) + 1024)
        new = (src * n + dst)[src != dst]
        del src, dst
        key = torch.unique(torch.cat([key, new]))
        del new
    if key.numel() > edges:                             # drop the surplus at random
        key = key[torch.randperm(key.numel(), generator=gen, device="cuda")[:edges]]
    loops = torch.arange(n, dtype=torch.int64, device="cuda") * (n + 1)
    key = torch.cat([key, loops]).sort().values
    rows = key // n
    cols = key - rows * n
    del key
    deg = torch.bincount(rows, minlength=n)
    indptr = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(deg, 0, out=indptr[1:])
    if case["graph"] == "hub":
        values = 1.0 - torch.rand(case["nnz"], generator=gen, device="cuda")
    else:                                               # GCN normalisation
        inv = deg.float().rsqrt()
        values = inv[rows] * inv[cols]
    return indptr.int(), cols.int(), values


def _degrees(case):
    """The expected degrees of a power-law graph, ascending, on the host."""
    n, edges = case["nodes"], case["nnz"] - case["nodes"]
    alpha = 1.0 / (case["gamma"] - 1.0)
    w = (np.arange(n, dtype=np.float64) + _powerlaw_offset(n, edges, case["max_degree"], alpha)) ** -alpha
    return np.sort(w * (edges / w.sum()))


# ---------------------------------------------------------------------------------------------------------------
# one case
# ---------------------------------------------------------------------------------------------------------------
def _stride(case):
    return (case["N"] + 31) // 32 * 32 if case.get("padded") else case["N"]


def prepare(case, seed):
    if case["call"] == "partition":
        rng = np.random.default_rng(seed)
        n = case["nodes"]
        indptr = np.zeros(n + 1, dtype=np.int64)
        np.cumsum(np.sort(rng.poisson(_degrees(case)) + 1), out=indptr[1:])
        capacity = n + 2 * case["nnz"] // pkg._lib.DEG_BOUND
        return {"case": case, "indptr": indptr.astype(np.int32), "block4": np.zeros((capacity, 4), dtype=np.int32)}
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    csr = _csr(case, gen)
    n, N, ld = case["nodes"], case["N"], _stride(case)

    def uniform(*shape):                                # features and weights in [-1, 1)
        return torch.rand(*shape, generator=gen, device="cuda").mul_(2.0).sub_(1.0)

    state = {"case": case, "csr": csr, "Y": torch.zeros(n, ld, device="cuda")}
    if case["call"] == "layer":
        state["X"] = uniform(n, case["K"])
        W = uniform(case["K"], N).mul_(case["K"] ** -0.5).cpu().numpy()
        bias = uniform(N).mul_(0.1).cpu().numpy()
    else:
        state["X"] = uniform(n, ld)
    if case["call"] != "new graph":
        state["op"] = pkg.AccelSpMM(*csr, n, device=True, n_rows=n, nnz=case["nnz"]).preprocess()
    if case["call"] == "layer":
        state["layer"] = pkg.GcnLayer(state["op"], W, bias, relu=True)
    elif case["call"] == "new values":
        state["values"] = uniform(case["nnz"])
    elif case.get("epilogue"):
        state["bias"] = uniform(N)
    return state


def run(state):
    case = state["case"]
    if case["call"] == "partition":
        indptr, block4, count = state["indptr"], state["block4"], ctypes.c_int64(0)
        pkg._lib.check(pkg.lib().accel_partition_gpu(
            pkg._lib.ptr(indptr, ctypes.c_int32), indptr.size - 1, pkg._lib.ptr(block4, ctypes.c_int32),
            block4.shape[0], ctypes.byref(count)))
        return block4, count.value
    X, Y, N = state["X"], state["Y"], case["N"]
    if case["call"] == "layer":
        state["layer"].forward(X, Y)
        return Y
    if case["call"] == "new graph":
        op = pkg.AccelSpMM(*state["csr"], case["nodes"], device=True, n_rows=case["nodes"], nnz=case["nnz"])
        op.preprocess()
        op.run(X, Y, N)
        op.close()
        return Y
    op = state["op"]
    if case["call"] == "new values":
        op.update_values_async(state["values"])
        op.run(X, Y, N)
    elif case.get("epilogue"):
        op.run_ex(X, Y, N, ld=_stride(case), bias=state["bias"], relu=True)
    elif case.get("padded"):
        op.run_strided(X, Y, N, _stride(case))
    else:
        op.run(X, Y, N)
    return Y


def _rows_per_block(d):
    """Rows of degree d in one entry of the partition's metadata (d up to 384)."""
    return np.select([d <= 32, d <= 64, d <= 96, d <= 128, d < 192], [12, 6, 4, 3, 2], 1)


def work(case):
    n, nnz = case["nodes"], case["nnz"]
    if case["call"] == "partition":                     # row pointers in, 16 bytes per entry out
        deg = np.rint(_degrees(case)).astype(np.int64) + 1
        d, count = np.unique(deg, return_counts=True)
        entries = np.where(d <= 384, -(-count // _rows_per_block(d)), count * -(-d // 384)).sum()
        return {"bytes": 4 * (n + 1) + 16 * int(entries), "flops": 0}
    N = case["N"]
    b = 4 * (n + 1) + 8 * nnz + 2 * 4 * n * N           # the matrix, X and Y
    f = 2 * nnz * N
    if case["call"] == "layer":                         # features and weights in the place of X
        K = case["K"]
        b += 4 * (n * K + K * N + N) - 4 * n * N
        f += 2 * n * K * N
    elif case.get("epilogue"):
        b += 4 * N
    return {"bytes": b, "flops": f}


def tolerance(case):
    if case["call"] == "partition":
        return "exact"
    return {"rel": 1e-5, "max": 1e-4}                   # fp32 sums in another order
