"""The framework's measured workloads: whole clusterings and the stages a program calls by themselves.

Every case is one call through the public entry points (grappolo_amd.engine,
grappolo_amd.active_set) on a seeded graph.  Graph kinds: "planted" (planted
partition, 16 entries per vertex, unit weights), "lfr" (power-law degrees 10 to
1000 and communities, weights uniform in [0.5, 2] or all 1) and "rmat"
(a/b/c/d 0.57/0.19/0.19/0.05, edge factor 16, symmetrised, unit weights; a
vertex count below the power of two keeps the edges among the lowest ids).
"""
import math
import random

import numpy as np
import torch

from grappolo_amd import active_set, engine, graph

DEV = "cuda"


def listed():
    return [
        # the smallest whole run (the smoke check's size): launches, host reads and step latency
        {"name": "run_planted_4k", "do": "run", "kind": "planted", "nv": 4096, "unit": True, "coloring": 1,
         "min_graph": 100},
        # a caller of the C API with host arrays: upload, run, labels back, on the 65,536-vertex configuration
        {"name": "run_planted_64k_host", "do": "run_host", "kind": "planted", "nv": 65536, "unit": True, "coloring": 1,
         "min_graph": 1000},
        # a weighted social-network-like graph, device resident: binned sweeps, then dense coarse phases
        {"name": "run_lfr_1m", "do": "run", "kind": "lfr", "nv": 1048576, "unit": False, "coloring": 1,
         "min_graph": 1000},
        # a hub-heavy graph of middling, odd size: persistent coarse sweeps from the first phase on
        {"name": "run_rmat_250k", "do": "run", "kind": "rmat", "nv": 250007, "unit": True, "coloring": 1,
         "min_graph": 1000},
        # the largest: the headline workload's generator at 4.2 million vertices, about 130 million entries
        {"name": "run_rmat_4m", "do": "run", "kind": "rmat", "nv": 4194304, "unit": True, "coloring": 1,
         "min_graph": 1000},
        # the uncolored driver (driverForGraphClustering without -c)
        {"name": "basic_lfr_200k", "do": "basic", "kind": "lfr", "nv": 200003, "unit": True, "no_map": False},
        # many small independent graphs in one call
        {"name": "basic_batch_128", "do": "batch", "graphs": 128},
        # the coloring alone (stage entry point)
        {"name": "color_rmat_1m", "do": "color", "kind": "rmat", "nv": 1048576, "unit": True},
        # quality of a given labelling, FP64 weights
        {"name": "modularity_lfr_1m", "do": "modularity", "kind": "lfr", "nv": 1048576, "unit": False},
        # the driver's vertex-following fold (-v): follow, renumber, contract
        {"name": "fold_rmat_1m", "do": "fold", "kind": "rmat", "nv": 1048576, "unit": True},
        # driverForClusterComparison on two labellings in device memory
        {"name": "compare_2m", "do": "compare", "nv": 2000003, "truth": 4000, "found": 3000},
        # the learned active set: loss and gradient of its network over trace rows
        {"name": "predictor_grad_256k", "do": "grad", "rows": 262144},
    ]


def _between(rng, lo, hi):
    """An odd whole number, log-uniform in [lo, hi]."""
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi)))) | 1


def draw(rng):
    do = rng.choice(["run", "run", "run", "run", "run_host", "basic", "batch", "color", "modularity", "fold", "compare",
                     "grad"])
    if do == "batch":
        return {"do": do, "graphs": _between(rng, 16, 160)}
    if do == "compare":
        return {"do": do, "nv": _between(rng, 20000, 4000000), "truth": _between(rng, 20, 8000),
                "found": _between(rng, 20, 8000)}
    if do == "grad":
        return {"do": do, "rows": _between(rng, 4096, 2000000)}
    kind = rng.choice(["planted", "lfr", "rmat"]) if do != "fold" else "rmat"  # the other kinds have nothing to fold
    top = {"planted": 500000, "lfr": 1000000, "rmat": 3000000}[kind]
    if do == "run_host":
        top = 200000
    c = {"do": do, "kind": kind, "nv": _between(rng, 3000 if kind != "rmat" else 10000, top),
         "unit": kind != "lfr" or rng.random() < 0.5}
    if do in ("run", "run_host"):
        c["coloring"] = rng.choice([1, 1, 1, 2, 3]) if kind != "rmat" else 1
        c["min_graph"] = rng.choice([100, 1000])
    if do == "basic":
        c["no_map"] = rng.random() < 0.3
    return c


# ------------------------------------------------------------------- inputs
def _csr(nv, key):
    """Unit-weight DeviceGraph of the entries row * nv + tail."""
    key = torch.sort(key).values
    off = torch.zeros(nv + 1, dtype=torch.int64, device=DEV)
    off[1:] = torch.cumsum(torch.bincount(key // nv, minlength=nv), 0)
    tails = key % nv
    w = torch.ones(tails.shape[0], dtype=torch.float64, device=DEV)
    return engine.DeviceGraph.from_tensors(off, tails, w, tails.shape[0] // 2)


def _renamed(dg, seed):
    """The same graph with its vertices in another order: as many folded vertices and entries whatever the seed."""
    nv = dg.numVertices
    to = torch.randperm(nv, generator=torch.Generator(device=DEV).manual_seed(seed), device=DEV)
    rows = torch.repeat_interleave(torch.arange(nv, device=DEV), dg.off[1:] - dg.off[:-1])
    return _csr(nv, to[rows] * nv + to[dg.tails])


def _rmat(nv, seed):
    """Symmetric CSR of an RMAT graph, built on the device."""
    scale = max(1, (nv - 1).bit_length())
    g = torch.Generator(device=DEV).manual_seed(seed)
    m = 16 << scale
    u = torch.zeros(m, dtype=torch.int64, device=DEV)
    v = torch.zeros_like(u)
    for _ in range(scale):
        r = torch.rand(m, generator=g, device=DEV)
        u = 2 * u + (r >= 0.76)
        v = 2 * v + (((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
    keep = (u != v) & (u < nv) & (v < nv)
    u, v = u[keep], v[keep]
    key = torch.unique(torch.minimum(u, v) * nv + torch.maximum(u, v))
    u, v = key // nv, key % nv
    return _csr(nv, torch.cat([key, v * nv + u]))


def _host_graph(case, seed):
    if case["kind"] == "planted":
        return graph.gen_planted(case["nv"], max(4, case["nv"] // 1024), 16, 0.3, seed=seed)
    lo, hi = (1.0, 1.0) if case["unit"] else (0.5, 2.0)
    return graph.gen_lfr(case["nv"], seed=seed, wlo=lo, whi=hi)


def _device_graph(case, seed):
    return _rmat(case["nv"], seed) if case["kind"] == "rmat" else engine.DeviceGraph(_host_graph(case, seed), DEV)


def prepare(case, seed):
    do = case["do"]
    gen = torch.Generator(device=DEV).manual_seed(seed)
    if do == "grad":
        # trace rows: features in about [-1, 1], one row in eight a mover
        feats = (torch.rand(case["rows"], 8, generator=gen, device=DEV) * 2 - 1).to(torch.bfloat16)
        labels = (torch.rand(case["rows"], generator=gen, device=DEV) < 0.125).to(torch.uint8)
        return {"case": case, "P": active_set.init_params(seed, DEV), "feats": feats.view(torch.int16), "labels": labels}
    if do == "compare":
        # a truth of skewed community sizes and a clustering that agrees with it on most vertices
        n = case["nv"]
        truth = (torch.rand(n, generator=gen, device=DEV).square() * case["truth"]).long()
        other = (torch.rand(n, generator=gen, device=DEV) * case["found"]).long()
        found = torch.where(torch.rand(n, generator=gen, device=DEV) < 0.7, truth % case["found"], other)
        truth[0] = found[0] = 0
        return {"case": case, "truth": truth, "found": found}
    if do == "batch":
        # the batched configuration: sizes log-uniform on [100, 50000], degrees 8 to 32, mixing 0.1 to 0.5
        rng = random.Random(5)  # the sizes are the configuration's, the graphs the seed's
        specs = []
        for i in range(case["graphs"]):
            nv = int(math.exp(rng.uniform(math.log(100), math.log(50000))))
            blocks = int(math.exp(rng.uniform(math.log(4), math.log(256))))
            specs.append((nv, min(blocks, nv), rng.uniform(8, 32), rng.uniform(0.1, 0.5), 1000 * seed + i))
        U, vbase = graph.union(graph.gen_planted_many(specs))
        dg = engine.DeviceGraph(U, DEV)
        return {"case": case, "dg": dg, "vbase": vbase, "C": torch.empty(dg.numVertices, dtype=torch.int64, device=DEV)}
    if do == "run_host":
        if case["kind"] == "rmat":
            return {"case": case, "G": _rmat(case["nv"], seed).to_host()}
        return {"case": case, "G": _host_graph(case, seed)}
    dg = _renamed(_rmat(case["nv"], 3), seed) if do == "fold" else _device_graph(case, seed)
    state = {"case": case, "dg": dg}
    if do == "color":
        state["colors"] = torch.empty(dg.numVertices, dtype=torch.int32, device=DEV)
    else:
        state["C"] = torch.full((dg.numVertices,), -1, dtype=torch.int64, device=DEV)
    if do == "modularity":
        # communities of about 64 consecutive vertices, one vertex in four elsewhere; isolated vertices have none
        nv = dg.numVertices
        ids = torch.arange(nv, device=DEV)
        stray = torch.rand(nv, generator=gen, device=DEV) < 0.25
        at = torch.where(stray, torch.randint(0, nv, (nv,), generator=gen, device=DEV), ids) // 64
        state["C"] = torch.where(dg.off[1:] > dg.off[:-1], at, -1)
    return state


# -------------------------------------------------------------------- passes
def run(state):
    case = state["case"]
    do = case["do"]
    if do == "run":
        st = engine.run_colored_dev(state["dg"], state["C"], coloring=case["coloring"], minGraphSize=case["min_graph"])
        return {"labels": state["C"], "modularity": st["final_modularity"], "iterations": st["total_iterations"]}
    if do == "run_host":
        C, st = engine.runMultiPhaseColoring(state["G"], coloring=case["coloring"], minGraphSize=case["min_graph"])
        return {"labels": C, "modularity": st["final_modularity"], "iterations": st["total_iterations"]}
    if do == "basic":
        st = engine.run_basic_dev(state["dg"], state["C"], basicOpt=int(case["no_map"]))
        return {"labels": state["C"], "modularity": st["final_modularity"], "iterations": st["total_iterations"]}
    if do == "batch":
        r = engine.run_basic_batch_dev(state["dg"], state["vbase"], state["C"])
        return {"labels": state["C"], "modularity": r["final_modularity"], "iterations": r["total_iterations"]}
    if do == "color":
        largest, _ = engine.color_dev(state["dg"], state["colors"])
        return {"colors": state["colors"], "largest": largest}
    if do == "modularity":
        return {"modularity": engine.modularity_dev(state["dg"], state["C"])}
    if do == "fold":
        dg, folded = engine.vertex_following_prepass_dev(state["dg"])
        return {"off": dg.off, "tails": dg.tails, "weights": dg.w, "folded": folded}
    if do == "compare":
        return engine.compare_dev(state["truth"], state["found"])
    loss, grad = active_set.grad_dev(state["P"], state["feats"], state["labels"], pos_weight=7.0)
    return {"loss": loss, "grad": grad}


def _entries(case):
    """About the directed entries of the case's graph."""
    return {"planted": 16, "lfr": 24.6, "rmat": 30}[case["kind"]] * case["nv"]


def work(case):
    do = case["do"]
    if do == "grad":
        # 16 bytes of features and a label per row; 4608 multiply-adds a row forward, twice that backward
        return {"bytes": 17 * case["rows"] + 8 * 4801, "flops": 3 * 2 * 4672 * case["rows"]}
    if do == "compare":
        return {"bytes": 16 * case["nv"], "flops": 0}
    if do == "batch":
        nv = 8030 * case["graphs"]  # mean of the log-uniform sizes
        return {"bytes": 16 * 20 * nv + 16 * nv, "flops": 0}
    # the graph once: tail and weight per entry (the coloring reads no weights), an offset and a label per vertex
    per_entry = 8 if do == "color" else 16
    return {"bytes": per_entry * _entries(case) + 16 * case["nv"], "flops": 0}


def tolerance(case):
    do = case["do"]
    if do in ("color", "fold"):
        return "exact"  # whole numbers, and sums of whole numbers
    if do == "grad":
        return {"rel": 1e-2}  # BF16 weights and activations, FP32 sums
    if do == "compare":
        return {"rel": 1e-13}  # counts are exact; a few double operations on them
    if do in ("run", "run_host") and not case["unit"]:
        # FP64 sums in another order can flip a vertex whose two best gains
        # agree to rounding, and what follows from it
        return {"rel": 1e-4, "differ": 0.01}
    return {"rel": 1e-12}  # FP64 sums over up to 2e8 terms in another order; labels are exact


# ----------------------------------------------------- the same in plain torch
def _exact_modularity(dg, C):
    nv = dg.numVertices
    rows = torch.repeat_interleave(torch.arange(nv, device=DEV), dg.off[1:] - dg.off[:-1])
    k = torch.zeros(nv, dtype=torch.float64, device=DEV).index_add_(0, rows, dg.w)
    total = k.sum()
    inside = dg.w[C[rows] == C[dg.tails]].sum()
    has = C >= 0
    a = torch.zeros(nv, dtype=torch.float64, device=DEV).index_add_(0, C[has], k[has])
    return float(inside / total - (a / total).square().sum())


def _exact_fold(dg):
    nv = dg.numVertices
    deg = dg.off[1:] - dg.off[:-1]
    rows = torch.repeat_interleave(torch.arange(nv, device=DEV), deg)
    ids = torch.arange(nv, device=DEV)
    to = dg.tails[dg.off[:-1].clamp(max=max(dg.nnz - 1, 0))]
    follows = (deg == 1) & ((deg[to] > 1) | (ids > to))
    C = torch.where(deg == 0, -1, torch.where(follows, to, ids))
    folded = int(((deg == 0) | follows).sum())
    # clusters in order of their first vertex
    first = torch.full((nv,), nv, dtype=torch.int64, device=DEV)
    has = C >= 0
    first.scatter_reduce_(0, C[has], ids[has], "amin")
    heads = torch.zeros(nv, dtype=torch.int64, device=DEV)
    heads[first[first < nv]] = 1
    rank = torch.cumsum(heads, 0) - 1
    k = int(heads.sum())
    L = torch.where(has, rank[first[C.clamp(min=0)].clamp(max=nv - 1)], -1)
    a, b, w = L[rows], L[dg.tails], dg.w.trunc()
    # a pair inside one cluster counts once per entry, one across once per direction
    key, at = torch.unique(a * k + b, return_inverse=True)
    sums = torch.zeros(key.shape[0], dtype=torch.float64, device=DEV).index_add_(0, at, w)
    off = torch.zeros(k + 1, dtype=torch.int64, device=DEV)
    off[1:] = torch.cumsum(torch.bincount(key // k, minlength=k), 0)
    return {"off": off, "tails": key % k, "weights": sums, "folded": folded}


def _gini(sizes):
    s = torch.sort(sizes.double()).values
    n = s.shape[0]
    i = torch.arange(1, n + 1, device=DEV, dtype=torch.float64)
    return float(2 * (i * s).sum() / (n * s.sum()) - (n + 1) / n)


def _exact_grad(state):
    P = state["P"].double().requires_grad_(True)
    X = state["feats"].view(torch.bfloat16).double()
    y = state["labels"].double()
    loss = torch.zeros((), dtype=torch.float64, device=DEV)
    n = X.shape[0]
    w1, b1, w2 = P[:512].view(8, 64), P[512:576], P[576:4672].view(64, 64)
    b2, w3, b3 = P[4672:4736], P[4736:4800], P[4800]
    for lo in range(0, n, 1 << 18):
        x, t = X[lo:lo + (1 << 18)], y[lo:lo + (1 << 18)]
        z = torch.relu(torch.relu(x @ w1 + b1) @ w2 + b2) @ w3 + b3
        each = 7.0 * t * torch.nn.functional.softplus(-z) + (1 - t) * torch.nn.functional.softplus(z)
        part = each.sum() / n
        part.backward()
        loss = loss + part.detach()
    return {"loss": float(loss), "grad": P.grad}


def exact(case, seed):
    do = case["do"]
    if do not in ("modularity", "fold", "compare", "grad"):
        return None  # a run's labels and its quality have no value apart from the method
    state = prepare(case, seed)
    if do == "modularity":
        return {"modularity": _exact_modularity(state["dg"], state["C"])}
    if do == "fold":
        return _exact_fold(state["dg"])
    if do == "grad":
        return _exact_grad(state)
    a, b = state["truth"], state["found"]
    na, nb = int(a.max()) + 1, int(b.max()) + 1
    pairs = lambda c: int((c * (c - 1) // 2).sum())  # noqa: E731
    ca, cb = torch.bincount(a, minlength=na), torch.bincount(b, minlength=nb)
    same = pairs(torch.bincount(a * nb + b))
    split, merged = pairs(ca) - same, pairs(cb) - same
    p, r = same / (same + merged), same / (same + split)
    return {"nC1": na, "nC2": nb, "SameSame": same, "SameDiff": split, "DiffSame": merged, "Agree": None, "precision": p,
            "recall": r, "fScore": 2 * p * r / (p + r), "gini1": _gini(ca), "gini2": _gini(cb)}
