"""The measured work: triangle counts as a program of this library asks for them.

A case is one call (or one round of calls) through the Python binding, on
inputs made from a seed:

  count     a resident graph counted whole, with the autotuner's spread,
            bitmap length, kernel and block shape for it: the library's main
            call, over its range of sizes, skewed (R-MAT) and flat
            (Erdos-Renyi), with 4- and 8-byte row offsets
  range     one of `parts` equal wedge ranges of a resident graph: what one
            GPU of several, or one step of a chunked count, does
  drop_in   the reference's own call tc_GPU: a host CSR in, the count out,
            everything allocated, copied and freed inside the call
  batch     many graphs resident as one set, replayed as one launch
  serve     a round of requests through the server: all submitted, then all
            waited for
  build     an edge list in host memory built into an oriented resident
            graph on the GPU and counted once

prepare() makes what such a program holds before the call: the resident
graph, batch or server with its context, or the host arrays.  Every state has
a context of its own, as every thread of a program has.
"""
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "wedge-parallel-triangle-counting_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import workloads  # noqa: E402
import wtc  # noqa: E402

# Distinct oriented edges of an R-MAT graph per vertex of 2^scale (edge
# factor 16) and its wedges, measured at seed 1; work() interpolates by them.
_RMAT_EDGES = {12: 11.9, 16: 14.0, 20: 14.97, 24: 15.52, 28: 15.78}
_RMAT_LOG2_WEDGES = {12: 19.6, 16: 24.8, 20: 30.2, 24: 35.3, 28: 40.3}


def listed():
    return [
        # a tiny skewed graph: launches and latency
        {"name": "count rmat12", "kind": "count", "family": "rmat", "scale": 12, "edge_factor": 16, "offset_bytes": 0},
        # a small one, below the sizes where the split count starts
        {"name": "count rmat16", "kind": "count", "family": "rmat", "scale": 16, "edge_factor": 16, "offset_bytes": 0},
        # the middle of the skewed range, where the benchmark's sweep of s and a lies
        {"name": "count rmat20", "kind": "count", "family": "rmat", "scale": 20, "edge_factor": 16, "offset_bytes": 0},
        # 8-byte row offsets, the layout of the reference's big-graph programs
        {"name": "count rmat22 o8", "kind": "count", "family": "rmat", "scale": 22, "edge_factor": 16,
         "offset_bytes": 8},
        # the headline benchmark's graph size
        {"name": "count rmat24", "kind": "count", "family": "rmat", "scale": 24, "edge_factor": 16, "offset_bytes": 0},
        # the largest whose states fit the card several times over, 8-byte offsets
        {"name": "count rmat26 o8", "kind": "count", "family": "rmat", "scale": 26, "edge_factor": 16,
         "offset_bytes": 8},
        # flat degrees at an odd size: mesh-like and random networks
        {"name": "count er 1m", "kind": "count", "family": "er", "n": 1000003, "degree": 16, "offset_bytes": 0},
        # the second quarter of a graph's wedges: one of four GPUs
        {"name": "range rmat21 2of4", "kind": "range", "family": "rmat", "scale": 21, "edge_factor": 16,
         "offset_bytes": 0, "part": 1, "parts": 4},
        # the reference's usage example through its own call, with its default s and a
        {"name": "drop_in chung-lu", "kind": "drop_in", "n": 262144, "edges": 900000, "spread": 5, "a": 8192},
        # the batching workload: Erdos-Renyi and Barabasi-Albert graphs, n log-uniform in [64, 65536]
        {"name": "batch 256", "kind": "batch", "graphs": 256},
        # a round of the serving mix: three requests for each of R-MAT 10..18, interleaved
        {"name": "serve rmat10-18", "kind": "serve", "lo": 10, "hi": 18, "rounds": 3},
        # edges as a program collects them, to a resident graph and its count
        {"name": "build rmat18", "kind": "build", "scale": 18, "edge_factor": 16},
    ]


def draw(rng):
    """A case of the same ranges; counts are the most frequent, as in use."""
    kind = rng.choice(["count", "count", "count", "count", "range", "drop_in", "batch", "serve", "build"])
    if kind in ("count", "range"):
        ob = rng.choice([0, 0, 8])
        if rng.random() < 0.3:
            c = {"kind": kind, "family": "er", "n": int(round(2 ** rng.uniform(12, 21.5))) | 1,
                 "degree": rng.randint(6, 40), "offset_bytes": ob}
        else:
            c = {"kind": kind, "family": "rmat", "scale": rng.randint(11, 23), "edge_factor": rng.randint(6, 20),
                 "offset_bytes": ob}
        if kind == "range":
            parts = rng.randint(2, 8)
            c.update(part=rng.randrange(parts), parts=parts)
        return c
    if kind == "drop_in":
        n = int(round(2 ** rng.uniform(12, 19)))
        return {"kind": kind, "n": n, "edges": int(n * rng.uniform(2.0, 8.0)), "spread": rng.choice([1, 3, 5, 8]),
                "a": rng.choice([0, 4096, 8192, 16384])}
    if kind == "batch":
        return {"kind": kind, "graphs": rng.randint(8, 300)}
    if kind == "serve":
        lo = rng.randint(10, 14)
        return {"kind": kind, "lo": lo, "hi": lo + rng.randint(2, 5), "rounds": rng.randint(1, 4)}
    return {"kind": kind, "scale": rng.randint(12, 18), "edge_factor": rng.randint(6, 20)}


def _er_pairs(n, degree, seed):
    """n*degree/2 uniform pairs: G(n, p) with that mean degree but for the few repeats."""
    r = np.random.default_rng(seed)
    return r.integers(0, n, size=(n * degree // 2, 2), dtype=np.uint32)


def _resident(case, seed):
    """The context and resident graph of a count or range case, tuned."""
    ctx = wtc.Context(0)
    if case["family"] == "rmat":
        dg = wtc.DeviceGraph.gen_rmat(ctx, case["scale"], case["edge_factor"], seed=seed + 1,
                                      offset_bytes=case["offset_bytes"])
    else:
        dg = wtc.DeviceGraph.from_pairs(ctx, _er_pairs(case["n"], case["degree"], seed), case["offset_bytes"])
    if dg.m <= 1 << 26:
        wedges = dg.download().wedges()
    else:  # a first count tells it sooner than a copy of the whole graph
        ctx.set_count_kernel(wtc.KERNEL_SPLIT)
        wedges = dg.count(8, 65536, stats=True)[1].wedges
    t = wtc.autotune_shape(dg.n, dg.m, wedges)
    ctx.use_tuned(t)
    return {"ctx": ctx, "dg": dg, "wedges": wedges, "s": int(t.spread), "a": int(t.adjacency_matrix_len)}


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("count", "range"):
        st = _resident(case, seed)
        st["kind"] = "count"
        st["lo"], st["hi"] = 0, 2 ** 64 - 1
        if kind == "range":
            st["lo"] = st["wedges"] * case["part"] // case["parts"]
            st["hi"] = st["wedges"] * (case["part"] + 1) // case["parts"]
        return st
    if kind == "drop_in":
        g = wtc.preprocess(wtc.gen_chung_lu(case["n"], target_edges=case["edges"], seed=seed))
        return {"kind": kind, "g": g, "s": case["spread"], "a": case["a"]}
    if kind == "batch":
        graphs = workloads.batch_graphs(case["graphs"], workloads.BATCH_BASE_SEED + 100003 * (seed % 10007))
        ctx = wtc.Context(0)
        ctx.use_tuned(wtc.autotune_shape(graphs[0].n, graphs[0].m, graphs[0].wedges(), batch=True))
        tune = [wtc.autotune(g.n, g.m, g.wedges(), batch=True) for g in graphs]
        return {"kind": kind, "ctx": ctx, "batch": wtc.Batch(ctx, graphs), "s": [t[0] for t in tune],
                "a": [t[1] for t in tune]}
    if kind == "serve":
        ctx = wtc.Context(0)
        srv = wtc.Server(hbm_budget_bytes=2 << 30)
        gids, params = [], []
        for scale in range(case["lo"], case["hi"] + 1):
            dg = wtc.DeviceGraph.gen_rmat(ctx, scale, 16, seed=seed + 31 * scale)
            g = dg.download()
            dg.free()
            gids.append(srv.register(g))
            params.append(wtc.autotune(g.n, g.m, g.wedges()))
        ctx.close()
        order = [i for _ in range(case["rounds"]) for i in range(len(gids))]
        return {"kind": kind, "srv": srv, "gids": gids, "params": params, "order": order}
    ctx = wtc.Context(0)
    ctx.set_count_kernel(wtc.KERNEL_SPLIT)
    return {"kind": "build", "ctx": ctx,
            "pairs": wtc.gen_rmat_pairs(case["scale"], case["edge_factor"], seed=seed + 1)}


def run(state):
    kind = state["kind"]
    if kind == "count":
        return state["dg"].count(state["s"], state["a"], state["lo"], state["hi"])
    if kind == "drop_in":
        return wtc.tc_gpu(state["g"], state["s"], state["a"])
    if kind == "batch":
        return state["batch"].count(state["s"], state["a"])
    if kind == "serve":
        srv = state["srv"]
        rids = [srv.submit(state["gids"][i], *state["params"][i]) for i in state["order"]]
        return [srv.wait(r)[0] for r in rids]
    dg = wtc.DeviceGraph.from_pairs(state["ctx"], state["pairs"])
    return {"triangles": dg.count(8, min(8192, (dg.n + 31) // 32 * 32)), "n": dg.n, "m": dg.m}


def _between(table, x):
    """Linear in the scale between the table's entries, the ends continued."""
    ks = sorted(table)
    i = max(0, min(len(ks) - 2, sum(k <= x for k in ks) - 1))
    k0, k1 = ks[i], ks[i + 1]
    return table[k0] + (table[k1] - table[k0]) * (x - k0) / (k1 - k0)


def _rmat_size(scale, edge_factor):
    """(n, m, W) of an R-MAT graph, from the measured tables; wedges grow
    with the square of the edge factor."""
    m = _between(_RMAT_EDGES, scale) * edge_factor / 16 * 2.0 ** scale
    return 2.0 ** scale, m, 2.0 ** _between(_RMAT_LOG2_WEDGES, scale) * (edge_factor / 16) ** 2


def work(case):
    """Bytes: the graph read once and the count written (build: the pairs
    read, the graph written).  Operations: one lookup and one addition per
    wedge, which is what the wedge-parallel count is made of."""
    kind = case["kind"]
    if kind in ("count", "range"):
        if case["family"] == "rmat":
            n, m, w = _rmat_size(case["scale"], case["edge_factor"])
        else:
            n, m = float(case["n"]), case["n"] * case["degree"] / 2.0
            # oriented by degree, a flat graph's rows hold about half of each degree
            w = n * ((case["degree"] / 2.0) ** 2 * 1.1) / 2.0
        share = 1.0 / case.get("parts", 1)
        return {"bytes": ((case["offset_bytes"] or 4) * n + 4 * m) * (share if kind == "range" else 1.0) + 8,
                "flops": 2 * w * share}
    if kind == "drop_in":
        return {"bytes": 4.0 * case["n"] + 4.0 * case["edges"] + 8, "flops": 3.2 * case["edges"]}
    if kind == "batch":
        # per graph on average: n 9,400, m 165,000, 1.9e6 wedges
        return {"bytes": case["graphs"] * (4 * 9.4e3 + 4 * 1.65e5 + 8), "flops": 2 * case["graphs"] * 1.9e6}
    if kind == "serve":
        sizes = [_rmat_size(s, 16) for s in range(case["lo"], case["hi"] + 1)]
        return {"bytes": case["rounds"] * sum(4 * n + 4 * m + 8 for n, m, _ in sizes),
                "flops": 2 * case["rounds"] * sum(w for _, _, w in sizes)}
    n, m, w = _rmat_size(case["scale"], case["edge_factor"])
    return {"bytes": 8.0 * case["edge_factor"] * 2 ** case["scale"] + 8 * n + 4 * m + 8, "flops": 2 * w}


def exact(case, seed):
    """The count by a dense product of 64-bit matrices, for the graphs small
    enough: every triangle closes six walks of length three."""
    if case["kind"] != "count" or case["family"] != "rmat" or case["scale"] > 13:
        return None
    g = wtc.gen_rmat(case["scale"], case["edge_factor"], seed=seed + 1)  # the input alone
    deg = torch.from_numpy(np.diff(g.row_ptr.astype(np.int64)))
    src = torch.repeat_interleave(torch.arange(g.n), deg)
    a = torch.zeros((g.n, g.n), dtype=torch.float64, device="cuda")
    a[src.cuda(), torch.from_numpy(g.col_ind.astype(np.int64)).cuda()] = 1.0
    return int(round(float(((a @ a) * a).sum()))) // 6
