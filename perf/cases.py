"""Workloads for timing the framework through its public entry points.

Two kinds of work: exact subgraph counts (whole graphs, shards of a graph,
device-resident graphs, captured replays, the `pm` interface) and the tuner's
learned cost model (train, then rank candidates). Every case is a plain dict:

  graph     "er" | "rmat" | "cl" (Erdos-Renyi, R-MAT, Chung-Lu)
  n         vertices (a power of two for "rmat")
  degree    mean degree (er, cl); edges drawn per vertex (rmat)
  patterns  names joined with "+" ("k4+k5"), or "all5": every connected
            5-vertex pattern in one batched plan
  mode      "unique" | "labeled" | "reference"
  entry     "count" (Plan.count), "replay" (captured once, then replayed),
            "roots" (Plan.count_shard), "edges" (Plan.count_shard_edges),
            "pm" (DeviceContext + Executor.perform_search),
            "device" (clique_counts_noalloc on a graph in device memory)
  config    "default", or "tuned": the kernel config the tuner picked for
            cliques on R-MAT scale 20

and for the cost model: entry "fit", rows (measured configs), steps (Adam
steps), candidates (configs to rank afterwards).
"""
import math

import numpy as np
import torch

from graphautotune_amd import core, workloads
from graphautotune_amd.tuning.features import FEATURES
from graphautotune_amd.tuning.mlp import MLPCostModel

PATTERNS = dict(workloads.NAMED, c4="0101101001011010", diamond="0111101111001100", p4="0100101001010010")

# what the tuner settled on for K4 + K5 on R-MAT scale 20
TUNED = {"block_waves": 2, "waves_per_cu": 8, "queue_chunk": 4, "slot_capacity": 64, "intersect_strategy": 0,
         "gallop_ratio": 4, "search_linear_threshold": 16, "vertex_store": 0}

HIDDEN = 256  # the cost model's width


def _count(name, graph, n, degree, patterns, mode="unique", entry="count", config="default", **more):
    return dict({"name": name, "graph": graph, "n": n, "degree": degree, "patterns": patterns, "mode": mode,
                 "entry": entry, "config": config}, **more)


def listed():
    return [
        # the smallest call: triangles of a sparse random graph, a latency test
        _count("triangle_er10k", "er", 10000, 16, "triangle", mode="labeled"),
        # cycles and paths of a larger sparse graph without hubs
        _count("c4_p4_er100k", "er", 100003, 16, "c4+p4"),
        # the clique benchmark: 4- and 5-cliques of a skewed graph, tuned
        _count("k4k5_rmat20", "rmat", 1 << 20, 16, "k4+k5", config="tuned"),
        # cliques as a user runs them first: default config, a power-law graph
        _count("k345_cl262k", "cl", 262144, 24, "triangle+k4+k5"),
        # a serving loop's cliques on a graph it keeps in device memory
        _count("k3to6_device_rmat16", "rmat", 1 << 16, 16, "", entry="device", kmax=6),
        # an ordinary clique count captured once and replayed
        _count("k4_replay_rmat14", "rmat", 1 << 14, 16, "k4", entry="replay", replays=8),
        # 5-vertex patterns with an inclusion-exclusion tail on power-law graphs
        _count("house_cl65k", "cl", 65536, 24, "house"),
        # long cycles: the deepest loops for a 5-vertex pattern, the longest call here
        _count("c5_rmat13", "rmat", 1 << 13, 16, "c5"),
        # the reference's own value through the interface of its `pm` program
        _count("pm_house_rmat14", "rmat", 1 << 14, 16, "house", mode="reference", entry="pm"),
        # every connected 5-vertex pattern at once (motif census) on a small graph
        _count("all5_rmat10", "rmat", 1 << 10, 16, "all5"),
        # one process's share of a large graph: a range of mid-degree roots
        _count("house_roots_cl1m", "cl", 1000003, 24, "house", entry="roots", lo=0.004, hi=0.0042),
        # the tuner's cost model: fit on measured configs, rank the candidates
        {"name": "cost_model_fit", "entry": "fit", "rows": 325, "steps": 400, "candidates": 2048},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["clique", "clique", "device", "five", "five", "pm", "shard", "sparse", "fit"])
    if kind == "fit":
        return {"entry": "fit", "rows": _log_int(rng, 16, 770), "steps": rng.randrange(100, 401),
                "candidates": _log_int(rng, 25, 4000)}
    if kind == "sparse":
        c = _count("", "er", _log_int(rng, 1000, 200000), rng.randrange(4, 25), rng.choice(["triangle", "c4", "c4+p4", "house"]),
                   mode=rng.choice(["unique", "labeled"]))
    elif kind == "clique":
        pats = rng.choice(["triangle", "k4", "k5", "k4+k5", "triangle+k4+k5"])
        conf = rng.choice(["default", "tuned"])
        if rng.random() < 0.5:
            c = _count("", "rmat", 1 << rng.randrange(9, 19), rng.choice([8, 16, 24]), pats, config=conf)
        else:
            c = _count("", "cl", _log_int(rng, 2000, 400000), rng.randrange(8, 33), pats, config=conf)
        if rng.random() < 0.3:
            c.update(entry="replay", replays=rng.randrange(2, 9))
    elif kind == "device":
        kmax = rng.randrange(3, 7)
        c = _count("", "rmat", 1 << rng.randrange(9, 18 if kmax < 6 else 16), rng.choice([8, 16]), "", entry="device",
                   kmax=kmax)
    elif kind == "five":
        pats = rng.choice(["house", "c5", "diamond", "house+c5", "all5"])
        top = {"house": 14, "diamond": 15, "c5": 12, "house+c5": 12, "all5": 10}[pats]
        if rng.random() < 0.5:
            c = _count("", "rmat", 1 << rng.randrange(7, top + 1), 16, pats)
        else:
            c = _count("", "cl", _log_int(rng, 500, 1 << (top - 1)), rng.randrange(8, 25), pats)
    elif kind == "pm":
        pats = rng.choice(["triangle", "k4", "house", "c5"])
        c = _count("", "rmat", 1 << rng.randrange(7, 12 if pats == "c5" else 14), 16, pats, mode="reference", entry="pm")
    else:
        lo = rng.uniform(0.002, 0.5)
        c = _count("", "cl", _log_int(rng, 50000, 500000), 24, rng.choice(["house", "k5", "diamond"]),
                   entry="roots", lo=lo, hi=lo + 0.0005)
        if c["patterns"] != "k5" and rng.random() < 0.5:
            c["entry"] = "edges"
    del c["name"]
    return c


def _graph(case, seed):
    n = case["n"]
    if case["graph"] == "er":
        return core.Graph.erdos_renyi(n, case["degree"] / (n - 1), seed)
    if case["graph"] == "rmat":
        return core.Graph.rmat(n.bit_length() - 1, case["degree"], 0.57, 0.19, 0.19, seed)
    return core.Graph.chung_lu(n, float(case["degree"]), 2.1, 50000, seed)


def _patterns(case):
    if case["patterns"] == "all5":
        return list(workloads.connected_patterns(5))
    return [PATTERNS[p] for p in case["patterns"].split("+")]


def _degree_ordered(graph):
    """The graph's CSR with vertex i the i-th by descending degree."""
    off, adj = (np.asarray(a) for a in graph.csr())
    deg = np.diff(off)
    order = np.argsort(-deg, kind="stable")
    rank = np.empty(len(order), dtype=np.int32)
    rank[order] = np.arange(len(order), dtype=np.int32)
    src = np.repeat(rank, deg)
    dst = rank[adj]
    k = np.lexsort((dst, src))
    new_off = np.concatenate([[0], np.cumsum(deg[order])]).astype(np.int64)
    return new_off, dst[k].astype(np.int32)


def _fit_inputs(case, seed):
    """Feature rows like the tuner's (sparse 0/1 bits and small counts) and
    runtimes that depend on them, over about two orders of magnitude."""
    rng = np.random.default_rng(seed)

    def rows(k):
        x = (rng.random((k, FEATURES)) < 0.25).astype(np.float32)
        x[:, FEATURES // 2:FEATURES // 2 + 16] = rng.random((k, 16), dtype=np.float32)
        return x

    X, Xc = rows(case["rows"]), rows(case["candidates"])
    w = rng.normal(size=FEATURES)
    secs = np.exp(0.25 * (X.astype(np.float64) @ w) + 0.05 * rng.normal(size=len(X)) - 4.0)
    p0 = []
    for fan_in, cols in ((FEATURES, HIDDEN), (HIDDEN, HIDDEN), (HIDDEN, 1)):
        lim = math.sqrt(6.0 / fan_in)
        p0 += [rng.uniform(-lim, lim, size=fan_in * cols), np.zeros(cols)]
    return X, secs, Xc, np.concatenate(p0).astype(np.float32)


def prepare(case, seed):
    if case["entry"] == "fit":
        X, secs, Xc, p0 = _fit_inputs(case, seed)
        return {"case": case, "X": X, "seconds": secs, "Xc": Xc, "p0": p0}
    g = _graph(case, seed)
    config = dict(TUNED) if case["config"] == "tuned" else None
    st = {"case": case, "config": config}
    if case["entry"] == "device":
        off, adj = _degree_ordered(g)
        st.update(off=torch.from_numpy(off).cuda(), adj=torch.from_numpy(adj).cuda(), n=len(off) - 1)
        return st
    if case["entry"] == "pm":
        st["context"] = core.DeviceContext(core.Schedule(core.Pattern(_patterns(case)[0])), g).to_device()
        st["executor"] = core.Executor(g.max_degree(), core.GPU_DEVICE)
        return st
    st["plan"] = core.Plan(g, _patterns(case), case["mode"])
    if case["entry"] in ("roots", "edges"):
        lo, hi = int(case["lo"] * case["n"]), max(1, int(case["hi"] * case["n"]))
        if case["entry"] == "edges":
            off = st["plan"].run_offsets()
            lo, hi = int(off[lo]), int(off[hi])
        st.update(lo=lo, hi=hi)
    return st


def run(state):
    case, entry = state["case"], state["case"]["entry"]
    if entry == "fit":
        model = MLPCostModel(FEATURES, HIDDEN)
        model.set_params(state["p0"])
        model.fit(state["X"], state["seconds"], steps=case["steps"])
        return [model.params(), model.predict(state["Xc"])]
    if entry == "device":
        return core.clique_counts_noalloc(state["off"].data_ptr(), state["adj"].data_ptr(), state["n"], case["kmax"],
                                          state["config"])
    if entry == "pm":
        return state["executor"].perform_search(state["context"])
    if entry == "roots":
        return state["plan"].count_shard(state["lo"], state["hi"], state["config"])[0]
    if entry == "edges":
        return state["plan"].count_shard_edges(state["lo"], state["hi"], state["config"])[0]
    return state["plan"].count(state["config"], graph_replays=case.get("replays", 0))[0]


def work(case):
    if case["entry"] == "fit":
        weights = FEATURES * HIDDEN + HIDDEN * HIDDEN + HIDDEN
        params = weights + 2 * HIDDEN + 1
        rows, cands = case["rows"], case["candidates"]
        # forward, and backward (weight gradients, and inputs of layers 2 and 3)
        flops = 2 * rows * case["steps"] * (2 * weights + HIDDEN * HIDDEN + HIDDEN) + 2 * cands * weights
        return {"bytes": 4 * (rows * (FEATURES + 1) + cands * (FEATURES + 1) + 2 * params), "flops": flops}
    # the graph read once, the counts written; integer work, no flops
    g = _graph(case, 1)
    frac = case["hi"] - case["lo"] if case["entry"] in ("roots", "edges") else 1.0
    times = case.get("replays", 1)
    return {"bytes": int(times * frac * (8 * (case["n"] + 1) + 4 * g.e_cnt())) + 8, "flops": 0}


def exact(case, seed):
    """The cost model's training in 64 bits; counts are whole numbers and
    have no such value."""
    if case["entry"] != "fit":
        return None
    X, secs, Xc, p = _fit_inputs(case, seed)
    y = np.log(np.maximum(secs, 1e-9))
    mu, sd = float(y.mean()), float(y.std() + 1e-6)
    X, t, p = X.astype(np.float64), ((y - mu) / sd).astype(np.float32).astype(np.float64), p.astype(np.float64)
    shapes = [(FEATURES, HIDDEN), (HIDDEN,), (HIDDEN, HIDDEN), (HIDDEN,), (HIDDEN, 1), (1,)]

    def views(v):
        out, o = [], 0
        for s in shapes:
            k = int(np.prod(s))
            out.append(v[o:o + k].reshape(s))
            o += k
        return out

    def forward(A):
        W1, b1, W2, b2, W3, b3 = views(p)
        z1 = A @ W1 + b1
        a1 = np.maximum(z1, 0.0)
        z2 = a1 @ W2 + b2
        a2 = np.maximum(z2, 0.0)
        return (a2 @ W3 + b3)[:, 0], z1, a1, z2, a2

    m, v = np.zeros_like(p), np.zeros_like(p)
    for k in range(1, case["steps"] + 1):
        _, _, W2, _, W3, _ = views(p)
        out, z1, a1, z2, a2 = forward(X)
        e = out - t
        dy = (2.0 * e / len(X))[:, None]
        d2 = (dy @ W3.T) * (z2 > 0)
        d1 = (d2 @ W2.T) * (z1 > 0)
        g = np.concatenate([x.ravel() for x in (X.T @ d1, d1.sum(0), a1.T @ d2, d2.sum(0), a2.T @ dy, dy.sum(0))])
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        p -= 2e-3 * (m / (1 - 0.9 ** k)) / (np.sqrt(v / (1 - 0.999 ** k)) + 1e-8)
    return [p, np.exp(forward(Xc.astype(np.float64))[0] * sd + mu)]
