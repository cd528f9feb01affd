"""The work this framework is measured by: whole calls of its public entry points.

Every graph is undirected and made from the seed: R-MAT (edge factor 8 or 16,
a in [0.45, 0.65], b = c, d = 0.05; 0.57/0.19/0.19/0.05 where nothing else is
said), Erdos-Renyi, or a 4-neighbour grid with 2% of its edges deleted. A
user's program holds the graph on the GPU (fastcon.Graph) and its queries in
host arrays, so that is what prepare() makes; run() is one call, or one loop
of calls, as such a program writes it, and returns everything the calls
answer. Answers are whole numbers (levels, verdicts, distances, counts),
except for the scheduler's training, whose parameters and loss exact()
recomputes in 64 bits.

Kinds of work (the "kind" of a case):
  bfs       one BFS per root, every level array read back
  bfs_n     one BFS per root in a loop (the reference's cudaBFS4K_N): the
            levels stay on the GPU, each visit's counts come back, and the
            last visit's levels are fetched
  st        s-t queries, one call each
  st_many   a list of s-t queries, each visited on its own
  batch     a list of s-t queries in bit-parallel waves of 64
  build     the canonical CSR of an edge list, built on the GPU
  train     scheduler training on traced rows
"""
import os
import sys

import numpy as np

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fast-con_amd"))

import fastcon as fc  # noqa: E402

POLICIES = {"plain": fc.POLICY_PLAIN, "heuristic": fc.POLICY_HEURISTIC, "learned": fc.POLICY_LEARNED}


def rmat(scale, ef=16, a=0.57):
    return {"graph": "rmat", "scale": scale, "ef": ef, "a": a}


def grid(rows, cols):
    return {"graph": "grid", "rows": rows, "cols": cols}


def er(vertices, degree):
    return {"graph": "er", "vertices": vertices, "degree": degree}


def listed():
    return [
        # eight BFS trees of a small graph, levels on the host: an analysis
        # script's inner loop, where the latency of a call counts
        dict(name="bfs_rmat16", kind="bfs", n=8, **rmat(16)),
        # the Graph500-style BFS run: 64 roots on 4M vertices
        dict(name="bfs_rmat22", kind="bfs_n", n=64, **rmat(22)),
        # BFS of a road-like graph: some 4,000 levels of small frontiers
        dict(name="bfs_grid2048", kind="bfs", n=1, **grid(2048, 2048)),
        # the smallest call, one query on a small graph, sixteen times
        dict(name="st_rmat16", kind="st", n=16, **rmat(16)),
        # a list of queries answered one by one
        dict(name="st_rmat22", kind="st_many", n=1024, **rmat(22)),
        # long shortest paths: thousands of levels of small frontiers
        dict(name="st_grid4096", kind="st_many", n=8, **grid(4096, 4096)),
        # the smallest batch: one wave, on a sparse graph with 64-bit offsets
        dict(name="batch_er2m", kind="batch", n=64, policy="heuristic", off64=True, **er(2097152, 8)),
        # the serving workload: 1,024 queries per call
        dict(name="batch_rmat22", kind="batch", n=1024, policy="heuristic", **rmat(22)),
        # the largest: 16,384 queries of uneven reach, 64-bit offsets
        dict(name="batch_rmat24", kind="batch", n=16384, policy="heuristic", off64=True, uneven=True, **rmat(24)),
        # batched queries on a road-like graph, learned schedule
        dict(name="batch_grid2048", kind="batch", n=256, policy="learned", **grid(2048, 2048)),
        # the first step of a program that reads a graph file: 4M edges, ids
        # skewed towards the low end, a tenth of the lines duplicates
        dict(name="build_4m", kind="build", n=4194304, vertices=1048576),
        # training the scheduler on the rows of a tracing run
        dict(name="train_1796", kind="train", n=1796, epochs=200, weighting=1),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["bfs", "bfs_n", "st", "st_many", "batch", "batch", "batch", "build", "train"])
    if kind == "train":
        return dict(kind=kind, n=_log_int(rng, 60, 3000), epochs=_log_int(rng, 20, 200), weighting=rng.randrange(2))
    if kind == "build":
        n = _log_int(rng, 20000, 4194304)
        return dict(kind=kind, n=n, vertices=_log_int(rng, n // 8 + 1000, n + 1000))
    graph = rng.choice(["rmat", "rmat", "grid", "er"])
    if graph == "rmat":
        c = rmat(rng.randint(13, 22), rng.choice([8, 16]), round(rng.uniform(0.45, 0.65), 3))
    elif graph == "grid":
        c = grid(_log_int(rng, 150, 2048), _log_int(rng, 150, 2048))
    else:
        c = er(_log_int(rng, 30000, 3000000), round(rng.uniform(5.0, 16.0), 2))
    c["kind"] = kind
    if kind == "bfs":
        c["n"] = rng.randint(1, 4)
    elif kind == "bfs_n":
        c["n"] = rng.randint(1, 4) if graph == "grid" else _log_int(rng, 2, 64)
    elif kind == "st_many":
        c["n"] = rng.randint(2, 8) if graph == "grid" else _log_int(rng, 2, 1024)
    elif kind == "batch":
        c["n"] = _log_int(rng, 10, 256) if graph == "grid" else _log_int(rng, 10, 4096)
        c["policy"] = rng.choice(["heuristic", "heuristic", "learned", "plain"])
        c["uneven"] = graph != "grid" and rng.random() < 0.3
    else:
        c["n"] = rng.randint(2, 16)
    c["off64"] = rng.random() < 0.25
    return c


def _host_graph(case, seed):
    if case["graph"] == "rmat":
        bc = (0.95 - case["a"]) / 2
        return fc.gen_rmat_gpu(case["scale"], case["ef"], case["a"], bc, bc, seed=seed + 1)
    if case["graph"] == "grid":
        return fc.gen_grid(case["rows"], case["cols"], 0.02, seed + 1)
    return fc.gen_er(case["vertices"], case["degree"], seed + 1)


def _pairs(case, hg, g, seed):
    """n query pairs: on a grid at Manhattan distances from a quarter
    to one and a half times its mean side, elsewhere among the vertices of degree > 0, and with
    "uneven" 30% of them with one endpoint outside the giant component."""
    n = case["n"]
    rng = np.random.default_rng(seed + 2)
    if case["graph"] == "grid":
        rows, cols = case["rows"], case["cols"]
        side = (rows + cols) / 2
        s, t = [], []
        while len(s) < n:
            p = rng.integers(0, [rows, cols, rows, cols])
            if side / 4 <= abs(p[0] - p[2]) + abs(p[1] - p[3]) <= 1.5 * side:
                s.append(p[0] * cols + p[1])
                t.append(p[2] * cols + p[3])
        return np.array(s, np.int32), np.array(t, np.int32)
    if case.get("uneven"):
        lv, _, _ = g.bfs(int(np.argmax(hg.degree())))
        giant = np.flatnonzero(lv >= 0).astype(np.int32)
        small = np.flatnonzero((lv < 0) & (hg.degree() > 0)).astype(np.int32)
        s, t = rng.choice(giant, n), rng.choice(giant, n)
        far = rng.random(n) < 0.3
        if len(small):
            t[far] = rng.choice(small, int(far.sum()))
        return s, t
    r = rng.choice(np.flatnonzero(hg.degree() > 0).astype(np.int32), 2 * n)
    return r[:n].copy(), r[n:].copy()


def _edges(case, seed):
    """An edge list as files hold it: a tenth of its lines repeat another
    edge the other way round, the rest are distinct edges."""
    rng = np.random.default_rng(seed + 1)
    n, V = case["n"], case["vertices"]
    distinct = n - n // 10
    keys = np.empty(0, np.int64)
    while len(keys) < distinct:
        u = rng.random((2, distinct + distinct // 4), np.float32)
        u = np.minimum(u * np.sqrt(u) * V, V - 1).astype(np.int64)
        lo, hi = u.min(axis=0), u.max(axis=0)
        keys = np.unique(np.concatenate([keys, (lo * V + hi)[lo < hi]]))
    keys = rng.permutation(keys)[:distinct]
    e = np.stack([keys // V, keys % V], axis=1)
    return np.concatenate([e, e[: n // 10, ::-1]])


def _rows(case, seed):
    """Rows as a tracing run gives them: features in [0, 1], and the costs of
    the nine actions in microseconds, spread over two decades, that follow
    the features with some noise."""
    rng = np.random.default_rng(seed + 3)
    x = rng.random((case["n"], fc.SCHED_FEATURES)).astype(np.float32)
    mix = rng.normal(0.0, 0.5, (fc.SCHED_FEATURES, fc.SCHED_ACTIONS))
    cost = np.exp(4.0 + 2.0 * x[:, :1] + x @ mix + rng.normal(0.0, 0.05, (case["n"], fc.SCHED_ACTIONS)))
    return x, cost.astype(np.float32)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "build":
        return dict(case=case, edges=_edges(case, seed))
    if kind == "train":
        x, cost = _rows(case, seed)
        return dict(case=case, g=fc.Graph(fc.gen_grid(8, 8, 0.0, 1)), x=x, cost=cost, seed=seed + 4)
    hg = _host_graph(case, seed)
    g = fc.Graph(hg, force64=case.get("off64", False))
    state = dict(case=case, g=g)
    if kind in ("bfs", "bfs_n"):
        roots = np.random.default_rng(seed + 2).choice(np.flatnonzero(hg.degree() > 0), case["n"])
        state["roots"] = [int(r) for r in roots]
    else:
        state["s"], state["t"] = _pairs(case, hg, g, seed)
        if case.get("policy") == "learned":
            fc.load_default_sched_params(g)
    return state


def run(state):
    case, g = state["case"], state.get("g")
    kind = case["kind"]
    if kind == "build":
        hg = fc.csr_from_edges_gpu(state["edges"], case["vertices"])
        return {"offsets": hg.offsets, "columns": hg.columns}
    if kind == "bfs":
        return [g.bfs(r)[0] for r in state["roots"]]
    if kind == "bfs_n":
        counts = []
        for r in state["roots"]:
            st = g.bfs(r, levels=False)[2]
            counts.append((st["visited_vertices"], st["visited_edges"], st["levels"]))
        return {"counts": np.array(counts, np.int64), "levels": g.levels()}
    if kind == "st":
        got = [g.stcon(int(a), int(b)) for a, b in zip(state["s"], state["t"])]
        return {"connected": np.array([r[0] for r in got]), "dist": np.array([r[1] for r in got])}
    if kind == "st_many":
        r = g.stcon_many(state["s"], state["t"])
        return {"connected": r.connected, "dist": r.dist}
    if kind == "batch":
        r = g.stcon_batch(state["s"], state["t"], policy=POLICIES[case["policy"]])
        return {"connected": r.connected, "dist": r.dist}
    loss = g.sched_train(state["x"], state["cost"], epochs=case["epochs"], lr=3e-3, seed=state["seed"],
                         weighting=case["weighting"])
    return {"params": g.sched_get_params(), "loss": loss}


def _size(case):
    """(vertices, directed edges) of the case's graph, as expected."""
    if case["graph"] == "rmat":
        return 1 << case["scale"], 2 * case["ef"] << case["scale"]
    if case["graph"] == "grid":
        return case["rows"] * case["cols"], int(3.92 * case["rows"] * case["cols"])
    return case["vertices"], int(case["vertices"] * case["degree"])


def work(case):
    """Bytes of one pass. A BFS reads the graph (offsets and columns) and
    writes a level per vertex. A query of an R-MAT or Erdos-Renyi graph reads
    at least its two roots' lists and the lists of one root's neighbours (4
    bytes a column), and has to look at what they lead to (8 bytes: a state
    word); its frontiers meet there. A query of a grid covers two diamonds
    that meet half way: about d^2 vertices at distance d, each with its
    offsets, four columns and a state word (32 bytes). A batch shares what
    its queries read, which cannot be more than the graph once per wave. A
    build reads the pairs (16 bytes each) and writes offsets and columns.
    Training reads every row once an epoch, in and out of two hidden layers
    of 32."""
    n = case["n"]
    if case["kind"] == "build":
        return {"bytes": 16.0 * n + 8.0 * case["vertices"] + 8.0 * n, "flops": 0}
    if case["kind"] == "train":
        flops = 6.0 * (12 * 32 + 32 * 32 + 32 * 9) * n * case["epochs"]
        return {"bytes": 4.0 * n * (12 + 9), "flops": flops}
    V, E = _size(case)
    o = 8 if case.get("off64") else 4
    graph = float(o * V + 4 * E)
    if case["kind"] in ("bfs", "bfs_n"):
        return {"bytes": n * (graph + 4.0 * V), "flops": 0}
    if case["graph"] == "grid":
        d = 0.7 * (case["rows"] + case["cols"]) / 2
        return {"bytes": 32.0 * n * d * d + 16.0 * n, "flops": 0}
    mean = E / V
    per_query = 12.0 * (2 * mean + mean * mean)
    waves = (n + 63) // 64
    total = n * per_query if case["kind"] != "batch" else min(n * per_query, waves * graph)
    return {"bytes": total + 16.0 * n, "flops": 0}


def _init_params(seed):
    """The seeded Xavier-uniform start of the training (biases zero)."""
    mask = (1 << 64) - 1
    st = (seed * 0x9E3779B97F4A7C15 + 1) & mask
    out = []
    for fan_out, fan_in in ((32, 12), (32, 32), (9, 32)):
        lim = (6.0 / (fan_in + fan_out)) ** 0.5
        w = np.empty(fan_out * fan_in, np.float32)
        for i in range(len(w)):
            st = (st + 0x9E3779B97F4A7C15) & mask
            z = st
            z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & mask
            z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
            z ^= z >> 31
            w[i] = (2.0 * ((z >> 11) / 9007199254740992.0) - 1.0) * lim
        out += [w.reshape(fan_out, fan_in).astype(np.float64), np.zeros(fan_out)]
    return out


def exact(case, seed):
    """The training in 64 bits (full batch, Adam); the other answers are whole numbers."""
    if case["kind"] != "train":
        return None
    x, cost = (v.astype(np.float64) for v in _rows(case, seed))
    target = np.log(cost)
    target -= target.mean(axis=1, keepdims=True)
    weight = np.ones(len(x))
    if case["weighting"] == fc.SCHED_WEIGHT_TIME:
        weight = cost.min(axis=1)
        weight /= weight.mean()
    weight = (weight / weight.sum())[:, None]
    p = _init_params(seed + 4)
    m = [np.zeros_like(a) for a in p]
    v = [np.zeros_like(a) for a in p]

    def forward():
        h1 = np.maximum(x @ p[0].T + p[1], 0.0)
        h2 = np.maximum(h1 @ p[2].T + p[3], 0.0)
        return h1, h2, h2 @ p[4].T + p[5] - target

    b1, b2, lr, eps = 0.9, 0.999, 3e-3, 1e-8
    for e in range(1, case["epochs"] + 1):
        h1, h2, d = forward()
        dy = d * weight
        d2 = (dy @ p[4]) * (h2 > 0)
        d1 = (d2 @ p[2]) * (h1 > 0)
        grads = [d1.T @ x, d1.sum(0), d2.T @ h1, d2.sum(0), dy.T @ h2, dy.sum(0)]
        for k, g in enumerate(grads):
            m[k] = b1 * m[k] + (1 - b1) * g
            v[k] = b2 * v[k] + (1 - b2) * g * g
            p[k] -= lr * (m[k] / (1 - b1 ** e)) / (np.sqrt(v[k] / (1 - b2 ** e)) + eps)
    d = forward()[2]
    return {"params": np.concatenate([a.reshape(-1) for a in p]), "loss": float(0.5 * (weight * d * d).sum())}
