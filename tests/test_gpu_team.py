"""The team engines (team.hpp). fc_stcon_batch in one launch, a wave machine per
XCD or half of one: distances against the host BFS at the edges of its wave
and machine counts, with every kind of step forced on small graphs, and the
graphs it must leave to the launch engine. Plain queries, one per XCD at a
time: distances and every counter against the launch engine's."""
import numpy as np
import pytest

from conftest import oracle_pair_dists

pytestmark = pytest.mark.gpu

FORCED = ["FASTCON_HUB_MIN_EDGES", "FASTCON_BRIDGE_MIN_EDGES", "FASTCON_FILTER_MIN_EDGES",
          "FASTCON_FILTER_MIN_VERTICES"]


def _graphs(fc):
    hub = np.concatenate([[[0, i] for i in range(1, 1500)], [[1, i] for i in range(1400, 2800)],
                          [[i, i + 1] for i in range(2800, 3000)], [[2799, 2800]]])
    return {
        "rmat9": lambda: fc.gen_rmat(9, 16, seed=3),
        "rmat13": lambda: fc.gen_rmat(13, 16, seed=4),
        "rmat12-sparse": lambda: fc.gen_rmat(12, 2, a=0.6, b=0.175, c=0.175, seed=5),
        "two-hubs-and-a-tail": lambda: fc.csr_from_edges(hub, 3100),
        "er4000": lambda: fc.gen_er(4000, 3.0, 6),
        "grid60": lambda: fc.gen_grid(60, 61, 0.1, 7),
        "K300": lambda: fc.csr_from_edges(np.array([[i, j] for i in range(300) for j in range(i)]), 300),
    }


@pytest.mark.parametrize("name", ["rmat9", "rmat13", "rmat12-sparse", "two-hubs-and-a-tail", "er4000", "grid60", "K300"])
@pytest.mark.parametrize("forced", [False, True])
def test_team_distances(fc, orc, monkeypatch, name, forced):
    if forced:  # every level meets the thresholds of every step
        for v in FORCED:
            monkeypatch.setenv(v, "1")
    hg = _graphs(fc)[name]()
    rng = np.random.default_rng(11)
    s = rng.integers(0, hg.V, 1100).astype(np.int32)
    t = rng.integers(0, hg.V, 1100).astype(np.int32)
    t[5] = s[5]
    exp = oracle_pair_dists(orc, hg, s, t)
    for off64, keep_ids in ((False, False), (True, False), (False, True)):
        with fc.Graph(hg, force64=off64, keep_ids=keep_ids) as g:
            fc.load_default_sched_params(g)
            for n in (1, 2, 7, 8, 9, 63, 64, 65, 127, 513, 1100):
                for pol in (fc.POLICY_HEURISTIC, fc.POLICY_PLAIN, fc.POLICY_LEARNED):
                    r = g.stcon_batch(s[:n], t[:n], policy=pol, learn_margin=0.0)
                    assert r.stats["launches"] == 1
                    assert np.array_equal(r.dist, exp[:n]), (name, off64, keep_ids, n, pol)
                    assert np.array_equal(r.connected, (exp[:n] >= 0).astype(np.int32))


@pytest.mark.parametrize("teams", ["1", "2"])
def test_team_counts_and_widths(fc, orc, monkeypatch, teams):
    """One and two machines per XCD, fixed widths and hub chunks, repeated
    calls on one graph (each leaves its workspace clean)."""
    monkeypatch.setenv("FASTCON_BATCH_TEAMS", teams)
    hg = fc.gen_rmat(12, 16, seed=8)
    rng = np.random.default_rng(12)
    s = rng.integers(0, hg.V, 700).astype(np.int32)
    t = rng.integers(0, hg.V, 700).astype(np.int32)
    exp = oracle_pair_dists(orc, hg, s, t)
    with fc.Graph(hg) as g:
        for vw, tile in ((0, 0), (4, 64), (8, 0), (16, 256), (32, 1024), (64, 65536)):
            for n in (700, 33):
                assert np.array_equal(g.stcon_batch(s[:n], t[:n], vw=vw, tile=tile).dist, exp[:n]), (vw, tile, n)


def test_directed_graphs_keep_the_launch_engine(fc, monkeypatch):
    """Directed CSRs are accepted as before: their answers depend on the
    order of the steps, so they stay with the engine whose order they had."""
    rng = np.random.default_rng(13)
    e = rng.integers(0, 400, (3000, 2))
    order = np.argsort(e[:, 0], kind="stable")
    off = np.zeros(401, np.int64)
    np.add.at(off, e[:, 0] + 1, 1)
    hg = fc.HostGraph(np.cumsum(off), e[order, 1].astype(np.int32), directed=True)
    s = rng.integers(0, 400, 200).astype(np.int32)
    t = rng.integers(0, 400, 200).astype(np.int32)
    with fc.Graph(hg) as g:
        for pol in (fc.POLICY_HEURISTIC, fc.POLICY_PLAIN):
            a = g.stcon_batch(s, t, policy=pol)
            b = g.stcon_batch(s, t, policy=pol, lanes=3)
            assert a.stats["launches"] > 1
            assert np.array_equal(a.dist, b.dist)


@pytest.mark.parametrize("name", ["rmat9", "rmat13", "rmat12-sparse", "two-hubs-and-a-tail", "er4000", "grid60", "K300"])
def test_plain_teams(fc, orc, monkeypatch, name):
    hg = _graphs(fc)[name]()
    rng = np.random.default_rng(21)
    s = rng.integers(0, hg.V, 1500).astype(np.int32)
    t = rng.integers(0, hg.V, 1500).astype(np.int32)
    t[::97] = s[::97]
    exp = oracle_pair_dists(orc, hg, s, t)
    for off64, keep_ids in ((False, False), (True, False), (False, True)):
        monkeypatch.setenv("FASTCON_PLAIN_TEAMS", "0")
        with fc.Graph(hg, force64=off64, keep_ids=keep_ids) as g:
            ref = {n: g.stcon_many(s[:n], t[:n]) for n in (1, 2, 9, 1500)}
            one = [g.stcon(int(a), int(b)) for a, b in zip(s[1:6], t[1:6])]
        monkeypatch.delenv("FASTCON_PLAIN_TEAMS")
        with fc.Graph(hg, force64=off64, keep_ids=keep_ids) as g:
            for _ in range(2):  # a second pass meets the first one's state words
                for n, r in ref.items():
                    x = g.stcon_many(s[:n], t[:n])
                    assert np.array_equal(x.dist, exp[:n]) and np.array_equal(x.connected, r.connected)
                    for k in ("levels", "depth", "visited_vertices", "visited_edges", "expanded_vertices",
                              "expanded_edges", "topdown_levels", "max_frontier"):
                        assert x.stats[k] == r.stats[k], (name, n, k)
            for (c, d, m, _), a, b in zip(one, s[1:6], t[1:6]):
                assert g.stcon(int(a), int(b))[:3] == (c, d, m)


def _narrow_graphs(fc):
    def edges(V, e):
        u, v = np.concatenate([e, e[:, ::-1]]).T
        order = np.lexsort((v, u))
        off = np.concatenate([[0], np.cumsum(np.bincount(u, minlength=V))])
        return fc.HostGraph(off, v[order].astype(np.int32))

    def tree():  # binary: twice as wide at each level, beyond a narrow visit's 65,534 vertices
        k = np.arange(1, 1 << 18)
        return edges(1 << 18, np.stack([(k - 1) // 2, k], 1))

    def ladder():  # 16 rungs wide, one list of 300 that its block publishes
        k = np.arange(3000 * 16).reshape(3000, 16)
        e = [np.stack([k[:-1].ravel(), k[1:].ravel()], 1), np.stack([k[:, :-1].ravel(), k[:, 1:].ravel()], 1)]
        e.append(np.stack([np.full(300, k[1500, 0]), 3000 * 16 + np.arange(300)], 1))
        return edges(3000 * 16 + 300, np.concatenate(e))

    return {"path": lambda: fc.gen_grid(1, 3000, 0.0, 1), "grid7x900": lambda: fc.gen_grid(7, 900, 0.05, 2),
            "grid500": lambda: fc.gen_grid(500, 500, 0.02, 3), "er-degree-3": lambda: fc.gen_er(100000, 3.0, 4),
            "tree": tree, "ladder": ladder}


@pytest.mark.parametrize("name", ["path", "grid7x900", "grid500", "er-degree-3", "tree", "ladder"])
def test_narrow_visits(fc, orc, monkeypatch, name):
    hg = _narrow_graphs(fc)[name]()
    rng = np.random.default_rng(31)
    s = np.concatenate([[0], rng.integers(0, hg.V, 39)]).astype(np.int32)
    t = rng.integers(0, hg.V, 40).astype(np.int32)
    t[::13] = s[::13]
    exp = oracle_pair_dists(orc, hg, s, t)
    keys = ("levels", "visited_vertices", "visited_edges", "expanded_vertices", "expanded_edges", "max_frontier")
    for off64, keep_ids in ((False, False), (True, False), (False, True)):
        monkeypatch.setenv("FASTCON_PLAIN_TEAMS", "0")
        with fc.Graph(hg, force64=off64, keep_ids=keep_ids) as g:
            ref = [g.bfs(int(r), parents=True) for r in s[:3]]
            st = {n: g.stcon_many(s[:n], t[:n]) for n in (1, 2, 40)}
        monkeypatch.delenv("FASTCON_PLAIN_TEAMS")
        with fc.Graph(hg, force64=off64, keep_ids=keep_ids) as g:
            for r, (lv, _, stats) in zip(s, ref):  # the root 0 is the tree's: too wide from there
                for parents in (True, False):
                    x = g.bfs(int(r), parents=parents)
                    assert np.array_equal(x[0], lv)
                    for k in keys:
                        assert x[2][k] == stats[k], (name, k)
                    if parents:
                        assert orc.validate_bfs_tree(hg.offsets, hg.columns, int(r), x[0], x[1]) == 0
                        assert np.array_equal(x[1] < 0, lv < 0)
            for n, r in st.items():
                x = g.stcon_many(s[:n], t[:n])
                assert np.array_equal(x.dist, exp[:n]) and np.array_equal(x.connected, r.connected)
                for k in keys + ("depth", "topdown_levels"):
                    assert x.stats[k] == r.stats[k], (name, n, k)


def _mesh(fc, n):  # n x n x n
    k = np.arange(n ** 3).reshape(n, n, n)
    e = [np.stack([a.ravel(), b.ravel()], 1)
         for a, b in ((k[:-1], k[1:]), (k[:, :-1], k[:, 1:]), (k[:, :, :-1], k[:, :, 1:]))]
    e = np.concatenate(e)
    u, v = np.concatenate([e, e[:, ::-1]]).T
    order = np.lexsort((v, u))
    off = np.concatenate([[0], np.cumsum(np.bincount(u, minlength=n ** 3))])
    return fc.HostGraph(off, v[order].astype(np.int32))


@pytest.mark.parametrize("name,one_launch,launches", [
    ("rmat16", (1, 8, 1024), (64,)), ("er100k", (1, 64, 256), ()), ("er1m", (8, 256), (64, 128)),
    ("grid300", (1, 64), ()), ("mesh48", (1, 256), (64,))])
def test_plain_batches_by_width(fc, orc, name, one_launch, launches):
    """The plain schedule's waves of 64 run in one launch where they are narrow
    or many, else by launches: the same distances and counters on both."""
    hg = {"rmat16": lambda: fc.gen_rmat(16, 16, seed=9), "er100k": lambda: fc.gen_er(100000, 8.0, 9),
          "er1m": lambda: fc.gen_er(1000000, 16.0, 9), "grid300": lambda: fc.gen_grid(300, 300, 0.02, 9),
          "mesh48": lambda: _mesh(fc, 48)}[name]()
    rng = np.random.default_rng(51)
    s = rng.integers(0, hg.V, 1024).astype(np.int32)
    t = rng.integers(0, hg.V, 1024).astype(np.int32)
    exp = oracle_pair_dists(orc, hg, s[:16], t[:16])
    with fc.Graph(hg) as g:
        for n in one_launch + launches:
            r = g.stcon_batch(s[:n], t[:n], policy=fc.POLICY_PLAIN)
            assert (r.stats["launches"] == 1) == (n in one_launch), n
            k = min(n, 16)
            assert np.array_equal(r.dist[:k], exp[:k])
            ref = g.stcon_batch(s[:n], t[:n], policy=fc.POLICY_PLAIN, lanes=1, tile=256)
            assert np.array_equal(r.dist, ref.dist)
            for key in ("waves", "levels", "active_vertices", "active_edges", "touched_vertices"):
                assert r.stats[key] == ref.stats[key], (n, key)


@pytest.mark.parametrize("name", ["rmat19", "star", "two"])
def test_wide_levels_go_to_the_whole_gpu(fc, orc, monkeypatch, name):
    """Queries that a team gives up at a wide level (rmat19), at the root
    (star: 400,000 edges at level 0) or all of them (two: unconnected, and
    more than half of a call) come back with the launches' answers and
    counters, and so do the others of the call."""
    def star():
        k = np.arange(1, 400001)
        off = np.concatenate([[0, 400000], 400000 + np.arange(1, 400001)])
        return fc.HostGraph(off, np.concatenate([k, np.zeros(400000)]).astype(np.int32))

    def two():
        h = fc.gen_er(200000, 16.0, 5)
        return fc.HostGraph(np.concatenate([h.offsets, h.offsets[1:] + h.E]), np.concatenate([h.columns, h.columns + h.V]))

    hg = {"rmat19": lambda: fc.gen_rmat(19, 16, seed=61), "star": star, "two": two}[name]()
    rng = np.random.default_rng(62)
    s = rng.integers(0, hg.V // 2, 40).astype(np.int32)
    t = rng.integers(hg.V // 2, hg.V, 40).astype(np.int32)
    if name == "star":
        s[1::2] = 0
    keys = ("levels", "depth", "visited_vertices", "visited_edges", "expanded_vertices", "expanded_edges",
            "topdown_levels", "max_frontier")
    monkeypatch.setenv("FASTCON_PLAIN_TEAMS", "0")
    with fc.Graph(hg) as g:
        if name == "rmat19":  # the heaviest of many first
            s, t = rng.integers(0, hg.V, (2, 300)).astype(np.int32)
            work = [g.stcon(int(a), int(b))[3]["expanded_edges"] for a, b in zip(s, t)]
            top = np.argsort(work)[::-1][:40]
            assert work[top[0]] > 1 << 19
            s, t = s[top], t[top]
        ref = {n: g.stcon_many(s[:n], t[:n]) for n in (1, 2, 3, 9, 40)}
    monkeypatch.delenv("FASTCON_PLAIN_TEAMS")
    assert np.array_equal(ref[9].dist, oracle_pair_dists(orc, hg, s[:9], t[:9]))
    launches = {}
    with fc.Graph(hg) as g:
        for _ in range(2):
            for n, r in ref.items():
                x = g.stcon_many(s[:n], t[:n])
                launches[n] = x.stats["launches"]
                assert np.array_equal(x.dist, r.dist) and np.array_equal(x.connected, r.connected), n
                for k in keys:
                    assert x.stats[k] == r.stats[k], (n, k)
    assert max(launches[2], launches[3]) > 1  # some were given up


def test_two_callers_at_a_time(fc, orc):
    """One graph per thread is a supported use: one-launch calls that find the
    GPU taken, or a part of it, and launches between them, answer as they do
    alone."""
    from concurrent.futures import ThreadPoolExecutor

    def work(hg, seed):
        rng = np.random.default_rng(seed)
        s, t = rng.integers(0, hg.V, (2, 300)).astype(np.int32)
        return hg, s, t, oracle_pair_dists(orc, hg, s, t, workers=4), orc.bfs(hg.offsets, hg.columns, int(s[0]))[0]

    def call(w):
        hg, s, t, exp, lv = w
        with fc.Graph(hg) as g:
            for k in range(12):
                n = (300, 40, 9, 2)[k % 4]
                assert np.array_equal(g.stcon_batch(s[:n], t[:n]).dist, exp[:n])
                assert np.array_equal(g.stcon_many(s[:n], t[:n]).dist, exp[:n])
                assert np.array_equal(g.stcon_batch(s[:n], t[:n], policy=fc.POLICY_PLAIN, lanes=2, tile=256).dist, exp[:n])
                assert np.array_equal(g.bfs(int(s[0]))[0], lv)
                assert g.stcon(int(s[k]), int(t[k]))[1] == exp[k]
        return True

    graphs = [work(fc.gen_rmat(14, 16, seed=71), 1), work(fc.gen_grid(150, 150, 0.02, 72), 2)]
    for pair in ((graphs[0], graphs[1]), (graphs[0], graphs[0]), (graphs[1], graphs[1])):
        with ThreadPoolExecutor(2) as ex:
            assert all(ex.map(call, pair))


def test_hub_steps_answer_queries(fc, orc, monkeypatch):
    """A hub step answers, before the bridge step of the same levels, the
    queries whose balls meet at a top vertex: fewer are left to the bridges,
    and the distances are the same."""
    hg = fc.gen_rmat(13, 16, seed=91)
    s, t = np.random.default_rng(92).integers(0, hg.V, (2, 512)).astype(np.int32)
    exp = oracle_pair_dists(orc, hg, s, t)
    monkeypatch.setenv("FASTCON_BRIDGE_MIN_EDGES", "1")
    got = {}
    with fc.Graph(hg) as g:
        for least in ("1", str(1 << 56)):
            monkeypatch.setenv("FASTCON_HUB_MIN_EDGES", least)
            r = g.stcon_batch(s, t)
            assert r.stats["launches"] == 1 and np.array_equal(r.dist, exp)
            got[least] = r.stats
    assert got["1"]["bridged"] < got[str(1 << 56)]["bridged"]


def _directed(fc, V, degree, seed):
    rng = np.random.default_rng(seed)
    e = np.unique(np.stack([np.repeat(np.arange(V), degree), rng.integers(0, V, V * degree)], 1), axis=0)
    off = np.concatenate([[0], np.cumsum(np.bincount(e[:, 0], minlength=V))])
    return fc.HostGraph(off, e[:, 1].astype(np.int32), directed=True)


@pytest.mark.parametrize("degree", [2, 8])
def test_plain_visits_of_directed_graphs(fc, orc, monkeypatch, degree):
    """Queries and BFS inside one launch on directed graphs (degree 2: narrow
    visits, 8: eight queries at a time) as by launches."""
    hg = _directed(fc, 30000, degree, 101)
    s, t = np.random.default_rng(102).integers(0, hg.V, (2, 300)).astype(np.int32)
    keys = ("levels", "depth", "visited_vertices", "visited_edges", "expanded_vertices", "expanded_edges", "max_frontier")
    monkeypatch.setenv("FASTCON_PLAIN_TEAMS", "0")
    with fc.Graph(hg) as g:
        ref = {n: g.stcon_many(s[:n], t[:n]) for n in (1, 2, 9, 300)}
        lv = g.bfs(int(s[0]))[0]
    monkeypatch.delenv("FASTCON_PLAIN_TEAMS")
    assert np.array_equal(lv, orc.bfs(hg.offsets, hg.columns, int(s[0]))[0])
    for off64, keep_ids in ((False, False), (True, False), (False, True)):
        with fc.Graph(hg, force64=off64, keep_ids=keep_ids) as g:
            for n, r in ref.items():
                x = g.stcon_many(s[:n], t[:n])
                assert np.array_equal(x.dist, r.dist) and np.array_equal(x.connected, r.connected)
                for k in keys:
                    assert x.stats[k] == r.stats[k], (n, k)
            assert np.array_equal(g.bfs(int(s[0]))[0], lv)


def test_plain_batches_of_directed_graphs(fc):
    """The plain schedule on a directed graph against a host visit by its
    rules: both balls grow along the edges at each step, and the first meet
    sets the distance."""
    hg = _directed(fc, 2000, 3, 103)
    out = [set(hg.columns[hg.offsets[v]:hg.offsets[v + 1]].tolist()) for v in range(hg.V)]

    def visit(a, b):
        if a == b:
            return 0
        ball, front = [{a}, {b}], [{a}, {b}]
        for step in range(hg.V):
            new = [set().union(*(out[v] for v in front[x])) - ball[x] for x in (0, 1)]
            if new[0] & ball[1] or new[1] & ball[0]:
                return 2 * step + 1
            if new[0] & new[1]:
                return 2 * step + 2
            if not new[0] or not new[1]:
                return -1
            ball, front = [ball[x] | new[x] for x in (0, 1)], new

    s, t = np.random.default_rng(104).integers(0, hg.V, (2, 200)).astype(np.int32)
    t[::50] = s[::50]
    exp = [visit(int(a), int(b)) for a, b in zip(s, t)]
    with fc.Graph(hg) as g:
        r = g.stcon_batch(s, t, policy=fc.POLICY_PLAIN)
        assert r.stats["launches"] > 1 and list(r.dist) == exp


def test_learned_bottom_up_steps_of_teams(fc, orc):
    """At margin 0 the network proposes bottom-up steps wherever they are cheap
    for the whole GPU. A team takes them only where the heuristic would: on a
    sparse random graph nowhere, so the work stays near the heuristic's."""
    hg = fc.gen_er(100000, 8.0, 105)
    s, t = np.random.default_rng(106).integers(0, hg.V, (2, 64)).astype(np.int32)
    exp = oracle_pair_dists(orc, hg, s, t)
    with fc.Graph(hg) as g:
        assert fc.load_default_sched_params(g)
        h = g.stcon_batch(s, t)
        for margin in (0.0, 0.25, 1.0):
            r = g.stcon_batch(s, t, policy=fc.POLICY_LEARNED, learn_margin=margin)
            assert r.stats["launches"] == 1 and np.array_equal(r.dist, exp)
            # a step scans at most its frontier, a bottom-up step every vertex
            assert r.stats["active_vertices"] < h.stats["active_vertices"] + hg.V // 2
