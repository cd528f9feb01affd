"""GPU kernels of the learned scheduler against the CPU oracle (forward,
gradient, one training step), the trace of the batched engine (answers
unchanged, costs positive, heuristic action recorded), and what a trained
network gains over the schedules without it."""
import sys

import numpy as np
import pytest

from oracle import mlp

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _oracle_dist(orc, hg, s, t):
    return np.array([orc.stcon(hg.offsets, hg.columns, a, b)[1] for a, b in zip(s, t)], np.int32)


def _data(seed, n=300):
    rng = np.random.default_rng(seed)
    w = (rng.normal(0, 0.3, mlp.P)).astype(np.float32)
    X = rng.uniform(0, 1, (n, mlp.F)).astype(np.float32)
    T = rng.normal(0, 1, (n, mlp.A)).astype(np.float32)
    return w, X, T


def test_forward_and_gradient_match_oracle(fc):
    hg = fc.gen_grid(8, 8, 0.0, 1)
    with fc.Graph(hg) as g:
        for seed in (1, 2):
            w, X, T = _data(seed)
            g.sched_set_params(w)
            say(f"sched forward/gradient seed={seed}")
            y = g.sched_forward(X)
            yo = mlp.forward(w, X)
            assert np.allclose(y, yo, rtol=1e-5, atol=1e-5)
            loss, grad = g.sched_gradient(X, T)
            lo, go = mlp.loss_grad(w, X, T)
            assert abs(loss - lo) <= 1e-5 * max(1.0, lo)
            scale = np.abs(go).max()
            assert np.abs(grad - go).max() <= 1e-4 * scale, np.abs(grad - go).max() / scale
            # row-weighted loss (some rows weigh nothing)
            wr = np.random.default_rng(seed + 10).uniform(0.0, 4.0, len(X)).astype(np.float32)
            wr[::7] = 0.0
            say(f"sched weighted gradient seed={seed}")
            loss, grad = g.sched_gradient(X, T, wr)
            lo, go = mlp.loss_grad(w, X, T, wr)
            assert abs(loss - lo) <= 1e-5 * max(1.0, lo)
            scale = np.abs(go).max()
            assert np.abs(grad - go).max() <= 1e-4 * scale, np.abs(grad - go).max() / scale
        # bad weights are rejected
        with pytest.raises(fc.FastconError):
            g.sched_gradient(X, T, np.full(len(X), -1.0, np.float32))
        with pytest.raises(fc.FastconError):
            g.sched_gradient(X, T, np.zeros(len(X), np.float32))


@pytest.mark.parametrize("weighting", ["uniform", "time"])
def test_one_training_step_matches_oracle(fc, weighting):
    """fc_sched_train with one epoch = seeded init + one Adam step on the
    full batch; the result equals the oracle's, with rows weighted alike or
    by the time at stake."""
    hg = fc.gen_grid(8, 8, 0.0, 1)
    rng = np.random.default_rng(4)
    X = rng.uniform(0, 1, (200, mlp.F)).astype(np.float32)
    cost = np.exp(rng.normal(3, 1, (200, mlp.A))).astype(np.float32)
    T = mlp.row_targets(cost)
    wr = mlp.row_weights(cost) if weighting == "time" else None
    code = fc.SCHED_WEIGHT_TIME if weighting == "time" else fc.SCHED_WEIGHT_UNIFORM
    w0 = mlp.init_params(11).astype(np.float64)
    l0, g0 = mlp.loss_grad(w0, X, T, wr)
    w1, _, _ = mlp.adam_step(w0, g0, np.zeros(mlp.P), np.zeros(mlp.P), 1, 1e-3)
    with fc.Graph(hg) as g:
        say(f"sched train one epoch weighting={weighting}")
        g.sched_train(X, cost, epochs=1, lr=1e-3, seed=11, weighting=code)
        w = g.sched_get_params()
    # Adam's first step is lr*sign(g): compare wherever g is not so small
    # that float32 rounding could flip its sign
    big = np.abs(g0) > 1e-4 * np.abs(g0).max()
    close = np.abs(w - w1) <= 2e-6
    assert close[big].all()
    assert close.mean() > 0.95
    if weighting == "time":  # the weighting moved the step somewhere
        _, gu = mlp.loss_grad(w0, X, T)
        assert (np.sign(gu[big]) != np.sign(g0[big])).any()


def test_training_reduces_loss(fc):
    hg = fc.gen_grid(8, 8, 0.0, 1)
    rng = np.random.default_rng(8)
    X = rng.uniform(0, 1, (400, mlp.F)).astype(np.float32)
    # costs that depend on the features: action a is cheap when x[a] is small
    clean = np.exp(2.0 * X[:, :mlp.A])
    cost = (clean * np.exp(0.1 * rng.normal(size=(400, mlp.A)))).astype(np.float32)
    T = mlp.row_targets(cost)
    with fc.Graph(hg) as g:
        l1 = g.sched_train(X, cost, epochs=1, lr=3e-3, seed=2)
        l2 = g.sched_train(X, cost, epochs=400, lr=3e-3, seed=2)
        w = g.sched_get_params()
    assert l2 < 0.25 * l1
    lo, _ = mlp.loss_grad(w.astype(np.float64), X, T)
    assert abs(lo - l2) <= 1e-3 * max(1.0, lo)
    # judged on the noise-free costs: with nine actions the label noise alone
    # moves the noisy argmin off the true one on about a fifth of the rows
    pick = mlp.argmin_actions(w, X)
    assert (pick == np.argmin(clean, 1)).mean() > 0.9
    rows = np.arange(len(X))
    assert np.mean(clean[rows, pick] / clean.min(axis=1) - 1.0) < 0.01


def test_trace_keeps_answers_and_times_every_action(fc, orc):
    hg = fc.gen_rmat(14, 16, seed=3)
    r = hg.sample_roots(256, 5)
    s, t = r[:128], r[128:]
    exp = _oracle_dist(orc, hg, s, t)
    with fc.Graph(hg) as g:
        say("sched trace rmat14")
        feats, cost, heur, wave, dist = g.sched_trace(s, t, cap=4096)
        assert np.array_equal(dist, exp)
        assert len(feats) >= 2 and set(wave) == {0, 1}
        assert (cost > 0).all() and np.isfinite(cost).all()
        assert ((heur >= 0) & (heur < mlp.A)).all()
        assert np.isfinite(feats).all()
        # the traced batch still answers correctly afterwards, under every policy
        for pol in (0, 1):
            assert np.array_equal(g.stcon_batch(s, t, policy=pol).dist, exp)


def test_trained_network_against_heuristic_and_plain(fc, orc):
    """The shipped trained parameters at their validated margin, on a graph
    and queries they were not trained on: every answer equals the oracle's;
    the learned schedule beats the plain schedule (both frontiers top-down
    every step, the reference's order of work); and against the heuristic,
    the method without the network, it gains nothing: at the shipped margin
    the network takes the heuristic's decisions on held-out graphs and adds
    only its inference, about 1-5% of a batch. The measured ratio is printed;
    the test bounds the overhead at 10%."""
    hg = fc.gen_rmat(20, 16, 0.57, 0.19, 0.19, seed=77)
    r = hg.sample_roots(1024, 78)
    s, t = r[:512], r[512:]
    exp = _oracle_dist(orc, hg, s[:48], t[:48])
    with fc.Graph(hg) as g:
        assert fc.load_default_sched_params(g)
        ms = {}
        for name, pol in (("plain", fc.POLICY_PLAIN), ("heuristic", fc.POLICY_HEURISTIC),
                          ("learned", fc.POLICY_LEARNED)):
            g.stcon_batch(s, t, policy=pol)
            times = []
            for _ in range(5):
                res = g.stcon_batch(s, t, policy=pol)
                assert np.array_equal(res.dist[:48], exp), name
                times.append(res.stats["time_ms"])
            ms[name] = float(np.median(times))
        say(f"rmat20 512 queries, ms per batch: {ms}; learned vs plain {ms['plain'] / ms['learned']:.2f}x, "
            f"learned vs heuristic {ms['heuristic'] / ms['learned']:.3f}x")
        assert ms["learned"] * 1.05 < ms["plain"]
        assert ms["learned"] < 1.10 * ms["heuristic"]


@pytest.mark.parametrize("n", [1, 3, 15, 16, 17, 63, 64, 65, 255, 256, 257, 287, 288, 511, 513, 3001])
def test_gradient_at_the_edges_of_the_row_tiles(fc, n):
    """Row counts around the 16-row blocks of the forward/backward pass and
    the 256-row tiles (and 32-row steps) of the parameter sums. The bound is
    the one of a recursive FP32 sum, (terms + 1) * 2^-24 * sum |term|, for
    the n rows and the at most 117 FMAs behind each term."""
    w, X, T = _data(40 + n, n)
    wr = np.random.default_rng(n).uniform(0.0, 4.0, n).astype(np.float32)
    wr[0] = 1.0
    lo, go = mlp.loss_grad(w, X, T, wr)
    aw = np.abs(w.astype(np.float64))
    W1, b1 = aw[:384].reshape(32, 12), aw[384:416]
    W2, b2 = aw[416:1440].reshape(32, 32), aw[1440:1472]
    W3, b3 = aw[1472:1760].reshape(9, 32), aw[1760:]
    h1 = np.abs(X).astype(np.float64) @ W1.T + b1
    h2 = h1 @ W2.T + b2
    dy = (h2 @ W3.T + b3 + np.abs(T)) * (wr / wr.astype(np.float64).sum())[:, None]
    d2 = dy @ W3
    d1 = d2 @ W2
    size = np.concatenate([x.reshape(-1) for x in (d1.T @ np.abs(X), d1.sum(0), d2.T @ h1, d2.sum(0), dy.T @ h2,
                                                   dy.sum(0))])
    with fc.Graph(fc.gen_grid(8, 8, 0.0, 1)) as g:
        g.sched_set_params(w)
        say(f"sched gradient n={n}")
        loss, grad = g.sched_gradient(X, T, wr)
        assert np.all(np.abs(grad - go) <= (n + 118) * 2.0 ** -24 * size)
        assert abs(loss - lo) <= (n + 118) * 2.0 ** -24 * float((dy * (h2 @ W3.T + b3 + np.abs(T))).sum())
