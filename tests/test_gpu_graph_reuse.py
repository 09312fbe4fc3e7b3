"""Captured pipelines are shared by all batches that are cut alike: results
of a context that goes back and forth between designs, batch sizes and
objectives equal, bit for bit, those of a context that evaluates each alone
(the arithmetic does not depend on what ran before)."""
import numpy as np
import pytest

import libkriging_amd as lk

pytestmark = pytest.mark.gpu


def design(n, d, seed):
    rng = np.random.default_rng(seed)
    X = rng.uniform(size=(n, d))
    return X, np.cos(3.0 * X).sum(axis=1) + 0.1 * rng.normal(size=n), np.exp(rng.uniform(-1.5, 0.0, size=(70, d)))


def test_back_and_forth_between_designs():
    ctx = lk.Context(0)
    # same blocks and dimension, different designs; ragged; other dimensions;
    # batches that outgrow the tables; more shapes than are kept captured
    cases = [(100, 3, 1), (110, 3, 2), (128, 3, 3), (129, 3, 4), (300, 5, 5), (61, 2, 6)]
    made = [(design(*c), c) for c in cases]
    ids = [ctx.problem(X, y, np.ones((len(y), 1)), "exp") for (X, y, _), _ in made]
    want = {}
    rng = np.random.default_rng(0)
    batches = [1, 2, 3, 5, 8, 9, 16, 17, 33, 70]
    for step in range(60):
        k = int(rng.integers(len(ids)))
        nb = batches[int(rng.integers(len(batches)))]
        grad = bool(rng.integers(2))
        (X, y, th), _ = made[k]
        ll, g, st, _ = ctx.ll_grad_batch(ids[k], th[:nb], grad)
        assert np.all(st == 0)
        if (k, nb, grad) not in want:
            one = lk.Context(0)
            p1 = one.problem(X, y, np.ones((len(y), 1)), "exp")
            want[k, nb, grad] = one.ll_grad_batch(p1, th[:nb], grad)[:2]
            one.close()
        l1, g1 = want[k, nb, grad]
        assert np.array_equal(ll, l1)
        assert (g is None and g1 is None) or np.array_equal(g, g1)


def test_failed_and_inactive_items_report_status():
    # an item whose jitter ladder fails, beside good ones, between batches
    # of other designs (its status comes back through the same table)
    ctx = lk.Context(0)
    X, y, th = design(40, 2, 9)
    X2 = np.vstack([X, X])  # duplicated points: singular without jitter
    y2 = np.concatenate([y, y])
    a = ctx.problem(X, y, np.ones((40, 1)), "exp")
    b = ctx.problem(X2, y2, np.ones((80, 1)), "gauss")
    for _ in range(3):
        ctx.set_chol_config(num_nugget=0.0)
        ll, _, st, _ = ctx.ll_grad_batch([a, b, a], np.vstack([th[0], [3.0, 3.0], th[1]]), True)
        assert st[0] == 0 and st[2] == 0 and st[1] != 0
        ctx.set_chol_config()
        ll2, _, st2, inc2 = ctx.ll_grad_batch([a, b, a], np.vstack([th[0], [3.0, 3.0], th[1]]), True)
        assert np.all(st2 == 0) and inc2[1] > 0 and inc2[0] == 0
        assert ll2[0] == ll[0] and ll2[2] == ll[2]


def test_objectives_in_turn():
    X, y, th = design(90, 3, 11)
    k = lk.Kriging("matern3_2")
    k.fit(y, X, "constant", False, "none", "LL", {"theta": th[0]})
    first = None
    for _ in range(3):
        got = (k.logLikelihoodFun(th[1], False)[0], k.logLikelihoodFun(th[1], True), k.leaveOneOutFun(th[1], False)[0],
               k.leaveOneOutFun(th[1], True), k.logMargPostFun(th[1], False)[0], k.logMargPostFun(th[1], True))
        assert got[0] == got[1][0] and got[2] == got[3][0] and got[4] == got[5][0]
        if first is None:
            first = got
        for i in (1, 3, 5):
            assert got[i][0] == first[i][0] and np.array_equal(got[i][1], first[i][1])
