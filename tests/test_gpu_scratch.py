"""Predictions take their device and pinned memory from blocks that earlier
calls have used: results must not depend on what ran before, from which
model or thread."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def fixed(kernel, d, n, seed, regmodel="constant"):
    import libkriging_amd as lk
    rng = np.random.default_rng(seed)
    X = rng.uniform(size=(n, d))
    y = np.sum(np.sin(3 * X), axis=1)
    k = lk.Kriging(kernel)
    k.fit(y, X, regmodel, False, "none", "LL", {"theta": [0.4] * d, "is_theta_estim": False})
    return k


def calls():
    a, b = fixed("matern5_2", 2, 150, 1, "linear"), fixed("exp", 5, 700, 2)
    rng = np.random.default_rng(3)
    P = {m: (rng.uniform(size=(m, 2)), rng.uniform(size=(m, 5))) for m in (1, 63, 64, 200, 1500)}
    out = []
    for m in (200, 1, 1500, 64, 63):
        out.append(lambda m=m: a.predict(P[m][0], True, m <= 200, True))
        out.append(lambda m=m: b.predict(P[m][1], True, False, False))
    return out


def same(u, v):
    for p, q in zip(u, v):
        if p is None or q is None:
            assert p is None and q is None
        else:
            np.testing.assert_array_equal(np.asarray(p), np.asarray(q))


def test_reused_blocks_leave_no_trace():
    fs = calls()
    first = [f() for f in fs]
    for order in (range(len(fs)), reversed(range(len(fs)))):
        for q in order:
            same(fs[q](), first[q])


def test_concurrent_predictions():
    fs = calls()
    first = [f() for f in fs]
    with ThreadPoolExecutor(4) as ex:
        for got, want in zip(ex.map(lambda q: fs[q % len(fs)](), range(4 * len(fs))), first * 4):
            same(got, want)
