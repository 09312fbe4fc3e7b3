"""Launches with few tiles run their updates and L^-1 levels on quarter tiles,
launches with many on whole ones: the same slot must come out the same, bit
for bit, alone (few) and in a batch that is over the lines (many)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,batch", [(129, 300), (193, 150), (320, 40), (513, 24), (1000, 8)])
def test_alone_as_in_a_batch(n, batch):
    import libkriging_amd as lk
    rng = np.random.default_rng(n)
    X = rng.uniform(size=(n, 3))
    y = np.sum(np.sin(3 * X), axis=1)
    th = np.exp(rng.uniform(np.log(0.2), 0.3, size=(batch, 3)))
    ctx = lk.Context(0)
    pid = ctx.problem(X, y, np.ones((n, 1)), "exp")
    ll, g, st, _ = ctx.ll_grad_batch(pid, th, True)
    assert np.all(st == 0)
    for b in (0, batch - 1):
        l1, g1, _, _ = ctx.ll_grad_batch(pid, th[b:b + 1], True)
        assert l1[0] == ll[b] and np.array_equal(g1[0], g[b])
    ctx.close()
