"""The forms that only launches of many workgroups take, against the same work
alone, bit for bit: 64-row workgroups below the Cholesky's squares, with and
without refinement of their rows, and the leave-one-out B on whole tiles."""
import numpy as np
import pytest

import libkriging_amd as lk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel,alpha", [("matern3_2", 1.0), ("gauss", 1.0 - 1e-7)])
def test_rows_of_64(kernel, alpha):
    # 9 blocks, 56 items: 4 x 7 x 56 = 1568 and 4 x 5 x 56 = 1120 groups of 16
    # rows below the first two squares, past the line of 1024
    n, items, d = 530, 56, 3
    rng = np.random.default_rng(5)
    X = rng.uniform(size=(n, d))
    th = np.exp(rng.uniform(np.log(0.2), 0.0, size=(items, d)))
    ctx = lk.Context(0)
    ctx.set_chol_config(rcond_check=False, max_inc=0)
    pid = ctx.problem(X, rng.normal(size=n), np.ones((n, 1)), kernel, "nugget")
    gamma = np.hstack([th, np.full((items, 1), alpha)])
    ll, g, st, inc = ctx.ll_grad_batch(pid, gamma, True)
    assert np.all(st == 0) and np.all(inc == 0)
    factors = [ctx.read_item(i, 0) for i in range(items)]
    if kernel == "gauss":  # either block of the first square is past the threshold of 1e4 in some items
        for k in (0, 64):
            B = [L[k:k + 64, k:k + 64] for L in factors]
            assert sum(64 * np.max(np.abs(D)) * np.max(np.abs(np.linalg.inv(D))) > 1e4 for D in B) >= 10
    for i in range(items):
        l1, g1, _, _ = ctx.ll_grad_batch(pid, gamma[i:i + 1], True)
        assert l1[0] == ll[i] and np.array_equal(g1[0], g[i]), i
        assert np.array_equal(ctx.read_item(0, 0), factors[i]), i
    ctx.close()


def test_loo_on_whole_tiles():
    # 11 blocks, 66 tiles; 8 starts of one fit are 528 tiles, past the line of 512
    n, d = 700, 2
    rng = np.random.default_rng(7)
    X = rng.uniform(size=(n, d))
    y = np.sum(np.sin(3 * X), axis=1) + 0.1 * rng.normal(size=n)
    th = np.exp(rng.uniform(np.log(0.05), 0.0, size=(8, d)))
    fit = lambda t: lk.Kriging(y, X, "matern3_2", "constant", False, "BFGS%d" % len(t), "LOO", {"theta": t})
    alone = [fit(th[i:i + 1]) for i in range(8)]
    values = [k.leaveOneOut() for k in alone]
    best = alone[int(np.argmin(values))]
    assert np.array_equal(fit(th).theta(), best.theta())


@pytest.mark.parametrize("n,m", [(700, 1100), (300, 200)])  # 594 tiles of 64 x 64, 60
def test_derivatives_against_dense(n, m):
    # d/dx of the simple-kriging formulas in 64 bits, by a general solver
    d, theta = 2, np.array([0.3, 0.5])
    rng = np.random.default_rng(n)
    X, Xn = rng.uniform(size=(n, d)), rng.uniform(size=(m, d))
    y = np.sum(np.sin(3 * X), axis=1)
    k = lk.Kriging("matern3_2")
    k.fit(y, X, "none", False, "none", "LL",
          {"theta": list(theta), "is_theta_estim": False, "sigma2": 1.2, "is_sigma2_estim": False})
    _, sd, _, dm, ds = k.predict(Xn, True, False, True)
    corr = lambda A, B: np.prod((1 + (u := np.sqrt(3) * np.abs(A[:, None] - B[None]) / theta)) * np.exp(-u), axis=2)
    R, r = corr(X, X), corr(X, Xn)
    tol = 1e3 * np.linalg.cond(R) * np.finfo(float).eps
    Riy, Rir = np.linalg.solve(R, y), np.linalg.solve(R, r)
    for q in range(d):
        u = np.sqrt(3) / theta[q] * (Xn[None, :, q] - X[:, None, q])
        dr = -r * np.sqrt(3) / theta[q] * u / (1 + np.abs(u))
        assert np.max(np.abs(dm[:, q] - dr.T @ Riy)) <= tol * np.max(np.abs(dm))
        dvar = -2 * 1.2 * np.sum(dr * Rir, axis=0)
        assert np.max(np.abs(2 * sd * ds[:, q] - dvar)) <= tol * np.max(np.abs(dvar))
