"""The blocked factorisation's kernels at the sizes where their tiles end:
one and two 64-row blocks per diagonal square, the remainders of both, the
rows below them in 16- and 64-row workgroups, and the 256-row groups of the
inverse.  Oracles: numpy's Cholesky and triangular inverse.

Tolerances: a computed factor satisfies |A - L L'| <= gamma_(n+1) |L||L'|
elementwise (Higham, Accuracy and Stability, Thm 10.3), so with unit diagonal
|A - L L'|_max <= (n + 1) eps; products with the explicit inverse of a
well-conditioned diagonal block add a few times cond(L_kk) <= 30 here: 64 (n +
1) eps is used."""
import numpy as np
import pytest

import libkriging_amd as lk

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps
SIZES = [1, 2, 15, 16, 17, 48, 63, 64, 65, 80, 127, 128, 129, 191, 192, 193, 255, 256, 257, 320, 385, 511, 513, 640]


def spd(n, seed=0):
    rng = np.random.default_rng(seed + n)
    X = rng.uniform(size=(n, 3))
    R = np.exp(-np.sum(np.abs(X[:, None, :] - X[None, :, :]), axis=2) / 0.3)
    return 0.9 * R + 0.1 * np.eye(n)


@pytest.mark.parametrize("n", SIZES)
def test_factor_at_block_edges(n):
    A = spd(n)
    L = lk.linalg.chol_safe(A)
    assert np.all(np.triu(L, 1) == 0.0)
    assert np.max(np.abs(A - L @ L.T)) <= 64 * (n + 1) * EPS


@pytest.mark.parametrize("n", [40, 64, 100, 128, 200, 260, 400])
def test_inverse_factor(n):
    # the inverse inside the 256-row groups and across them, through a model's
    # factors: L^-1 F* relations of the committed model
    rng = np.random.default_rng(n)
    ctx = lk.Context(0)
    X = rng.uniform(size=(n, 3))
    pid = ctx.problem(X, rng.normal(size=n), np.ones((n, 1)), "exp")
    ctx.ll_grad_batch(pid, np.full((1, 3), 0.3), False)
    L, Li = ctx.read_item(0, 0), ctx.read_item(0, 1)
    # |L Li - I| <= gamma_n |L||Li| elementwise for a product-formed inverse,
    # a few levels of products: 64 n eps |L||Li|
    bound = 64 * n * EPS * (np.abs(L) @ np.abs(Li)) + EPS
    assert np.all(np.abs(L @ Li - np.eye(n)) <= bound)


@pytest.mark.parametrize("items", [1, 7, 24])
def test_row_workgroup_sizes_agree(items):
    # 24 items of 9 blocks run the rows below the squares in 64-row
    # workgroups, one item in 16-row ones: the same arithmetic
    n = 530
    rng = np.random.default_rng(5)
    X = rng.uniform(size=(n, 4))
    y = rng.normal(size=n)
    th = np.exp(rng.uniform(np.log(0.2), 0.0, size=(items, 4)))
    ctx = lk.Context(0)
    pid = ctx.problem(X, y, np.ones((n, 1)), "matern3_2")
    ll, g, st, _ = ctx.ll_grad_batch(pid, th, True)
    assert np.all(st == 0)
    for i in range(items):
        l1, g1, _, _ = ctx.ll_grad_batch(pid, th[i:i + 1], True)
        assert l1[0] == ll[i] and np.array_equal(g1[0], g[i])


@pytest.mark.parametrize("row", [0, 5, 16, 33, 63, 64, 70, 100, 127, 128, 150])
def test_bad_pivot_is_found_in_every_panel(row):
    n = 160
    A = spd(n)
    A[row, row] = -1.0
    lk.set_num_nugget(0.0)
    try:
        with pytest.raises(RuntimeError):
            lk.linalg.chol_safe(A)
    finally:
        lk.set_num_nugget(1e-10)


@pytest.mark.parametrize("n", [70, 128, 200, 300])
def test_ill_conditioned_diagonal_blocks(n):
    # cond(L_kk) well past the refinement threshold in every block: a factor
    # with geometric diagonal, whose backward error stays at the level above
    # times the refined products' small constant
    rng = np.random.default_rng(n)
    L0 = np.tril(rng.uniform(-1.0, 1.0, size=(n, n)), -1) / np.sqrt(n)
    L0 += np.diag(10.0 ** (-5.0 * (np.arange(n) % 64) / 63.0))
    A = L0 @ L0.T
    L, inc = lk.linalg.chol_safe(A, return_inc=True)
    p10 = sum(1e-10 * 10.0 ** q for q in range(inc))
    B = A + p10 * np.eye(n)
    scale = np.sqrt(np.outer(np.diag(B), np.diag(B)))
    assert np.max(np.abs(B - L @ L.T) / scale) <= 256 * (n + 1) * EPS


@pytest.mark.parametrize("n", [5, 64, 65, 128, 130, 300])
def test_given_factor(n):
    # factor mode: only the inverses are formed; rcond(L)^2 in the 1-norm is
    # never above the exact one's by more than rounding, and never below a
    # tenth of it for these factors (the estimator is sharp on them)
    L = np.linalg.cholesky(spd(n))
    r = lk.linalg.rcond_chol(L)
    exact = (1.0 / (np.linalg.norm(L, 1) * np.linalg.norm(np.linalg.inv(L), 1))) ** 2
    assert exact * (1 - 1e-10) <= r <= 100 * exact
