"""Prediction on both tile sizes of its products and over the trend widths of
its sums: the 32 x 32 and the 64 x 64 tiles (512 tiles of 64 x 64 apart), with
remainders in rows and points, one pass over [M | z] and several."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


@pytest.mark.parametrize("n,m,d,regmodel,cov,deriv", [
    (7, 1, 1, "constant", True, True),
    (64, 65, 2, "none", True, True),
    (129, 33, 6, "linear", True, True),     # 7 columns of [M | z]: two passes
    (200, 130, 12, "linear", True, False),  # 14: three
    (300, 700, 3, "linear", False, True),   # 5 x 11 x 4 = 220 tiles
    (700, 1100, 2, "constant", False, True),  # 11 x 18 x 3 = 594: 64 x 64
    (1000, 2100, 4, "constant", False, False),  # 16 x 33 = 528: 64 x 64
    (90, 2100, 3, "constant", True, False),  # 561 covariance tiles of 64 x 64
])
def test_tiles_and_trends(n, m, d, regmodel, cov, deriv):
    import libkriging_amd as lk
    rng = np.random.default_rng(n + m)
    X, Xn = rng.uniform(size=(n, d)), rng.uniform(size=(m, d))
    y = np.sum(np.sin(3 * X), axis=1)
    theta = np.full(d, 0.4 * np.sqrt(d))
    k = lk.Kriging("matern5_2")
    k.fit(y, X, regmodel, False, "none", "LL", {"theta": list(theta), "is_theta_estim": False, "sigma2": 1.2,
                                               "is_sigma2_estim": False})
    mean, sd, cv, dm, ds = k.predict(Xn, True, cov, deriv)
    # the universal-kriging formulas in 64 bits, by a general solver
    R = O.corr_mat("matern5_2", X, X, theta)
    r = O.corr_mat("matern5_2", X, Xn, theta)
    one = lambda A: np.ones((len(A), 1))
    F, Fn = {"none": (np.zeros((n, 0)), np.zeros((m, 0))), "constant": (one(X), one(Xn)),
             "linear": (np.hstack([one(X), X]), np.hstack([one(Xn), Xn]))}[regmodel]
    Ri = np.linalg.solve(R, np.hstack([r, F, y[:, None]]))
    Rir, RiF, Riy = Ri[:, :m], Ri[:, m:-1], Ri[:, -1]
    G = F.T @ RiF
    beta = np.linalg.solve(G, F.T @ Riy) if F.shape[1] else np.zeros(0)
    res = Riy - RiF @ beta
    E = Fn - r.T @ RiF
    S = np.linalg.solve(G, E.T) if F.shape[1] else np.zeros((0, m))
    c = np.linalg.cond(R)
    tol = max(1e-11, 1e3 * c * EPS)
    scale = max(1.0, np.max(np.abs(y)))
    assert np.max(np.abs(mean - (Fn @ beta + r.T @ res))) <= tol * scale
    var = 1.0 - np.sum(r * Rir, axis=0) + np.sum(E.T * S, axis=0)
    assert np.max(np.abs(sd ** 2 / 1.2 - np.maximum(var, 0.0))) <= tol
    if cov:
        C = O.corr_mat("matern5_2", Xn, Xn, theta) - r.T @ Rir + E @ S
        assert np.max(np.abs(cv / 1.2 - C)) <= tol
        np.testing.assert_array_equal(cv, cv.T)
    if deriv:
        # central differences of the same call: step h, error h^2 f''' and tol / h
        h = 1e-4
        for q in range(min(d, 2)):
            e = np.zeros(d)
            e[q] = h
            up, dn = k.predict(Xn + e, True, False, False), k.predict(Xn - e, True, False, False)
            assert np.max(np.abs(dm[:, q] - (up[0] - dn[0]) / (2 * h))) <= max(1e-4, tol / h) * scale
            dvar = (up[1] ** 2 - dn[1] ** 2) / (2 * h)
            assert np.max(np.abs(2 * sd * ds[:, q] - dvar)) <= max(1e-4, tol / h)
