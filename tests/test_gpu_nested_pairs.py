"""The group-pair sums of the NK aggregation over the widths its kernels are
cut at: 16, 32 and 64 points in registers, 128 to 512 through the LDS, more in
whole tiles and a rest; dimensions on both sides of what is kept in registers;
groups of one point, of one tile, and of several with a remainder."""
import numpy as np
import pytest

from oracle import nested as NKO
from oracle import oracle as O

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps
WIDTHS = [1, 16, 17, 32, 33, 64, 65, 128, 129, 300, 385, 512, 513, 576, 580, 650]


@pytest.mark.parametrize("kernel,d,sizes", [
    ("matern3_2", 5, [64, 65, 200, 1, 130]),
    ("matern5_2", 8, [17, 129]),
    ("exp", 9, [3, 66, 128]),
    ("gauss", 32, [1, 1, 40, 70]),
    ("exp", 1, [5] * 12),
    ("exp", 3, [3] * 64),  # the largest system solved in LDS
    ("exp", 3, [3] * 65),
])
def test_pair_widths(kernel, d, sizes):
    import libkriging_amd as lk
    rng = np.random.default_rng(100 + d)
    n = sum(sizes)
    X = rng.uniform(size=(n, d))
    y = np.sum(np.sin(3 * X), axis=1)
    gof = np.repeat(np.arange(len(sizes)), sizes).astype(np.int32)
    theta = [0.3 * np.sqrt(d) if kernel != "gauss" else 0.1 * d] * d
    nk = lk.NestedKriging(kernel)
    nk.fit_groups(y, X, gof, "constant", "none", "LL",
                  {"theta": theta, "is_theta_estim": False, "sigma2": 1.3, "is_sigma2_estim": False,
                   "beta": [0.2], "is_beta_estim": False})
    G = [np.asarray(g, dtype=np.int64) for g in nk.groups()]
    Xn = rng.uniform(size=(max(WIDTHS), d))
    m_o, s_o = NKO.predict_nk(X, y, G, nk.theta(), 1.3, 0.2, kernel, Xn)
    # the aggregation solves with the groups' matrices and, per point, with one
    # between their predictors that no eigenvalue of the joint matrix undercuts
    c = np.linalg.cond(O.corr_mat(kernel, X, X, nk.theta()) + 1e-10 * np.eye(n))
    tol = max(1e-11, 1e3 * c * EPS)
    for m in WIDTHS:
        mean, sd = nk.predict(Xn[:m], True)
        em = np.max(np.abs(mean - m_o[:m])) / max(1.0, np.max(np.abs(m_o)))
        es = np.max(np.abs(sd ** 2 - s_o[:m] ** 2)) / 1.3
        assert em <= tol and es <= tol, (m, em, es, tol)
        if m == max(WIDTHS):
            # the same points in chunks of another width
            nk.set_predict_chunk(70)
            m2, s2 = nk.predict(Xn[:m], True)
            assert np.max(np.abs(m2 - mean)) <= tol * max(1.0, np.max(np.abs(m_o)))
            assert np.max(np.abs(s2 ** 2 - sd ** 2)) <= tol * 1.3
