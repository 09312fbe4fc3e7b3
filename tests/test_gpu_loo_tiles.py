"""The leave-one-out gradient's B on quarter tiles (up to 512 tiles) and on
whole ones (n = 2100: 561 tiles), at the edges of tiles, against central
differences of the objective, which does not use B."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3, 64, 65, 130, 700, 2100])
@pytest.mark.parametrize("regmodel", ["constant", "linear"])
def test_gradient_against_differences(n, regmodel):
    import libkriging_amd as lk
    if regmodel == "linear" and n < 10:
        pytest.skip("fewer points than trend columns leave no residual")
    d = 3
    rng = np.random.default_rng(n)
    X = rng.uniform(size=(n, d))
    y = np.sum(np.sin(3 * X), axis=1)
    k = lk.Kriging("matern3_2")
    k.fit(y, X, regmodel, False, "none", "LOO", {"theta": [0.5] * d, "is_theta_estim": False})
    th = np.array([0.3, 0.5, 0.8])
    v, g = k.leaveOneOutFun(th, True)
    h = 1e-5
    for q in range(d):
        e = np.zeros(d)
        e[q] = h
        num = (k.leaveOneOutFun(th + e)[0] - k.leaveOneOutFun(th - e)[0]) / (2 * h)
        # step error h^2 f''' / 6 and rounding cond eps f / h, both below 1e-5 f
        assert abs(g[q] - num) <= 1e-4 * max(abs(v), np.max(np.abs(g)))
