"""The NK aggregation at a point is the same, bit for bit, whatever other
points the call has and however it is cut into chunks: over the forms of the
pair kernel for few and for many points and the slices of its row tiles."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel,d,sizes", [
    ("matern3_2", 5, [64, 65, 200, 1, 130, 700]),
    ("matern5_2", 8, [1100, 129]),
    ("exp", 9, [300] * 9),
    ("gauss", 20, [150, 40, 70]),
    ("exp", 2, [70] * 70),  # 2 415 pairs
])
def test_points_alone(kernel, d, sizes):
    import libkriging_amd as lk
    rng = np.random.default_rng(d)
    X = rng.uniform(size=(sum(sizes), d))
    gof = np.repeat(np.arange(len(sizes)), sizes).astype(np.int32)
    nk = lk.NestedKriging(kernel)
    nk.fit_groups(np.sum(np.sin(3 * X), axis=1), X, gof, "constant", "none", "LL",
                  {"theta": [0.3 * np.sqrt(d) if kernel != "gauss" else 0.1 * d] * d, "is_theta_estim": False,
                   "sigma2": 1.3, "is_sigma2_estim": False, "beta": [0.2], "is_beta_estim": False})
    Xn = rng.uniform(size=(1200, d))
    mean, sd = nk.predict(Xn, True)
    for m in (1, 16, 17, 32, 33, 64, 129, 500, 512, 513, 1025):
        m1, s1 = nk.predict(Xn[-m:], True)
        assert np.array_equal(m1, mean[-m:]) and np.array_equal(s1, sd[-m:]), m
    for chunk in (30, 70, 600):
        nk.set_predict_chunk(chunk)
        m1, s1 = nk.predict(Xn, True)
        assert np.array_equal(m1, mean) and np.array_equal(s1, sd), chunk
