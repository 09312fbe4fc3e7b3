"""A point's prediction is the same, bit for bit, whatever other points the
call has: over the lines between the tile sizes of the products (512 tiles of
64 x 64), and over the forms, slices and chunks of the nested aggregation."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def model(n, d, regmodel="constant"):
    import libkriging_amd as lk
    rng = np.random.default_rng(n + d)
    X = rng.uniform(size=(n, d))
    k = lk.Kriging("matern5_2")
    k.fit(np.sum(np.sin(3 * X), axis=1), X, regmodel, False, "none", "LL",
          {"theta": [0.4 * np.sqrt(d)] * d, "is_theta_estim": False, "sigma2": 1.2, "is_sigma2_estim": False})
    return k, rng


@pytest.mark.parametrize("n,d,many,few", [
    (1000, 4, 2100, [1, 33, 64, 500]),  # 528 tiles; fewer
    (700, 2, 3100, [1, 65, 2900]),      # 539
    (129, 6, 8192, [1, 100]),           # 384
])
def test_mean_and_stdev(n, d, many, few):
    k, rng = model(n, d, "linear")
    Xn = rng.uniform(size=(many, d))
    mean, sd = k.predict(Xn, True, False, False)[:2]
    for m in few:
        m1, s1 = k.predict(Xn[-m:], True, False, False)[:2]
        assert np.array_equal(m1, mean[-m:]) and np.array_equal(s1, sd[-m:]), m


@pytest.mark.parametrize("n,d,many,few", [(700, 2, 1100, [1, 100, 500]), (90, 3, 600, [7])])
def test_derivatives(n, d, many, few):
    k, rng = model(n, d, "linear")
    Xn = rng.uniform(size=(many, d))
    dm, ds = k.predict(Xn, True, False, True)[3:]
    for m in few:
        d1, s1 = k.predict(Xn[-m:], True, False, True)[3:]
        assert np.array_equal(d1, dm[-m:]) and np.array_equal(s1, ds[-m:]), m


@pytest.mark.parametrize("n,d,many,few", [(90, 3, 2100, [1, 65, 500]), (300, 20, 2047, [64])])
def test_covariance(n, d, many, few):
    # 561 covariance tiles of 64 x 64 (2047 points: 528); fewer
    k, rng = model(n, d)
    Xn = rng.uniform(size=(many, d))
    cov = k.predict(Xn, True, True, False)[2]
    assert np.array_equal(cov, cov.T)
    for m in few:
        assert np.array_equal(k.predict(Xn[-m:], True, True, False)[2], cov[-m:, -m:]), m
