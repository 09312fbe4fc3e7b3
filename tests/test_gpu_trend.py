"""The trend's normal equations, summed per 64-row block and solved by every
workgroup of the GLS kernel: widths from none to the largest, row counts at
the edges of the 64- and 256-row units.  Oracle: numpy in the orthogonal form
(QR of the whitened trend).  Both solve with F*'F* or its R factor, so the
results agree to cond(F*)^2 eps (normal equations, here and in the reference,
KrigingImpl.cpp:105-121); cond(F*) is computed and used with a factor 64 n
for the sums."""
import numpy as np
import pytest
import scipy.linalg as sla

import libkriging_amd as lk

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


@pytest.mark.parametrize("n,d,p", [(1, 1, 0), (5, 1, 1), (63, 2, 1), (64, 3, 4), (65, 1, 2), (130, 4, 0), (200, 8, 9),
                                   (255, 20, 21), (257, 22, 23), (300, 32, 33), (520, 9, 10), (1030, 16, 17)])
def test_gls_against_qr(n, d, p):
    rng = np.random.default_rng(n + d)
    X = rng.uniform(size=(n, d))
    y = 3.0 + rng.normal(size=n)
    F = np.column_stack([np.ones(n), X])[:, :p]
    th = 0.7 * np.ones((1, d)) * np.sqrt(d)
    ctx = lk.Context(0)
    pid = ctx.problem(X, y, F, "exp")
    ll, _, st, _ = ctx.ll_grad_batch(pid, th, False)
    assert st[0] == 0
    R = np.exp(-np.sum(np.abs(X[:, None] - X[None]) / th[0], axis=2))
    L = np.linalg.cholesky(R)
    Fs = sla.solve_triangular(L, F, lower=True)
    ys = sla.solve_triangular(L, y, lower=True)
    if p > 0:
        Q, _ = np.linalg.qr(Fs)
        E = ys - Q @ (Q.T @ ys)
        cond = np.linalg.cond(Fs)
    else:
        E, cond = ys, 1.0
    tol = 64 * n * EPS * cond ** 2 * max(1.0, np.linalg.cond(L))
    got = ctx.read_item(0, 4)
    assert np.linalg.norm(got - E) <= tol * np.linalg.norm(ys)
    s2 = E @ E / n
    want = -0.5 * (n * np.log(2 * np.pi * s2) + 2 * np.sum(np.log(np.diag(L))) + n)
    # d ll / d |E| = -n / |E|
    assert abs(ll[0] - want) <= n * tol * np.linalg.norm(ys) / np.linalg.norm(E) + 64 * n * EPS * abs(want)
