"""The work this framework is used for, as timed cases.

`listed()` names them, `draw(rng)` gives more of the same ranges, `prepare`
makes what a program holds before the call, `run` is one call through the
public entry points, `work` what it cannot do without and `exact` the same
result in plain torch, in 64 bits on the host.

Kinds:
  ll       the log-likelihood and its gradient at given parameters: one
           vector (what an external optimiser asks for) or a batch
           (multistart), through one Context kept by the program
  uneven   the same for several designs of different sizes in one batch
           (the submodels of a nested model)
  loo      the leave-one-out objective and its gradient
  fit      a whole multistart fit
  predict  mean and standard deviation at new points, optionally their
           covariance and derivatives
  nested   the aggregated prediction of a nested model
Designs are uniform in the unit cube.  gauss kernels, and every kernel in few
dimensions, come with a nugget: without one the correlation matrix is
numerically singular and two correct programs differ in most digits.
"""
import functools
import math

import numpy as np
import torch

import libkriging_amd as lk

KERNELS = ("gauss", "exp", "matern3_2", "matern5_2")


def listed():
    return [
        # a small model's likelihood, the unit step of a small fit: latency
        dict(name="ll_n200_d3_gauss_nugget", kind="ll", n=200, d=3, kernel="gauss", trend="constant", nugget=0.01,
             batch=1),
        # one evaluation of a medium model, as an external optimiser calls it
        dict(name="ll_n1000_d6_exp", kind="ll", n=1000, d=6, kernel="exp", trend="constant", nugget=0.0, batch=1),
        # the 64-start fit's step: one batched evaluation of all starts
        dict(name="ll_batch64_n1024_d6_exp", kind="ll", n=1024, d=6, kernel="exp", trend="constant", nugget=0.0,
             batch=64),
        # a large model with a linear trend
        dict(name="ll_n4096_d8_matern52_linear", kind="ll", n=4096, d=8, kernel="matern5_2", trend="linear",
             nugget=0.0, batch=1),
        # the largest single evaluation
        dict(name="ll_n8192_d10_gauss_nugget", kind="ll", n=8192, d=10, kernel="gauss", trend="constant",
             nugget=0.01, batch=1),
        # the submodels of a nested model in one batch, 300 to 1450 points each
        dict(name="uneven48_d5_matern32", kind="uneven", groups=48, d=5, kernel="matern3_2", nmin=300, nmax=1450),
        # the other fit objective
        dict(name="loo_n1500_d5_matern32", kind="loo", n=1500, d=5, kernel="matern3_2", trend="constant"),
        # a whole fit of a small model
        dict(name="fit_n300_d4_matern32_bfgs10", kind="fit", n=300, d=4, kernel="matern3_2", starts=10),
        # a small model's prediction on a plotting grid
        dict(name="predict_n200_m1000_d3", kind="predict", n=200, m=1000, d=3, kernel="gauss", trend="constant",
             nugget=0.01, cov=False, deriv=False),
        # a large model's prediction
        dict(name="predict_n3001_m5003_d6", kind="predict", n=3001, m=5003, d=6, kernel="exp", trend="constant",
             nugget=0.0, cov=False, deriv=False),
        # joint prediction with derivatives, as Bayesian optimisation asks for
        dict(name="predict_cov_deriv_n1000_m500_d4", kind="predict", n=1000, m=500, d=4, kernel="matern5_2",
             trend="linear", nugget=0.01, cov=True, deriv=True),
        # a nested model's prediction
        dict(name="nested_n20000_g32_m500_d5", kind="nested", n=20000, groups=32, m=500, d=5, kernel="matern3_2"),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["ll", "ll", "ll", "ll", "uneven", "loo", "fit", "predict", "predict", "nested"])
    d = rng.randint(1, 12)
    kernel = rng.choice(KERNELS)
    trend = rng.choice(["none", "constant", "constant", "linear"])
    nugget = 0.01 if kernel == "gauss" or d <= 4 or rng.random() < 0.3 else 0.0
    if kind == "ll":
        n = _log_uniform(rng, 50, 6000)
        most = max(1, min(64, int(1.5e11 / float(n) ** 3)))
        batch = 1 if rng.random() < 0.4 else _log_uniform(rng, 1, most)
        return dict(kind="ll", n=n, d=d, kernel=kernel, trend=trend, nugget=nugget, batch=batch)
    if kind == "uneven":
        lo = _log_uniform(rng, 60, 400)
        return dict(kind="uneven", groups=rng.randint(3, 48), d=rng.randint(5, 8),
                    kernel=rng.choice(["exp", "matern3_2"]), nmin=lo, nmax=lo * rng.randint(2, 4) - rng.randint(0, 40))
    if kind == "loo":
        return dict(kind="loo", n=_log_uniform(rng, 50, 2500), d=rng.randint(5, 10),
                    kernel=rng.choice(["exp", "matern3_2"]), trend=rng.choice(["constant", "linear"]))
    if kind == "fit":
        return dict(kind="fit", n=_log_uniform(rng, 50, 500), d=rng.randint(3, 6),
                    kernel=rng.choice(["exp", "matern3_2"]), starts=rng.randint(1, 12))
    if kind == "predict":
        cov, deriv = rng.random() < 0.3, rng.random() < 0.3
        n = _log_uniform(rng, 50, 2000 if cov or deriv else 4000)
        m = _log_uniform(rng, 1, 1200 if cov or deriv else 6000)
        return dict(kind="predict", n=n, m=m, d=min(d, 6) if deriv else d, kernel=kernel, trend=trend,
                    nugget=nugget, cov=cov, deriv=deriv)
    groups = rng.randint(3, 32)
    return dict(kind="nested", n=groups * _log_uniform(rng, 100, 600) + rng.randint(0, 63), groups=groups,
                m=_log_uniform(rng, 1, 500), d=rng.randint(4, 7), kernel=rng.choice(["exp", "matern3_2"]))


# -- inputs -------------------------------------------------------------------

def _design(rng, n, d):
    X = rng.uniform(size=(n, d))
    y = np.prod(1.0 + 0.5 * np.cos(3.0 * X), axis=1) + rng.normal(0.0, 1e-2, size=n)
    return X, y


def _theta(rng, d, shape=()):
    return np.exp(rng.uniform(math.log(0.2), math.log(1.0), size=tuple(shape) + (d,)))


def _trend(X, trend):
    n = X.shape[0]
    if trend == "none":
        return np.zeros((n, 0))
    return np.ones((n, 1)) if trend == "constant" else np.column_stack([np.ones(n), X])


def _sizes(case):
    """group sizes of an uneven batch: the same for every seed"""
    r = np.random.default_rng(case["groups"])
    s = np.exp(r.normal(math.log((case["nmin"] + case["nmax"]) / 2.5), 0.5, size=case["groups"]))
    return np.clip(s.astype(int), case["nmin"], case["nmax"])


def _inputs(case, seed):
    rng = np.random.default_rng(seed)
    kind, d = case["kind"], case["d"]
    if kind == "uneven":
        designs = [_design(rng, int(n), d) for n in _sizes(case)]
        return dict(designs=designs, theta=_theta(rng, d, (len(designs),)))
    X, y = _design(rng, case["n"], d)
    out = dict(X=X, y=y, theta=_theta(rng, d, (case["batch"],) if kind == "ll" else ()))
    if kind == "nested":
        out["group_of"] = rng.permutation(np.arange(case["n"]) % case["groups"]).astype(np.int32)
    if "m" in case:
        out["Xn"] = rng.uniform(size=(case["m"], d))
    return out


# -- the program under test ---------------------------------------------------

@functools.lru_cache(maxsize=None)
def _context():
    """one context per process, as a program keeps it"""
    return lk.Context(0)


class _Problems:
    """designs resident on the GPU for as long as this object lives"""

    def __init__(self, ctx, designs, kernel, noise, trend):
        self.ctx = ctx
        self.ids = [ctx.problem(X, y, _trend(X, trend), kernel, noise) for X, y in designs]

    def __del__(self):
        for i in self.ids:
            self.ctx.drop_problem(i)


def _model(case, inp):
    nug = case.get("nugget", 0.0) > 0.0
    m = lk.Kriging(case["kernel"], "nugget" if nug else "none")
    par = {"theta": inp["theta"]}
    if nug:
        par.update(sigma2=1.0, nugget=case["nugget"])
    m.fit(inp["y"], inp["X"], case["trend"], False, "none", "LL", par)
    return m


def prepare(case, seed):
    inp = _inputs(case, seed)
    kind = case["kind"]
    state = dict(case=case)
    if kind == "ll":
        nug = case["nugget"] > 0.0
        gamma = inp["theta"]
        if nug:
            gamma = np.column_stack([gamma, np.full(len(gamma), 1.0 / (1.0 + case["nugget"]))])
        state.update(problems=_Problems(_context(), [(inp["X"], inp["y"])], case["kernel"],
                                        "nugget" if nug else "none", case["trend"]), gamma=gamma)
    elif kind == "uneven":
        state.update(problems=_Problems(_context(), inp["designs"], case["kernel"], "none", "constant"),
                     gamma=inp["theta"])
    elif kind == "loo":
        state.update(model=_model(case, inp), theta=inp["theta"])
    elif kind == "fit":
        state.update(X=inp["X"], y=inp["y"])
    elif kind == "predict":
        state.update(model=_model(case, inp), Xn=inp["Xn"])
    else:
        m = lk.NestedKriging(case["kernel"])
        m.fit_groups(inp["y"], inp["X"], inp["group_of"], "constant", "none", "LL", {"theta": inp["theta"]})
        state.update(model=m, Xn=inp["Xn"])
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("ll", "uneven"):
        p = state["problems"]
        ids = p.ids[0] if kind == "ll" else p.ids
        ll, grad, status, _ = p.ctx.ll_grad_batch(ids, state["gamma"], True)
        return dict(ll=ll, grad=grad, status=status)
    if kind == "loo":
        v, g = state["model"].leaveOneOutFun(state["theta"], True)
        return dict(loo=v, grad=g)
    if kind == "fit":
        k = lk.Kriging(state["y"], state["X"], case["kernel"], "constant", False, "BFGS%d" % case["starts"], "LL")
        return dict(theta=k.theta(), sigma2=k.sigma2(), beta=k.beta(), ll=k.logLikelihood())
    if kind == "predict":
        mean, sd, cov, dm, ds = state["model"].predict(state["Xn"], True, case["cov"], case["deriv"])
        out = dict(mean=mean, stdev=sd)
        if case["cov"]:
            out["cov"] = cov
        if case["deriv"]:
            out.update(mean_deriv=dm, stdev_deriv=ds)
        return out
    mean, sd = state["model"].predict(state["Xn"], True)
    return dict(mean=mean, stdev=sd)


# -- what a call cannot do without --------------------------------------------

def _trend_width(case):
    return {"none": 0, "constant": 1, "linear": 1 + case["d"]}[case.get("trend", "constant")]


def work(case):
    """A likelihood with its gradient takes n^3 flops (factor, inverse factor
    and R^-1, a third each) and n^2 (p + 3) for its matrix-vector products;
    matrices that are made inside the call count no bytes."""
    kind, d = case["kind"], case["d"]
    p = _trend_width(case)

    def ll(n):
        return float(n) ** 3 + float(n) ** 2 * (p + 3)

    if kind == "uneven":
        s = _sizes(case)
        return dict(bytes=8.0 * sum(int(n) * (d + 2) for n in s), flops=sum(ll(int(n)) for n in s))
    n = case["n"]
    data = 8.0 * n * (d + 1 + p)
    if kind == "ll":
        return dict(bytes=data + 16.0 * case["batch"] * (d + 1), flops=case["batch"] * ll(n))
    if kind == "loo":
        # factor, inverse, B and B diag(a) B
        return dict(bytes=data, flops=2.0 * float(n) ** 3 + float(n) ** 2 * (2 * p + 6))
    if kind == "fit":
        # about ten evaluations per start
        return dict(bytes=data, flops=10.0 * case["starts"] * ll(n))
    m = case["m"]
    if kind == "predict":
        rows = m * (1 + d) if case["deriv"] else m
        flops = float(n) ** 2 * rows + 2.0 * n * rows * (p + 2)
        out = 16.0 * rows
        if case["cov"]:
            flops += float(m) ** 2 * n
            out += 8.0 * m * m
        return dict(bytes=data + 4.0 * n * n + 8.0 * m * d + out, flops=flops)
    sizes = np.bincount(np.arange(n) % case["groups"])
    own = float(np.sum(sizes.astype(float) ** 2))
    return dict(bytes=8.0 * n * (d + 1) + 4.0 * own + 8.0 * m * (d + 2),
                flops=m * (float(n) ** 2 - own + 2.0 * own) + m * case["groups"] ** 3 / 3.0)


# -- the same in plain torch, 64 bits -----------------------------------------

def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a))


def _corr(kernel, X1, X2, theta):
    """tensor-product kernel values k(x1_i - x2_j)"""
    R, s = None, None
    for k in range(X1.shape[1]):
        u = (X1[:, k, None] - X2[None, :, k]) / theta[k]
        if kernel == "gauss":
            t, q = 0.5 * u * u, None
        elif kernel == "exp":
            t, q = u.abs(), None
        elif kernel == "matern3_2":
            t = math.sqrt(3.0) * u.abs()
            q = 1.0 + t
        else:
            t = math.sqrt(5.0) * u.abs()
            q = 1.0 + t + t * t / 3.0
        s = t if s is None else s + t
        if q is not None:
            R = q if R is None else R * q
    return torch.exp(-s) if R is None else R * torch.exp(-s)


def _dlog(kernel, dx, th):
    """d ln k / d theta for one coordinate's differences"""
    if kernel == "gauss":
        return dx * dx / th ** 3
    if kernel == "exp":
        return dx.abs() / th ** 2
    if kernel == "matern3_2":
        u = math.sqrt(3.0) * dx.abs() / th
        return u * u / (1.0 + u) / th
    u = math.sqrt(5.0) * dx.abs() / th
    b = u * u / 3.0
    return (1.0 + u) * b / (1.0 + u + b) / th


def _gls(R, y, F):
    """(L, M = L^-1 F, z = L^-1 (y - F beta), beta)"""
    L = torch.linalg.cholesky(R)
    M = torch.linalg.solve_triangular(L, F, upper=False) if F.shape[1] else F
    ys = torch.linalg.solve_triangular(L, y[:, None], upper=False)
    beta = torch.linalg.solve(M.T @ M, M.T @ ys) if F.shape[1] else torch.zeros(0, 1, dtype=y.dtype)
    return L, M, (ys - M @ beta)[:, 0], beta[:, 0]


def _with_nugget(C, alpha):
    R = alpha * C
    R.fill_diagonal_(1.0)
    return R


def _ll_exact(X, y, F, kernel, theta, alpha):
    n, d = X.shape
    C = _corr(kernel, X, X, theta)
    R = _with_nugget(C, 1.0 if alpha is None else alpha)
    L, M, z, _ = _gls(R, y, F)
    s2 = z @ z / n
    ll = -0.5 * (n * torch.log(2.0 * math.pi * s2) + 2.0 * torch.log(torch.diagonal(L)).sum() + n)
    x = torch.linalg.solve_triangular(L.T, z[:, None], upper=True)[:, 0]
    W = torch.outer(x, x) / s2
    W -= torch.cholesky_inverse(L)
    W.fill_diagonal_(0.0)
    g = np.zeros(d + (alpha is not None))
    if alpha is not None:
        g[d] = 0.5 * float((W * C).sum())
    W *= R
    for k in range(d):
        g[k] = 0.5 * float((W * _dlog(kernel, X[:, k, None] - X[None, :, k], theta[k])).sum())
    return float(ll), g


def _predict_exact(case, inp):
    X, y, Xn, theta = (_t(inp[k]) for k in ("X", "y", "Xn", "theta"))
    alpha = 1.0 / (1.0 + case["nugget"])
    F = _t(_trend(inp["X"], case["trend"]))
    R = _with_nugget(_corr(case["kernel"], X, X, theta), alpha)
    L, M, z, beta = _gls(R, y, F)
    vs = z @ z / X.shape[0]
    Rs = torch.linalg.cholesky(M.T @ M) if F.shape[1] else None
    Xn.requires_grad_(case["deriv"])

    def trend(Xq):
        one = torch.ones(Xq.shape[0], 1, dtype=Xq.dtype)
        return {"none": one[:, :0], "constant": one, "linear": torch.cat([one, Xq], 1)}[case["trend"]]

    C = torch.linalg.solve_triangular(L, alpha * _corr(case["kernel"], X, Xn, theta), upper=False)
    Fn = trend(Xn)
    mean = Fn @ beta + C.T @ z
    var = 1.0 - (C * C).sum(0)
    E = None
    if F.shape[1]:
        E = torch.linalg.solve_triangular(Rs, (Fn - C.T @ M).T, upper=False)
        var = var + (E * E).sum(0)
    sd = torch.sqrt(vs * var.clamp(min=0.0))
    out = dict(mean=mean.detach(), stdev=sd.detach())
    if case["cov"]:
        Rnn = _with_nugget(_corr(case["kernel"], Xn, Xn, theta).detach(), alpha)
        out["cov"] = (vs * (Rnn - C.T @ C + (E.T @ E if E is not None else 0.0))).detach()
    if case["deriv"]:
        out["mean_deriv"] = torch.autograd.grad(mean.sum(), Xn, retain_graph=True)[0]
        out["stdev_deriv"] = torch.autograd.grad(sd.sum(), Xn)[0]
    return out


def _loo_exact(case, inp):
    X, y = _t(inp["X"]), _t(inp["y"])
    F = _t(_trend(inp["X"], case["trend"]))
    theta = _t(inp["theta"]).requires_grad_(True)
    n = X.shape[0]
    R = _corr(case["kernel"], X, X, theta)
    R = R - torch.diag(torch.diagonal(R)) + torch.eye(n, dtype=R.dtype)
    Ri = torch.cholesky_inverse(torch.linalg.cholesky(R))
    RF = Ri @ F
    B = Ri - RF @ torch.linalg.solve(F.T @ RF, RF.T)
    err = (B @ y) / torch.diagonal(B)
    loo = (err @ err) / n
    return dict(loo=float(loo.detach()), grad=torch.autograd.grad(loo, theta)[0])


def _nested_exact(case, inp):
    """Rulliere et al.'s aggregation of simple-kriging submodels, the common
    variance and mean being the groups' own, weighted by their sizes"""
    X, y, Xn, theta = (_t(inp[k]) for k in ("X", "y", "Xn", "theta"))
    kernel, p, m, jitter = case["kernel"], case["groups"], case["m"], 1e-10
    groups = [torch.from_numpy(np.flatnonzero(inp["group_of"] == g)) for g in range(p)]
    chol, s2, b0 = [], 0.0, 0.0
    for idx in groups:
        R = _corr(kernel, X[idx], X[idx], theta)
        _, _, z, beta = _gls(R, y[idx], torch.ones(len(idx), 1, dtype=X.dtype))
        w = len(idx) / float(case["n"])
        s2, b0 = s2 + w * float(z @ z) / len(idx), b0 + w * float(beta[0])
        R.diagonal().add_(jitter)
        chol.append(torch.linalg.cholesky(R))
    W, mu, own = [], [], []
    for idx, L in zip(groups, chol):
        c = _corr(kernel, X[idx], Xn, theta)
        w = torch.cholesky_solve(c, L)
        W.append(w)
        mu.append(w.T @ (y[idx] - b0))
        own.append((c * w).sum(0))
    K = torch.zeros(m, p, p, dtype=X.dtype)
    for i in range(p):
        K[:, i, i] = own[i] + jitter
        later = range(i + 1, p)
        if not later:
            continue
        # all later groups at once: R(X_i, X_later) in one piece
        idx = torch.cat([groups[j] for j in later])
        Rij = _corr(kernel, X[groups[i]], X[idx], theta)
        at = 0
        for j in later:
            v = (W[i] * (Rij[:, at:at + len(groups[j])] @ W[j])).sum(0)
            at += len(groups[j])
            K[:, i, j] = v
            K[:, j, i] = v
    kM = torch.diagonal(K, dim1=1, dim2=2)
    w = torch.linalg.solve(K, kM[:, :, None])[:, :, 0]
    mean = b0 + (w * torch.stack(mu, 1)).sum(1)
    var = s2 * (1.0 - (w * kM).sum(1)).clamp(min=0.0)
    return dict(mean=mean, stdev=torch.sqrt(var))


def exact(case, seed):
    inp = _inputs(case, seed)
    kind = case["kind"]
    if kind == "fit":
        return None  # where an iteration stops is no formula
    if kind == "predict":
        return _predict_exact(case, inp)
    if kind == "loo":
        return _loo_exact(case, inp)
    if kind == "nested":
        return _nested_exact(case, inp)
    if kind == "uneven":
        jobs = [(X, y, inp["theta"][i]) for i, (X, y) in enumerate(inp["designs"])]
    else:
        jobs = [(inp["X"], inp["y"], th) for th in inp["theta"]]
    alpha = 1.0 / (1.0 + case["nugget"]) if case.get("nugget", 0.0) > 0.0 else None
    got = [_ll_exact(_t(X), _t(y), _t(_trend(X, case.get("trend", "constant"))), case["kernel"], _t(th), alpha)
           for X, y, th in jobs]
    return dict(ll=np.array([v for v, _ in got]), grad=np.array([g for _, g in got]), status=None)
