"""Work that a user of gpjax_amd has it do, from the smallest call to the largest.

Sizes are those of the package's own workloads (``gpjax_amd/workloads.py``) where it
has one, generic and ragged (no multiple of a tile) elsewhere.  Every case goes through the
public entry points: ``conjugate_mll`` / ``conjugate_loocv`` / ``collapsed_elbo``
with their gradients, ``fit``, ``ConjugatePosterior.predict``, the batched MLL and
the kernels' ``cross_covariance`` / ``gram``.  float64 is the package's default;
"mixed" is its large-problem option.

A case is a dict of plain values; ``kind`` names the path:

  mll, loocv   n, d, kernel, ard, precision         objective and its gradient
  fit          n, d, kernel, ard, steps, graph      a short Adam run
  predict      n, d, kernel, ard, t, full           predictive (full: and log-prob)
  elbo         n, m, d, kernel, ard, precision      collapsed ELBO, gradient with Z
  batched      count, nmin, nmax, d                 many small GPs, MLL and gradients
  cov          n, m, d, kernel, ard                 cross-covariance (m = 0: gram)
"""

from __future__ import annotations

import math

import torch

import gpjax_amd as gpx
from gpjax_amd.batched import BatchedConjugateMLL

KERNELS = ("rbf", "matern12", "matern32", "matern52")
JITTER = 1e-6


def listed():
    return [
        # the surrogate of a Bayesian-optimisation loop: one objective + gradient
        # on a handful of points; launches and host work are all there is
        dict(name="mll_100", kind="mll", n=100, d=4, kernel="rbf", ard=True, precision="fp64"),
        # training a small regression model with the package's own fit loop
        dict(name="fit_300", kind="fit", n=300, d=3, kernel="matern52", ard=True, steps=25,
             graph=False),
        # the plain regression example (workloads.exact_small): one training step
        dict(name="mll_2000", kind="mll", n=2000, d=1, kernel="rbf", ard=False,
             precision="fp64"),
        # the same model's predictive at 500 test points, scored on held-out targets
        dict(name="predict_2000_500", kind="predict", n=2000, d=1, kernel="rbf", ard=False,
             t=500, full=True),
        # leave-one-out objective at a ragged size
        dict(name="loocv_3001", kind="loocv", n=3001, d=8, kernel="matern52", ard=True,
             precision="fp64"),
        # workloads.exact_matern: a training step of a large exact GP in float64
        dict(name="mll_16384", kind="mll", n=16384, d=8, kernel="matern52", ard=True,
             precision="fp64"),
        # workloads.exact_large: the largest exact GP, in the mixed-precision option
        dict(name="mll_65536_mixed", kind="mll", n=65536, d=16, kernel="rbf", ard=True,
             precision="mixed"),
        # predictive variances over a large grid of test points
        dict(name="predict_diag_8192", kind="predict", n=8192, d=8, kernel="matern52", ard=True,
             t=100003, full=False),
        # a sparse GP of everyday size: training step with the inducing inputs
        dict(name="elbo_50021_500", kind="elbo", n=50021, m=500, d=8, kernel="matern32",
             ard=True, precision="fp64"),
        # workloads.sparse: a million points, 2,048 inducing inputs, mixed precision
        dict(name="elbo_1e6_2048_mixed", kind="elbo", n=1_000_000, m=2048, d=8,
             kernel="matern32", ard=True, precision="mixed"),
        # workloads.batched: thousands of small GPs of uneven size in one call
        dict(name="batched_4096", kind="batched", count=4096, nmin=32, nmax=1024, d=4),
        # the kernel matrix itself, for callers that do their own algebra
        dict(name="cross_cov_10007", kind="cov", n=10007, m=4099, d=8, kernel="rbf", ard=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mll", "mll", "mll", "mll", "fit", "predict", "predict", "loocv", "elbo",
                       "elbo", "batched", "cov"])
    kernel = rng.choice(KERNELS)
    ard = rng.random() < 0.7
    if kind == "mll":
        mixed = rng.random() < 0.25
        n = _log_int(rng, 4096, 40000) if mixed else _log_int(rng, 20, 16384)
        d = rng.randint(8, 20) if mixed else rng.randint(1, 20)
        return dict(kind=kind, n=n, d=d, kernel="rbf" if mixed else kernel, ard=ard,
                    precision="mixed" if mixed else "fp64")
    if kind == "loocv":
        return dict(kind=kind, n=_log_int(rng, 50, 10000), d=rng.randint(1, 16), kernel=kernel,
                    ard=ard, precision="fp64")
    if kind == "fit":
        return dict(kind=kind, n=_log_int(rng, 50, 1500), d=rng.randint(1, 8), kernel=kernel,
                    ard=ard, steps=rng.randint(10, 40), graph=rng.random() < 0.5)
    if kind == "predict":
        full = rng.random() < 0.5
        n = _log_int(rng, 50, 12000)
        t = _log_int(rng, 10, 2000) if full else _log_int(rng, 1000, 100000)
        return dict(kind=kind, n=n, d=rng.randint(1, 16), kernel=kernel, ard=ard, t=t, full=full)
    if kind == "elbo":
        mixed = rng.random() < 0.4
        n = _log_int(rng, 20000, 800000) if mixed else _log_int(rng, 1000, 300000)
        m = _log_int(rng, 256, 2048) if mixed else _log_int(rng, 20, 2048)
        return dict(kind=kind, n=n, m=min(m, n // 2), d=rng.randint(6, 16),
                    kernel="matern32" if mixed else rng.choice(KERNELS), ard=True,
                    precision="mixed" if mixed else "fp64")
    if kind == "batched":
        nmin = _log_int(rng, 8, 128)
        return dict(kind=kind, count=_log_int(rng, 16, 3000), nmin=nmin,
                    nmax=nmin + _log_int(rng, 32, 1000), d=rng.randint(1, 8))
    n = _log_int(rng, 100, 15000)
    m = 0 if rng.random() < 0.5 else _log_int(rng, 100, 15000)
    return dict(kind="cov", n=n, m=m, d=rng.randint(1, 20), kernel=kernel, ard=ard)


# ---- inputs -------------------------------------------------------------------

def _uniform(g, lo, hi, *shape):
    return lo + (hi - lo) * torch.rand(*shape, generator=g, dtype=torch.float64, device="cuda")


def _log_uniform(g, lo, hi, *shape):
    return torch.exp(_uniform(g, math.log(lo), math.log(hi), *shape))


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, dtype=torch.float64, device="cuda")


def _inputs(case, seed):
    """Everything the case's call reads, as float64 tensors on the GPU."""
    g = torch.Generator(device="cuda").manual_seed(1_000_003 * seed + 17)
    kind, d = case["kind"], case["d"]
    if kind == "batched":
        cpu = torch.Generator().manual_seed(1_000_003 * seed + 17)
        sizes = torch.randint(case["nmin"], case["nmax"] + 1, (case["count"],), generator=cpu)
        B = case["count"]
        X = torch.rand(int(sizes.sum()), d, generator=cpu, dtype=torch.float64)
        e = torch.randn(X.shape[0], generator=cpu, dtype=torch.float64)

        def logu(lo, hi, *shape):
            u = torch.rand(*shape, generator=cpu, dtype=torch.float64)
            return torch.exp(math.log(lo) + (math.log(hi) - math.log(lo)) * u)

        ls, var, sd = logu(0.1, 1.0, B, d), logu(0.5, 2.0, B), logu(0.02, 0.2, B)
        y = torch.sin(6 * X[:, 0]) + X[:, -1] ** 2 + sd.repeat_interleave(sizes) * e
        return dict(sizes=sizes.tolist(), X=X, y=y, ls=ls, var=var, sd=sd)
    n = case["n"]
    nls = d if case["ard"] else 1
    if kind == "elbo":
        X = _uniform(g, 0.0, 1.0, n, d)
        Z = X[torch.randperm(n, generator=g, device="cuda")[:case["m"]]].clone()
        ls, sd = _uniform(g, 0.1, 0.3, nls) * math.sqrt(d / 8), 0.2
        y = torch.sin(2 * math.pi * X).sum(1) + sd * _normal(g, n)
        return dict(X=X, y=y, Z=Z, ls=ls, var=1.0, sd=sd)
    if d == 1:
        X = _uniform(g, -3.0, 3.0, n, 1)
        ls, var, sd = torch.full((1,), 0.5, dtype=torch.float64, device="cuda"), 1.0, 0.1
        f = torch.sin(3 * X[:, 0]) + torch.cos(2 * X[:, 0])
    else:
        X = _normal(g, n, d) * _uniform(g, 0.5, 2.0, d)
        ls, var, sd = _log_uniform(g, 1.0, 4.0, nls) * math.sqrt(d / 16), 1.2, 0.1
        # a draw from the prior through random Fourier features
        F = 512
        W = _normal(g, d, F) / ls.reshape(-1, 1)
        w = _normal(g, 2 * F)
        f = torch.empty(n, dtype=torch.float64, device="cuda")
        for i in range(0, n, 16384):
            p = X[i:i + 16384] @ W
            f[i:i + 16384] = (torch.cos(p) @ w[:F] + torch.sin(p) @ w[F:]) * math.sqrt(var / F)
    y = f + sd * _normal(g, n)
    out = dict(X=X, y=y, ls=ls if case["ard"] else ls[0], var=var, sd=sd)
    if kind == "predict":
        t = case["t"]
        if d == 1:
            out["T"] = torch.linspace(-3.5, 3.5, t, dtype=torch.float64, device="cuda")[:, None]
            fT = torch.sin(3 * out["T"][:, 0]) + torch.cos(2 * out["T"][:, 0])
        else:
            out["T"] = _normal(g, t, d) * X.std(0)
            fT = torch.zeros(t, dtype=torch.float64, device="cuda")
        out["yT"] = fT + sd * _normal(g, t)
    if kind == "cov":
        out["Z"] = _normal(g, max(1, case["m"]), d)
    return out


def _kernel(case, a):
    cls = {"rbf": gpx.kernels.RBF, "matern12": gpx.kernels.Matern12,
           "matern32": gpx.kernels.Matern32, "matern52": gpx.kernels.Matern52}[case["kernel"]]
    return cls(lengthscale=a["ls"], variance=a["var"])


def _posterior(case, a):
    prior = gpx.gps.Prior(kernel=_kernel(case, a), mean_function=gpx.mean_functions.Zero(),
                          jitter=JITTER)
    lik = gpx.likelihoods.Gaussian(num_datapoints=a["X"].shape[0], obs_stddev=a["sd"])
    return prior * lik


def prepare(case, seed):
    a = _inputs(case, seed)
    kind = case["kind"]
    if kind == "batched":
        Xs = [x.numpy() for x in a["X"].split(a["sizes"])]
        ys = [y.numpy() for y in a["y"].split(a["sizes"])]
        model = BatchedConjugateMLL(Xs, ys, kernel="rbf", lengthscale=a["ls"],
                                    variance=a["var"], obs_stddev=a["sd"], jitter=JITTER)
        return dict(case=case, model=model)
    if kind == "cov":
        return dict(case=case, kernel=_kernel(case, a), X=a["X"], Z=a["Z"])
    if kind == "fit":
        return dict(case=case, a=a, data=gpx.Dataset(X=a["X"], y=a["y"][:, None]))
    post = _posterior(case, a)
    s = dict(case=case, post=post, data=gpx.Dataset(X=a["X"], y=a["y"][:, None]))
    if kind == "elbo":
        s["q"] = gpx.variational_families.CollapsedVariationalGaussian(
            posterior=post, inducing_inputs=a["Z"], jitter=JITTER)
    if kind == "predict":
        s.update(T=a["T"], yT=a["yT"])
    return s


# ---- one pass -----------------------------------------------------------------

def _theta(post):
    k = post.prior.kernel
    return [k.lengthscale.value, k.variance.value, post.likelihood.obs_stddev.value]


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind in ("mll", "loocv"):
        f = gpx.objectives.conjugate_mll if kind == "mll" else gpx.objectives.conjugate_loocv
        v = f(s["post"], s["data"], precision=case["precision"])
        return [v.detach(), *torch.autograd.grad(v, _theta(s["post"]))]
    if kind == "elbo":
        v = gpx.objectives.collapsed_elbo(s["q"], s["data"], precision=case["precision"])
        wrt = _theta(s["post"]) + [s["q"].inducing_inputs.value]
        return [v.detach(), *torch.autograd.grad(v, wrt)]
    if kind == "predict":
        dist = s["post"].predict(s["T"], s["data"], full_covariance=case["full"])
        if not case["full"]:
            return [dist.mean, dist.variance]
        obs = s["post"].likelihood(dist)
        return [dist.mean, dist.covariance(), obs.log_prob(s["yT"])]
    if kind == "batched":
        m = s["model"]
        v = m.mll()
        return [v.detach(), *torch.autograd.grad(v.sum(), [m.lengthscale.value, m.variance.value,
                                                           m.obs_stddev.value])]
    if kind == "cov":
        k = s["kernel"]
        return k.gram(s["X"]) if case["m"] == 0 else k.cross_covariance(s["X"], s["Z"])
    post = _posterior(case, s["a"])   # a training run starts from its initial values
    post, history = gpx.fit(
        model=post, objective=lambda p, dat: -gpx.objectives.conjugate_mll(p, dat),
        train_data=s["data"], num_iters=case["steps"], learning_rate=0.02,
        capture_graph=case["graph"])
    return [history, *[p.detach() for p in _theta(post)]]


# ---- what one pass cannot do without --------------------------------------------

def work(case):
    kind, d = case["kind"], case["d"]
    if kind == "batched":
        # E[n^3] and E[n] of sizes uniform on nmin .. nmax
        lo, hi, B = case["nmin"], case["nmax"], case["count"]
        w = range(lo, hi + 1)
        return {"bytes": 8.0 * B * (sum(w) / len(w) * (d + 1) + 2 * d + 10),
                "flops": B * sum(float(n) ** 3 for n in w) / len(w)}
    n = float(case["n"])
    read = 8.0 * n * (d + 1)
    if kind == "mll":      # factor, inverse factor, Sigma^-1: n^3 / 3 each
        return {"bytes": read, "flops": n ** 3}
    if kind == "loocv":    # and the product Sigma^-1 diag(c) Sigma^-1 over lower tiles
        return {"bytes": read, "flops": 2 * n ** 3}
    if kind == "fit":
        return {"bytes": read, "flops": case["steps"] * n ** 3}
    if kind == "predict":
        t = float(case["t"])
        if case["full"]:   # factor, L^-1 Kxt, its Gram, the factor of the T x T covariance
            return {"bytes": read + 8 * t * (d + 1) + 8 * t * t,
                    "flops": n ** 3 / 3 + n * n * t + n * t * t + t ** 3 / 3}
        return {"bytes": read + 8 * t * (d + 2), "flops": n ** 3 / 3 + n * n * t}
    if kind == "elbo":     # P (lower half), G_P Kzx, the M x M algebra
        m = float(case["m"])
        return {"bytes": read + 16 * m * d, "flops": 3 * n * m * m + 6 * m ** 3}
    m = float(case["m"]) or n
    return {"bytes": 8 * (n + m) * d + 8 * n * m, "flops": n * m * (3.0 * d + 20)}


# ---- 64-bit values from plain torch ----------------------------------------------

def _k_and_factor(kernel, d2):
    """k(rho) and F(rho), dk/dl_d = var F u_d / l_d with u_d = (x_d - z_d)^2 / l_d^2."""
    if kernel == "rbf":
        k = torch.exp(-0.5 * d2)
        return k, k
    r = torch.sqrt(torch.clamp(d2, min=1e-36))
    if kernel == "matern12":
        e = torch.exp(-r)
        return e, torch.where(d2 > 1e-36, e / r, torch.zeros_like(e))
    if kernel == "matern32":
        e = torch.exp(-math.sqrt(3.0) * r)
        return (1 + math.sqrt(3.0) * r) * e, 3 * e
    e = torch.exp(-math.sqrt(5.0) * r)
    return ((1 + math.sqrt(5.0) * r + 5.0 / 3.0 * r * r) * e,
            5.0 / 3.0 * (1 + math.sqrt(5.0) * r) * e)


def _d2(A, B):
    """Squared distances by direct differences (leading batch dimensions allowed)."""
    out = torch.zeros(*A.shape[:-1], B.shape[-2], dtype=torch.float64, device=A.device)
    for q in range(A.shape[-1]):
        out += (A[..., :, None, q] - B[..., None, :, q]) ** 2
    return out


def _chol_inverse(S):
    """log|S| and S^-1 (leading batch dimensions allowed)."""
    L = torch.linalg.cholesky(S)
    eye = torch.eye(S.shape[-1], dtype=S.dtype, device=S.device).expand_as(S)
    X = torch.linalg.solve_triangular(L, eye.contiguous(), upper=False)
    return 2 * torch.log(torch.diagonal(L, dim1=-2, dim2=-1)).sum(-1), X.mT.contiguous() @ X


def _exact_grads(W, k, F, U, ls, var, sd, ard):
    """1/2 tr(W dSigma) for the lengthscales, the variance and the noise."""
    G = W * F
    g = torch.stack([(G * (U[..., :, None, q] - U[..., None, :, q]) ** 2).sum((-2, -1))
                     for q in range(U.shape[-1])], -1)
    if not ard:
        g = g.sum(-1)
    v = var[..., None] if ard and torch.is_tensor(var) and var.ndim else var
    tr = torch.diagonal(W, dim1=-2, dim2=-1).sum(-1)
    return [0.5 * v * g / ls, 0.5 * (W * k).sum((-2, -1)), sd * tr]


def _exact_objective(case, X, y, ls, var, sd, loo):
    n = X.shape[0]
    U = X / ls
    k, F = _k_and_factor(case["kernel"], _d2(U, U))
    S = var * k
    S.diagonal().add_(JITTER + sd * sd)
    logdet, Si = _chol_inverse(S)
    a = Si @ y
    if not loo:
        v = -0.5 * (n * math.log(2 * math.pi) + logdet + y @ a)
        W = torch.outer(a, a) - Si
    else:
        dg = torch.diagonal(Si)
        v = (-0.5 * math.log(2 * math.pi) + 0.5 * torch.log(dg) - 0.5 * a * a / dg).sum()
        w = Si @ (a / dg)
        c2 = 1 / dg + (a / dg) ** 2
        W = torch.outer(a, w) + torch.outer(w, a) - (Si * c2) @ Si
    return [v, *_exact_grads(W, k, F, U, ls, var, sd, case["ard"])]


def _exact_fit(case, a):
    """Adam on the softplus-unconstrained lengthscale(s), variance and noise."""
    dev = a["X"].device
    vals = [torch.as_tensor(v, dtype=torch.float64).to(dev) for v in (a["ls"], a["var"], a["sd"])]
    raw = [v + torch.log(-torch.expm1(-v)) for v in vals]
    mom = [[torch.zeros_like(r), torch.zeros_like(r)] for r in raw]
    hist = []
    for t in range(1, case["steps"] + 1):
        vals = [torch.nn.functional.softplus(r, threshold=50.0) for r in raw]
        o = _exact_objective(case, a["X"], a["y"], *vals, loo=False)
        hist.append(-o[0])
        for j in range(3):
            g = -o[1 + j].reshape(raw[j].shape) * torch.sigmoid(raw[j])
            mom[j][0] = 0.9 * mom[j][0] + 0.1 * g
            mom[j][1] = 0.999 * mom[j][1] + 0.001 * g * g
            mh, vh = mom[j][0] / (1 - 0.9 ** t), mom[j][1] / (1 - 0.999 ** t)
            raw[j] = raw[j] - 0.02 * mh / (torch.sqrt(vh) + 1e-8)
    vals = [torch.nn.functional.softplus(r, threshold=50.0) for r in raw]
    return [torch.stack(hist), *vals]


def _exact_elbo(case, a):
    X, y, Z, ls, var, s = a["X"], a["y"], a["Z"], a["ls"], a["var"], a["sd"] ** 2
    n, m = X.shape[0], Z.shape[0]
    UX, UZ = X / ls, Z / ls
    P = torch.zeros(m, m, dtype=torch.float64, device=X.device)
    b = torch.zeros(m, dtype=torch.float64, device=X.device)
    step = 32768
    for i in range(0, n, step):
        K = var * _k_and_factor(case["kernel"], _d2(UZ, UX[i:i + step]))[0]
        P += K @ K.mT.contiguous()
        b += K @ y[i:i + step]
    kz, Fz = _k_and_factor(case["kernel"], _d2(UZ, UZ))
    Kzz = var * kz
    Kzz.diagonal().add_(JITTER)
    ldK, Ki = _chol_inverse(Kzz)
    ldC, Ci = _chol_inverse(Kzz + P / s)
    c = Ci @ b
    rr = y @ y
    trKP = (Ki * P).sum()
    v = 0.5 * (-n * math.log(2 * math.pi * s) - (ldC - ldK) - (rr - b @ c / s) / s
               - n * var / s + trKP / s)
    cc = torch.outer(c, c)
    GP = (Ki - Ci) / s - cc / s ** 3
    GK = Ki - Ci - cc / s ** 2 - Ki @ P @ Ki / s
    gl = torch.zeros_like(ls)
    gv = 0.5 * (GK * kz).sum() - 0.5 * n / s
    gZ = torch.zeros_like(Z)

    def add(W, F, A, scale):
        G = W * F
        for q in range(A.shape[1]):
            df = UZ[:, None, q] - A[None, :, q]
            Gd = G * df
            gl[q] += scale * (Gd * df).sum()
            gZ[:, q] += Gd.sum(1)

    add(GK, Fz, UZ, 0.5)
    for i in range(0, n, step):
        k, F = _k_and_factor(case["kernel"], _d2(UZ, UX[i:i + step]))
        W = GP @ (var * k) + torch.outer(c / s ** 2, y[i:i + step])
        gv = gv + (W * k).sum()
        add(W, F, UX[i:i + step], 1.0)
    gs = (-n / s + (Ci * P).sum() / s ** 2 + rr / s ** 2 + c @ P @ c / s ** 4
          - 2 * b @ c / s ** 3 + n * var / s ** 2 - trKP / s ** 2)
    return [v, var * gl / ls, gv, gs * a["sd"], -var * gZ / ls]


def _exact_batched(case, a):
    sizes = a["sizes"]
    off = [0]
    for n in sizes:
        off.append(off[-1] + n)
    B, d = len(sizes), case["d"]
    v = torch.empty(B, dtype=torch.float64, device="cuda")
    gl = torch.empty(B, d, dtype=torch.float64, device="cuda")
    gv, gs = torch.empty_like(v), torch.empty_like(v)
    X, y = a["X"].cuda(), a["y"].cuda()
    ls, var, sd = a["ls"].cuda(), a["var"].cuda(), a["sd"].cuda()
    by_size = sorted(range(B), key=lambda p: sizes[p])
    for i in range(0, B, 64):
        idx = by_size[i:i + 64]
        N = sizes[idx[-1]]
        U = torch.zeros(len(idx), N, d, dtype=torch.float64, device="cuda")
        Y = torch.zeros(len(idx), N, dtype=torch.float64, device="cuda")
        on = torch.zeros(len(idx), N, dtype=torch.float64, device="cuda")
        for j, p in enumerate(idx):
            U[j, :sizes[p]] = X[off[p]:off[p + 1]] / ls[p]
            Y[j, :sizes[p]] = y[off[p]:off[p + 1]]
            on[j, :sizes[p]] = 1
        at = torch.tensor(idx, device="cuda")
        k, F = _k_and_factor("rbf", _d2(U, U))
        both = on[:, :, None] * on[:, None, :]
        k, F = k * both, F * both
        S = var[at, None, None] * k
        torch.diagonal(S, dim1=-2, dim2=-1).add_(
            on * (JITTER + sd[at, None] ** 2) + (1 - on))
        logdet, Si = _chol_inverse(S)
        al = (Si @ Y[:, :, None])[..., 0]
        W = (al[:, :, None] * al[:, None, :] - Si) * both
        v[at] = -0.5 * (on.sum(1) * math.log(2 * math.pi) + logdet + (Y * al).sum(1))
        gl[at], gv[at], gs[at] = _exact_grads(W, k, F, U, ls[at], var[at], sd[at], True)
    return [v, gl, gv, gs]


def exact(case, seed):
    kind = case["kind"]
    n = case.get("n", 0)
    # beyond these sizes the plain evaluation takes too long or too much memory
    if kind in ("mll", "loocv", "predict") and n > 10000:
        return None
    if kind == "elbo" and float(n) * case["m"] > 3e8:
        return None
    if kind == "batched" and case["count"] > 600:
        return None
    a = _inputs(case, seed)
    if kind == "batched":
        return _exact_batched(case, a)
    if kind == "elbo":
        return _exact_elbo(case, a)
    if kind == "fit":
        return _exact_fit(case, a)
    if kind in ("mll", "loocv"):
        return _exact_objective(case, a["X"], a["y"], a["ls"], a["var"], a["sd"],
                                kind == "loocv")
    U = a["X"] / a["ls"]
    if kind == "cov":
        V = U if case["m"] == 0 else a["Z"] / a["ls"]
        return a["var"] * _k_and_factor(case["kernel"], _d2(U, V))[0]
    S = a["var"] * _k_and_factor(case["kernel"], _d2(U, U))[0]
    S.diagonal().add_(JITTER + a["sd"] ** 2)
    L = torch.linalg.cholesky(S)
    del S
    al = torch.cholesky_solve(a["y"][:, None], L)[:, 0]
    T = a["T"] / a["ls"]
    if not case["full"]:
        mean, var = [], []
        for i in range(0, case["t"], 8192):
            K = a["var"] * _k_and_factor(case["kernel"], _d2(U, T[i:i + 8192]))[0]
            mean.append(K.mT @ al)
            A = torch.linalg.solve_triangular(L, K, upper=False)
            var.append(a["var"] + JITTER - (A * A).sum(0))
        return [torch.cat(mean), torch.cat(var)]
    K = a["var"] * _k_and_factor(case["kernel"], _d2(U, T))[0]
    A = torch.linalg.solve_triangular(L, K, upper=False)
    cov = a["var"] * _k_and_factor(case["kernel"], _d2(T, T))[0]
    cov.diagonal().add_(JITTER)
    cov = cov - A.mT.contiguous() @ A
    mean = K.mT @ al
    obs = cov.clone()
    obs.diagonal().add_(a["sd"] ** 2)
    Lo = torch.linalg.cholesky(obs)
    z = torch.linalg.solve_triangular(Lo, (a["yT"] - mean)[:, None], upper=False)[:, 0]
    lp = -0.5 * (case["t"] * math.log(2 * math.pi)
                 + 2 * torch.log(torch.diagonal(Lo)).sum() + z @ z)
    return [mean, cov, lp]
