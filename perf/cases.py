"""Performance cases of the exact-GP path on one GPU.

A case is one call (or the few calls that belong together) that a program
using this framework makes, through its public entry points:

  gp          gprat_amd.GP.predict_with_uncertainty: the drop-in API, fit and
              prediction in one call on host lists
  once        capi.Context.predict(variance=True): the same call on arrays
  gradient    capi.Context.loss_gradient: the device half of one Adam step
  cholesky    capi.Context.cholesky: the factor as the reference's tiles
  resident    capi.Context.fit, then Model.predict and Model.loss: a resident
              model, FP64 or mixed precision (with the refined variance)
  predict     Model.predict on a model fitted before (serving)
  posterior   Model.predict_full_cov on a model fitted before
  batch       capi.Batch over many GPs of uneven size, its losses, and
              predictions from a few of them

Inputs are the mass-spring-damper series of the benchmark configurations
(gprat_amd.datagen) from the case's seed; they are host arrays, as every
program of the reference passes them.
"""
import math

import numpy as np
import torch

import gprat_amd
from gprat_amd import capi, datagen

# the hyperparameters of the benchmark configurations: lengthscale 1,
# vertical lengthscale 1, and this noise variance
NOISE, NOISE_LONG_WINDOW = 0.1, 0.05

_CONTEXT = None


def _context():
    """The process's one library context (streams and device pool)."""
    global _CONTEXT
    if _CONTEXT is None:
        _CONTEXT = capi.Context(0, 1)
    return _CONTEXT


def listed():
    return [
        # the reference's own test data set size (4 tiles of 32, 8
        # regressors): the smallest call, bound by launches and latency
        {"name": "gp_n128_m128", "family": "gp", "tiles": 4, "tile": 32, "m": 128, "n_reg": 8, "noise": NOISE},
        # the plain configuration (4 tiles of 256): an ordinary small fit and prediction
        {"name": "once_n1024_m1024", "family": "once", "tiles": 4, "tile": 256, "m": 1024, "n_reg": 8, "noise": NOISE},
        # one optimisation step of the plain configuration: loss and gradient
        {"name": "gradient_n1024", "family": "gradient", "tiles": 4, "tile": 256, "n_reg": 8, "noise": NOISE},
        # the factor itself, returned to the host tile by tile
        {"name": "cholesky_n2048", "family": "cholesky", "tiles": 8, "tile": 256, "n_reg": 8, "noise": NOISE},
        # sizes that fit no tile: a resident FP64 model and its first prediction
        {"name": "resident_n5003_m777", "family": "resident", "n": 5003, "m": 777, "n_reg": 7, "noise": NOISE, "mixed": False},
        # the large FP64 configuration: fit and prediction in one call
        {"name": "once_n16384_m4096", "family": "once", "tiles": 32, "tile": 512, "m": 4096, "n_reg": 8, "noise": NOISE},
        # one optimisation step at that size
        {"name": "gradient_n16384", "family": "gradient", "tiles": 32, "tile": 512, "n_reg": 8, "noise": NOISE},
        # the mixed-precision configuration: fit, alpha and variance refined
        {"name": "mixed_n32768_m8192", "family": "resident", "n": 32768, "m": 8192, "n_reg": 16, "noise": NOISE_LONG_WINDOW,
         "mixed": True},
        # serving: a handful of points from a resident FP64 model
        {"name": "predict_n8192_m16", "family": "predict", "n": 8192, "m": 16, "n_reg": 8, "noise": NOISE, "mixed": False},
        # serving: an ordinary request against a mixed-precision model
        {"name": "predict_mixed_n12000_m1500", "family": "predict", "n": 12000, "m": 1500, "n_reg": 8, "noise": NOISE, "mixed": True},
        # the whole posterior covariance (sampling from the posterior)
        {"name": "posterior_n3000_m501", "family": "posterior", "n": 3000, "m": 501, "n_reg": 8, "noise": NOISE, "mixed": False},
        # many small GPs of uneven size in one call, the batched
        # configuration's distributions of size, window and hyperparameters
        {"name": "batch_512", "family": "batch", "count": 512, "n_min": 64, "n_max": 2048},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["gp", "once", "once", "gradient", "gradient", "cholesky", "resident", "resident", "predict", "predict",
                         "posterior", "batch"])
    n_reg = rng.choice([4, 7, 8, 8, 16, 20])
    noise = rng.choice([NOISE, NOISE_LONG_WINDOW])
    case = {"family": family, "n_reg": n_reg, "noise": noise}
    if family in ("gp", "once", "gradient", "cholesky"):
        top = {"gp": 1024, "once": 16384, "gradient": 16384, "cholesky": 4096}[family]
        n = _log_int(rng, 128, top)
        tiles = rng.choice([1, 3, 4, 8, 16])
        case.update(tiles=tiles, tile=max(8, n // tiles))
        if family in ("gp", "once"):
            case["m"] = _log_int(rng, 1, 1024 if family == "gp" else 4096)
    elif family == "resident":
        mixed = rng.random() < 0.5
        case.update(n=_log_int(rng, 2049 if mixed else 128, 16384), m=_log_int(rng, 1, 4096), mixed=mixed)
    elif family == "predict":
        mixed = rng.random() < 0.5
        case.update(n=_log_int(rng, 2049 if mixed else 256, 20000), m=_log_int(rng, 1, 4096), mixed=mixed)
    elif family == "posterior":
        case.update(n=_log_int(rng, 128, 8192), m=_log_int(rng, 16, 1024), mixed=False)
    else:
        case = {"family": "batch", "count": _log_int(rng, 16, 512), "n_min": 64, "n_max": rng.choice([256, 1024, 2048])}
    return case


def _size(case):
    return case["n"] if "n" in case else case["tiles"] * case["tile"]


def _theta(case):
    return [1.0, 1.0, case["noise"]]


def _problem(case, seed):
    return datagen.gp_problem(_size(case), case.get("m", 1), case["n_reg"], 2 * seed + 1000, 2 * seed + 1001)


def _batch_problems(case, seed):
    """(train_in, train_out, n, n_reg, theta) per GP: n log-uniform, n_reg
    from {4, 8, 16}, hyperparameters log-uniform; all series advance together."""
    g = np.random.default_rng(seed)
    count = case["count"]
    n = np.exp(g.uniform(math.log(case["n_min"]), math.log(case["n_max"]), count)).astype(int)
    n_reg = g.choice([4, 8, 16], count)

    def log_uniform(lo, hi):
        return np.exp(g.uniform(math.log(lo), math.log(hi), count))

    theta = np.stack([log_uniform(0.3, 3.0), log_uniform(0.5, 2.0), log_uniform(0.01, 0.3)], axis=1)
    longest = int(n.max())
    u = g.uniform(-1.0, 1.0, (longest, count))
    y = np.empty_like(u)
    x, v = np.zeros(count), np.zeros(count)
    for t in range(longest):
        v = v + 0.05 * (u[t] - x - 0.5 * v)
        x = x + 0.05 * v
        y[t] = x
    y += 0.01 * g.standard_normal(y.shape)
    return [(datagen.padded_input(u[:n[i], i], int(n_reg[i])), np.ascontiguousarray(y[:n[i], i]), int(n[i]), int(n_reg[i]),
             theta[i].tolist()) for i in range(count)]


# points of each of the first GPs that a batch's program predicts at
BATCH_PREDICTED, BATCH_POINTS = 4, 64


def _batch_points(seed, n_reg):
    return datagen.padded_input(np.random.default_rng([seed, 1]).uniform(-1.0, 1.0, BATCH_POINTS), n_reg)


def prepare(case, seed):
    family = case["family"]
    state = {"case": case, "ctx": _context()}
    if family == "batch":
        state["problems"] = _batch_problems(case, seed)
        state["points"] = [_batch_points(seed, p[3]) for p in state["problems"][:BATCH_PREDICTED]]
        return state
    x, y, z = _problem(case, seed)
    state.update(x=x, y=y, z=z, theta=_theta(case))
    if family == "gp":
        # a GP object in use: its target's context exists (the loss was looked at)
        state["z"] = z.tolist()
        state["gp"] = gprat_amd.GP(x.tolist(), y.tolist(), case["tiles"], case["tile"], case["n_reg"], _theta(case), [True, True, True])
        state["gp"].compute_loss()
    elif family in ("predict", "posterior"):
        state["model"] = state["ctx"].fit(x, y, case["n"], case["n_reg"], _theta(case), _precision(case))
    return state


def _precision(case):
    return capi.PRECISION_MIXED if case["mixed"] else capi.PRECISION_FP64


def run(state):
    case, ctx = state["case"], state["ctx"]
    family = case["family"]
    if family == "gp":
        mean, var = state["gp"].predict_with_uncertainty(state["z"], 1, case["m"])
        return np.array(mean), np.array(var)
    if family == "once":
        return ctx.predict(state["x"], state["y"], state["z"], state["theta"], case["tiles"], case["tile"], 1, case["m"], case["n_reg"],
                           variance=True)
    if family == "gradient":
        return ctx.loss_gradient(state["x"], state["y"], state["theta"], case["tiles"], case["tile"], case["n_reg"])
    if family == "cholesky":
        return ctx.cholesky(state["x"], state["theta"], case["tiles"], case["tile"], case["n_reg"])
    if family == "resident":
        model = ctx.fit(state["x"], state["y"], case["n"], case["n_reg"], state["theta"], _precision(case))
        mean, var = model.predict(state["z"], case["m"])
        loss = model.loss()
        model.release()
        return mean, var, loss
    if family == "predict":
        return state["model"].predict(state["z"], case["m"])
    if family == "posterior":
        return state["model"].predict_full_cov(state["z"], case["m"])
    batch = capi.Batch(ctx, state["problems"])
    out = [batch.losses()]
    for i, z in enumerate(state["points"]):
        out.extend(batch.predict(i, z, BATCH_POINTS))
    batch.release()
    return out


def _entries(n, m, n_reg):
    """Flops of n * m covariance entries: the window's distance and an exponential."""
    return n * m * (3.0 * n_reg + 20.0)


def _fit_work(n, n_reg):
    return n ** 3 / 3.0 + 2.0 * n ** 2 + _entries(n, n / 2, n_reg)


def work(case):
    """Bytes: series, targets and a resident factor read once, results
    written once. Flops: entries of K and K*, the factorisation (n^3 / 3), a
    triangular solve per test point, K^-1 for the gradient (2 n^3 / 3)."""
    family = case["family"]
    if family == "batch":
        problems = _batch_sizes(case)
        flops = sum(_fit_work(n, r) for n, r in problems)
        flops += sum(n ** 2 * BATCH_POINTS + _entries(n, BATCH_POINTS, r) for n, r in problems[:BATCH_PREDICTED])
        return {"bytes": 8.0 * (sum(2 * n + r for n, r in problems) + len(problems) + 3 * BATCH_PREDICTED * BATCH_POINTS), "flops": flops}
    n, m, r = _size(case), case.get("m", 0), case["n_reg"]
    flops, values = 0.0, 2.0 * n + r
    if family in ("gp", "once", "resident"):
        flops = _fit_work(n, r) + n ** 2 * m + _entries(n, m, r) + 2.0 * n * m
        values += 3.0 * m
        if family == "resident" and case["mixed"]:
            # the refined variance: a backward solve and an FP64 residual product more
            flops += 2.0 * n ** 2 * m
    elif family == "gradient":
        flops = n ** 3 + 2.0 * n ** 2 + _entries(n, n, r)
        values += 4.0
    elif family == "cholesky":
        flops = n ** 3 / 3.0 + _entries(n, n / 2, r)
        values += case["tiles"] * (case["tiles"] + 1) / 2 * case["tile"] ** 2
    elif family == "predict":
        flops = n ** 2 * m * (3.0 if case["mixed"] else 1.0) + _entries(n, m, r) + 2.0 * n * m
        values += n ** 2 / 2.0 + 3.0 * m
    else:
        flops = n ** 2 * m + float(n) * m * m + _entries(n, m, r) + _entries(m, m / 2, r)
        values += n ** 2 / 2.0 + 2.0 * m + m * m
    return {"bytes": 8.0 * values, "flops": flops}


def _batch_sizes(case, seed=0):
    g = np.random.default_rng(seed)
    n = np.exp(g.uniform(math.log(case["n_min"]), math.log(case["n_max"]), case["count"])).astype(int)
    return list(zip(n.tolist(), g.choice([4, 8, 16], case["count"]).tolist()))


# ---- the same results in plain torch, 64 bits --------------------------------

_CHUNK = 4096  # rows of a covariance block formed at a time


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _sqdist(a, na, b, nb, n_reg):
    """Squared distances of the windows a[i .. i + n_reg) and b[j .. j + n_reg)."""
    d = torch.zeros(na, nb, dtype=torch.float64, device=a.device)
    for i in range(0, na, _CHUNK):
        e = min(na, i + _CHUNK)
        for k in range(n_reg):
            d[i:e] += (a[i + k:e + k, None] - b[None, k:nb + k]).square_()
    return d


def _kernel(a, na, b, nb, n_reg, theta):
    d = _sqdist(a, na, b, nb, n_reg)
    return d.mul_(-0.5 / theta[0] ** 2).exp_().mul_(theta[1])


def _forward(L, B):
    """L^-1 B by blocks of rows (B is overwritten)."""
    n = L.shape[0]
    for i in range(0, n, _CHUNK):
        e = min(n, i + _CHUNK)
        B[i:e] = torch.linalg.solve_triangular(L[i:e, i:e].contiguous(), B[i:e].contiguous(), upper=False)
        if e < n:
            B[e:] -= L[e:, i:e] @ B[i:e]
    return B


def _exact_fit(x, y, n, n_reg, theta):
    dev = _device()
    x, y = (torch.as_tensor(np.asarray(v), dtype=torch.float64, device=dev) for v in (x, y))
    K = _kernel(x, n, x, n, n_reg, theta)
    K.diagonal().add_(theta[2])
    L = torch.linalg.cholesky(K)
    del K
    beta = _forward(L, y[:n, None].clone())
    return x, y[:n], L, beta


def _exact_loss(L, beta, n):
    return float(0.5 * (beta.square().sum() + 2.0 * L.diagonal().log().sum() + n * math.log(2.0 * math.pi)) / n)


def _exact_predict(x, L, beta, z, n, m, n_reg, theta):
    z = torch.as_tensor(np.asarray(z), dtype=torch.float64, device=x.device)
    V = _forward(L, _kernel(x, n, z, m, n_reg, theta))
    return z, V, (V * beta).sum(0)


def exact(case, seed):
    family = case["family"]
    if family == "batch":
        problems = _batch_problems(case, seed)
        losses, predictions = [], []
        for i, (x, y, n, r, theta) in enumerate(problems):
            xt, _, L, beta = _exact_fit(x, y, n, r, theta)
            losses.append(_exact_loss(L, beta, n))
            if i < BATCH_PREDICTED:
                _, V, mean = _exact_predict(xt, L, beta, _batch_points(seed, r), n, BATCH_POINTS, r, theta)
                predictions += [mean.cpu().numpy(), (theta[1] - V.square().sum(0)).cpu().numpy()]
        return [np.array(losses)] + predictions
    n, r, theta = _size(case), case["n_reg"], _theta(case)
    x, y, z = _problem(case, seed)
    if family == "cholesky":
        xt = torch.as_tensor(x, dtype=torch.float64, device=_device())
        K = _kernel(xt, n, xt, n, r, theta)
        K.diagonal().add_(theta[2])
        L = torch.linalg.cholesky(K)
        b, out = case["tile"], []
        for i in range(case["tiles"]):
            for j in range(i + 1):
                t = L[i * b:(i + 1) * b, j * b:(j + 1) * b]
                out.append(t if j < i else t.tril() + K[i * b:(i + 1) * b, j * b:(j + 1) * b].triu(1))
        return torch.stack(out).cpu().numpy()
    xt, yt, L, beta = _exact_fit(x, y, n, r, theta)
    if family == "gradient":
        alpha = torch.linalg.solve_triangular(L.T, beta, upper=True)
        Kinv = torch.cholesky_inverse(L)
        loss = _exact_loss(L, beta, n)
        del L
        # dK/du in softplus space: u = log(exp(theta) - 1), the noise shifted by 1e-6
        slope = [1.0 - math.exp(-theta[0]), 1.0 - math.exp(-theta[1]), 1.0 - math.exp(1e-6 - theta[2])]
        d = _sqdist(xt, n, xt, n, r)
        e = (d * (-0.5 / theta[0] ** 2)).exp_()
        trace_noise = float(Kinv.diagonal().sum())
        Kinv.sub_(alpha @ alpha.T)
        g_v = float((Kinv * e).sum()) * slope[1]
        g_l = float(Kinv.mul_(e.mul_(d)).sum()) * theta[1] / theta[0] ** 3 * slope[0]
        g_n = (trace_noise - float(alpha.square().sum())) * slope[2]
        return loss, np.array([g_l, g_v, g_n]) * 0.5 / n
    m = case["m"]
    zt, V, mean = _exact_predict(xt, L, beta, z, n, m, r, theta)
    if family == "posterior":
        cov = _kernel(zt, m, zt, m, r, theta) - V.T @ V
        return mean.cpu().numpy(), cov.cpu().numpy()
    var = theta[1] - V.square().sum(0)
    out = (mean.cpu().numpy(), var.cpu().numpy())
    return out + (_exact_loss(L, beta, n),) if family == "resident" else out
