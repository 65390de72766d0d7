"""The workloads that this package is timed on, through its public entry points.

listed() gives the fixed cases, draw() further ones of the same ranges, prepare() what a program holds before
the call (inputs made from a seed, resident models), run() one pass, work() the bytes and operations a pass
cannot do without, and exact() the pass in 64 bits with plain torch.

Rows are synthetic systematics as in decontamination_amd.synth: lognormal and Gaussian columns and the sine and
cosine of a random colatitude, each standardised. Densities are galaxy counts over coverage, zeros among them.
Maps that are searched are trained on a few thousand of such rows by a plain torch batch SOM.
"""
import ctypes
import math

import numpy as np
import torch

import decontamination_amd as dam
from decontamination_amd import _lib, synth
from decontamination_amd.runtime import Accumulator, DeviceArray, Model, get_context
from decontamination_amd.serving import SOMServer, pinned_empty

ROWS_64 = 12_582_912    # all pixels of a HEALPix map with nside 1024
ROWS_100 = 50_331_648   # nside 2048


def listed():
    return [
        # One object list against a trained map, from host memory: the smallest request; launches and latency.
        _case("winners_small", "winners_host", n=1000, m=32, cols=32, dim=16),
        # A catalogue resident on the device, with a dimension and a length that fit no tile.
        _case("winners_ragged", "winners", n=1_000_003, m=64, cols=64, dim=13),
        # Weighted activation map of a nside 256 footprint over many systematics.
        _case("activation_wide", "activation", n=786_432, m=32, cols=32, dim=40, rho=True),
        # Quantisation and topographic errors of a nside 512 footprint on a rectangular square-grid map.
        _case("errors_square", "errors", n=3_145_728, m=90, cols=70, dim=20, topology="square", arithmetic="fp64"),
        # A whole small training from host memory: 10x10 square map, 8 features, 10 epochs.
        _case("train_small", "train_host", n=100_000, m=10, cols=10, dim=8, topology="square", epochs=10),
        # The headline training: the first epochs of a 20-epoch schedule on a nside 1024 footprint.
        _case("epochs_64", "epochs", n=ROWS_64, m=64, cols=64, dim=16, epochs=3, arithmetic="fp64"),
        # The large map: the first two epochs on a nside 2048 footprint, weighted by the density.
        _case("epochs_100", "epochs", n=ROWS_100, m=100, cols=100, dim=32, epochs=2, rho=True),
        # Training by number of vectors, where sigma shrinks with every sample.
        _case("vectors", "vectors", n=100_000, m=32, cols=32, dim=16),
        # A float64 SOM: two weighted epochs.
        _case("epochs_f64", "epochs", n=1_048_576, m=64, cols=64, dim=16, epochs=2, rho=True, f64=True),
        # Covariance of the PCA initialisation, weighted by the density.
        _case("covariance", "covariance", n=ROWS_64, m=1, cols=1, dim=16, rho=True),
        # Galaxy number density maps of the footprint from its winners.
        _case("gndm", "gndm", n=ROWS_64, m=64, cols=64, dim=16, rho=True),
        # Requests of uneven sizes to two resident maps, sent together, as a serving process meets them.
        _case("serve_mixed", "serve", n=250_000, m=64, cols=64, dim=32, requests=12),
    ]


def draw(rng):
    kind = rng.choice(["winners_host", "winners", "winners", "activation", "errors", "train_host", "epochs", "epochs",
                       "epochs", "vectors", "covariance", "gndm", "serve"])
    dim = rng.choice([8, 16, 16, 32, rng.randint(5, 32), rng.randint(33, 64)])
    m, cols = rng.randint(16, 100), rng.randint(16, 100)
    if rng.random() < 0.4:
        m = cols = rng.choice([32, 64, 100])
    opts = {"dim": dim, "m": m, "cols": cols, "topology": rng.choice(["hexagonal", "hexagonal", "square"]),
            "arithmetic": rng.choice(["ref32", "fp64"]), "rho": rng.random() < 0.5}
    if kind == "winners_host":
        return _case(None, kind, n=_log(rng, 500, 300_000), **opts)
    if kind == "train_host":
        m, cols = rng.randint(8, 24), rng.randint(8, 24)
        return _case(None, kind, n=_log(rng, 20_000, 400_000), epochs=rng.randint(5, 12),
                     **dict(opts, m=m, cols=cols, dim=min(dim, 16)))
    if kind == "vectors":
        return _case(None, kind, n=_log(rng, 10_000, 200_000), **dict(opts, m=min(m, 48), cols=min(cols, 48)))
    if kind == "epochs" and rng.random() < 0.35:
        return _case(None, kind, n=_log(rng, 50_000, 1_000_000), epochs=rng.randint(1, 3), f64=True,
                     **dict(opts, m=min(m, 64), cols=min(cols, 64), dim=min(dim, 32), arithmetic="fp64"))
    if kind == "epochs":
        return _case(None, kind, n=_log(rng, 100_000, 12_000_000), epochs=rng.randint(1, 3), **opts)
    if kind == "covariance":
        return _case(None, kind, n=_log(rng, 100_000, ROWS_64), **dict(opts, m=1, cols=1))
    if kind == "gndm":
        return _case(None, kind, n=_log(rng, 100_000, ROWS_64), **dict(opts, rho=True))
    if kind == "serve":
        return _case(None, kind, n=_log(rng, 20_000, 250_000), requests=rng.randint(6, 16),
                     **dict(opts, dim=min(dim, 32), m=min(m, 64), cols=min(cols, 64)))
    return _case(None, kind, n=_log(rng, 20_000, 4_000_000), **opts)


def _case(name, kind, **opts):
    c = {"kind": kind, "topology": "hexagonal", "arithmetic": "ref32", "rho": False, "f64": False, "epochs": 1,
         "requests": 0, **opts}
    return c if name is None else {"name": name, **c}


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# ---------------------------------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed & 0x7FFFFFFF)


def _rows(g, n, dim, dtype=torch.float32):
    """n synthetic systematics rows: about half lognormal(0, 0.5) columns, Gaussian ones, sin and cos of theta."""
    x = torch.empty((n, dim), dtype=dtype, device="cuda")
    ln = max(1, (dim - 2) // 2 + 1)
    mu, sd = math.exp(0.125), math.sqrt((math.exp(0.25) - 1.0) * math.exp(0.25))
    for b in range(0, n, 1 << 22):
        v = x[b:b + (1 << 22)]
        v.normal_(generator=g)
        v[:, :ln] = (torch.exp(0.5 * v[:, :ln]) - mu) / sd
        z = torch.rand(v.shape[0], dtype=dtype, device="cuda", generator=g) * 2.0 - 1.0
        v[:, dim - 2] = (torch.sqrt(1.0 - z * z) - math.pi / 4.0) / math.sqrt(2.0 / 3.0 - math.pi ** 2 / 16.0)
        v[:, dim - 1] = z * math.sqrt(3.0)
    return x


def _density(g, n):
    """Galaxy counts of a pixel over its coverage (FP64)."""
    counts = torch.poisson(torch.full((n,), 3.0, device="cuda"), generator=g).double()
    return counts / (0.5 + 0.5 * torch.rand(n, dtype=torch.float64, device="cuda", generator=g))


def _grid(case):
    """FP64 neuron positions (m * cols, 2)."""
    a = torch.arange(case["m"], dtype=torch.float64, device="cuda")[:, None]
    b = torch.arange(case["cols"], dtype=torch.float64, device="cuda")[None, :]
    if case["topology"] == "square":
        x, y = a + 0 * b, b + 0 * a
    else:
        x, y = a + 0.5 * (b % 2), b * 0.8660254037844386 + 0 * a
    return torch.stack([x, y], dim=2).reshape(-1, 2)


def _apart(a, b):
    """Squared distances between two lists of positions."""
    return (a[:, None, 0] - b[None, :, 0]) ** 2 + (a[:, None, 1] - b[None, :, 1]) ** 2


def _trained(case, seed, epochs=6, sample=8192):
    """FP32 weights of a map trained on a sample of rows, as a searched map is."""
    g = _generator(seed + 77)
    x = _rows(g, sample, case["dim"]).double()
    w = torch.rand((case["m"] * case["cols"], case["dim"]), dtype=torch.float64, device="cuda", generator=g)
    t = _grid(case)
    d2 = _apart(t, t)
    for e in range(epochs):
        sigma = max(case["m"], case["cols"]) / 2.0 / (1.0 + 2.0 * e / (epochs - 1))
        near = _nearest(x, w)[0]
        hit = torch.nn.functional.one_hot(near, w.shape[0]).double()
        h = torch.exp(-d2 / (2.0 * sigma * sigma))
        w = (h @ (hit.T @ x)) / (h @ hit.sum(0))[:, None]
    return w.float()


def _start_weights(case, seed):
    """Initial weights of a training, uniform in [0, 1) as init_rand draws them."""
    dt = torch.float64 if case["f64"] else torch.float32
    return torch.rand((case["m"] * case["cols"], case["dim"]), dtype=dt, device="cuda", generator=_generator(seed + 55))


def _inputs(case, seed):
    """(rows, density or None, weights) of a case on the GPU."""
    g = _generator(seed)
    kind, n, dim = case["kind"], case["n"], case["dim"]
    if kind == "gndm":
        # neighbouring pixels see different systematics: winners spread over the map, a few neurons without any
        mn = case["m"] * case["cols"]
        u = torch.rand(n, dtype=torch.float64, device="cuda", generator=g)
        return (u * u * 0.98 * mn).to(torch.int32), _density(g, n), None
    if kind == "train_host":
        x = torch.from_numpy(synth.mixture_dataset(n, dim, seed=seed)).cuda()
    else:
        x = _rows(g, n, dim, torch.float64 if case["f64"] else torch.float32)
    rho = _density(g, n) if case["rho"] else None
    if kind == "covariance":
        return x, rho, None
    return x, rho, (_start_weights if kind in ("train_host", "epochs", "vectors") else _trained)(case, seed)


def _schedule(case):
    """(epochs of the schedule, sigma0)."""
    return (case["epochs"] if case["kind"] == "train_host" else 20), max(case["m"], case["cols"]) / 2.0


def _requests(case):
    """(model, kind, rows) of the requests of a serving case: sizes from 1,000 rows up in equal ratios, ragged."""
    k = case["requests"]
    ratio = max(1.0, case["n"] / 1000.0) ** (1.0 / (k - 1))
    return [(i % 2, "activation" if i % 3 == 2 else "winners", int(1000 * ratio ** ((i * 5) % k)) + i) for i in range(k)]


def _serve_maps(case):
    """The two resident maps of a serving case."""
    return [dict(case), dict(case, m=32, cols=32, dim=min(16, case["dim"]))]


def _som(case, weights):
    som = dam.SOM_Batch(case["m"], case["cols"], case["dim"], topology=case["topology"],
                        dtype=np.float64 if case["f64"] else np.float32,
                        **({} if case["f64"] else {"arithmetic": case["arithmetic"]}))
    som.weights[...] = weights.cpu().numpy()
    return som


# ---------------------------------------------------------------------------------------------------------------
# A program's state and one pass
# ---------------------------------------------------------------------------------------------------------------
def prepare(case, seed):
    kind, mn, dim = case["kind"], case["m"] * case["cols"], case["dim"]
    ctx = get_context(0)
    s = {"case": case, "ctx": ctx}
    if kind == "serve":
        soms = [_som(c, _trained(c, seed + 1000 * i)) for i, c in enumerate(_serve_maps(case))]
        s["server"] = SOMServer(soms, memory_budget=1 << 30, arithmetic=case["arithmetic"])
        s["requests"] = []
        for i, (model, what, n) in enumerate(_requests(case)):
            x = pinned_empty((n, soms[model].dim), np.float32)
            x[...] = _rows(_generator(seed + 1 + i), n, soms[model].dim).cpu().numpy()
            s["requests"].append((model, what, x))
        return s
    x, rho, w = _inputs(case, seed)
    if kind in ("winners_host", "train_host"):
        s["som"], s["x"], s["w"] = _som(case, w), x.cpu().numpy(), w.cpu().numpy()
        s["rho"] = None if rho is None else rho.cpu().numpy()
        return s
    s["x"], s["rho"] = x, rho
    s["rho_ptr"] = None if rho is None else rho.data_ptr()
    if kind == "gndm":
        s["maps"] = torch.empty((3, mn), dtype=torch.float32, device="cuda")
        s["gndm"] = torch.empty(case["n"], dtype=torch.float32, device="cuda")
        return s
    if kind == "covariance":
        return s
    som = _som(case, w)
    s["codes"] = _lib.PRECISIONS[som.precision], _lib.ARITHMETICS[som.arithmetic]
    s["model"] = Model(ctx, som.m, som.n, dim, som.topology, som._topography, dtype=som.dtype)
    s["model"].set_weights(som.weights)
    s["w"] = w
    if kind == "winners":
        s["out"] = torch.empty(case["n"], dtype=torch.int32, device="cuda")
    elif kind == "activation":
        s["result"] = DeviceArray.zeros(ctx, (som.m, som.n), np.float64)
    elif kind == "errors":
        s["errors"] = DeviceArray.zeros(ctx, (3,), np.float64)
    else:
        s["acc"] = Accumulator(s["model"])
        s["history"] = DeviceArray.empty(ctx, (case["epochs"], mn, dim), som.dtype)
        s["errors"] = DeviceArray.zeros(ctx, (case["epochs"], 3), np.float64)
    return s


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    n, dim = case["n"], case["dim"]
    if kind == "winners_host":
        return s["som"].get_winners(s["x"])
    if kind == "train_host":
        som = s["som"]
        som.weights[...] = s["w"]
        som.train(s["x"], dataset_weights=s["rho"], n_epochs=case["epochs"])
        return [som.weights.copy(), som.quantization_errors, som.topographic_errors]
    if kind == "winners":
        s["model"].find_bmus(s["x"].data_ptr(), n, s["out"].data_ptr(), *s["codes"])
        return s["out"]
    if kind == "activation":
        s["result"].fill_zero()
        s["model"].count_bmus(s["x"].data_ptr(), s["rho_ptr"], n, s["result"].ptr, *s["codes"])
        return s["result"].copy_to_host()
    if kind == "errors":
        s["errors"].fill_zero()
        s["model"].compute_errors(s["x"].data_ptr(), s["rho_ptr"], n, s["errors"].ptr, *s["codes"])
        e = s["errors"].copy_to_host()
        return [e[0] / e[2], e[1] / e[2]]
    if kind == "epochs":
        total, sigma0 = _schedule(case)
        s["model"].set_weights(s["w"].data_ptr())
        s["errors"].fill_zero()
        for e in range(case["epochs"]):
            s["acc"].reset()
            s["acc"].epoch_accumulate(s["x"].data_ptr(), s["rho_ptr"], n, *s["codes"],
                                      s["errors"].view_ptr(3 * (e - 1)) if e > 0 else None)
            s["acc"].epoch_update(e, total, sigma0, s["history"].view_ptr(e * case["m"] * case["cols"] * dim))
        return [s["history"].copy_to_host(), s["errors"].copy_to_host()]
    if kind == "vectors":
        s["model"].set_weights(s["w"].data_ptr())
        s["acc"].reset()
        s["acc"].iter_accumulate(s["x"].data_ptr(), s["rho_ptr"], n, 0, n, _schedule(case)[1], *s["codes"])
        s["acc"].iter_update(s["history"].ptr)
        return s["history"].copy_to_host()
    if kind == "covariance":
        out = np.empty(1 + dim + dim * dim)
        _lib.call("somhip_covariance_chunk", s["ctx"].handle, _lib.vp(s["x"].data_ptr()), 0,
                  None if s["rho_ptr"] is None else _lib.vp(s["rho_ptr"]), n, dim, _lib.vp(out))
        return [out[:1], out[1:1 + dim], out[1 + dim:]]
    if kind == "gndm":
        p = [ctypes.c_void_p(s["maps"][i].data_ptr()) for i in range(3)]
        _lib.call("somhip_gndm", s["ctx"].handle, _lib.vp(s["x"].data_ptr()), _lib.vp(s["rho_ptr"]), n,
                  case["m"] * case["cols"], *p, _lib.vp(s["gndm"].data_ptr()))
        return [s["maps"], s["gndm"]]
    tickets = [s["server"].submit(model, what, x) for model, what, x in s["requests"]]
    return [s["server"].wait(t)[0] for t in tickets]


# ---------------------------------------------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------------------------------------------
def work(case):
    kind, n, mn, dim = case["kind"], case["n"], case["m"] * case["cols"], case["dim"]
    size = 8 if case["f64"] else 4
    row = size * dim + (8 if case["rho"] else 0)
    search = 2.0 * mn * dim
    if kind == "covariance":
        return {"bytes": n * row, "flops": n * 2.0 * dim * (dim + 1)}
    if kind == "gndm":
        return {"bytes": n * 16.0 + 12.0 * mn, "flops": 3.0 * n}
    if kind == "serve":
        maps = _serve_maps(case)
        todo = [(maps[model], what, k) for model, what, k in _requests(case)]
        return {"bytes": sum(k * (4.0 * c["dim"] + (4 if what == "winners" else 0)) for c, what, k in todo),
                "flops": sum(2.0 * k * c["m"] * c["cols"] * c["dim"] for c, what, k in todo)}
    if kind in ("epochs", "train_host"):
        e = case["epochs"]
        # search, sums and the separable neighbourhood update
        flops = e * (n * (search + 2.0 * (dim + 1)) + 2.0 * mn * (case["m"] + case["cols"]) * (dim + 1))
        return {"bytes": e * (n * row + 2.0 * size * mn * dim), "flops": flops}
    if kind == "vectors":
        # every vector has a neighbourhood of its own
        return {"bytes": n * row + 2.0 * size * mn * dim, "flops": n * (search + 2.0 * mn * (dim + 1) + 6.0 * mn)}
    out = 4 * n if kind.startswith("winners") else 8 * mn
    return {"bytes": n * row + size * mn * dim + out, "flops": n * search}


# ---------------------------------------------------------------------------------------------------------------
# The same in 64 bits, with torch alone
# ---------------------------------------------------------------------------------------------------------------
def _nearest(x, w, second=False):
    """(first, second or None, squared distance of the first) of every row among the rows of w, in FP64."""
    w = w.double()
    w2 = (w * w).sum(1)[None, :]
    step = max(1, (1 << 29) // w.shape[0])
    first = torch.empty(x.shape[0], dtype=torch.int64, device="cuda")
    other = torch.empty_like(first) if second else None
    d1 = torch.empty(x.shape[0], dtype=torch.float64, device="cuda")
    for b in range(0, x.shape[0], step):
        v = x[b:b + step].double()
        d = torch.addmm(w2, v, w.T, alpha=-2.0)
        i = d.argmin(1)
        first[b:b + step] = i
        d1[b:b + step] = ((v - w[i]) ** 2).sum(1)
        if second:
            d.scatter_(1, i[:, None], math.inf)
            other[b:b + step] = d.argmin(1)
    return first, other, d1


def _error_sums(case, first, other, d1, rho):
    # positions and their differences in the type of the map: neighbours of a hexagonal map lie at the penalty itself
    t = _grid(case) if case["f64"] else _grid(case).float()
    tt = t[first] - t[other]
    apart = (tt * tt).double().sum(1) > (2.0 if case["topology"] == "square" else 1.0)
    r = torch.ones_like(d1) if rho is None else rho
    return [float((r * d1.sqrt()).sum()), float((r * apart).sum()), float(r.sum())]


def _sums(x, rho, near, mn):
    """Per-neuron sums of rho * (row, 1)."""
    total = torch.zeros((mn, x.shape[1] + 1), dtype=torch.float64, device="cuda")
    for b in range(0, x.shape[0], 1 << 22):
        v = x[b:b + (1 << 22)].double()
        v = torch.cat([v, torch.ones_like(v[:, :1])], 1)
        if rho is not None:
            v *= rho[b:b + (1 << 22), None]
        total.index_add_(0, near[b:b + (1 << 22)], v)
    return total


def exact(case, seed):
    kind, mn, dim = case["kind"], case["m"] * case["cols"], case["dim"]
    if kind in ("winners", "winners_host"):
        return None  # indices alone
    if kind == "epochs" and case["n"] * mn * case["epochs"] > 2e11:
        return None  # minutes of FP64 scans
    if kind == "serve":
        maps = _serve_maps(case)
        weights = [_trained(c, seed + 1000 * i) for i, c in enumerate(maps)]
        out = []
        for i, (model, what, n) in enumerate(_requests(case)):
            c = maps[model]
            near = _nearest(_rows(_generator(seed + 1 + i), n, c["dim"]), weights[model])[0]
            counts = torch.bincount(near, minlength=c["m"] * c["cols"]).double().reshape(c["m"], c["cols"])
            out.append(counts.cpu().numpy() if what == "activation" else None)
        return out
    x, rho, w = _inputs(case, seed)
    if kind == "gndm":
        near = x.long()
        cat = torch.zeros(mn, dtype=torch.float64, device="cuda").index_add_(0, near, rho)
        foot = torch.bincount(near, minlength=mn).double()
        gnd = torch.where(foot > 0, cat / foot, torch.full_like(cat, math.nan))
        return [torch.stack([cat, foot, gnd]), gnd[near]]
    if kind == "covariance":
        r = torch.ones(x.shape[0], dtype=torch.float64, device="cuda") if rho is None else rho
        total = r.sum()
        mean = torch.stack([(r * x[:, k].double()).sum() for k in range(dim)]) / total
        d = x.double() - mean
        m2 = (d * r[:, None]).T @ d
        return [total.reshape(1), mean, m2.reshape(-1)]
    if kind == "activation":
        near = _nearest(x, w)[0]
        r = torch.ones(x.shape[0], dtype=torch.float64, device="cuda") if rho is None else rho
        return torch.zeros(mn, dtype=torch.float64, device="cuda").index_add_(0, near, r).reshape(case["m"], case["cols"])
    if kind == "errors":
        e = _error_sums(case, *_nearest(x, w, second=True), rho)
        return [e[0] / e[2], e[1] / e[2]]
    t = _grid(case)
    total, sigma0 = _schedule(case)
    if kind == "vectors":
        near = _nearest(x, w)[0]
        num = torch.zeros((mn, dim + 1), dtype=torch.float64, device="cuda")
        for b in range(0, x.shape[0], 1 << 15):
            v = x[b:b + (1 << 15)].double()
            v = torch.cat([v, torch.ones_like(v[:, :1])], 1)
            if rho is not None:
                v *= rho[b:b + (1 << 15), None]
            i = torch.arange(b, b + v.shape[0], dtype=torch.float64, device="cuda")
            sigma = sigma0 / (1.0 + 2.0 * i / x.shape[0])
            d2 = _apart(t, t[near[b:b + (1 << 15)]])
            num += torch.exp(-d2 / (2.0 * sigma * sigma)[None, :]) @ v
        return (num[:, :dim] / num[:, dim:]).reshape(1, mn, dim)
    # epochs and train_host: weights after every epoch; errors of epoch e belong to the weights it gave
    d2 = _apart(t, t)
    w = w.double()
    host = kind == "train_host"
    history, errors = [], []
    for e in range(case["epochs"]):
        near, other, d1 = _nearest(x, w, second=e > 0)
        if e > 0:
            errors.append(_error_sums(case, near, other, d1, rho))
        h = torch.exp(-d2 / (2.0 * (sigma0 / (1.0 + 2.0 * e / total)) ** 2))
        num = h @ _sums(x, rho, near, mn)
        w = num[:, :dim] / num[:, dim:]
        history.append(w)
    if not host:
        return [torch.stack(history), np.array(errors + [[0.0, 0.0, 0.0]])]
    errors.append(_error_sums(case, *_nearest(x, w, second=True), rho))
    q, p = np.array([v[0] / v[2] for v in errors]), np.array([v[1] / v[2] for v in errors])
    return [history[int(np.nanargmin(q))], q, p]
