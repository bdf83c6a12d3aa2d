"""Workloads of the Lomb-Scargle engine, for timing it and comparing its outputs between versions.

A case is a dict of plain values.  Three kinds of calls are covered, each through the package's public entry points:

  host    ``lombscarglegpu.lombscargle`` on host arrays, the drop-in call (arrays in, object ids, periods and the whole
          periodogram out);
  sweep   ``device.SweepPlan`` on device tensors: a batch with its periodogram, or a search that keeps only the peaks,
          optionally followed by ``grad.refine_peaks``;
  grad    ``grad.power`` forward and backward.

Light curves follow gpu_lomb_scargle_amd/synth.py: nightly sampling over ``span`` days, a sinusoid plus noise, observation
counts log-normal around ``median``.  They are drawn on the GPU here, so that a batch is made in milliseconds.
"""
import math

import numpy as np
import torch

from gpu_lomb_scargle_amd import _native, device, grad, synth
from gpu_lomb_scargle_amd.lombscarglegpu import lombscargle

FORMS = {"plain": _native.FORM_PLAIN, "split": _native.FORM_SPLIT, "split32": _native.FORM_SPLIT32}
TORCH = {"float": torch.float32, "double": torch.float64}
TWO_PI = 2.0 * math.pi
GRID = (synth.OMEGA_MIN / TWO_PI, synth.OMEGA_MAX / TWO_PI)  # cycles/day of the batch workloads


def _case(name=None, **kw):
    c = {"kind": "sweep", "form": "split32", "dtype": "double", "gen": False, "objects": 1, "median": 140, "sigma": 0.6,
         "lo": 20, "hi": 1000, "span": 1800, "nf": 100000, "pgram": True, "top_k": 1, "persistent": False, "refine": False,
         "fmin": GRID[0], "fmax": GRID[1]}
    if name:
        c["name"] = name
    c.update(kw)
    return c


def listed():
    return [
        # The first call of a new user, and of a script that goes through its stars one by one: one sparse light curve,
        # every option at its default, the grid from the observing window.  Latency is all there is.
        _case("one_star_default", kind="host", form="plain", dtype="float", median=29, sigma=0.0, lo=5, span=120, nf=0,
              fmin=0.1, fmax=10.0),
        # The drop-in example on SDSS Stripe 82: 136 stars of ~52 observations, float build, error bars.
        _case("catalogue_float_errors", kind="host", form="plain", dtype="float", gen=True, objects=136, median=50,
              sigma=0.3, lo=10, hi=120, span=2700, nf=100000, fmin=0.1, fmax=10.0),
        # One well-sampled star with error bars in the double build, as the reference's 8205 example.
        _case("one_star_double_errors", kind="host", form="plain", dtype="double", gen=True, median=3555, sigma=0.0,
              lo=5, hi=5000, nf=200000, fmin=0.5, fmax=24.0),
        # The reference's arithmetic on device tensors: what a parity run and a new data set's first pass use.
        _case("plain_double_batch", form="plain", objects=100, nf=100003),
        # FP64 sums without the software sin/cos: the accurate fast form.
        _case("split_double_batch", form="split", objects=200, nf=200000),
        # The benchmark: 1000 objects x 10^6 bins in the fast form, FP64 in and out, periodogram written.
        _case("batch_double", objects=1000, nf=1000000),
        # The same batch as the reference's float build has it.
        _case("batch_float", dtype="float", objects=1000, nf=1000000),
        # Error bars per observation, float, bins from the ten-per-resolution-element rule the wrapper's "auto" uses.
        _case("errors_float_auto_grid", dtype="float", gen=True, objects=250, nf=429119, span=1800),
        # A survey's period search: uneven light curves, three best peaks, no periodogram, persistent schedule.
        _case("survey_top3", objects=8000, median=60, sigma=1.0, lo=5, hi=5000, nf=200000, pgram=False, top_k=3,
              persistent=True),
        # Search, then refine below the grid spacing: best bin of a fine grid, Newton steps from it.
        _case("search_and_refine", gen=True, objects=1000, median=200, sigma=0.5, lo=5, hi=5000, span=2000, nf=500000,
              pgram=False, refine=True),
        # One long light curve in the fast form: too few work items to fill the chip by themselves.
        _case("one_star_fast", median=3555, sigma=0.0, lo=5, hi=5000, nf=100000),
        # A fit that differentiates the power of every star: forward and backward at one frequency each.
        _case("gradients", kind="grad", gen=True, objects=4096, median=200, sigma=0.5, lo=5, hi=5000, span=2000, nf=0,
              pgram=False),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges; its terms (observations x bins) stay below the listed ones of its kind."""
    kind = rng.choice(["host", "plain", "split", "batch", "batch", "batch", "search", "search", "single", "grad"])
    gen = rng.random() < 0.5
    dtype = rng.choice(["float", "double"])
    span = rng.choice([400, 1000, 1800, 2000, 2700])
    median = _logint(rng, 25, 300)
    if kind == "grad":
        return _case(kind="grad", gen=gen, dtype=dtype, objects=_logint(rng, 64, 4096), median=median, sigma=0.5, lo=5,
                     hi=5000, span=span, nf=0, pgram=False)
    if kind == "single":
        nf = _logint(rng, 5000, 200000)
        return _case(gen=gen, dtype=dtype, median=_logint(rng, 200, 5000), sigma=0.0, lo=5, hi=5000, span=span, nf=nf)
    nf = _logint(rng, 10000, 1000000)
    most = {"host": 7e8, "plain": 1.5e9, "split": 6e9, "batch": 1.5e11, "search": 1.2e11}[kind]
    rows = most / nf
    objects = max(1, min(_logint(rng, 4, 1000 if kind != "search" else 8000), int(rows / (1.3 * median))))
    if kind == "host":
        return _case(kind="host", form="plain", dtype=dtype, gen=gen, objects=min(objects, max(1, int(1.5e7 / nf))),
                     median=median, sigma=0.3, lo=5, span=span, nf=nf, fmin=0.1, fmax=10.0)
    if kind in ("plain", "split"):
        return _case(form=kind, dtype="double", gen=gen, objects=objects, median=median, span=span, nf=nf)
    if kind == "search":
        return _case(gen=gen, dtype=dtype, objects=objects, median=median, sigma=0.8, lo=5, hi=5000, span=span, nf=nf,
                     pgram=False, top_k=rng.choice([1, 3]), persistent=rng.random() < 0.5)
    return _case(gen=gen, dtype=dtype, objects=objects, median=median, span=span, nf=nf)


# ----------------------------------------------------------------------------------------------------------------------
# Inputs
# ----------------------------------------------------------------------------------------------------------------------
def _counts(c):
    """Observations per object: part of the case, the same for every seed."""
    return synth.lognormal_counts(np.random.default_rng(1001), c["objects"], c["median"], c["sigma"], c["lo"], c["hi"])


def _light_curves(c, seed):
    """Light curves of the case on the GPU: t, y, dy (None without error bars), row offsets, true periods."""
    counts = _counts(c)
    dev = torch.device("cuda")
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed))

    def uniform(n, a, b):
        return a + (b - a) * torch.rand(n, dtype=torch.float64, device=dev, generator=g)

    off = device.offsets_from_counts(counts, dev)
    K, n = len(counts), int(counts.sum())
    obj = torch.repeat_interleave(torch.arange(K, device=dev), torch.as_tensor(counts, device=dev))
    nights = torch.randint(0, c["span"] + 1, (n,), device=dev, generator=g).to(torch.float64)
    t = nights + uniform(n, 0.0, 0.3)
    key = 1e5 * obj.to(torch.float64) + t
    t = t[torch.argsort(key)]
    if c["nf"] == 0:  # the observing window fixes the automatic grid: the same number of bins for every seed
        t[off[:-1]], t[off[1:] - 1] = 0.0, float(c["span"])
    P = torch.exp(uniform(K, math.log(0.05), math.log(10.0)))
    phase = uniform(K, 0.0, TWO_PI)
    wave = torch.sin(TWO_PI * t / P[obj] + phase[obj])
    noise = torch.randn(n, dtype=torch.float64, device=dev, generator=g)
    if c["gen"]:
        dy = torch.exp(uniform(n, math.log(0.01), math.log(0.2)))
        y = uniform(K, 15.0, 20.0)[obj] + synth.AMPLITUDE_WITH_ERROR * wave + dy * noise
    else:
        dy = None
        y = wave + 0.3 * noise
        # normalised on the host, where the sums have one order: the inputs are the same bits each time
        first, host = np.concatenate([[0], np.cumsum(counts)[:-1]]), y.cpu().numpy()
        host = host - np.repeat(np.add.reduceat(host, first) / counts, counts)
        host = host / np.repeat(np.sqrt(np.add.reduceat(host * host, first) / counts), counts)
        y = torch.from_numpy(host).to(dev)
    td = TORCH[c["dtype"]]
    return t.to(td), y.to(td), None if dy is None else dy.to(td), off, P


def _bins(c, t):
    """Number of bins: the case's, or the wrapper's rule for one object."""
    return c["nf"] or int((c["fmax"] - c["fmin"]) / (0.1 / float(t[-1] - t[0])))


def _omega0(c, P):
    """A frequency near each star's own (a few parts in 10^4 off), as a fit in progress has it."""
    return (TWO_PI / P) * (1.0 + 2e-4 * torch.sin(torch.arange(len(P), device=P.device, dtype=torch.float64)))


def prepare(case, seed):
    c = dict(case)
    t, y, dy, off, P = _light_curves(c, seed)
    if c["kind"] == "host":
        host = [None if x is None else x.to(torch.float64).cpu().numpy() for x in (t, y, dy)]
        ids = np.repeat(np.arange(c["objects"]), np.diff(off.cpu().numpy()))
        return {"case": c, "ids": ids, "t": host[0], "y": host[1], "dy": host[2]}
    if c["kind"] == "grad":
        leaves = [x.detach().clone().requires_grad_(True) for x in (_omega0(c, P), y) + ((dy,) if c["gen"] else ())]
        weight = torch.linspace(0.5, 1.5, c["objects"], dtype=torch.float64, device=t.device)
        return {"case": c, "t": t, "off": off, "leaves": leaves, "weight": weight}
    plan = device.SweepPlan(
        t, y, dy, off, min_freq=TWO_PI * c["fmin"], max_freq=TWO_PI * c["fmax"], num_freqs=c["nf"],
        variant=_native.GENERALIZED if c["gen"] else _native.STANDARD, form=FORMS[c["form"]], pgram=c["pgram"],
        top_k=c["top_k"], schedule=_native.SCHEDULE_PERSISTENT if c["persistent"] else _native.SCHEDULE_GRID)
    return {"case": c, "plan": plan}


def run(state):
    c = state["case"]
    if c["kind"] == "host":
        # the wrapper pre-centres a double magnitude array in place: a program that keeps its data passes a copy
        _, periods, pgrams = lombscargle(state["ids"], state["t"], state["y"].copy(), c["fmin"], c["fmax"], c["gen"], "GPU",
                                         state["dy"], c["nf"] or "auto", c["dtype"])
        return {"periods": periods, "pgram": pgrams}
    variant = _native.GENERALIZED if c["gen"] else _native.STANDARD
    if c["kind"] == "grad":
        omega, y = state["leaves"][:2]
        dy = state["leaves"][2] if c["gen"] else None
        P = grad.power(omega, state["t"], y, dy, state["off"], variant)
        return [P.detach()] + list(torch.autograd.grad(P, state["leaves"], state["weight"]))
    plan = state["plan"]
    plan.run()
    out = plan.results()
    if c["refine"]:
        step = TWO_PI * (c["fmax"] - c["fmin"]) / c["nf"]
        omega0 = TWO_PI * c["fmin"] + step * out["index"][:, 0].to(torch.float64)
        omega, power, iterations = grad.refine_peaks(omega0, plan.t, plan.y, plan.dy, plan.offsets, variant, max_step=step)
        out.update(omega=omega, refined=power, iterations=iterations)
    return out


def work(case):
    """Bytes: observations in, outputs out.  Flops: a direct evaluation's complex multiply-adds (two sums per term, three
    with error bars), or the 18 weighted sums per observation of a power with derivatives."""
    c = dict(case)
    rows = float(_counts(c).sum())
    size = 4 if c["dtype"] == "float" else 8
    inputs = rows * size * (3 if c["gen"] else 2)
    if c["kind"] == "grad":
        return {"bytes": 2 * inputs + 32.0 * c["objects"], "flops": 2 * 36.0 * rows}
    nf = c["nf"] or int((c["fmax"] - c["fmin"]) * 10 * c["span"])
    written = size * float(c["objects"]) * nf if c["pgram"] else 20.0 * c["objects"] * c["top_k"]
    return {"bytes": inputs + written, "flops": (24.0 if c["gen"] else 16.0) * rows * nf}


# ----------------------------------------------------------------------------------------------------------------------
# The same outputs in 64 bits, from torch alone
# ----------------------------------------------------------------------------------------------------------------------
def _power(XC, XS, C, S, CC, CS, W, Y, YY, gen):
    """Power from the sums of y c, y s, c, s, c c, c s, 1, y, y y over (weighted) observations."""
    if gen:
        c, s, y = C / W, S / W, Y / W
        cc, cs = CC / W - c * c, CS / W - c * s
        ss = 1.0 - CC / W - s * s
        xc, xs = XC / W - y * c, XS / W - y * s
        yy = YY / W - y * y
        return (ss * xc * xc - 2 * cs * xc * xs + cc * xs * xs) / ((cc * ss - cs * cs) * yy)
    SS = W - CC
    var = YY / W - (Y / W) ** 2
    return (SS * XC * XC - 2 * CS * XC * XS + CC * XS * XS) / (2 * (CC * SS - CS * CS)) * (2.0 / (W * var))


def _exact_pgram(t, y, dy, f, gen):
    """Periodogram of one object in float64 at ordinary frequencies f."""
    w = torch.ones_like(t) if dy is None else dy ** -2
    tc = t - 0.5 * (t.min() + t.max())
    y = y - (w * y).sum() / w.sum() if gen else y
    right = torch.stack([w * y, w], 1)
    quad = torch.stack([0.5 * w], 1)
    W, Y, YY = w.sum(), (w * y).sum(), (w * y * y).sum()
    out = torch.empty_like(f)
    step = max(1, int(4e8 // (8 * len(t))))
    for a in range(0, len(f), step):
        ph = torch.outer(f[a:a + step], tc)
        ph -= torch.round(ph)
        ph *= TWO_PI
        c, s = torch.cos(ph), torch.sin(ph)
        left, low = c @ right, s @ right
        cs = (2.0 * c * s) @ quad
        c *= c
        cc = c @ (2.0 * quad)
        out[a:a + step] = _power(left[:, 0], low[:, 0], left[:, 1], low[:, 1], cc[:, 0], cs[:, 0], W, Y, YY, gen)
    return out


def _point_power(omega, t, y, dy, off, gen):
    """Power of every object at its own omega, differentiable."""
    K = len(omega)
    obj = torch.repeat_interleave(torch.arange(K, device=t.device), off[1:] - off[:-1])
    w = torch.ones_like(t) if dy is None else dy ** -2

    def total(x):
        return torch.zeros(K, dtype=torch.float64, device=t.device).index_add(0, obj, x)

    lo = torch.full((K,), math.inf, dtype=torch.float64, device=t.device).scatter_reduce(0, obj, t, "amin")
    hi = torch.full((K,), -math.inf, dtype=torch.float64, device=t.device).scatter_reduce(0, obj, t, "amax")
    if gen:
        y = y - (total(w * y) / total(w)).detach()[obj]
    ph = omega[obj] * (t - (0.5 * (lo + hi))[obj])
    c, s = torch.cos(ph), torch.sin(ph)
    sums = [total(x) for x in (w * y * c, w * y * s, w * c, w * s, w * c * c, w * c * s, w, w * y, w * y * y)]
    return _power(*sums, gen)


def _refined(omega, t, y, dy, off, gen, max_step):
    """Newton steps on the power from omega, bounded by max_step and taken uphill."""
    for _ in range(30):
        w = omega.clone().requires_grad_(True)
        d1 = torch.autograd.grad(_point_power(w, t, y, dy, off, gen).sum(), w, create_graph=True)[0]
        d2 = torch.autograd.grad(d1.sum(), w)[0]
        d1 = d1.detach()
        step = -d1 / d2
        far = ~(d2 < 0) | ~torch.isfinite(step) | (step.abs() > max_step)
        omega = omega + torch.where(far, max_step * torch.sign(d1), step)
    return omega


def exact(case, seed):
    c = dict(case)
    t, y, dy, off, P = _light_curves(c, seed)
    t, y, dy = t.double(), y.double(), None if dy is None else dy.double()
    gen, K = c["gen"], c["objects"]
    if c["kind"] == "grad":
        leaves = [x.detach().clone().requires_grad_(True) for x in (_omega0(c, P), y) + ((dy,) if gen else ())]
        power = _point_power(leaves[0], t, leaves[1], leaves[2] if gen else None, off, gen)
        weight = torch.linspace(0.5, 1.5, K, dtype=torch.float64, device=t.device)
        return [power.detach()] + list(torch.autograd.grad(power, leaves, weight))
    nf = _bins(c, t)
    if float(len(t)) * nf > 2.5e11:
        return None
    f = c["fmin"] + (c["fmax"] - c["fmin"]) / nf * torch.arange(nf, dtype=torch.float64, device=t.device)
    rows = off.tolist()
    kept = torch.empty(K, nf, dtype=torch.float64, device=t.device) if c["pgram"] else None
    top = torch.empty(K, c["top_k"], dtype=torch.float64, device=t.device)
    best = torch.empty(K, dtype=torch.int64, device=t.device)
    for k in range(K):
        a, b = rows[k], rows[k + 1]
        p = _exact_pgram(t[a:b], y[a:b], None if dy is None else dy[a:b], f, gen)
        if kept is not None:
            kept[k] = p
        high = torch.topk(torch.nan_to_num(p, nan=0.0), c["top_k"])
        top[k], best[k] = high.values, high.indices[0]
    if c["kind"] == "host":
        return {"periods": None, "pgram": kept}
    # which of two nearly equal bins is the best one is no computed number: index and period have no exact value
    out = {"index": None, "power": top, "period": None}
    if kept is not None:
        out["pgram"] = kept
    if c["refine"]:
        step = TWO_PI * (c["fmax"] - c["fmin"]) / nf
        omega = _refined(TWO_PI * c["fmin"] + step * best, t, y, dy, off, gen, step)
        out.update(omega=omega, refined=_point_power(omega, t, y, dy, off, gen), iterations=None)
    return out
