"""The work a user has this framework do, as cases to be timed.

Two kinds of call make up that work:

  * simulations ("sim"): a batch is initialised on an engine the program keeps
    (t = 0 census, tables), its days are run and its time series read back.
    This is simulation(), one likelihood evaluation of the MCMC driver, and
    one training batch of fit.simulate_weekly().  Every pass draws the same
    census again, so a pass does the same work each time;
  * the surrogate MLP (6 parameters -> weekly log-incidence): forward passes
    (host rows or device buffers), input gradients, loss gradients and
    training epochs.

A pass goes through the public entry points only, on handles (engine,
surrogate) that the program created before.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from arbo_gpu_fit_amd import abi, configs
from arbo_gpu_fit_amd.data import community_sizes, mosquito_shares
from arbo_gpu_fit_amd.engine import Engine, SimSpec
from arbo_gpu_fit_amd.surrogate import Surrogate

SERIES = ("n_count", "m_count", "n_infected", "n_incidence", "n_one_subpop")
MODELS = ("lattice", "reference", "climate", "fit", "batch", "cities")


def _sim(name, model, sims, grid, humans, days, graph=True, keep=False):
    """model: the parameter set (see _specs); sims simulations of grid x grid
    communities (for "batch" the mean side of the drawn lattices) with about
    `humans` humans per community, `days` days; graph: day loop replayed as
    hipGraphs; keep: the per-community series, infection histories and
    age-of-infection rings are kept, and they and the census read back."""
    return {"name": name, "kind": "sim", "model": model, "sims": sims, "grid": grid, "humans": humans,
            "days": days, "graph": graph, "keep": keep}


def _mlp(name, kind, rows, hidden=256, depth=4, outputs=260, epochs=0):
    return {"name": name, "kind": kind, "rows": rows, "hidden": hidden, "depth": depth, "outputs": outputs,
            "epochs": epochs}


def listed():
    return [
        # the 10x10 lattice, 1e5 humans, one year: the smallest simulation a
        # user runs (a first look, a unit test), bound by launches
        _sim("lattice 10x10", "lattice", 1, 10, 1000, 365),
        # the reference's own parameter set (one serotype, introductions,
        # stochastic-rounding counts) on ragged communities with every output
        # file's data kept and the census read back, launched day by day
        _sim("reference set kept", "reference", 1, 17, 300, 200, graph=False, keep=True),
        # a fit of the climate coefficients: 16 chains' proposals, one year of
        # days whose parameters and lifetimes change daily
        _sim("climate fit", "climate", 16, 12, 400, 363),
        # one iteration of the 64-chain fit: 1e6 humans in 32x32 communities
        # per chain, 260 weeks
        _sim("fit iteration", "fit", 64, 32, 977, 1819),
        # the 100x100 lattice, 1e7 humans, prior immunity, ten years
        _sim("lattice 100x100", "lattice", 1, 100, 1000, 3650),
        # a batch of simulations of uneven lattices and communities, through
        # its epidemic: the training data of the surrogate and the benchmark
        _sim("uneven batch", "batch", 64, 53, 1100, 150, graph=False),
        # few large communities (cities of 3,000 to 21,000 humans), whose
        # bitmaps need several waves each
        _sim("cities", "cities", 1, 7, 9000, 180),
        # surrogate: a serving loop's device-buffer call, 64 rows
        _mlp("device forward 64", "noalloc", 64),
        # the first stage of screened delayed acceptance, 64 chains
        _mlp("forward 64", "forward", 64),
        # a Langevin step's gradient, 64 chains
        _mlp("input gradient 64", "input_grad", 64),
        # validation of a trained network, the largest batch train_surrogate
        # allows
        _mlp("forward 4096", "forward", 4096),
        # training on 50,000 runs in minibatches of 512 (the last one ragged)
        _mlp("training", "train", 50000, epochs=2),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: any model or surrogate call, sizes spread on a log
    scale over the ranges the listed cases span."""
    case = _drawn(rng)
    del case["name"]
    return case


def _drawn(rng):
    kind = rng.choice(["sim", "sim", "sim", "noalloc", "forward", "input_grad", "loss_grad", "train"])
    if kind != "sim":
        hidden = rng.choice([64, 96, 128, 200, 256])
        depth = rng.randint(2, 4)
        outputs = rng.randint(20, 260)
        if kind == "train":
            return _mlp("", kind, _log_int(rng, 3000, 50000), hidden, depth, outputs, rng.randint(1, 2))
        top = {"loss_grad": 512}.get(kind, 4096)
        return _mlp("", kind, _log_int(rng, 1 if kind != "loss_grad" else 30, top), hidden, depth, outputs)
    model = rng.choice(MODELS)
    if model == "lattice":
        c = _sim("", model, 1, _log_int(rng, 10, 100), _log_int(rng, 200, 1500), _log_int(rng, 120, 1800))
    elif model == "reference":
        c = _sim("", model, 1, _log_int(rng, 4, 30), _log_int(rng, 50, 800), _log_int(rng, 60, 300),
                 graph=rng.random() < 0.5, keep=rng.random() < 0.5)
    elif model == "climate":
        c = _sim("", model, rng.randint(1, 20), _log_int(rng, 5, 20), _log_int(rng, 100, 800), 7 * rng.randint(20, 60) - 1)
    elif model == "fit":
        c = _sim("", model, rng.randint(4, 64), _log_int(rng, 12, 32), _log_int(rng, 200, 1200), 7 * rng.randint(26, 156) - 1)
    elif model == "batch":
        c = _sim("", model, rng.randint(6, 48), _log_int(rng, 25, 53), _log_int(rng, 400, 1300), _log_int(rng, 30, 150),
                 graph=rng.random() < 0.5)
    else:
        c = _sim("", model, 1, rng.randint(2, 8), _log_int(rng, 4000, 10000), _log_int(rng, 40, 180))
    return c


# --- simulations -----------------------------------------------------------

def _specs(case, seed):
    r = np.random.Generator(np.random.PCG64([seed, 1]))
    n, g, hum, days = case["sims"], case["grid"], case["humans"], case["days"]
    out = []
    for i in range(n):
        sd = int(r.integers(0, 2 ** 63))
        if case["model"] == "lattice":          # the plain workload: Beta(2,5) prior immunity
            out.append(SimSpec(g, g, np.full(g * g, hum, np.uint32), configs.base_params(immunity_mode=1), sd))
        elif case["model"] == "reference":      # degree-heterogeneous sizes, infections seeded and introduced
            humans = community_sizes(g, g, hum * g * g, 1.0, seed=g, neighbourhood=4)   # the place is the same
            p = configs.reference_params(seed_frac_h=0.01, seed_frac_m=0.01, beta_hm=0.4, beta_mh=0.4)
            out.append(SimSpec(g, g, humans, p, sd))
        elif case["model"] == "climate":        # coefficients of the reference's fitted set, drawn as proposals
            cl = configs.seasonal_climate(days + 1, biting_rate=0.5, scale_eip=float(r.uniform(2.0, 3.0)),
                                          scale_mle=float(r.uniform(2.5, 3.5)), scale_cc=float(r.uniform(0.6, 1.4)),
                                          scale_humidity=float(r.uniform(0.6, 1.4)),
                                          min_mos_to_human=float(r.uniform(2.0, 4.0)))
            p = configs.reference_params(n_serotypes=2, seed_frac_h=0.01, seed_frac_m=0.01)
            out.append(SimSpec(g, g, np.full(g * g, hum, np.uint32), p, sd, climate=cl,
                               mosq_share=mosquito_shares(g, g, 0.5, neighbourhood=4)))
        elif case["model"] == "fit":            # proposals from the fit's priors
            p = configs.base_params(beta_hm=float(r.uniform(0.05, 0.6)), beta_mh=float(r.uniform(0.05, 0.6)),
                                    long_distance=float(10 ** r.uniform(-3, -1)), season_amp=float(r.uniform(0, 0.9)),
                                    season_phase=float(r.uniform(0, 2 * math.pi)))
            out.append(SimSpec(g, g, np.full(g * g, hum, np.uint32), p, sd))
        elif case["model"] == "batch":          # sides log-uniform over a factor 2 either way, ragged communities
            gi = max(2, int(round(g * math.exp(r.uniform(-0.69, 0.63)))))
            humans = r.integers(max(1, hum // 5), hum * 9 // 5, gi * gi).astype(np.uint32)
            p = configs.base_params(beta_hm=float(r.uniform(0.05, 0.6)), beta_mh=float(r.uniform(0.05, 0.6)),
                                    long_distance=float(10 ** r.uniform(-3, -1)), season_amp=float(r.uniform(0, 0.9)),
                                    season_phase=float(r.uniform(0, 2 * math.pi)))
            out.append(SimSpec(gi, gi, humans, p, sd))
        else:                                   # cities: log-uniform sizes within the slot limit (3 slots a human)
            humans = np.minimum(21000, np.exp(r.uniform(math.log(hum / 3), math.log(hum * 2.3), g * g))).astype(np.uint32)
            out.append(SimSpec(g, g, humans, configs.base_params(long_distance=0.05), sd))
    return out


def _prepare_sim(case, seed):
    flags = (abi.F_GRAPH if case["graph"] else 0) | ((abi.F_SPATIAL | abi.F_AOI) if case["keep"] else 0)
    return {"case": case, "engine": Engine(flags=flags), "specs": _specs(case, seed)}


def _run_sim(st):
    eng, case, n = st["engine"], st["case"], st["case"]["sims"]
    eng.init(st["specs"], case["days"])
    eng.step(case["days"])
    got = [eng.series(i) for i in range(n)]
    out = {k: np.stack([s[k] for s in got]) for k in SERIES}
    if case["keep"]:
        for i in range(n):
            out["kept %d" % i] = {"spatial": eng.spatial(i), "history": eng.history(i), "aoi": eng.aoi(i),
                                  "state": eng.state(i)}
    return out


# --- the surrogate ---------------------------------------------------------

BATCH, RATE = 512, 1e-5   # the training's minibatch and the last rate of its schedule


def _widths(case):
    return [6] + [case["hidden"]] * case["depth"] + [case["outputs"]]


def _network(case, seed):
    """Flat float32 parameters (He-normal weights, small biases, output biases
    at weekly log-means of tens to hundreds of cases)."""
    r = np.random.Generator(np.random.PCG64([seed, 2]))
    w, parts = _widths(case), []
    for k, n in zip(w[:-1], w[1:]):
        scale = math.sqrt(2.0 / k) * (1.0 if n != w[-1] else 0.5)
        parts.append(r.normal(0.0, scale, (n, k)).ravel())
        parts.append(r.normal(0.0, 0.05, n))
    week = np.arange(w[-1])
    parts[-1] = 4.0 + 1.2 * np.sin(2 * math.pi * week / 52.0 + r.uniform(0, 6.28)) + r.normal(0.0, 0.1, w[-1])
    return np.concatenate(parts).astype(np.float32)


def _rows(case, seed):
    """Feature rows on [-1, 1] and Poisson counts of a mean that depends on
    them."""
    r = np.random.Generator(np.random.PCG64([seed, 3]))
    n, out = case["rows"], case["outputs"]
    x = r.uniform(-1.0, 1.0, (n, 6)).astype(np.float32)
    if case["kind"] in ("noalloc", "forward"):
        return x, None
    if case["kind"] == "input_grad":   # d log-likelihood / d log mean: of the order of the counts' noise
        return x, (r.normal(0.0, 1.0, (n, out)) * np.exp(r.normal(1.0, 0.8, (n, 1)))).astype(np.float32)
    c = r.normal(0.0, 0.5, 6)
    level = 4.0 + x @ c
    season = 1.2 * np.sin(2 * math.pi * np.arange(out) / 52.0 + r.uniform(0, 6.28))
    return x, r.poisson(np.exp(level)[:, None] * np.exp(season)).astype(np.float32)


_STREAM = []


def _serving_stream():
    """The one stream of a serving loop: calls that share the library's
    scratch activations must not overlap."""
    if not _STREAM:
        _STREAM.append(torch.cuda.Stream())
    return _STREAM[0]


def _prepare_mlp(case, seed):
    sur = Surrogate(_widths(case), max_batch=4096, seed=seed & 0xFFFF)
    sur.set_params(_network(case, seed))
    x, y = _rows(case, seed)
    st = {"case": case, "sur": sur, "x": x, "y": y, "seed": seed & 0xFFFF}
    if case["kind"] == "noalloc":
        st["stream"] = _serving_stream()
        st["dx"] = torch.from_numpy(x).cuda()
        st["dout"] = torch.empty((case["rows"], case["outputs"]), dtype=torch.float32, device="cuda")
    return st


def _run_mlp(st):
    sur, kind, x, y = st["sur"], st["case"]["kind"], st["x"], st["y"]
    if kind == "forward":
        return sur.forward(x)
    if kind == "noalloc":   # the C entry point for device buffers
        stream = ctypes.c_void_p(st["stream"].cuda_stream)
        rc = sur.lib.arbo_sur_forward_noalloc(sur._h, x.shape[0], ctypes.c_void_p(st["dx"].data_ptr()),
                                              ctypes.c_void_p(st["dout"].data_ptr()), stream)
        if rc:
            raise RuntimeError("arbo_sur_forward_noalloc: %d" % rc)
        return st["dout"]
    if kind == "input_grad":
        out, dx = sur.input_grad(x, y)
        return {"out": out, "dx": dx}
    if kind == "loss_grad":   # the loss in the network's own precision
        loss, g = sur.loss_grad(x, y)
        return {"loss": np.float32(loss), "grad": g}
    hist = sur.train(x, y, epochs=st["case"]["epochs"], batch=BATCH, lr=RATE, seed=st["seed"])
    return {"loss": hist.astype(np.float32), "params": sur.get_params()}


def prepare(case, seed):
    return _prepare_sim(case, seed) if case["kind"] == "sim" else _prepare_mlp(case, seed)


def run(state):
    return _run_sim(state) if state["case"]["kind"] == "sim" else _run_mlp(state)


# --- what a pass cannot do without -----------------------------------------

def work(case):
    """Simulations: the census is written once and then, every day, each
    human's word (4 bytes) and each living mosquito's word (2 bytes) looked
    at once; the series come out.  Surrogate: the float32 network's products;
    parameters, rows and results moved once (training: parameters, gradients
    and moments once per minibatch, the rows once per epoch)."""
    if case["kind"] == "sim":
        comm = case["sims"] * case["grid"] ** 2 * (1.24 if case["model"] == "batch" else 1.0)
        humans = float(comm) * case["humans"]
        mosq = 2.0 * humans
        s = 4 * case["sims"] * (case["days"] + 1) * 14
        kept = 16.0 * humans if case["keep"] else 0.0
        return {"bytes": 10 * humans + 4 * mosq + case["days"] * (4 * humans + 2 * mosq) + s + kept, "flops": 0.0}
    w, n = _widths(case), case["rows"]
    mm = float(sum(a * b for a, b in zip(w[:-1], w[1:])))
    first = float(w[0] * w[1])
    params = 4.0 * (mm + sum(w[1:]))
    io = 4.0 * n * (w[0] + w[-1])
    if case["kind"] in ("forward", "noalloc"):
        return {"bytes": params + io, "flops": 2 * mm * n}
    if case["kind"] == "input_grad":
        return {"bytes": params + 2 * io, "flops": 4 * mm * n}
    if case["kind"] == "loss_grad":
        return {"bytes": 2 * params + io, "flops": (6 * mm - 2 * first) * n}
    steps = case["epochs"] * -(-n // BATCH)
    return {"bytes": 7 * params * steps + io * case["epochs"], "flops": case["epochs"] * (6 * mm - 2 * first) * n}


# --- 64-bit values of the surrogate's outputs ------------------------------

def _layers64(case, seed):
    p = torch.from_numpy(_network(case, seed)).double().cuda()
    out, o = [], 0
    w = _widths(case)
    for k, n in zip(w[:-1], w[1:]):
        out.append([p[o:o + n * k].reshape(n, k).clone(), p[o + n * k:o + n * k + n].clone()])
        o += n * k + n
    return out


def _forward64(layers, x):
    hs, zs = [x], []
    for i, (W, b) in enumerate(layers):
        zs.append(hs[-1] @ W.T + b)
        if i + 1 < len(layers):
            hs.append(0.5 * zs[-1] * (1.0 + torch.erf(zs[-1] / math.sqrt(2.0))))
    return hs, zs


def _backward64(layers, hs, zs, dz):
    grads = [None] * len(layers)
    for i in range(len(layers) - 1, -1, -1):
        grads[i] = [dz.T @ hs[i], dz.sum(0)]
        dz = dz @ layers[i][0]
        if i:
            z = zs[i - 1]
            dz = dz * (0.5 * (1.0 + torch.erf(z / math.sqrt(2.0)))
                       + z * torch.exp(-0.5 * z * z) / math.sqrt(2.0 * math.pi))
    return grads, dz


def _loss64(layers, x, y):
    hs, zs = _forward64(layers, x)
    e = torch.exp(zs[-1])
    total = float((e - y * zs[-1]).sum())
    grads, _ = _backward64(layers, hs, zs, (e - y) / y.numel())
    return total, grads


def _flat(pairs):
    return torch.cat([t.reshape(-1) for pair in pairs for t in pair]).cpu().numpy()


def _shuffle(n, epoch, seed):
    """The documented order of an epoch's rows: Fisher-Yates from the last
    row down, row i swapped with floor(r (i + 1) / 2^32), r the first word of
    Philox4x32-10 (Salmon et al. 2011) at counter (i, epoch, 7, 0)."""
    m = np.uint64(0xFFFFFFFF)
    c = [np.arange(n, dtype=np.uint64)] + [np.full(n, v, np.uint64) for v in (epoch, 7, 0)]
    k0, k1 = seed & 0xFFFFFFFF, seed >> 32
    for _ in range(10):
        a, b = c[0] * np.uint64(0xD2511F53), c[2] * np.uint64(0xCD9E8D57)
        c = [(b >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), b & m, (a >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), a & m]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    j = ((c[0] * (np.arange(n, dtype=np.uint64) + np.uint64(1))) >> np.uint64(32)).tolist()
    perm = list(range(n))
    for i in range(n - 1, 0, -1):
        perm[i], perm[j[i]] = perm[j[i]], perm[i]
    return perm


def _train64(case, seed, layers, x, y):
    flat = [t for pair in layers for t in pair]
    m, v = [torch.zeros_like(t) for t in flat], [torch.zeros_like(t) for t in flat]
    step, hist, n = 0, [], case["rows"]
    for epoch in range(case["epochs"]):
        order = torch.tensor(_shuffle(n, epoch, seed & 0xFFFF), device=x.device)
        total = 0.0
        for o in range(0, n, BATCH):
            rows = order[o:o + BATCH]
            part, grads = _loss64(layers, x[rows], y[rows])
            total += part
            step += 1
            for p, g, a, b in zip(flat, [t for pair in grads for t in pair], m, v):
                a.mul_(0.9).add_(g, alpha=0.1)
                b.mul_(0.999).addcmul_(g, g, value=0.001)
                p.sub_(RATE * (a / (1.0 - 0.9 ** step)) / ((b / (1.0 - 0.999 ** step)).sqrt() + 1e-8))
        hist.append(total / y.numel())
    return {"loss": np.array(hist), "params": _flat(layers)}


def exact(case, seed):
    """None for simulations: their outputs are whole numbers."""
    if case["kind"] == "sim":
        return None
    layers = _layers64(case, seed)
    x, y = (None if a is None else torch.from_numpy(a).double().cuda() for a in _rows(case, seed))
    if case["kind"] == "train":
        return _train64(case, seed, layers, x, y)
    if case["kind"] == "loss_grad":
        total, grads = _loss64(layers, x, y)
        return {"loss": total / y.numel(), "grad": _flat(grads)}
    hs, zs = _forward64(layers, x)
    if case["kind"] == "input_grad":
        _, dx = _backward64(layers, hs, zs, y)
        return {"out": zs[-1].cpu().numpy(), "dx": dx.cpu().numpy()}
    return zs[-1].cpu().numpy()
