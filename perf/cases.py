"""Performance cases of the framework: the work that its users have it do,
through the public entry points of parallelcmacionize_amd.

Kinds of case (every pass takes host data in and gives host data back where
the entry point does):

  buffer  one subgrid, one packet buffer (Context.interact_batch)
  list    an explicit packet list through the whole grid
          (Context.transport_packets)
  solve   the plain iteration of a medium: fields in, a number of transports
          with their ionization updates, neutral fractions out
  set     a set of independent problems (Batch.iteration)
  net     one inference or one loss and gradient of the warm-start network
  train   training steps of the warm-start network
  warm    cheap passes and the learned warm start on a new medium

`exact` restates what the entry points compute in 64 bits (numpy and torch
only): the lattice walk, the emission, the ionization balance, the network.
"""
import math
import os

import numpy as np
import torch

import parallelcmacionize_amd as cmi
from parallelcmacionize_amd import warmstart

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NET_FILE = os.path.join(ROOT, "parallelcmacionize_amd", "data", "warmstart_clumpy256.npz")

PC = 3.086e16
SIGMA = 6.3e-22       # m^2
ALPHA = 2.7e-19       # m^3 s^-1
MEAN_N = 1.0e8        # m^-3
X0 = 1.0e-6
BOX = (-5 * PC, -5 * PC, -5 * PC, 10 * PC, 10 * PC, 10 * PC)
EDGES = (32, 48, 64, 96, 128)   # problem sizes of the sets
FACE_X_N = 22                   # entry through the lower x face


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def _solve(name, ncell, nsub, packets, iterations, sources, medium, precision, reemit=0.0):
    c = {"kind": "solve", "nx": ncell[0], "ny": ncell[1], "nz": ncell[2],
         "sx": nsub[0], "sy": nsub[1], "sz": nsub[2], "packets": packets,
         "iterations": iterations, "sources": sources, "medium": medium,
         "precision": precision, "reemit": reemit}
    return dict(c, name=name) if name else c


def _list(name, ncell, nsub, packets, precision):
    c = {"kind": "list", "nx": ncell[0], "ny": ncell[1], "nz": ncell[2],
         "sx": nsub[0], "sy": nsub[1], "sz": nsub[2], "packets": packets,
         "precision": precision}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the reference's unit of work: one 200-packet PhotonBuffer walked
        # through one subgrid; the smallest call, all latency
        {"name": "buffer_200", "kind": "buffer", "cells": 16, "nsub": 2, "packets": 200,
         "walk": "interact", "entry": 0},
        # a caller's own packets (not emitted on the device) in the
        # reference's arithmetic: the bit-exact mode
        _list("list_fp64_128", (128, 128, 128), (4, 4, 4), 300000, "fp64"),
        # the same interface on the production engine
        _list("list_fp32_128", (128, 128, 128), (8, 8, 8), 2000000, "fp32"),
        # the reference's own test problem at its own size: a 64^3 Stromgren
        # sphere, 1e6 packets, 10 iterations; launches and latency count
        _solve("stromgren_64", (64, 64, 64), (4, 4, 4), 1000000, 10, 1, "uniform", "fp32"),
        # an ordinary medium on a lattice that is neither cubic nor a power
        # of two (40 x 24 x 24 subgrids, non-cubic cells)
        _solve("solve_ragged", (120, 96, 72), (3, 4, 3), 3000000, 5, 5, "clumpy", "fp32"),
        # diffuse reemission (alpha_1 / alpha_A = 0.364)
        _solve("reemission_128", (128, 128, 128), (8, 8, 8), 5000000, 3, 1, "uniform", "fp32",
               0.364),
        # a solve in the reference's arithmetic, as a check run of a new setup
        _solve("solve_fp64_64", (64, 64, 64), (4, 4, 4), 1000000, 3, 4, "clumpy", "fp64"),
        # the headline workload: 256^3 clumpy, 1e8 packets, 10 iterations
        _solve("clumpy_256", (256, 256, 256), (4, 4, 4), 100000000, 10, 8, "clumpy", "fp32"),
        # a parameter study: uneven problems iterated together
        {"name": "set_24", "kind": "set", "problems": 24, "layout": 5, "iterations": 2},
        # the trainer's step: batches of 4 whole 64^3 crops
        {"name": "train_64", "kind": "train", "batch": 4, "crop": 64, "sample": 64,
         "samples": 12, "steps": 8},
        # a gradient on a ragged volume (validation, fine-tuning on crops)
        {"name": "grad_ragged", "kind": "net", "backward": True, "batch": 2, "d": 40, "h": 72,
         "w": 96},
        # the learned warm start of a new 256^3 medium: 5 cheap passes, then
        # the network
        {"name": "warm_256", "kind": "warm", "cells": 256, "nsub": 4, "packets": 10000000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _lattice(rng, most):
    """Subgrid edges of use (powers of two and not) and 1 .. 8 subgrids per
    axis, at most `most` cells per axis and 8 cells at least in all."""
    ncell, nsub = [], []
    for _ in range(3):
        edge = rng.choice((8, 12, 16, 16, 20, 24, 32, 32, 40, 48, 64))
        edge = min(edge, most)
        n = rng.randint(1, max(1, min(8, most // edge)))
        ncell.append(edge * n)
        nsub.append(n)
    return ncell, nsub


def draw(rng):
    kind = rng.choice(("buffer", "list", "list", "solve", "solve", "solve", "set", "net", "net",
                       "train", "warm"))
    if kind == "buffer":
        return {"kind": kind, "cells": rng.choice((8, 12, 16, 20, 32, 48, 64)),
                "nsub": rng.randint(1, 4), "packets": _log_int(rng, 1, 100000),
                "walk": rng.choice(("interact", "propagate", "optical_depth")),
                "entry": rng.choice((0, FACE_X_N))}
    if kind == "list":
        precision = rng.choice(("fp64", "fp32"))
        ncell, nsub = _lattice(rng, 160)
        return _list(None, ncell, nsub,
                     _log_int(rng, 100, 500000 if precision == "fp64" else 2000000), precision)
    if kind == "solve":
        precision = rng.choice(("fp64", "fp32", "fp32", "fp32"))
        ncell, nsub = _lattice(rng, 96 if precision == "fp64" else 256)
        medium = rng.choice(("uniform", "clumpy", "clumpy"))
        return _solve(None, ncell, nsub,
                      _log_int(rng, 10000, 2000000 if precision == "fp64" else 30000000),
                      rng.randint(1, 5), 1 if medium == "uniform" else rng.randint(1, 16),
                      medium, precision, rng.choice((0.0, 0.0, 0.364)))
    if kind == "set":
        return {"kind": kind, "problems": _log_int(rng, 2, 32), "layout": rng.randint(1, 10000),
                "iterations": rng.randint(1, 4)}
    if kind == "net":
        return {"kind": kind, "backward": rng.random() < 0.5, "batch": 1, "d": rng.randint(8, 128),
                "h": rng.randint(8, 128), "w": 32 * rng.randint(1, 4)}
    if kind == "train":
        crop = rng.choice((32, 64, 64))
        return {"kind": kind, "batch": rng.randint(1, 4), "crop": crop,
                "sample": rng.choice((crop, 64)), "samples": rng.randint(2, 12),
                "steps": rng.randint(1, 8)}
    cells = rng.choice((64, 96, 128, 160, 192, 224))
    return {"kind": kind, "cells": cells, "nsub": 4, "packets": _log_int(rng, 100000, 5000000)}


# ---------------------------------------------------------------------------
# Inputs (the same for prepare and exact)
# ---------------------------------------------------------------------------
def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _random_field(shape, seed):
    """Zero-mean unit-variance Gaussian random field, P(k) ~ k^(-11/3)."""
    dev = _device()
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    white = torch.randn(shape, generator=gen, device=dev, dtype=torch.float64)
    f = torch.fft.rfftn(white)
    k2 = torch.zeros((1, 1, 1), device=dev, dtype=torch.float64)
    for a, n in enumerate(shape):
        k = (torch.fft.rfftfreq(n) if a == 2 else torch.fft.fftfreq(n)).to(dev, torch.float64)
        view = [1, 1, 1]
        view[a] = -1
        k2 = k2 + (k * k).reshape(view)
    k2[0, 0, 0] = 1.0
    amp = k2 ** (-11.0 / 12.0)
    amp[0, 0, 0] = 0.0
    g = torch.fft.irfftn(f * amp, s=tuple(shape))
    g = g - g.mean()
    return g / g.std()


def _density(shape, medium, seed, sigma_ln=1.0):
    if medium == "uniform":
        return torch.full(tuple(shape), MEAN_N, dtype=torch.float64, device=_device())
    g = _random_field(shape, seed)
    return MEAN_N * torch.exp(sigma_ln * g - 0.5 * sigma_ln * sigma_ln)


def _to_subgrids(a, nsub):
    """(nx, ny, nz) lattice -> flat subgrid-major order (torch)."""
    n = a.shape
    b = a.reshape(nsub[0], n[0] // nsub[0], nsub[1], n[1] // nsub[1], nsub[2], n[2] // nsub[2])
    return b.permute(0, 2, 4, 1, 3, 5).contiguous().reshape(-1)


def _host(t):
    return t.cpu().numpy()


def _shape(case):
    return ((case["nx"], case["ny"], case["nz"]), (case["sx"], case["sy"], case["sz"]))


def _sources(case, rng):
    """A star near the centre of the uniform medium (4.26e49 s^-1), or
    clusters anywhere in a clumpy one (log-uniform 1e48 .. 1e49 s^-1)."""
    if case.get("medium", "clumpy") == "uniform":
        pos = rng.uniform(-0.3 * PC, 0.3 * PC, (case["sources"], 3))
        return pos, np.full(case["sources"], 4.26e49)
    pos = np.array(BOX[:3]) + rng.uniform(0.02, 0.98, (case["sources"], 3)) * np.array(BOX[3:])
    return pos, 10 ** rng.uniform(48, 49, case["sources"])


def _solve_inputs(case, seed):
    rng = np.random.default_rng([1, seed])
    ncell, nsub = _shape(case)
    n = _density(ncell, case["medium"], seed)
    pos, lum = _sources(case, rng)
    return n, pos, lum, int(rng.integers(1, 1 << 40))


def _packets(count, lo, side, rng):
    p = np.zeros(count, cmi.PHOTON_DTYPE)
    p["pos"] = lo + rng.uniform(0, 1, (count, 3)) * side
    cost = rng.uniform(-1, 1, count)
    phi = rng.uniform(0, 2 * np.pi, count)
    sint = np.sqrt(1 - cost * cost)
    p["dir"] = np.stack([sint * np.cos(phi), sint * np.sin(phi), cost], axis=1)
    p["tau"] = rng.exponential(1.0, count)
    p["sigma"] = SIGMA
    p["weight"] = 1.0
    return p


def _list_inputs(case, seed):
    """A partly ionized clumpy medium and packets from anywhere in it."""
    rng = np.random.default_rng([2, seed])
    ncell, nsub = _shape(case)
    n = _density(ncell, "clumpy", seed)
    x = 10 ** (1.5 * _random_field(ncell, seed + 1) - 4.0).clamp(-7.0, 0.0)
    p = _packets(case["packets"], np.array(BOX[:3]), np.array(BOX[3:]), rng)
    u = (p["pos"] - np.array(BOX[:3])) / np.array(BOX[3:])
    s = np.minimum((u * np.array(nsub)).astype(np.int64), np.array(nsub) - 1)
    start = ((s[:, 0] * nsub[1] + s[:, 1]) * nsub[2] + s[:, 2]).astype(np.uint32)
    return n, x, p, start


def _buffer_inputs(case, seed):
    rng = np.random.default_rng([3, seed])
    edge, nsub = case["cells"], case["nsub"]
    shape = (edge * nsub,) * 3
    n = _density(shape, "clumpy", seed)
    x = 10 ** (1.5 * _random_field(shape, seed + 1) - 4.0).clamp(-7.0, 0.0)
    sub = int(rng.integers(0, nsub ** 3))
    s = np.array([sub // (nsub * nsub), (sub // nsub) % nsub, sub % nsub])
    side = BOX[3] / nsub
    lo = np.array(BOX[:3]) + s * side
    p = _packets(case["packets"], lo, np.full(3, side), rng)
    if case["entry"] == FACE_X_N:
        p["pos"][:, 0] = lo[0]
        p["dir"][:, 0] = np.abs(p["dir"][:, 0])
    return n, x, sub, s, lo, side, p


def _set_spec(case):
    rng = np.random.default_rng([4, case["layout"]])
    spec = []
    for _ in range(case["problems"]):
        n = int(rng.choice(EDGES))
        spec.append({"n": n, "side": n / 128 * 10 * PC, "sigma_ln": float(rng.uniform(0.5, 1.5)),
                     "sources": int(rng.integers(1, 17)),
                     "packets": int(np.clip(2 * n ** 3, 20000, 4000000))})
    return spec


def _set_inputs(case, seed):
    rng = np.random.default_rng([5, seed])
    out = []
    for q, s in enumerate(_set_spec(case)):
        n = _density((s["n"],) * 3, "clumpy", 1000 * seed + q, s["sigma_ln"])
        pos = rng.uniform(0.02, 0.98, (s["sources"], 3)) * s["side"]
        lum = 10 ** rng.uniform(48, 49, s["sources"]) * (s["n"] / 128) ** 3
        out.append((s, n, pos, lum))
    return out, int(rng.integers(1, 1 << 40))


LAYERS = ((2, 32, 32), (32, 32, 32), (32, 32, 32), (32, 1, 16))  # cin, cout, padded cout
NET_MEAN, NET_SCALE, NET_OUT = (8.0, -4.0), (2.0, 0.3), 8.0
NET_DILATION = (1, 2, 4, 8)


def _net_params(seed):
    """He-uniform weights and small biases in the master layout
    (W[27][padded cout][32], b[padded cout] per layer)."""
    rng = np.random.default_rng([6, seed])
    out = []
    for cin, cout, pad in LAYERS:
        w = np.zeros((27, pad, 32), np.float32)
        bound = math.sqrt(6.0 / (27 * cin))
        w[:, :cout, :cin] = rng.uniform(-bound, bound, (27, cout, cin))
        b = np.zeros(pad, np.float32)
        b[:cout] = rng.uniform(-0.05, 0.05, cout)
        out += [w.reshape(-1), b]
    return np.concatenate(out)


def _net_samples(count, shape, seed):
    """log10 n_H and the logit of a cheap x_n, and a smooth correction."""
    f = np.empty((count,) + tuple(shape) + (2,), np.float32)
    t = np.empty((count,) + tuple(shape), np.float32)
    for k in range(count):
        g = _random_field(shape, 100 * seed + 2 * k)
        h = _random_field(shape, 100 * seed + 2 * k + 1)
        f[k, ..., 0] = _host(8.0 + 0.43 * g)
        f[k, ..., 1] = _host((2.0 * g + 4.0 * h - 6.0).clamp(-16.0, 5.0))
        t[k] = _host(2.0 * torch.tanh(g) * torch.sigmoid(h) + 0.5 * h)
    return f, t


def _new_net(seed):
    net = cmi.WarmStartNet(seed=1)
    net.set_normalisation(NET_MEAN, NET_SCALE, NET_OUT)
    net.set_dilation(NET_DILATION)
    net.set_loss_weight(4.0)
    p = _net_params(seed)
    net.set_params(p)
    return net, p


def _warm_inputs(case, seed):
    rng = np.random.default_rng([7, seed])
    c = case["cells"]
    n = _density((c, c, c), "clumpy", seed)
    pos = np.array(BOX[:3]) + rng.uniform(0.02, 0.98, (8, 3)) * np.array(BOX[3:])
    return n, pos, 10 ** rng.uniform(48, 49, 8), int(rng.integers(1, 1 << 40))


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------
def _context(shape, nsub, precision):
    fp32 = precision == "fp32"
    ctx = cmi.Context(BOX, shape, nsub, cmi.PREC_FP32 if fp32 else cmi.PREC_FP64)
    ctx.set_engine(cmi.ENGINE_TILES if fp32 else cmi.ENGINE_WALK)
    ctx.set_kernel_timing(False)
    return ctx


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "buffer":
        n, x, s["sub"], _, _, _, s["p"] = _buffer_inputs(case, seed)
        nsub = (case["nsub"],) * 3
        s["ctx"] = _context(n.shape, nsub, "fp64")
        s["ctx"].set_fields(_host(_to_subgrids(n, nsub)), _host(_to_subgrids(x, nsub)))
    elif kind == "list":
        n, x, s["p"], s["start"] = _list_inputs(case, seed)
        nsub = _shape(case)[1]
        s["ctx"] = _context(n.shape, nsub, case["precision"])
        s["ctx"].set_fields(_host(_to_subgrids(n, nsub)), _host(_to_subgrids(x, nsub)))
    elif kind == "solve":
        n, pos, lum, s["seed"] = _solve_inputs(case, seed)
        nsub = _shape(case)[1]
        s["ctx"] = _context(n.shape, nsub, case["precision"])
        s["ctx"].set_sources(pos, lum)
        s["ctx"].set_reemission(case["reemit"])
        s["n"] = _host(_to_subgrids(n, nsub))
        s["x0"] = np.full(s["n"].size, X0)
        s["L"] = s["ctx"].total_luminosity()
    elif kind == "set":
        probs, s["seed"] = _set_inputs(case, seed)
        s["batch"] = cmi.Batch([[0, 0, 0] + [p[0]["side"]] * 3 for p in probs],
                               [[p[0]["n"]] * 3 for p in probs])
        for q, (_, _, pos, lum) in enumerate(probs):
            s["batch"].set_sources(q, pos, lum)
        s["n"] = [_host(p[1]) for p in probs]
        s["x0"] = [np.full(a.size, X0) for a in s["n"]]
        s["packets"] = np.array([p[0]["packets"] for p in probs], np.uint64)
    elif kind == "net":
        s["net"], _ = _new_net(seed)
        s["f"], s["t"] = _net_samples(case["batch"], (case["d"], case["h"], case["w"]), seed)
    elif kind == "train":
        s["net"], s["params"] = _new_net(seed)
        s["net"].add_samples(*_net_samples(case["samples"], (case["sample"],) * 3, seed))
        s["seed"] = seed + 17
    else:
        n, pos, lum, s["seed"] = _warm_inputs(case, seed)
        s["prob"] = warmstart.Problem(np.array(BOX), _host(n), pos, lum, nsub=case["nsub"])
        s["net"] = warmstart.load_net(NET_FILE)
        s["net"].pass_packets = case["packets"]
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "buffer":
        ctx = s["ctx"]
        if case["walk"] == "interact":
            ctx.reset_intensity()
        p, exits, crossings = ctx.interact_batch(s["sub"], case["entry"], s["p"], case["walk"])
        out = {"pos": p["pos"], "tau": p["tau"], "exits": exits, "crossings": crossings}
        if case["walk"] == "interact":
            out["J"] = ctx.get_fields()[0]
        return out
    if kind == "list":
        ctx = s["ctx"]
        ctx.reset_intensity()
        p, status, crossings, _, _ = ctx.transport_packets(s["p"], s["start"])
        return {"pos": p["pos"], "tau": p["tau"], "status": status, "crossings": crossings,
                "J": ctx.get_fields()[0]}
    if kind == "solve":
        ctx = s["ctx"]
        ctx.set_fields(s["n"], s["x0"])
        ctx.reset_intensity()
        l1, counts = [], []
        for it in range(case["iterations"]):
            st = ctx.transport(case["packets"], s["seed"], it, SIGMA)
            l1.append(ctx.update_ionization(s["L"], case["packets"], ALPHA, form=1))
            counts.append([st["crossings"], st["absorbed"], st["escaped"], st["reemitted"]])
        return {"x": ctx.get_fields()[1], "l1": np.array(l1), "counts": np.array(counts)}
    if kind == "set":
        b = s["batch"]
        for q in range(b.nprob):
            b.set_fields(q, s["n"][q], s["x0"][q])
        l1, crossings = [], []
        for it in range(case["iterations"]):
            r = b.iteration(s["packets"], s["seed"], it, ALPHA, form=1)
            l1.append(r["l1"])
            crossings.append(r["problem_crossings"].astype(np.int64))
        return {"x": [b.get_fields(q)[1] for q in range(b.nprob)], "l1": np.array(l1),
                "crossings": np.array(crossings)}
    if kind == "net":
        if case["backward"]:
            loss, grad = s["net"].loss_and_grad(s["f"], s["t"])
            return {"loss": loss, "grad": grad}
        return [s["net"].predict(s["f"][k]) for k in range(case["batch"])]
    if kind == "train":
        net = s["net"]
        net.set_params(s["params"])
        losses = net.train(case["steps"], case["batch"], [case["crop"]] * 3, 1e-3, s["seed"])
        return {"losses": losses, "params": net.params()}
    prob, net = s["prob"], s["net"]
    prob.reset()
    packets = warmstart.net_start(prob, net, s["seed"])
    net.warm_start(prob.ctx, prob.L, packets)
    return {"x": prob.ctx.get_fields()[1]}


# ---------------------------------------------------------------------------
# The least work of a pass
# ---------------------------------------------------------------------------
def _conv_flops(voxels):
    return 2.0 * 27 * voxels * sum(cin * cout for cin, cout, _ in LAYERS)


def work(case):
    """Fields and packets read and written once; about 12 operations per cell
    crossing, with an expected 0.45 lattice edges of crossings per packet."""
    kind = case["kind"]
    if kind == "buffer":
        return {"bytes": case["packets"] * (144 + 8) + 24 * case["cells"] ** 3,
                "flops": 12 * 0.6 * case["cells"] * case["packets"]}
    if kind in ("list", "solve"):
        cells = case["nx"] * case["ny"] * case["nz"]
        crossings = 0.45 * cells ** (1 / 3) * case["packets"]
        if kind == "list":
            return {"bytes": case["packets"] * (2 * 72 + 12) + 24 * cells,
                    "flops": 12 * crossings}
        return {"bytes": 24 * cells + 44 * cells * case["iterations"],
                "flops": 12 * crossings * case["iterations"] / (1 - case["reemit"])}
    if kind == "set":
        spec = _set_spec(case)
        cells = sum(p["n"] ** 3 for p in spec)
        crossings = sum(0.45 * p["n"] * p["packets"] for p in spec)
        return {"bytes": 24 * cells + 44 * cells * case["iterations"],
                "flops": 12 * crossings * case["iterations"]}
    if kind == "net":
        v = case["batch"] * case["d"] * case["h"] * case["w"]
        return {"bytes": 12 * v, "flops": (3 if case["backward"] else 1) * _conv_flops(v)}
    if kind == "train":
        v = case["batch"] * case["crop"] ** 3
        return {"bytes": 12 * v * case["steps"], "flops": 3 * _conv_flops(v) * case["steps"]}
    cells = case["cells"] ** 3
    return {"bytes": 24 * cells + 5 * 44 * cells,
            "flops": _conv_flops(cells) + 5 * 12 * 0.45 * case["cells"] * case["packets"]}


# ---------------------------------------------------------------------------
# The same results in 64 bits
# ---------------------------------------------------------------------------
def _philox(c, seed):
    """Philox4x32-10 of four int64 tensors holding 32-bit words."""
    mask = 0xFFFFFFFF
    k0, k1 = seed & mask, (seed >> 32) & mask

    def mul(m, v):
        lo, hi = m * (v & 0xFFFF), m * (v >> 16)
        mid = hi + (lo >> 16)
        return mid >> 16, ((mid & 0xFFFF) << 16) | (lo & 0xFFFF)

    for r in range(10):
        h0, l0 = mul(0xD2511F53, c[0])
        h1, l1 = mul(0xCD9E8D57, c[2])
        c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
        k0, k1 = (k0 + 0x9E3779B9) & mask, (k1 + 0xBB67AE85) & mask
    return c


def _uniform(hi, lo):
    return ((((hi >> 5) << 26) | (lo >> 6)).double() + 0.5) * 2.0 ** -53


def _split(lum, packets, seed, iteration):
    """Packets of each source: the floor of its share, the rest one each to
    the sources of the smallest keys."""
    total = 0.0
    for v in lum:
        total += float(v)
    counts = [int(float(v) / total * float(packets)) for v in lum]
    while sum(counts) > packets:
        counts[counts.index(max(counts))] -= 1
    i = torch.arange(len(counts), dtype=torch.int64)
    o = _philox([i, torch.zeros_like(i), torch.full_like(i, iteration),
                 torch.full_like(i, 0x5EED)], seed)
    order = torch.sort(_uniform(o[0], o[1]), stable=True)[1].tolist()
    for r in range(packets - sum(counts)):
        counts[order[r % len(counts)]] += 1
    return counts


def _emit(pos, counts, first, count, seed, iteration, problem=0):
    dev = _device()
    k = torch.arange(first, first + count, dtype=torch.int64, device=dev)
    c = [k & 0xFFFFFFFF, (k >> 32) ^ (problem << 20), torch.full_like(k, iteration)]
    r0 = _philox(c + [torch.zeros_like(k)], seed)
    r1 = _philox(c + [torch.ones_like(k)], seed)
    cost = 2.0 * _uniform(r0[0], r0[1]) - 1.0
    phi = 2.0 * math.pi * _uniform(r0[2], r0[3])
    sint = torch.sqrt((1.0 - cost * cost).clamp(min=0.0))
    d = torch.stack([sint * torch.cos(phi), sint * torch.sin(phi), cost])
    cum = torch.cumsum(torch.tensor(counts, device=dev), 0)
    src = torch.searchsorted(cum, k, right=True).clamp(max=len(counts) - 1)
    p = torch.from_numpy(np.ascontiguousarray(pos.T)).to(dev)[:, src]
    return p, d, -torch.log(_uniform(r1[0], r1[1]))


def _walk(lo, cell, shape, kappa, p, d, tau, J, stop=True):
    """Packets (3, n) through a lattice of opacities (per m): adds the path
    lengths to J (flat) and returns the final positions, the optical depth
    left on entering the last cell and after the whole of it (of the whole
    path, summed, without `stop`).  The sums are 64-bit integers of 2^-34 of
    a cell edge: a source's cell gets every one of its packets, and integer
    adds stay fast on one address."""
    dev = p.device
    unit = 2.0 ** 34 / max(cell)
    path = torch.zeros(J.numel(), dtype=torch.int64, device=dev)
    lo_t = torch.tensor(lo, dtype=torch.float64, device=dev)[:, None]
    cs = torch.tensor(cell, dtype=torch.float64, device=dev)[:, None]
    nc = torch.tensor(shape, dtype=torch.int64, device=dev)[:, None]
    stride = torch.tensor([shape[1] * shape[2], shape[2], 1], device=dev)[:, None]
    count = p.shape[1]
    out_p = p.clone()
    out_in = tau.clone()
    out_done = tau.clone()
    idx = torch.minimum(((p - lo_t) / cs).long(), nc - 1).clamp(min=0)
    up = d > 0
    tm = torch.where(d == 0, math.inf, (lo_t + (idx + up) * cs - p) / d)
    td = torch.where(d == 0, math.inf, cs / d.abs())
    left = torch.where(up, nc - idx, idx + 1)
    inc = torch.where(up, stride, -stride)
    st = {"tm": tm, "td": td, "left": left, "inc": inc, "cell": (idx * stride).sum(0),
          "t": torch.zeros_like(tau), "tau": tau.clone(), "id": torch.arange(count, device=dev),
          "live": torch.ones(count, dtype=torch.bool, device=dev)}
    del idx, up, tm, td, left, inc
    step = 0
    while st["id"].numel():
        ax = st["tm"].argmin(0, keepdim=True)
        tn = st["tm"].gather(0, ax)[0]
        seg = tn - st["t"]
        kap = kappa[st["cell"]]
        dtau = seg * kap
        ends = st["live"] & (dtau >= st["tau"]) if stop else torch.zeros_like(st["live"])
        s = torch.where(ends, st["tau"] / kap, seg) if stop else seg
        path.index_add_(0, st["cell"], torch.where(st["live"], s * unit, 0.0).round().long())
        st["left"].scatter_add_(0, ax, torch.full_like(ax, -1))
        gone = st["live"] & ~ends & (st["left"].gather(0, ax)[0] == 0)
        rest = st["tau"] - dtau if stop else st["tau"] + dtau
        over = ends | gone
        which = over.nonzero()[:, 0]
        ids = st["id"][which]
        out_p[:, ids] += (st["t"] + s)[which] * d[:, ids]
        out_in[ids] = torch.where(ends, st["tau"], rest)[which]
        out_done[ids] = rest[which]
        st["live"] &= ~over
        st["tau"] = rest
        st["t"] = tn
        st["cell"] = torch.where(st["live"], st["cell"] + st["inc"].gather(0, ax)[0], 0)
        st["tm"].scatter_add_(0, ax, st["td"].gather(0, ax))
        step += 1
        if step % 8 == 0:
            keep = st["live"].nonzero()[:, 0]
            if keep.numel() < 0.9 * st["id"].numel():
                st = {k: (v[:, keep] if v.dim() == 2 else v[keep]) for k, v in st.items()}
    J += path.double() / unit
    return out_p, out_in, out_done


def _balance(path, n, lum, packets, volume):
    """x_n of the path lengths (m) through cells of density n."""
    jH = lum / packets / volume * path * SIGMA
    b = jH / (n * ALPHA)
    x = 2.0 / (2.0 + b + torch.sqrt(b * (b + 4.0)))
    return torch.where(jH > 0, x, torch.ones_like(x))


def _iterate(lo, side, n, pos, lum, packets, seed, iterations, problem=0, split_seed=None):
    """Plain iterations from x_n = 1e-6 (iterations: the emission's iteration
    numbers); returns x_n and the mean changes."""
    shape = tuple(n.shape)
    cell = [side[a] / shape[a] for a in range(3)]
    flat = n.reshape(-1)
    x = torch.full_like(flat, X0)
    l1 = []
    total = float(np.sum(lum))
    for it in iterations:
        counts = _split(lum, packets, seed if split_seed is None else split_seed, it)
        J = torch.zeros_like(flat)
        kappa = SIGMA * flat * x
        for first in range(0, packets, 10000000):
            p, d, tau = _emit(pos, counts, first, min(10000000, packets - first), seed, it,
                              problem)
            _walk(lo, cell, shape, kappa, p, d, tau, J)
        new = _balance(J, flat, total, packets, cell[0] * cell[1] * cell[2])
        l1.append(float((new - x).abs().sum() / flat.numel()))
        x = new
    return x.reshape(shape), l1


def _normalised(f, mean, scale):
    f = torch.from_numpy(np.ascontiguousarray(f)).to(_device(), torch.float64)
    m = torch.tensor(np.asarray(mean, np.float64), device=f.device)
    return (f - m) * torch.tensor(np.asarray(scale, np.float64), device=f.device)


def _network(params, x, dilation):
    """(B, D, H, W, 2) -> (B, D, H, W): each layer as one product per plane
    with the 27 shifted inputs side by side, 32 planes at a time."""
    off = 0
    B, D, H, W = x.shape[:4]
    for l, (cin, cout, pad) in enumerate(LAYERS):
        w = params[off:off + 27 * pad * 32].reshape(27, pad, 32)[:, :cout, :cin]
        w = w.permute(0, 2, 1).reshape(27 * cin, cout)
        off += 27 * pad * 32
        b = params[off:off + pad][:cout]
        off += pad
        k = dilation[l]
        xp = torch.nn.functional.pad(x, (0, 0, k, k, k, k, k, k))
        planes = []
        for s in range(B):
            for z in range(0, D, 32):
                m = min(32, D - z)
                cols = torch.cat([xp[s, z + i:z + i + m, j:j + H, n:n + W]
                                  for i in (0, k, 2 * k) for j in (0, k, 2 * k)
                                  for n in (0, k, 2 * k)], dim=-1)
                y = torch.bmm(cols.reshape(m, H * W, 27 * cin),
                              w.expand(m, 27 * cin, cout).contiguous()) + b
                planes.append(torch.relu(y) if l < 3 else y)
        x = torch.cat(planes).reshape(B, D, H, W, cout)
    return x[..., 0]


def _loss(z, t):
    e = z - t
    return (torch.where(e > 0, 4.0, 1.0) * e * e).mean()


def exact(case, seed):
    with torch.no_grad():
        return _exact(case, seed)


def _exact(case, seed):
    kind = case["kind"]
    dev = _device()
    if kind == "buffer":
        n, x, sub, s, lo, side, p = _buffer_inputs(case, seed)
        e = case["cells"]
        cut = tuple(slice(int(v) * e, (int(v) + 1) * e) for v in s)
        kappa = (SIGMA * n * x)[cut].reshape(-1)
        J = torch.zeros_like(kappa)
        stop = case["walk"] != "optical_depth"
        pos, _, done = _walk(lo, [side / e] * 3, (e,) * 3, kappa,
                             torch.from_numpy(p["pos"].T.copy()).to(dev),
                             torch.from_numpy(p["dir"].T.copy()).to(dev),
                             torch.from_numpy(p["tau"].copy()).to(dev), J, stop)
        out = {"pos": pos.t(), "tau": done, "exits": None, "crossings": None}
        if case["walk"] == "interact":
            whole = torch.zeros(case["nsub"] ** 3, e ** 3, dtype=torch.float64, device=dev)
            whole[sub] = SIGMA * J
            out["J"] = whole.reshape(-1)
        return out
    if kind == "list":
        n, x, p, _ = _list_inputs(case, seed)
        ncell, nsub = _shape(case)
        J = torch.zeros_like(n).reshape(-1)
        pos, entering, done = _walk(BOX[:3], [BOX[3 + a] / ncell[a] for a in range(3)], ncell,
                                    (SIGMA * n * x).reshape(-1),
                                    torch.from_numpy(p["pos"].T.copy()).to(dev),
                                    torch.from_numpy(p["dir"].T.copy()).to(dev),
                                    torch.from_numpy(p["tau"].copy()).to(dev), J)
        # an absorbed packet comes back with the depth left on entering its
        # last cell (production engine) or after all of it (reference)
        return {"pos": pos.t(), "tau": entering if case["precision"] == "fp32" else done,
                "status": None, "crossings": None,
                "J": _to_subgrids(SIGMA * J.reshape(ncell), nsub)}
    if kind == "solve":
        # reemission draws are keyed by the walk's own roundings: no 64-bit
        # value; the largest solves take too long
        if case["reemit"] > 0 or case["packets"] * case["iterations"] > 1.6e8:
            return None
        n, pos, lum, key = _solve_inputs(case, seed)
        x, l1 = _iterate(BOX[:3], BOX[3:], n, pos, lum, case["packets"], key,
                         range(case["iterations"]))
        return {"x": _to_subgrids(x, _shape(case)[1]), "l1": np.array(l1), "counts": None}
    if kind == "set":
        if case["problems"] * case["iterations"] > 48:
            return None  # too long
        probs, key = _set_inputs(case, seed)
        xs, l1 = [], []
        for q, (s, n, pos, lum) in enumerate(probs):
            x, l = _iterate((0.0, 0.0, 0.0), (s["side"],) * 3, n, pos, lum, s["packets"], key,
                            range(case["iterations"]), q, key ^ q)
            xs.append(x)
            l1.append(l)
        return {"x": xs, "l1": np.array(l1).T, "crossings": None}
    if kind == "net":
        f, t = _net_samples(case["batch"], (case["d"], case["h"], case["w"]), seed)
        x = _normalised(f, NET_MEAN, NET_SCALE)
        p = torch.from_numpy(_net_params(seed)).to(dev, torch.float64)
        if not case["backward"]:
            return [z * NET_OUT for z in _network(p, x, NET_DILATION)]
        with torch.enable_grad():
            p.requires_grad_(True)
            loss = _loss(_network(p, x, NET_DILATION),
                         torch.from_numpy(t).to(dev, torch.float64) / NET_OUT)
            grad, = torch.autograd.grad(loss, p)
        return {"loss": float(loss), "grad": grad}
    if kind == "train":
        f, t = _net_samples(case["samples"], (case["sample"],) * 3, seed)
        f = _normalised(f, NET_MEAN, NET_SCALE)
        t = torch.from_numpy(t).to(dev, torch.float64) / NET_OUT
        p = torch.from_numpy(_net_params(seed)).to(dev, torch.float64)
        m, v, losses = torch.zeros_like(p), torch.zeros_like(p), []
        c, room = case["crop"], case["sample"] - case["crop"] + 1
        for s in range(case["steps"]):
            xs, ts = [], []
            for b in range(case["batch"]):
                r = _philox([torch.tensor([w]) for w in (s, b, s, 0x7A1E)], seed + 17)
                k, i, j, l = (int(r[0]) % case["samples"], int(r[1]) % room, int(r[2]) % room,
                              int(r[3]) % room)
                xs.append(f[k, i:i + c, j:j + c, l:l + c])
                ts.append(t[k, i:i + c, j:j + c, l:l + c])
            with torch.enable_grad():
                q = p.clone().requires_grad_(True)
                loss = _loss(_network(q, torch.stack(xs), NET_DILATION), torch.stack(ts))
                g, = torch.autograd.grad(loss, q)
            losses.append(float(loss))
            m = 0.9 * m + 0.1 * g
            v = 0.999 * v + 0.001 * g * g
            p = p - 1e-3 * (m / (1 - 0.9 ** (s + 1))) / (
                torch.sqrt(v / (1 - 0.999 ** (s + 1))) + 1e-8)
        return {"losses": np.array(losses), "params": p}
    # warm: the start rule is a threshold on the predicted logit, which the
    # network's BF16 roundings move cells across; the passes and the network
    # have their values in the other kinds
    return None
