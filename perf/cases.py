"""Performance cases of the colony step: what a user's program runs through the public entry points.

A pass of the stepping cases is one output frame: `steps` calls' worth of `mdStep` on the resident
colony (one `HipMD.step`), the drain check where the colony is open, and the download that the frame
writers and analysis read.  The training case is a block of Adam steps and the read-back of the
weights; the surrogate case a block of judged macro-steps and the download.

Families and what they stand for:
  sc2d       the 2D periodic soft-core colony of two-disc cells (motility, harmonic bond, FDT
             noise): the small colonies most runs consist of, where latency and launches count
  heun       two-disc FENE cells with Wiener noise under the stochastic Heun integrator
  theta      a single-disc Hertz colony with the theta cell cycle and divisions
  channel    a growing two-disc Hertz colony between channel walls, with divisions and drain
  bulk       the 3D mixed LJ / soft-core bulk: FP64 (parity mode), FP32 with the default stencil
             kernels, FP32 with one- and two-level neighbour lists (the largest runs)
  batch      an ensemble of growing soft-core colonies of uneven sizes, one launch for all
  surrogate  judged surrogate macro-steps on the 3D bulk, one-level lists
  train      Adam steps of the surrogate's network

`exact` restates each family in 64 bits with plain torch (own neighbour search, counter RNG, laws,
network), on the same inputs.
"""
import math

import numpy as np
import torch

from cil_cuda_amd import abi, configs
from cil_cuda_amd.colony import Colony, HipBatch, HipMD

F64, I64 = torch.float64, torch.int64


# ------------------------------------------------------------------------------------------
# Cases
# ------------------------------------------------------------------------------------------
def listed():
    return [
        # a colony of the first divisions of a run: nothing but latency
        {"name": "sc2d_150", "family": "sc2d", "n": 150, "steps": 500, "fp32": False, "skin": 0.0},
        # the 2000-cell colony in a 64 x 64 box, the everyday plain run in FP64
        {"name": "sc2d_2000", "family": "sc2d", "n": 2000, "steps": 500, "fp32": False, "skin": 0.0},
        # the reference's other integrator (two force passes per step)
        {"name": "heun_1100", "family": "heun", "n": 1100, "steps": 250},
        # the size of the reference's seeded single-disc run at its last frame
        {"name": "theta_934", "family": "theta", "n": 934, "steps": 500},
        # a channel colony on its way to 65,536 cells, FP64
        {"name": "channel_9000", "family": "channel", "n": 9000, "steps": 200},
        # parity-mode bulk of an odd size
        {"name": "bulk_fp64_30011", "family": "bulk", "n": 30011, "steps": 100, "mode": "fp64"},
        # FP32 without lists: what set-ups without set_neighbour_list run
        {"name": "bulk_stencil_131071", "family": "bulk", "n": 131071, "steps": 100, "mode": "stencil"},
        # one-level lists at the size of the CPU-baseline sample
        {"name": "bulk_list_131072", "family": "bulk", "n": 131072, "steps": 400, "mode": "list"},
        # the benchmark's workload: two-level lists, 1,048,576 particles
        {"name": "bulk_two_level_1m", "family": "bulk", "n": 1 << 20, "steps": 500, "mode": "two_level"},
        # a parameter scan: 32 colonies of 300-4000 cells
        {"name": "batch_32", "family": "batch", "colonies": 32, "lo": 300, "hi": 4000, "steps": 200},
        # 16 macro-steps, the last one judged
        {"name": "surrogate_262144", "family": "surrogate", "n": 1 << 18, "macro": 16},
        # a block of the training loop at its usual batch size
        {"name": "train_8192", "family": "train", "samples": 1 << 16, "batch": 8192, "adam": 32},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    fam = rng.choice(["sc2d", "sc2d", "heun", "theta", "channel", "bulk", "bulk", "bulk", "batch", "surrogate", "train"])
    if fam == "sc2d":
        fp32 = rng.random() < 0.5
        skin = rng.choice([0.0, 0.2, 0.3]) if fp32 else 0.0
        return {"family": fam, "n": _log_int(rng, 60, 20000), "steps": rng.randint(100, 500), "fp32": fp32, "skin": skin}
    if fam == "heun":
        return {"family": fam, "n": _log_int(rng, 60, 5000), "steps": rng.randint(60, 300)}
    if fam == "theta":
        return {"family": fam, "n": _log_int(rng, 60, 6000), "steps": rng.randint(100, 500)}
    if fam == "channel":
        return {"family": fam, "n": _log_int(rng, 300, 20000), "steps": rng.randint(50, 200)}
    if fam == "bulk":
        mode = rng.choice(["fp64", "stencil", "list", "two_level", "two_level"])
        hi = {"fp64": 60000, "stencil": 260000, "list": 500000, "two_level": 1000000}[mode]
        return {"family": fam, "n": _log_int(rng, 4000, hi), "steps": rng.randint(50, 200), "mode": mode}
    if fam == "batch":
        return {"family": fam, "colonies": rng.randint(3, 40), "lo": rng.randint(40, 400), "hi": rng.randint(800, 5000),
                "steps": rng.randint(60, 200)}
    if fam == "surrogate":
        return {"family": fam, "n": _log_int(rng, 20000, 400000), "macro": rng.choice([8, 16, 24])}
    return {"family": fam, "samples": _log_int(rng, 8000, 100000), "batch": _log_int(rng, 256, 16384),
            "adam": rng.randint(8, 32)}


# ------------------------------------------------------------------------------------------
# Inputs (from the seed alone; numpy and torch, none of the library's kernels)
# ------------------------------------------------------------------------------------------
def _grid2(n, width, a, rng, jitter):
    """n centres of a jittered square lattice of `width` columns of spacing a."""
    k = np.arange(n)
    return (np.stack([k % width, k // width], axis=1) + 0.5) * a + rng.uniform(-jitter, jitter, (n, 2))


def _two_disc(col, s, c, u, half, L):
    sp = col.species[s]
    n = c.shape[0]
    for e, sg in ((0, -1.0), (1, 1.0)):
        x = c + sg * half * u
        sp["pos"][:n, e] = np.mod(x, L) if L is not None else x


def _units(n, rng):
    a = rng.uniform(0, 2 * math.pi, n)
    return np.stack([np.cos(a), np.sin(a)], axis=1)


def _sc2d(n, seed, fp32):
    """configs.plain_2d_sc's parameters and density (2000 cells in 64 x 64) at any size."""
    rng = np.random.default_rng(seed)
    side = int(math.ceil(math.sqrt(n)))
    L = side * 1.431
    p, box, _ = configs.plain_2d_sc(n_cells=1, L=L, seed=seed % 1000 + 1,
                                    precision=abi.PREC_FP32 if fp32 else abi.PREC_FP64)
    col = Colony(2, 2, [n], ncells=[n])
    _two_disc(col, 0, _grid2(n, side, 1.431, rng, 0.15), _units(n, rng), 0.25, L)
    s = col.species[0]
    s["sigma"][:n] = rng.uniform(0.9, 1.1, (n, 2))
    s["rest_len"][:n] = 0.5
    s["state"][:n] = abi.CS_CRAWLING
    return p, box, col


def _heun(n, seed):
    """configs.binary_2d_fene's cells (FENE bond, rss-scaled motility, Wiener noise), not dividing."""
    rng = np.random.default_rng(seed)
    side = int(math.ceil(math.sqrt(n)))
    L = side * 1.63
    p, box, _ = configs.binary_2d_fene(n_cells=1, L=L, seed=seed % 1000 + 1, integrator=abi.INT_HEUN, capacity=4)
    p.division = abi.DIV_NONE
    col = Colony(2, 2, [n], ncells=[n])
    _two_disc(col, 0, _grid2(n, side, 1.63, rng, 0.15), _units(n, rng), 0.3, L)
    s = col.species[0]
    s["sigma"][:n] = [0.85, 0.95]
    s["state"][:n] = abi.CS_CRAWLING
    return p, box, col


def _theta(n, seed):
    """configs.theta_2d_hz with the time step and cycle span of the reference's seeded run."""
    rng = np.random.default_rng(seed)
    side = int(math.ceil(math.sqrt(n)))
    L = side * 1.6 + 1.0
    dt = 1e-5
    p, box, _ = configs.theta_2d_hz(n_cells=1, L=max(L, 8.0), seed=seed % 1000 + 1, dt=dt, capacity=4)
    sp = p.species[0]
    sp.division_tau.mu, sp.division_tau.sigma = 1.0, 0.1
    sp.cycle_tau_p = 0.1 / dt
    col = Colony(2, 1, [4 * n + 64], ncells=[n])
    s = col.species[0]
    s["pos"][:n, 0] = _grid2(n, side, 1.6, rng, 0.35)
    th = rng.uniform(0, 1, n)
    s["sigma"][:n, 0] = s["sigma_t"][:n] = np.sqrt(4 * np.exp2(th) * 0.9 / math.pi)
    s["vel"][:n, 0] = rng.normal(0, 0.1, (n, 2))
    s["state"][:n] = abi.CS_DIVIDING
    s["rho"][:n] = rng.uniform(0.7, 1.0, n)
    s["theta"][:n] = th
    s["ang_vel"][:n] = 1.0 / np.maximum(np.rint(rng.lognormal(0, 0.1, n) / dt), 1)
    return p, box, col


def _channel(n, seed):
    """configs.channel_2d_hz part way through its growth: cells of every length in the 40-wide channel."""
    rng = np.random.default_rng(seed)
    a, width = 2.3, 40.0
    rows = -(-n // 17)
    length = rows * a + 40.0
    p, box, _ = configs.channel_2d_hz(width=width, length=length, seed=seed % 1000 + 1, tau=5.0, kT=0.01, capacity=4)
    col = Colony(2, 2, [2 * n + 64], ncells=[n])
    c = _grid2(n, 17, a, rng, 0.2) + np.array([0.45, 20.0])
    l = rng.uniform(0.5, 2.0, n)
    ang = rng.normal(0.5 * math.pi, 0.6, n)
    u = np.stack([np.cos(ang), np.sin(ang)], axis=1)
    _two_disc(col, 0, c, u, 0.5 * l[:, None], None)
    s = col.species[0]
    s["pos"][:n, :, 0] = np.clip(s["pos"][:n, :, 0], 0.7, width - 0.7)
    s["sigma"][:n] = 1.0 + 0.05 * rng.normal(0, 1, (n, 2))
    s["rest_len"][:n] = l
    s["state"][:n] = abi.CS_CRAWLING
    return p, box, col


def _bulk(n, seed, mode, kT=0.05):
    """configs.bulk_3d_mixed's density, diameters, types and laws; overlaps pushed out in 64 bits."""
    p, box, _ = configs.bulk_3d_mixed(n=64, seed=seed % 1000 + 1, kT=kT,
                                      precision=abi.PREC_FP64 if mode == "fp64" else abi.PREC_FP32)
    L = configs.bulk_3d_box_length(n)
    for d in range(3):
        box.length[d] = L
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    side = int(math.ceil((n / 4) ** (1 / 3)))  # a perturbed FCC lattice with vacancies
    sites = torch.randperm(4 * side ** 3, generator=g, device=dev)[:n].sort().values
    cell, b = sites // 4, sites % 4
    base = torch.tensor([[0, 0, 0], [0.5, 0.5, 0], [0.5, 0, 0.5], [0, 0.5, 0.5]], dtype=F64, device=dev)
    x = torch.stack([cell // (side * side), cell // side % side, cell % side], 1).to(F64) + base[b] + 0.25
    x = x * (L / side) + 0.2 * torch.randn((n, 3), generator=g, device=dev, dtype=F64)
    sig = torch.exp(-0.5 * math.log(1.01) + math.sqrt(math.log(1.01)) * torch.randn(n, generator=g, device=dev, dtype=F64))
    spec = (torch.rand(n, generator=g, device=dev) < 0.5)
    x = torch.remainder(x, L)
    for _ in range(8):
        i, j = _pairs(x, [L] * 3, [1] * 3, 1.35)
        for _ in range(10):  # overlaps pushed apart; integer sums, so every run makes the same bits
            d = _min_image(x[j] - x[i], [L] * 3, [1] * 3)
            r = d.square().sum(1).sqrt()
            gap = torch.where(spec[i] | spec[j], 0.45, 0.495) * (sig[i] + sig[j]) - r
            w = (0.35 * gap.clamp(min=0.0) / r.clamp(min=1e-6))[:, None] * d
            q = torch.round(w * 2.0 ** 40).to(I64)
            acc = torch.zeros((n, 3), dtype=I64, device=dev)
            acc.index_add_(0, j, q)
            acc.index_add_(0, i, -q)
            x = torch.remainder(x + acc.to(F64) * 2.0 ** -40, L)
    x, sig, spec = x.cpu().numpy(), sig.cpu().numpy(), spec.cpu().numpy()
    n0 = int((~spec).sum())
    col = Colony(3, 1, [n0, n - n0], ncells=[n0, n - n0])
    for s, m in ((0, ~spec), (1, spec)):
        col.species[s]["pos"][:, 0] = x[m]
        col.species[s]["sigma"][:, 0] = sig[m]
    return p, box, col


def _ensemble(case, seed):
    """Growing soft-core colonies of uneven sizes, each with its own seed, motility, kT and growth."""
    rng = np.random.default_rng(seed)
    out = []
    for c in range(case["colonies"]):
        n = int(round(case["lo"] * (case["hi"] / case["lo"]) ** ((c * 0.618034) % 1.0)))
        side = int(math.ceil(math.sqrt(n)))
        L = side * 2.1
        p, box, _ = configs.plain_2d_sc(n_cells=1, L=L, seed=1000 + c, kT=rng.uniform(0.001, 0.05),
                                        motility=rng.uniform(0.0, 0.5), precision=abi.PREC_FP32)
        sp = p.species[0]
        sp.growth_rate, sp.l_div, sp.l_birth, sp.sigma_jitter = rng.uniform(0.02, 0.08), 2.0, 0.5, 0.05
        p.division = abi.DIV_LINEAR_GROWTH
        col = Colony(2, 2, [3 * n + 64], ncells=[n])
        _two_disc(col, 0, _grid2(n, side, 2.1, rng, 0.2), _units(n, rng), 0.25, L)
        s = col.species[0]
        s["sigma"][:n] = rng.uniform(0.9, 1.1, (n, 2))
        s["rest_len"][:n] = rng.uniform(0.5, 2.0, n)
        s["state"][:n] = abi.CS_CRAWLING
        out.append((p, box, col))
    return out


SETTLE = 64  # plain steps before the first macro-step, as a run equilibrates before it is judged


def _weights(seed, out=1.0):
    """Network parameters (W1, b1, W2, b2, W3, b3) uniform in +-1 / sqrt(fan_in), the last layer's times `out`
    (0.1: corrections of the size a trained network makes)."""
    rng = np.random.default_rng(seed)
    return [(g * rng.uniform(-1, 1, s) / math.sqrt(f)).astype(np.float32)
            for s, f, g in (((128, 72), 72, 1.0), ((128,), 72, 1.0), ((128, 128), 128, 1.0), ((128,), 128, 1.0),
                            ((3, 128), 128, out), ((3,), 128, out))]


def _flat(w):
    return np.concatenate([a.reshape(-1) for a in w])


def _bf16(x):
    return torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).to(torch.bfloat16).to(torch.float32).numpy()


def _samples(n, seed):
    """Training rows with the features' distributions, and corrections a smooth teacher makes of them."""
    rng = np.random.default_rng(seed)
    u = rng.normal(0, 1, (n, 16, 3))
    u /= np.linalg.norm(u, axis=2, keepdims=True)
    m = rng.lognormal(-0.005, 0.1, (n, 16, 1)) + 4.0 * (rng.random((n, 16, 1)) < 0.5)
    gap = 20.0 * np.sort(rng.gamma(2.0, 0.12, (n, 16, 1)), axis=1)
    own = np.stack([rng.lognormal(-0.005, 0.1, n), (rng.random(n) < 0.5).astype(float)], 1)
    X = _bf16(np.concatenate([np.concatenate([u * m, gap], 2).reshape(n, 64), own, rng.normal(0, 0.3, (n, 6))], 1))
    t = np.tanh(X.astype(np.float64) @ rng.normal(0, 0.04, (72, 3))) + 0.05 * rng.normal(0, 1, (n, 3))
    return X, (0.002 * t).astype(np.float32)


def _inputs(case, seed):
    f = case["family"]
    if f == "sc2d":
        return _sc2d(case["n"], seed, case["fp32"])
    if f == "bulk":
        return _bulk(case["n"], seed, case["mode"])
    if f == "surrogate":
        return _bulk(case["n"], seed, "list", kT=0.005)
    return {"heun": _heun, "theta": _theta, "channel": _channel}[f](case["n"], seed)


# ------------------------------------------------------------------------------------------
# A user's program: set-up and one pass
# ------------------------------------------------------------------------------------------
def _start(p, box, col, skin=0.0, inner=0.0):
    md = HipMD(p, box, [sp["capacity"] for sp in col.species])
    md.upload(col)
    if skin:
        md.set_neighbour_list(True, skin, 256, inner_skin=inner)
    md.forces(want=False)
    return md


def prepare(case, seed):
    f = case["family"]
    if f == "batch":
        sets = _ensemble(case, seed)
        members = [_start(*s) for s in sets]
        return {"case": case, "mds": members, "batch": HipBatch(members), "cols": [s[2] for s in sets],
                "ts": [0] * len(sets)}
    if f == "train":
        p, box, col = configs.bulk_3d_mixed(n=512, seed=1)
        md = HipMD(p, box, [sp["capacity"] for sp in col.species])
        md.surrogate_set_samples(*_samples(case["samples"], seed))
        md.mlp_set_params(_flat(_weights(seed + 1)))
        return {"case": case, "md": md, "seed": seed}
    p, box, col = _inputs(case, seed)
    skin, inner = case.get("skin", 0.0), 0.0
    if f == "surrogate" or case.get("mode") == "list":
        skin = 0.3
    elif case.get("mode") == "two_level":
        skin, inner = 0.6, 0.2
    md = _start(p, box, col, skin, inner)
    ts = 0
    if f == "surrogate":
        md.mlp_set_params(_flat(_weights(seed + 1, 0.1)))
        ts = md.step(SETTLE, 0)
    return {"case": case, "md": md, "col": col, "ts": ts}


FIELDS = {"theta": ("sigma", "sigma_t", "theta", "rho", "pressure"), "channel": ("sigma", "rest_len"),
          "batch": ("sigma", "rest_len")}


def _frame(md, col, family):
    md.download(col)
    if family in FIELDS:  # growing colonies: the host arrays at their capacity, and the counts
        s = col.species[0]
        return {"cells": np.array(col.ncells()), **{k: s[k] for k in ("pos", "vel", "frc") + FIELDS[family]}}
    return {k: col.flat(k) for k in ("pos", "vel", "frc")}


def run(state):
    case = state["case"]
    f = case["family"]
    if f == "train":
        losses = state["md"].surrogate_train(case["adam"], batch=case["batch"], lr=1e-3, seed=state["seed"])
        return {"losses": losses, "params": state["md"].mlp_get_params()}
    if f == "batch":
        state["ts"] = state["batch"].step(case["steps"], state["ts"])
        frames = [_frame(m, c, f) for m, c in zip(state["mds"], state["cols"])]
        return {k: np.concatenate([fr[k] for fr in frames]) for k in frames[0]}
    md = state["md"]
    if f == "surrogate":
        state["ts"], _ = md.surrogate_step(case["macro"], state["ts"], judge_every=16, tol=1e-3)
    else:
        state["ts"] = md.step(case["steps"], state["ts"])
    if f == "channel":
        md.check_positions()
    return _frame(md, state["col"], f)


def work(case):
    """Per step: positions read and written and diameters read once (FP64, as the boundary holds them),
    each interacting pair evaluated once; per frame: positions, velocities and forces out."""
    f = case["family"]
    if f == "train":
        b = case["batch"] * case["adam"]
        return {"bytes": b * (144 + 12) + case["adam"] * 26243 * 24, "flops": 3.0 * b * 2 * (72 * 128 + 128 * 128 + 384)}
    if f == "batch":
        n = 2 * case["colonies"] * (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
        d, steps, pairs = 2, case["steps"], 1.5
    elif f == "surrogate":
        d, steps, n, pairs = 3, case["macro"], case["n"], 27.0
    else:
        d = 3 if f == "bulk" else 2
        steps = case["steps"] * (2 if f == "heun" else 1)
        n = case["n"] * (1 if f in ("bulk", "theta") else 2)
        pairs = 11.0 if f == "bulk" else 2.0
    flops = steps * n * (pairs * 30 + 60)
    if f == "surrogate":
        flops += steps * n * 51968.0
    return {"bytes": float(steps * n * (16 * d + 8) + 24 * d * n), "flops": float(flops)}


def tolerance(case):
    """About four times the largest difference seen between summation orders (3 against 2 bins per cut-off)
    and from `exact`, over the frames' steps."""
    f = case["family"]
    if f == "train":  # BF16 operands; Adam moves weights of tiny gradients by whole steps either way
        return {"rel": 5e-3, "max": 0.5}
    if f == "surrogate":
        return {"rel": 5e-4, "max": 0.1}
    if case.get("mode") in ("stencil", "list", "two_level"):
        return {"rel": 1e-4, "max": 0.1}
    if f == "batch" or case.get("fp32"):
        return {"rel": 3e-6, "max": 1e-3}
    return {"rel": 1.2e-10, "max": 1e-7}


# ------------------------------------------------------------------------------------------
# The same in 64 bits with plain torch
# ------------------------------------------------------------------------------------------
def _min_image(d, L, pbc):
    d = d.clone()
    for k in range(d.shape[1]):
        if pbc[k]:
            d[:, k] -= L[k] * torch.round(d[:, k] / L[k])
    return d


def _pairs(x, L, pbc, rmax):
    """Pairs (i, j), each once, closer than rmax."""
    n, D = x.shape
    dev = x.device
    m = [max(1, int(L[d] / rmax)) for d in range(D)]
    if any(pbc[d] and m[d] < 3 for d in range(D)):
        i, j = torch.triu_indices(n, n, 1, device=dev)
        keep = _min_image(x[j] - x[i], L, pbc).square().sum(1) < rmax * rmax
        return i[keep], j[keep]
    bins = torch.stack([(x[:, d] * (m[d] / L[d])).floor().long().clamp(0, m[d] - 1) for d in range(D)], 1)
    key = bins[:, 0]
    for d in range(1, D):
        key = key * m[d] + bins[:, d]
    order = torch.argsort(key, stable=True)
    xs, bs, ks = x[order], bins[order], key[order]
    count = torch.bincount(ks, minlength=math.prod(m))
    start = torch.cumsum(count, 0) - count
    me = torch.arange(n, device=dev)
    out_i, out_j = [], []
    offsets = [()]
    for _ in range(D):
        offsets = [o + (s,) for o in offsets for s in (-1, 0, 1)]
    for o in offsets[len(offsets) // 2:]:  # the bin itself, then half of its neighbours
        ok = torch.ones(n, dtype=torch.bool, device=dev)
        nk = torch.zeros(n, dtype=I64, device=dev)
        for d in range(D):
            b = bs[:, d] + o[d]
            if pbc[d]:
                b = b % m[d]
            else:
                ok &= (b >= 0) & (b < m[d])
                b = b.clamp(0, m[d] - 1)
            nk = nk * m[d] + b
        own = not any(o)
        first = me + 1 if own else start[nk]
        cnt = torch.where(ok, start[nk] + count[nk] - first, torch.zeros_like(first))
        ends = torch.cumsum(cnt, 0)
        for lo in range(0, n, 1 << 18):  # chunks bound the memory of dense boxes
            c = cnt[lo:lo + (1 << 18)]
            total = int(c.sum())
            if not total:
                continue
            a = torch.repeat_interleave(me[lo:lo + (1 << 18)], c, output_size=total)
            q = torch.arange(total, device=dev) - (ends[a] - cnt[a] - (ends[lo] - cnt[lo])) + first[a]
            keep = _min_image(xs[q] - xs[a], L, pbc).square().sum(1) < rmax * rmax
            out_i.append(order[a[keep]])
            out_j.append(order[q[keep]])
    return torch.cat(out_i), torch.cat(out_j)


def _philox(c0, c1, c2, c3, seed):
    """Philox4x32-10 on int64 tensors holding 32-bit words."""
    M = 0xFFFFFFFF
    k0, k1 = seed & M, (seed >> 32) & M
    c0, c1, c2, c3 = (t.clone() if torch.is_tensor(t) else t for t in (c0, c1, c2, c3))
    z = torch.zeros_like(c0)
    c1, c2, c3 = z + c1, z + c2, z + c3
    for _ in range(10):
        p0, p1 = c0 * 0xD2511F53, c2 * 0xCD9E8D57
        c0, c1, c2, c3 = ((p1 >> 32) & M) ^ c1 ^ k0, p1 & M, ((p0 >> 32) & M) ^ c3 ^ k1, p0 & M
        k0, k1 = (k0 + 0x9E3779B9) & M, (k1 + 0xBB67AE85) & M
    return c0, c1, c2, c3


def _u53(lo, hi):
    return (((hi << 32) | lo) >> 11) & ((1 << 53) - 1)


def _uniform2(ids, ts, st, k, seed):
    a, b, c, d = _philox(ids, ts, st, k, seed)
    return _u53(a, b).to(F64) * 2.0 ** -53, _u53(c, d).to(F64) * 2.0 ** -53


def _normal2(ids, ts, st, k, seed):
    a, b, c, d = _philox(ids, ts, st, k, seed)
    u1 = (_u53(a, b) + 1).to(F64) * 2.0 ** -53
    r = torch.sqrt(-2.0 * torch.log(u1))
    t = 2.0 * math.pi * (_u53(c, d).to(F64) * 2.0 ** -53)
    return r * torch.cos(t), r * torch.sin(t)


class _Exact:
    """One species set's colony in 64 bits: state tensors per particle (cell-major) and the step."""

    def __init__(self, p, box, col):
        self.p, self.D, self.nE = p, p.dim, p.species[0].nelem
        dev = torch.device("cuda")
        self.L = [box.length[d] for d in range(self.D)]
        self.pbc = [box.periodic[d] for d in range(self.D)]
        t = lambda k: torch.from_numpy(np.ascontiguousarray(col.flat(k))).to(dev)  # noqa: E731
        self.x = t("pos").reshape(-1, self.D)
        self.v = t("vel").reshape(-1, self.D)
        self.sig = t("sigma").reshape(-1)
        self.cell = {k: t(k) for k in ("sigma_t", "theta", "rho", "ang_vel", "rest_len", "pressure")}
        nc = col.ncells()
        self.key = torch.cat([(s << 28) | torch.arange(c, device=dev) for s, c in enumerate(nc)])
        self.spec = torch.cat([torch.full((c * self.nE,), s, device=dev, dtype=I64) for s, c in enumerate(nc)])
        self.ts, self.phase, self.xref = 0, 0, None
        self.skin = 0.3 if self.D == 3 else 0.25

    # -- pair forces ----------------------------------------------------------------------
    def _cut(self, i, j):
        s = 0.5 * (self.sig[i] + self.sig[j])
        if self.D == 3:
            return torch.where((self.spec[i] == 0) & (self.spec[j] == 0), 2.5 * s, s)
        return s

    def _list(self):
        if self.xref is not None and self.xref.shape == self.x.shape:
            d = _min_image(self.x - self.xref, self.L, self.pbc).square().sum(1).max().sqrt()
            grown = (self.sig - self.sref).max().clamp(min=0.0)
            if float(d + grown * 1.25) < 0.5 * self.skin:
                return
        self.xref, self.sref = self.x.clone(), self.sig.clone()
        smax = float(self.sig.max())
        if self.D == 3:  # the wide search only among species-0 discs, the only long-range pairs
            a = torch.nonzero(self.spec == 0).reshape(-1)
            s0 = float(self.sig[a].max())
            i0, j0 = _pairs(self.x[a], self.L, self.pbc, 2.5 * s0 + self.skin)
            i0, j0 = a[i0], a[j0]
            i1, j1 = _pairs(self.x, self.L, self.pbc, smax + self.skin)
            far = (self.spec[i1] != 0) | (self.spec[j1] != 0)
            i, j = torch.cat([i0, i1[far]]), torch.cat([j0, j1[far]])
        else:
            i, j = _pairs(self.x, self.L, self.pbc, smax + self.skin)
        r = _min_image(self.x[j] - self.x[i], self.L, self.pbc).square().sum(1).sqrt()
        keep = r < self._cut(i, j) + self.skin
        if self.nE == 2:
            keep &= (i // 2) != (j // 2)
        self.i, self.j = i[keep], j[keep]

    def _pair_forces(self):
        self._list()
        i, j, p = self.i, self.j, self.p
        d = _min_image(self.x[j] - self.x[i], self.L, self.pbc)
        r2 = d.square().sum(1)
        r = r2.sqrt()
        si, sj = self.sig[i], self.sig[j]
        s = 0.5 * (si + sj)
        press = None
        if p.law[0][0] == abi.LAW_HZ:
            h = (s - r).clamp(min=0.0)
            E, nu = p.species[0].eps_core[0], p.species[0].sig_well[0]
            f = -h.pow(1.5) / (1.5 * (1 - nu * nu) / E * torch.sqrt(2 / si + 2 / sj))
            if p.pressure:
                ra, rb = 0.5 * si, 0.5 * sj
                a = 2 * torch.sqrt((ra * ra - (ra - (2 * rb * h - h * h) / (2 * (ra + rb - h))) ** 2).clamp(min=0.0))
                press = torch.where(a > 0, -f / a.clamp(min=1e-300), torch.zeros_like(f))
        else:
            y, xi = r - s, p.species[0].sig_well[0]
            f = torch.where((y < 0) & (y > -xi) & (r2 > (s - xi) ** 2), 6.0 * y * (y + xi) / xi ** 3 / r, torch.zeros_like(r))
            if self.D == 3:
                lj = (self.spec[i] == 0) & (self.spec[j] == 0)
                s6 = (s * s / r2) ** 3
                f = torch.where(lj, torch.where(r2 <= 6.25 * s * s, 24.0 * (s6 - 2 * s6 * s6) / r2, torch.zeros_like(r)), f)
        F = torch.zeros_like(self.x)
        fd = f[:, None] * d
        F.index_add_(0, i, fd)
        F.index_add_(0, j, -fd)
        if press is not None:
            pr = torch.zeros_like(self.sig)
            pr.index_add_(0, i, press)
            pr.index_add_(0, j, press)
            self.cell["new_pressure"] = pr
        return F

    def forces(self):
        """Total force at the current state (pair, intra-cell, walls, Wiener noise)."""
        p, sp, D = self.p, self.p.species[0], self.D
        F = self._pair_forces()
        if self.nE == 2:
            X = self.x.view(-1, 2, D)
            d = _min_image(X[:, 1] - X[:, 0], self.L, self.pbc)
            r2 = d.square().sum(1, keepdim=True)
            r = r2.sqrt()
            if sp.spring == abi.SPRING_HARMONIC:
                spring, axis, scf = -sp.k_harm * (r - self.cell["rest_len"][:, None]) / r, d / r, 1.0
            else:
                m = torch.maximum(self.sig.view(-1, 2).max(1, keepdim=True).values, torch.tensor(sp.r2max, device=r.device))
                q = m * sp.spring_ratio
                spring = torch.where(r2 <= q, sp.kappa_push * (r2 - q).abs(),
                                     -sp.kappa / (1 - ((r2 - q) / (m * (1 - sp.spring_ratio))) ** 2))
                axis, scf = d * (sp.rss / r), 2.0
            G = F.view(-1, 2, D)
            G[:, 0] -= sp.motility[0] * axis + spring * d * scf
            G[:, 1] += sp.motility[1] * axis + spring * d * scf
        elif sp.motility[0]:
            vl = self.v.norm(dim=1, keepdim=True)
            still = vl[:, 0] == 0
            if bool(still.any()):  # a disc at rest gets a random direction
                k = torch.nonzero(still).reshape(-1)
                z = torch.stack(_normal2(self.key[k] << 1, self.ts, 5, 0, p.seed), 1)
                self.v[k] = z / z.norm(dim=1, keepdim=True) * 1e-11
                vl = self.v.norm(dim=1, keepdim=True)
            F += sp.motility[0] * self.v / vl
        for w in range(p.nwalls):
            wl = p.walls[w]
            g = (self.x[:, wl.axis] - wl.x0) * (1 if wl.positive else -1) / self.sig
            q = g.clamp(min=0.82)
            i2 = 1 / (q * q)
            i6 = i2 ** 3
            f = torch.where(g <= wl.rcut, wl.epsilon * (2 * i6 - 1) * i6 * i2 / self.sig ** 2, torch.zeros_like(g))
            F[:, wl.axis] += f if wl.positive else -f
        if p.noise == abi.NOISE_CELL_WIENER:
            z = torch.stack(_normal2(self.key, self.ts, 1 + 8 * self.phase, 0, p.seed), 1) * sp.d_noise
            F += sp.zeta[0] * z.repeat_interleave(self.nE, 0)
        self.F = F
        if "new_pressure" in self.cell:
            self.cell["pressure"] = self.cell.pop("new_pressure")

    # -- moves ----------------------------------------------------------------------------
    def _wrap(self, x):
        return torch.stack([torch.remainder(x[:, d], self.L[d]) if self.pbc[d] else x[:, d] for d in range(self.D)], 1)

    def _mobility_dt(self):
        s0 = self.sig.view(-1, self.nE)[:, 0].repeat_interleave(self.nE)
        return (self.p.dt / (self.p.species[0].zeta[0] * math.pi * (s0 / 2) ** 2))[:, None]

    def noise(self, temp, ts):
        kT = self.p.species[0].kT
        if self.p.noise != abi.NOISE_FDT or not kT:
            return torch.zeros_like(self.x)
        e = torch.arange(self.nE, device=self.x.device).repeat(self.key.numel())
        ids = (self.key.repeat_interleave(self.nE) << 1) | e
        z = list(_normal2(ids, ts, 2, 0, self.p.seed))
        if self.D == 3:
            z.append(_normal2(ids, ts, 2, 1, self.p.seed)[0])
        return torch.sqrt(2 * kT * temp) * torch.stack(z, 1)

    def step(self):
        if self.p.integrator == abi.INT_HEUN:
            for phase in (1, 0):
                self.x = self._wrap(self.x + 0.5 * self.p.dt / self.p.species[0].zeta[0] * self.F)
                if phase == 0:
                    self.ts += 1
                self.phase = phase
                self.forces()
            return
        temp = self._mobility_dt()
        self.x = self._wrap(self.x + temp * self.F + self.noise(temp, self.ts))
        self.v = self.F * (temp / self.p.dt)
        self.ts += 1
        if self.p.division == abi.DIV_LINEAR_GROWTH:
            self._grow_linear()
        elif self.p.division == abi.DIV_THETA_CYCLE:
            self._grow_theta()
        self.forces()

    def _append(self, k, x_new, **cell):
        m = k.numel()
        self.x = torch.cat([self.x, x_new])
        self.v = torch.cat([self.v, torch.zeros_like(x_new)])
        self.key = torch.cat([self.key, self.key.numel() + torch.arange(m, device=k.device)])
        self.spec = torch.cat([self.spec, torch.zeros(m * self.nE, dtype=I64, device=k.device)])
        for f in self.cell:
            self.cell[f] = torch.cat([self.cell[f], cell.get(f, self.cell[f][k])])
        self.xref = None

    def _grow_linear(self):
        p, sp, c = self.p, self.p.species[0], self.cell
        c["rest_len"] = c["rest_len"] + sp.growth_rate * p.dt
        k = torch.nonzero(c["rest_len"] >= sp.l_div).reshape(-1)
        if not k.numel():
            return
        b, f = self.x[2 * k], self.x[2 * k + 1]
        u = _min_image(f - b, self.L, self.pbc)
        u = u / u.norm(dim=1, keepdim=True)
        keys = self.key[k]
        z = _normal2(keys, self.ts, 4, 0, p.seed) + _normal2(keys, self.ts, 4, 1, p.seed)
        z = [sp.sigma[q % 2] * (1 + sp.sigma_jitter * z[q]) for q in range(4)]
        c["rest_len"][k] = sp.l_birth
        self._append(k, torch.stack([self._wrap(f - sp.l_birth * u), f], 1).reshape(-1, self.D))
        self.x[2 * k + 1] = self._wrap(b + sp.l_birth * u)
        self.v[2 * k] = self.v[2 * k + 1] = 0.0
        self.sig[2 * k], self.sig[2 * k + 1] = z[0], z[1]
        self.sig = torch.cat([self.sig, torch.stack(z[2:], 1).reshape(-1)])

    def _grow_theta(self):
        p, sp, c = self.p, self.p.species[0], self.cell
        pn = c["pressure"].clamp(min=0.0) / sp.cycle_p0
        rho, av = c["rho"], c["ang_vel"]
        theta = c["theta"] + av * (sp.cycle_rmaxed_inv * rho).clamp(max=1.0)
        area = lambda s: math.pi * (s / 2) ** 2  # noqa: E731
        vt, vv = area(c["sigma_t"]), area(self.sig)
        c0 = av * math.log(2.0) + (sp.cycle_v_1 - 1) / sp.cycle_tau_v
        vt = vt + (c0 * rho - (vt - sp.cycle_v_s) / sp.cycle_v_s / sp.cycle_tau_v) * vt
        vv = vv - (vv - vt / (1 + sp.cycle_beta_vs * (p.osmotic_pi + pn))) / sp.cycle_tau_p
        c["sigma_t"], self.sig = 2 * torch.sqrt(vt / math.pi), 2 * torch.sqrt(vv / math.pi)
        rp = 1 - rho - pn
        c["rho"] = rho + rp / (sp.cycle_tau_r * torch.where(rp > 0, torch.ones_like(rp), sp.cycle_rho_ratio * torch.ones_like(rp))) * rho
        c["theta"] = theta
        k = torch.nonzero(theta >= 1).reshape(-1)
        if not k.numel():
            return
        keys = self.key[k]
        lm = self.sig[k]
        ld = lm / math.sqrt(2.0)
        al = _uniform2(keys, self.ts, 4, 0, p.seed)[0] * 2 * math.pi
        dr = (0.5 * (lm - ld))[:, None] * torch.stack([torch.sin(al), torch.cos(al)], 1)
        mu, sd = sp.division_tau.mu, sp.division_tau.sigma
        span = lambda z: 1.0 / torch.round(torch.exp(math.log(mu * mu / math.sqrt(mu * mu + sd * sd))  # noqa: E731
                                                     + math.sqrt(math.log(1 + sd * sd / (mu * mu))) * z) / p.dt)
        z = _normal2(keys, self.ts, 4, 2, p.seed)
        c["theta"][k] = 0.0
        c["sigma_t"][k] = ld
        av = c["ang_vel"].clone()
        av[k] = span(z[0])
        c["ang_vel"] = av
        m = self.x[k]
        self._append(k, self._wrap(m + dr), ang_vel=span(z[1]))
        self.x[k] = self._wrap(m - dr)
        self.v[k] = 0.0
        self.sig[k] = ld
        self.sig = torch.cat([self.sig, ld])

    def frame(self, family, col):
        shape = (-1, self.nE, self.D)
        out = {"pos": self.x.view(shape), "vel": self.v.view(shape), "frc": self.F.view(shape)}
        if family in FIELDS:
            for k in FIELDS[family]:
                out[k] = self.sig.view(-1, self.nE) if k == "sigma" else self.cell[k]
            n = self.key.numel()
            for k, a in out.items():  # the unused tail of the host arrays
                full = torch.from_numpy(col.species[0][k].copy()).to(a.device)
                full[:n] = a
                out[k] = full
            out["cells"] = torch.tensor([n])
        return out


def _net(w, X):
    h = torch.nn.functional.silu(X @ w[0].T + w[1])
    h = torch.nn.functional.silu(h @ w[2].T + w[3])
    return h @ w[4].T + w[5]


def _macro(e, w):
    """One surrogate macro-step of 8 Euler steps."""
    n = e.x.shape[0]
    temp = e._mobility_dt()
    b = 8 * temp * e.F
    z = sum(e.noise(temp, e.ts + k) for k in range(8))
    i, j = _pairs(e.x, e.L, e.pbc, 2.4)
    i, j = torch.cat([i, j]), torch.cat([j, i])
    r2 = _min_image(e.x[j] - e.x[i], e.L, e.pbc).square().sum(1)
    o = torch.argsort(r2)
    o = o[torch.argsort(i[o], stable=True)]
    cnt = torch.bincount(i, minlength=n)
    if int(cnt.min()) < 16:
        return False
    first = torch.cumsum(cnt, 0) - cnt
    j = j[o][first[:, None] + torch.arange(16, device=e.x.device)]
    d = _min_image((e.x[j] - e.x[:, None]).reshape(-1, 3), e.L, e.pbc).view(n, 16, 3)
    r = d.norm(dim=2, keepdim=True)
    m = e.sig[j] + 4.0 * e.spec[j]
    g = 20.0 * (r[:, :, 0] / (0.5 * (e.sig[:, None] + e.sig[j])) - 1)
    X = torch.cat([torch.cat([d / r * m[:, :, None], g[:, :, None]], 2).reshape(n, 64),
                   torch.stack([e.sig, e.spec.to(F64)], 1), b / 0.01, z / 0.01], 1)
    c = 0.002 * _net(w, X)
    c = c * (0.05 / c.norm(dim=1, keepdim=True).clamp(min=1e-30)).clamp(max=1.0)
    e.x = e._wrap(e.x + b + c + z)
    e.v = (b + c) / (8 * e.p.dt)
    e.ts += 8
    e.forces()
    return True


def _exact_train(case, seed):
    dev = torch.device("cuda")
    X, T = (torch.from_numpy(a).to(dev, F64) for a in _samples(case["samples"], seed))
    w = [torch.from_numpy(a).to(dev, F64).requires_grad_(True) for a in _weights(seed + 1)]
    m = [torch.zeros_like(a) for a in w]
    v = [torch.zeros_like(a) for a in w]
    n, losses = X.shape[0], []
    row = torch.arange(case["batch"], device=dev)
    for t in range(1, case["adam"] + 1):
        hi, lo, _, _ = _philox(row, t, 0x5EED, 7, seed)
        pick = ((hi % n) * ((1 << 32) % n) + lo % n) % n
        loss = 0.5 * (_net(w, X[pick]) - T[pick] / 0.002).square().mean()
        losses.append(loss.detach())
        for k, g in enumerate(torch.autograd.grad(loss, w)):
            m[k] = 0.9 * m[k] + 0.1 * g
            v[k] = 0.999 * v[k] + 0.001 * g * g
            with torch.no_grad():
                w[k] -= 1e-3 * (m[k] / (1 - 0.9 ** t)) / ((v[k] / (1 - 0.999 ** t)).sqrt() + 1e-8)
    return {"losses": torch.stack(losses), "params": torch.cat([a.detach().reshape(-1) for a in w])}


def exact(case, seed):
    f = case["family"]
    if f == "train":
        return _exact_train(case, seed)
    if f == "batch":
        frames = []
        for p, box, col in _ensemble(case, seed):
            e = _Exact(p, box, col)
            e.forces()
            for _ in range(case["steps"]):
                e.step()
            frames.append(e.frame(f, col))
        return {k: torch.cat([fr[k] for fr in frames]) for k in frames[0]}
    p, box, col = _inputs(case, seed)
    e = _Exact(p, box, col)
    e.forces()
    if f == "surrogate":
        for _ in range(SETTLE):
            e.step()
        w = [torch.from_numpy(a).to(e.x.device, F64) for a in _weights(seed + 1, 0.1)]
        for k in range(1, case["macro"] + 1):
            if k % 16:
                if not _macro(e, w):
                    return None
            else:  # judged: the plain integrator's result is kept
                for _ in range(8):
                    e.step()
        return e.frame(f, col)
    if case["n"] * case["steps"] > 2.5e8:
        return None  # over 20 seconds
    for _ in range(case["steps"]):
        e.step()
    if f == "channel" and bool(((e.x < 0) | (e.x >= torch.tensor(e.L, device=e.x.device))).any()):
        return None  # the drain moves cells: their order is not restated here
    return e.frame(f, col)
