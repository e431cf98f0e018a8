"""The work this framework is used for, as cases that can be timed and compared.

A case is one pass of a user's program through the public entry points: a run
of a collective or Selkov engine to its next output frame and the frame itself,
a batch of replicas advanced and averaged, a training run or a prediction of
the surrogate, a collision step of a Fortran driver through the per-procedure
drop-ins.  Sizes and physics are those of the repository's benchmark, tests,
sweep and reference inputs, or generic boxes of the same ranges.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from main_amd import dropin
from main_amd import systems as S
from main_amd.batch import CollectiveBatch
from main_amd.collective import CollectiveEngine, draws_per_collision
from main_amd.selkov import SelkovEngine
from main_amd.surrogate import Surrogate
from main_amd.tour import cell_tour

# the benchmark's solvent and dimer physics (10 per cell, skin 0.3, 50 MD steps a collision)
PHYS = dict(rhoa=10.0, Rc=2.0, Rn=4.0, Dcn=6.5, EbN=0.1, T=1.0 / 6.0, skinrad=0.3, MDt=0.01, MPCt=0.5,
            sort_step=500, k1=1e-3, react_box_type=7)
N_IN, N_OUT = 8, 2049   # the sweep's network: 8 parameters -> 64 x 32 field and the velocity
MAXS = 100              # member slots per cell in the reference's census arrays


def listed():
    return [
        # FP64 collective runs, device draws, one dimer, from one output frame to the next:
        # the sweep's box, the smallest in use (latency of the near engine),
        {"name": "collective_24", "kind": "collective", "x": 24, "y": 24, "z": 24, "dimers": 1, "n": 20,
         "host_draws": False, "split": False},
        # a ragged box in parity mode (the caller's own draws), two dimers, as a Fortran driver embeds the engine,
        {"name": "collective_ragged_host", "kind": "collective", "x": 45, "y": 37, "z": 29, "dimers": 2, "n": 10,
         "host_draws": True, "split": False},
        # the headline box, the largest
        {"name": "collective_100", "kind": "collective", "x": 100, "y": 100, "z": 100, "dimers": 1, "n": 50,
         "host_draws": False, "split": False},
        # many dimers: the reference's own input and the 100-dimer slab
        {"name": "dimers_20_reference", "kind": "collective", "x": 64, "y": 64, "z": 32, "dimers": 20, "n": 10,
         "host_draws": False, "split": False},
        {"name": "dimers_100_slab", "kind": "collective", "x": 200, "y": 200, "z": 10, "dimers": 100, "n": 10,
         "host_draws": False, "split": False},
        # one system in split precision storage
        {"name": "split_64", "kind": "collective", "x": 64, "y": 64, "z": 64, "dimers": 1, "n": 20,
         "host_draws": False, "split": True},
        # replicas: the sweep's FP64 batch of one box, and the split ensemble of uneven boxes (20 to 40 cells)
        {"name": "batch_fp64", "kind": "batch", "replicas": 64, "lo": 24, "hi": 24, "n": 10, "m": 10, "split": False},
        {"name": "batch_split", "kind": "batch", "replicas": 192, "lo": 20, "hi": 40, "n": 10, "m": 10,
         "split": True},
        # the Selkov simulator at the benchmark's box
        {"name": "selkov_50", "kind": "selkov", "L": 50, "n": 20},
        # the surrogate: epochs of the sweep's training (448 of 512 runs, the rest held out), screening of candidates
        {"name": "surrogate_train", "kind": "train", "rows": 448, "batch": 64, "hidden": 256, "layers": 3, "epochs": 5},
        {"name": "surrogate_predict", "kind": "predict", "rows": 8192, "hidden": 256, "layers": 3},
        # one collision step of the reference's driver through the drop-in procedures, host arrays
        {"name": "dropin_collision", "kind": "dropin", "x": 30, "y": 30, "z": 30},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _box(rng, lo, hi):
    """Edges around a log-uniform size, uneven."""
    side = _log(rng, lo, hi)
    return {k: int(min(hi, max(20, round(side * rng.uniform(0.85, 1.18))))) for k in "xyz"}


def draw(rng):
    kind = rng.choice(["collective", "collective", "collective", "many", "split", "batch", "batch_split", "selkov",
                       "train", "predict", "dropin"])
    if kind == "collective":
        return {"kind": "collective", **_box(rng, 22, 100), "dimers": 1, "n": rng.randint(5, 30),
                "host_draws": rng.random() < 0.2, "split": False}
    if kind == "split":
        return {"kind": "collective", **_box(rng, 24, 90), "dimers": 1, "n": rng.randint(5, 30),
                "host_draws": False, "split": True}
    if kind == "many":
        if rng.random() < 0.4:   # slabs, every dimer in the mid-plane
            x, y, z = rng.randint(60, 200), rng.randint(60, 200), 10
            nd = max(3, int(x * y / rng.uniform(420, 900)))
        else:
            x, y, z = rng.randint(40, 90), rng.randint(40, 90), rng.randint(28, 44)
            nd = max(3, int(x * y * z / rng.uniform(7000, 14000)))
        return {"kind": "collective", "x": x, "y": y, "z": z, "dimers": nd, "n": rng.randint(3, 12),
                "host_draws": False, "split": False}
    if kind in ("batch", "batch_split"):
        lo = rng.randint(20, 30)
        split = kind == "batch_split"
        return {"kind": "batch", "replicas": int(_log(rng, 8, 160 if split else 64)), "lo": lo,
                "hi": rng.randint(lo, 40 if split else 32), "n": rng.randint(4, 12), "m": rng.randint(4, 12),
                "split": split}
    if kind == "selkov":
        return {"kind": "selkov", "L": int(_log(rng, 24, 60)), "n": rng.randint(5, 25)}
    hidden, layers = rng.choice([64, 100, 128, 200, 256]), rng.randint(2, 4)
    if kind == "train":
        return {"kind": "train", "rows": rng.randint(96, 512), "batch": rng.choice([32, 50, 64, 96, 128]),
                "hidden": hidden, "layers": layers, "epochs": rng.randint(2, 6)}
    if kind == "predict":
        return {"kind": "predict", "rows": int(_log(rng, 1, 8192)), "hidden": hidden, "layers": layers}
    return {"kind": "dropin", "x": rng.randint(16, 40), "y": rng.randint(16, 40), "z": rng.randint(20, 32)}


# ------------------------------------------------------------------ inputs
@functools.lru_cache(maxsize=64)
def _tour(x, y, z):
    return cell_tour(x, y, z)


def _params(case):
    return S.collective_params(Lx=float(case["x"]), Ly=float(case["y"]), Lz=float(case["z"]),
                               numdims=case.get("dimers", 1), **PHYS)


def _engine(p, seed, rng_mode=1, split=False):
    e = CollectiveEngine(p, rng_mode=rng_mode, seed=seed, split=split)
    e.set_dimers(S.collective_dimers(p, seed=seed), tour=_tour(*(int(v) for v in p["box"])))
    e.init_solvent(seed)
    e.setup(do_sort=True)
    return e


def _network(case, seed):
    """He-uniform weights as a flat parameter vector (each layer's W, then b)."""
    dims = [N_IN] + [case["hidden"]] * case["layers"] + [N_OUT]
    rng = np.random.default_rng(seed + 1)
    flat = []
    for k, n in zip(dims[:-1], dims[1:]):
        flat += [rng.uniform(-1.0, 1.0, n * k) * math.sqrt(6.0 / k), rng.uniform(-0.1, 0.1, n)]
    return dims, np.concatenate(flat).astype(np.float32)


def _training_set(case, seed):
    """Standardized parameters, smooth targets with sampling noise, output weights."""
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((case["rows"], N_IN)).astype(np.float32)
    mix = rng.standard_normal((N_IN, N_OUT)) / math.sqrt(N_IN)
    t = (np.tanh(x @ mix) + 0.2 * rng.standard_normal((case["rows"], N_OUT))).astype(np.float32)
    return x, t, np.full(N_OUT, 1.0 / N_OUT, np.float32)


def _driver_state(case, seed):
    """Host arrays of the reference's driver at a collision step, in its kinds and layouts."""
    p = _params(case)
    s = S.collective_initial_state(p, seed=seed)
    rng = np.random.default_rng(seed + 1)
    s["flag"][:] = (rng.random(p["NT"]) < 0.3).astype(np.int32)   # a run under way: A and B solvent
    r2 = [(p[k] * p["cutoff"] + p["skinrad"]) ** 2 for k in ("Rc", "Rn")]
    inside = np.zeros(p["NT"], bool)
    for i in (0, 1):
        d = [s[k] - s[k + "d"][0, i] for k in ("x", "y", "z")]
        for c in (0, 1):
            d[c] -= p["box"][c] * np.rint(d[c] / p["box"][c])
        inside |= d[0] ** 2 + d[1] ** 2 + d[2] ** 2 <= r2[i]
    s["in"], s["out"] = (np.flatnonzero(m).astype(np.int64) + 1 for m in (inside, ~inside))
    s["draws"] = rng.random(draws_per_collision(p))
    mc, vol = p["mpcnumcell"], p["vol"]
    s["cells"] = {k: np.zeros(mc) for k in ("vxcm", "vycm", "vzcm", "tcs", "uvx", "uvy", "uvz")}
    s["ncn"] = np.zeros(p["NT"], np.int64)
    s["t"] = [np.zeros(vol, np.int64) for _ in range(3)]
    s["s"] = [np.zeros((vol, MAXS), np.int64, order="F") for _ in range(3)]
    return p, s


def prepare(case, seed):
    kind = case["kind"]
    if kind == "collective":
        p = _params(case)
        e = _engine(p, seed, 0 if case["host_draws"] else 1, case["split"])
        draws = None
        if case["host_draws"]:
            draws = np.random.default_rng(seed).random(case["n"] * draws_per_collision(p))
        return {"case": case, "engine": e, "draws": draws}
    if kind == "batch":
        rng = np.random.default_rng(seed)
        engines = []
        for r in range(case["replicas"]):
            L = int(rng.integers(case["lo"], case["hi"] + 1))
            p = S.collective_params(Lx=float(L), Ly=float(L), Lz=float(L), numdims=1,
                                    **{**PHYS, "EbN": float(rng.uniform(0.1, 1.0))})
            engines.append(_engine(p, seed + r, split=case["split"]))
        return {"case": case, "batch": CollectiveBatch(engines, tile=2048)}
    if kind == "selkov":
        p = S.selkov_params(L=float(case["L"]), rho=10.0, NG=int(0.8 * case["L"] ** 3))
        e = SelkovEngine(p, rng_mode=1, seed=seed)
        e.set_state(S.selkov_initial_state(p, seed=seed), cstep=0)
        return {"case": case, "engine": e}
    if kind in ("train", "predict"):
        net = Surrogate(n_in=N_IN, n_hidden=case["hidden"], n_layers=case["layers"], n_out=N_OUT, seed=seed)
        net.set_params(_network(case, seed)[1])
        return {"case": case, "net": net, "data": _training_set(case, seed) if kind == "train" else
                np.random.default_rng(seed).standard_normal((case["rows"], N_IN)).astype(np.float32)}
    p, s = _driver_state(case, seed)
    return {"case": case, "p": p, "s": s}


# ------------------------------------------------------------------ passes
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "collective":
        state["engine"].run(case["n"], state["draws"])
        return state["engine"].get_state()
    if kind == "batch":   # as the sweep: advance, then sample after every collision
        state["batch"].run(case["n"])
        counts, velocity = state["batch"].body_average(case["m"])
        return {"counts": counts, "velocity": velocity}
    if kind == "selkov":
        state["engine"].run(case["n"])
        return state["engine"].get_state()
    if kind == "train":
        x, t, w = state["data"]
        losses = state["net"].train_raw(x, t, w, batch=case["batch"], epochs=case["epochs"], lr=1e-3, seed=3)
        return {"losses": losses, "params": state["net"].params()}
    if kind == "predict":
        return state["net"].forward_raw(state["data"])
    p, s = state["p"], state["s"]
    mc, c = p["mpcnumcell"], s["cells"]
    tA, tB, tS = s["t"]
    sA, sB, sS = s["s"]
    dropin.distribute(p["NT"], 1, s["flag"], s["x"], s["y"], s["z"], s["xd"], s["yd"], s["zd"], p["box"], tA, tB, tS,
                      sA, sB, sS, (p["Rc"] * p["cutoff"]) ** 2, (p["Rn"] * p["cutoff"]) ** 2, s["out"].size, s["out"],
                      s["in"].size, s["in"])
    dropin.mpc_rotation(p["NT"], p["rotang"], mc, p["a0"], p["box"], s["x"], s["y"], s["z"], s["vx"], s["vy"],
                        s["vz"], c["vxcm"], c["vycm"], c["vzcm"], c["tcs"], s["ncn"], c["uvx"], c["uvy"], c["uvz"],
                        s["draws"])
    dropin.reaction_simple(p["MPCt"], p["rxnnumcell"], p["k1"], p["NT"], s["flag"], tB, sB, s["draws"][3 + 2 * mc:])
    return {"v": [s["vx"], s["vy"], s["vz"]], "cells": c, "cell": s["ncn"], "flag": s["flag"], "census": [tA, tB, tS]}


def work(case):
    """Bytes: the state read and written once a collision interval (FP64 100, split 57, Selkov 108 B a particle)
    and each output once; operations: streaming, cell index, sums and rotation, about 90 a particle and interval."""
    kind = case["kind"]
    if kind == "collective":
        nt = _params(case)["NT"]
        return {"bytes": nt * (case["n"] * (57 if case["split"] else 100) + 52.0), "flops": 90.0 * nt * case["n"]}
    if kind == "batch":
        nt = 10.0 * case["replicas"] * ((case["lo"] + case["hi"]) / 2.0) ** 3
        n = case["n"] + case["m"]
        return {"bytes": nt * n * (57.0 if case["split"] else 100.0), "flops": 90.0 * nt * n}
    if kind == "selkov":
        nt = 10.0 * case["L"] ** 3
        return {"bytes": nt * (case["n"] * 108.0 + 80.0), "flops": 90.0 * nt * case["n"]}
    if kind in ("train", "predict"):
        h, L = case["hidden"], case["layers"]
        weights = N_IN * h + (L - 1) * h * h + h * N_OUT
        rows = case["rows"]
        if kind == "predict":
            return {"bytes": 4.0 * (rows * (N_IN + N_OUT) + weights), "flops": 2.0 * rows * weights}
        steps = case["epochs"] * -(-rows // case["batch"])
        return {"bytes": 4.0 * (rows * case["epochs"] * (N_IN + N_OUT) + 6 * steps * weights),
                "flops": 6.0 * rows * case["epochs"] * weights}
    p = _params(case)
    nt, mc = p["NT"], p["mpcnumcell"]
    return {"bytes": nt * (48 + 4 + 8 + 24 + 8 + 4 + 8.0) + mc * (7 * 8 + 16 + 24 + 8.0), "flops": 90.0 * nt}


# ------------------------------------------------------------------ the same in plain 64-bit numbers
def _exact_layers(dims, flat):
    out, o = [], 0
    for k, n in zip(dims[:-1], dims[1:]):
        out.append([flat[o:o + n * k].reshape(n, k), flat[o + n * k:o + n * k + n]])
        o += n * k + n
    return out


def _exact_forward(layers, x):
    acts = [x]
    for i, (w, b) in enumerate(layers):
        z = acts[-1] @ w.T + b
        acts.append(torch.relu(z) if i + 1 < len(layers) else z)
    return acts


def _exact_train(case, seed):
    """Minibatch Adam over rows shuffled each epoch by a 64-bit linear congruential generator."""
    dims, flat = _network(case, seed)
    x, t, w = (torch.from_numpy(a).double() for a in _training_set(case, seed))
    p = torch.from_numpy(flat).double()
    m, v, step, losses, mask = torch.zeros_like(p), torch.zeros_like(p), 0, [], (1 << 64) - 1
    n = case["rows"]
    for ep in range(case["epochs"]):
        order, s = list(range(n)), (4 * 6364136223846793005 + ep * 1442695040888963407) & mask
        for i in range(n - 1, 0, -1):
            s = (s * 6364136223846793005 + 1442695040888963407) & mask
            j = (s >> 33) % (i + 1)
            order[i], order[j] = order[j], order[i]
        total = 0.0
        for b in range(0, n, case["batch"]):
            q = torch.tensor(order[b:b + case["batch"]])
            layers = _exact_layers(dims, p)
            acts = _exact_forward(layers, x[q])
            d = acts[-1] - t[q]
            total += float((w * d * d).sum())
            dz, grads = 2.0 * w * d / len(q), []
            for k in range(len(layers) - 1, -1, -1):
                grads[:0] = [(dz.T @ acts[k]).reshape(-1), dz.sum(0)]
                if k:
                    dz = (dz @ layers[k][0]) * (acts[k] > 0)
            g = torch.cat(grads)
            step += 1
            m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
            p = p - 1e-3 * (m / (1 - 0.9 ** step)) / ((v / (1 - 0.999 ** step)).sqrt() + 1e-8)
        losses.append(total / n)
    return {"losses": np.array(losses), "params": p.numpy()}


def _exact_driver(case, seed):
    """Shifted-grid cells, their mean velocities and axes, and the rotation about them."""
    p, s = _driver_state(case, seed)
    mc, d = p["mpcnumcell"], s["draws"]
    shift = d[:3] - 0.5
    bx, by = p["box"][0], p["box"][1]
    X, Y = (s[k] + shift[i] - b * np.floor((s[k] + shift[i]) / b) for i, (k, b) in enumerate((("x", bx), ("y", by))))
    Z = s["z"] + shift[2]
    Z = np.floor(Z + 1.0) if shift[2] < 0.0 else np.floor(Z)
    c = (np.floor(X) + bx * np.floor(Y) + bx * by * Z).astype(np.int64)
    n = np.bincount(c, minlength=mc)
    v = np.stack([s["vx"], s["vy"], s["vz"]])
    cm = np.stack([np.bincount(c, weights=a, minlength=mc) for a in v]) / np.maximum(n, 1)
    phi, th = 2.0 * math.pi * d[3:3 + 2 * mc:2], 2.0 * d[4:4 + 2 * mc:2] - 1.0
    u = np.stack([np.sqrt(1.0 - th * th) * np.cos(phi), np.sqrt(1.0 - th * th) * np.sin(phi), th])
    r, ax = v - cm[:, c], u[:, c]
    cs, sn = math.cos(p["rotang"]), math.sin(p["rotang"])
    r = cs * r + (1.0 - cs) * ax * (ax * r).sum(0) + sn * np.cross(ax, r, axis=0)
    keys = ("vxcm", "vycm", "vzcm", "tcs", "uvx", "uvy", "uvz")
    return {"v": list(cm[:, c] + r), "cells": dict(zip(keys, [*cm, n.astype(np.float64), *u])), "cell": None,
            "flag": None, "census": [None, None, None]}


def exact(case, seed):
    """The network and the drop-in collision in 64 bits.  The engines' runs have none: thousands of dependent MD
    steps and collisions with draws made on the device, minutes to hours in plain numpy."""
    if case["kind"] == "predict":
        dims, flat = _network(case, seed)
        x = torch.from_numpy(np.random.default_rng(seed).standard_normal((case["rows"], N_IN)).astype(np.float32))
        return _exact_forward(_exact_layers(dims, torch.from_numpy(flat).double()), x.double())[-1]
    if case["kind"] == "train":
        return _exact_train(case, seed)
    if case["kind"] == "dropin":
        return _exact_driver(case, seed)
    return None
