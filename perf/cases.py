"""Performance cases: the calls that programs built on this package make.

Every case goes through the public Python entry points (`procell`,
`procell.calibrate`).  `prepare` makes what such a program holds before the
call (inputs, plan, device tensors), `run` is one pass, `exact` computes the
relaxed estimator's outputs again in plain torch, in 64 bits, breadth first
(the plain method's outputs are whole numbers and need no such value).
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cuda-pro-cell_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import procell  # noqa: E402
from procell import calibrate  # noqa: E402


# ---------------------------------------------------------------------------
# The cases.  bins: histogram rows, log-spaced from 1 to 10**decades; cells:
# initial cells of one set; prolif / quiet: cell types; phi 0: the smallest
# populated value.
# ---------------------------------------------------------------------------
def listed():
    plain = {"decades": 5, "phi": 50.0, "t_max": 240.0, "prolif": 4, "quiet": 1}
    readme = {"decades": 4, "phi": 0.0, "t_max": 168.0, "prolif": 2, "quiet": 1}
    batch = {"decades": 4, "phi": 0.0, "prolif": 0, "quiet": 0, "bins": 256, "cells": 200_000, "sets": 256, "beta": 0.5}
    return [
        # one call from host buffers to host buffers, as the command line and
        # scripts make it: latency, set-up and launches
        {"name": "simulate_64x1e4", "kind": "simulate", "bins": 64, "cells": 10_000, **readme},
        # the same on a cytometer-sized histogram with an odd number of rows
        {"name": "simulate_1021x3e6", "kind": "simulate", "bins": 1021, "cells": 3_000_000, **plain},
        # repeated runs of one problem with new seeds (uncertainty of a
        # histogram): the standard small problem, the standard large one and
        # ten times that
        {"name": "plan_64x1e5", "kind": "plan", "bins": 64, "cells": 100_000, **readme},
        {"name": "plan_1024x1e7", "kind": "plan", "bins": 1024, "cells": 10_000_000, **plain},
        {"name": "plan_1024x1e8", "kind": "plan", "bins": 1024, "cells": 100_000_000, **plain},
        # a sweep over uneven parameter sets in one launch, every set's
        # histogram read back (derivative-free fits, parameter studies)
        {"name": "batch_512", "kind": "batch", "sets": 512, "cells": 30_000},
        # the relaxed estimator of one histogram: value only, and the
        # vector-Jacobian product for a caller's own loss
        {"name": "forward_256x1e6", "kind": "forward", "bins": 256, "cells": 1_000_000, "beta": 0.5, **readme},
        {"name": "adjoint_256x1e6", "kind": "adjoint", "bins": 256, "cells": 1_000_000, "beta": 0.5, **readme},
        # one gradient step's loss and gradient through torch.autograd on a
        # small sample: launches and host work beside a short walk
        {"name": "autograd_61x2e4", "kind": "autograd", "bins": 61, "cells": 20_000, "beta": 0.5, **readme},
        # h and its Jacobian for many sets at once (one Gauss-Newton iteration)
        {"name": "jacobian_64x2e5", "kind": "jacobian", **batch, "sets": 64},
        # on-device Adam over many sets: every cell per step, and a quarter of
        # the cells per step (one cycle of four steps between reads)
        {"name": "calibrate_256x2e5", "kind": "calibrate", "stride": 1, "steps": 1, **batch},
        {"name": "calibrate_256x2e5_stride4", "kind": "calibrate", "stride": 4, "steps": 4, **batch},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["simulate", "plan", "plan", "batch", "forward", "adjoint", "autograd", "jacobian", "calibrate",
                       "calibrate"])
    if kind == "batch":
        return {"kind": kind, "sets": _log_int(rng, 8, 512), "cells": _log_int(rng, 3_000, 100_000)}
    case = {"kind": kind, "bins": _log_int(rng, 33, 1024), "decades": rng.choice([3, 4, 5])}
    if kind in ("simulate", "plan"):
        case["cells"] = _log_int(rng, 1_000, 10_000_000)
        case["phi"] = rng.choice([0.0, round(rng.uniform(1.0, 100.0), 2)])
        case["t_max"] = round(rng.uniform(72.0, 240.0), 1)
        case["prolif"], case["quiet"] = rng.randint(1, 4), rng.randint(0, 1)
        return case
    case["phi"] = 0.0
    case["beta"] = rng.choice([0.25, 0.5, 1.0])
    if kind in ("jacobian", "calibrate"):
        case["sets"] = _log_int(rng, 2, 256)
        case["cells"] = _log_int(rng, 5_000, 200_000)
        case["bins"] = min(case["bins"], 400)
        case["prolif"] = case["quiet"] = 0
        if kind == "calibrate":
            case["stride"] = rng.choice([1, 1, 2, 4, 8])
            case["steps"] = case["stride"]
        return case
    case["cells"] = _log_int(rng, 5_000, 1_500_000)
    case["t_max"] = round(rng.uniform(96.0, 200.0), 1)
    case["prolif"], case["quiet"] = rng.randint(1, 3), rng.randint(0, 1)
    return case


# ---------------------------------------------------------------------------
# Inputs: the form (populated rows, numbers of types, phi, t_max) from the
# case, so that a case's outputs keep their shapes; counts, types and random
# streams from the seed.
# ---------------------------------------------------------------------------
def _histogram(rng, bins, decades, cells):
    v = 10.0 ** (decades * np.arange(bins) / max(bins - 1, 1))
    lam = np.exp(-((np.log(v) - math.log(800.0)) ** 2) / 2.0)
    lam *= cells / lam.sum()
    return v, np.where(lam >= 0.5, np.maximum(rng.poisson(lam), 1), 0).astype(np.uint64)


def _types(rng, n, quiet, lo, hi, sd_lo, sd_hi):
    mean = rng.uniform(lo, hi, size=n)
    sd = rng.uniform(sd_lo, sd_hi, size=n) * mean
    if quiet:
        mean, sd = np.append(mean, -1.0), np.append(sd, -1.0)
    return mean, sd, rng.dirichlet(np.full(len(mean), 2.0))


def _inputs(case, seed):
    """The parameter sets of a case: a list of dicts of plain arrays and numbers."""
    rng, form = np.random.default_rng([int(seed), 11]), np.random.default_rng(10)
    out = []
    for _ in range(case.get("sets", 1)):
        if case["kind"] == "batch":
            # uneven sets: cells lognormal over a factor of a thousand
            cells = case["cells"] * 10.0 ** float(np.clip(form.normal(0.0, 0.75), -1.5, 1.5))
            v, c = _histogram(rng, int(form.integers(128, 1025)), 5, cells)
            n = int(form.integers(1, 6))
            quiet = n >= 2 and bool(form.integers(0, 2))
            mean, sd, p = _types(rng, n - int(quiet), quiet, 24.0, 120.0, 0.15, 0.5)
            t_max, phi = float(form.uniform(72.0, 336.0)), float(form.uniform(1.0, 100.0))
        else:
            v, c = _histogram(rng, case["bins"], case["decades"], case["cells"])
            if "sets" in case:
                n = int(form.integers(1, 4))
                quiet = n == 1 or bool(form.integers(0, 2))
                t_max = float(form.uniform(96.0, 240.0))
            else:
                n, quiet, t_max = case["prolif"], case["quiet"], case["t_max"]
            mean, sd, p = _types(rng, n, quiet, 30.0, 100.0, 0.2, 0.4)
            phi = case["phi"]
        out.append({"values": v, "counts": c, "mean": mean, "sd": sd, "proportion": p, "t_max": t_max,
                    "phi": phi, "seed": int(rng.integers(1, 2**62))})
    return out


def _nonzero(s):
    keep = s["counts"] > 0
    v, n = s["values"][keep], s["counts"][keep].astype(np.int64)
    phi = s["phi"] if s["phi"] > 0 else float(v.min())
    cap = np.zeros(len(v), dtype=np.int64)
    f = v / 2
    while (f > phi).any():
        cap += f > phi
        f = f / 2
    return v, n, phi, cap


def _bins(s):
    """Output values (ascending) and the bin of every (row, generation), -1 for none."""
    v, _, phi, cap = _nonzero(s)
    k = np.arange(int(cap.max()) + 1)
    f = v[:, None] / 2.0 ** k[None, :]
    ok = (k[None, :] <= cap[:, None]) & ((k[None, :] > 0) | (f >= phi))
    bins = np.unique(np.concatenate([x[x >= phi] for x in (v[:, None] / 2.0 ** np.arange(k[-1] + 2)).T]))
    at = np.searchsorted(bins, np.where(ok, f, bins[0]))
    return bins, np.where(ok, at, -1)


def _target(s, true):
    """A histogram to fit: what the types `true` leave at t_max, by the normal
    approximation of the division times, on the set's output values."""
    v, n, _, _ = _nonzero(s)
    bins, at = _bins(s)
    w = np.zeros(at.shape[1])
    for m, sd, p in zip(*true):
        before = 1.0
        for k in range(len(w)):
            if m < 0:
                w[0] += p
                break
            var = (7.0 / 3.0) * sd * sd + m * m / 12.0 + k * sd * sd
            after = 0.5 * math.erfc(-(s["t_max"] - (1.5 + k) * m) / math.sqrt(2.0 * var))
            w[k] += p * 2.0 ** k * max(0.0, before - after)
            before = after
    count = np.zeros(len(bins))
    np.add.at(count, at[at >= 0], np.rint(n[:, None] * w[None, :])[at >= 0])
    keep = count > 0
    return bins[keep], count[keep].astype(np.int64)


def _fit(case, seed):
    """Sets with perturbed starting types, and the targets their types came from."""
    sets = _inputs(case, seed)
    rng = np.random.default_rng([int(seed), 12])
    targets = []
    for s in sets:
        true = (s["mean"], s["sd"], s["proportion"])
        targets.append(_target(s, true))
        n, move = len(true[0]), true[0] >= 0
        s["mean"] = np.where(move, true[0] * rng.uniform(0.85, 1.15, n), -1.0)
        s["sd"] = np.where(move, true[1] * rng.uniform(0.85, 1.15, n), -1.0)
        s["proportion"] = 0.5 * true[2] + 0.5 / n
        s["proportion"] /= s["proportion"].sum()
    return sets, targets


def _problem(s):
    return procell.Problem(s["values"], s["counts"], s["proportion"], s["mean"], s["sd"], s["t_max"], s["phi"], s["seed"])


def _theta(sets):
    return np.concatenate([np.concatenate([s["mean"], s["sd"], s["proportion"]]) for s in sets])


def _cotangent(shape, seed):
    g = torch.Generator().manual_seed(int(seed) + 77)
    return torch.rand(shape, dtype=torch.float64, generator=g) - 0.25


LR = 0.02


def prepare(case, seed):
    kind, dev = case["kind"], "cuda"
    st = {"kind": kind, "case": case}
    if kind in ("simulate", "plan"):
        st["prob"] = _problem(_inputs(case, seed)[0])
        st["seed"] = st["prob"].params.seed
        st["capacity"] = st["prob"].output_capacity()
        if kind == "plan":
            st["plan"] = procell.Plan(st["prob"])
    elif kind == "batch":
        sets = _inputs(case, seed)
        st["plan"] = procell.Batch([_problem(s) for s in sets])
        st["capacity"] = [p.output_capacity() for p in st["plan"].problems]
        st["seeds"] = np.array([s["seed"] for s in sets], dtype=np.uint64)
    elif kind in ("forward", "adjoint"):
        s = _inputs(case, seed)[0]
        st["plan"] = procell.Relaxed(_problem(s), case["beta"])
        st["theta"] = torch.tensor(_theta([s]), device=dev).reshape(3, -1)
        st["h"] = torch.empty(st["plan"].shape, dtype=torch.float64, device=dev)
        st["g"] = _cotangent(st["plan"].shape, seed).to(dev)
        st["grad"] = torch.empty_like(st["theta"])
    elif kind == "autograd":
        sets, targets = _fit(case, seed)
        prob = _problem(sets[0])
        st["plan"] = procell.Relaxed(prob, case["beta"])
        st["theta"] = torch.tensor(_theta(sets), device=dev).reshape(3, -1)
        st["bins"] = calibrate.BinMap(prob, st["plan"].shape[1], dev)
        st["target"] = torch.tensor(calibrate.target_histogram(st["bins"].bins, *targets[0]), device=dev)
    elif kind == "jacobian":
        sets = _inputs(case, seed)
        st["plan"] = procell.RelaxedBatch([_problem(s) for s in sets], case["beta"])
        st["theta"] = torch.tensor(_theta(sets), device=dev)
        st["h"] = torch.empty(st["plan"].h_total, dtype=torch.float64, device=dev)
        st["jac"] = torch.empty((2, st["plan"].h_total), dtype=torch.float64, device=dev)
    else:
        sets, targets = _fit(case, seed)
        st["plan"] = procell.Calibration([_problem(s) for s in sets], case["beta"], targets, lr=LR,
                                         cell_stride=case["stride"])
    return st


def _rows(results, what, capacity):
    """One column of the results' histograms, end to end, each at its capacity (zeros past its last row)."""
    width = [1 if what != "type_count" else r.type_count.shape[1] for r in results]
    out = np.zeros(sum(c * w for c, w in zip(capacity, width)), dtype=getattr(results[0], what).dtype)
    at = 0
    for r, c, w in zip(results, capacity, width):
        col = getattr(r, what).reshape(-1)
        out[at:at + len(col)] = col
        at += c * w
    return out


def _outputs(results, capacity):
    out = {k: _rows(results, k, capacity) for k in ("value", "count", "type_count")}
    out["divisions"] = np.array([r.stats["divisions"] for r in results])
    if results[0].raw_tally is not None:
        out["tally"] = results[0].raw_tally
    return out


def run(st):
    kind = st["kind"]
    if kind == "simulate":
        return _outputs([procell.simulate(st["prob"])], [st["capacity"]])
    plan = st["plan"]
    if kind == "plan":
        plan.run(st["seed"])
        return _outputs([plan.result()], [st["capacity"]])
    if kind == "batch":
        plan.run(st["seeds"])
        res = [plan.result(i, want_raw=False) for i in range(len(plan.problems))]
        return _outputs(res, st["capacity"])
    if kind == "forward":
        plan.forward(st["theta"], st["h"])
        return st["h"]
    if kind == "adjoint":
        plan.backward(st["theta"], st["g"], st["grad"])
        return st["grad"]
    if kind == "autograd":
        theta = st["theta"].detach().requires_grad_(True)
        loss = calibrate.normalized_l2(st["bins"](calibrate.relaxed_tally(plan, theta)), st["target"])
        loss.backward()
        return {"loss": loss.detach(), "grad": theta.grad}
    if kind == "jacobian":
        plan.jacobian(st["theta"], st["h"], st["jac"])
        return {"h": st["h"], "jac": st["jac"]}
    plan.step(st["case"]["steps"])
    theta, (loss, _) = plan.theta(), plan.loss()
    return {"theta": np.concatenate([t.reshape(-1) for t in theta]), "loss": loss}


# ---------------------------------------------------------------------------
# The work of one pass: per division or expansion the random block, the
# normal pair and the bookkeeping (180 lane operations), and for the relaxed
# estimator two sigmoids, records and tangents.
# ---------------------------------------------------------------------------
def _divisions(t_max, cap, relaxed):
    """Divisions of one cell of a middling type (mean 60, sd 18): P(D_k <= t) 2^k."""
    m, sd, e = 60.0, 18.0, 0.0
    for k in range(cap):
        mu, var = (1.5 + k) * m, (7.0 / 3.0 + k) * sd * sd + m * m / 12.0
        e += 2.0 ** k * 0.5 * math.erfc((mu - t_max - (10.0 if relaxed else 0.0)) / math.sqrt(2.0 * var))
    return e


def work(case):
    kind = case["kind"]
    sets = case.get("sets", 1)
    types = case.get("prolif", 0) + case.get("quiet", 0) or 3
    bins, phi = case.get("bins", 576), case.get("phi", 50.0) or 10.0
    cap = max(1, int(math.log2(800.0 / phi)) + 1)
    deep = case.get("decades", 5) * 3.33 + 1
    entries = sets * bins * deep * types
    relaxed = kind in ("forward", "adjoint", "autograd", "jacobian", "calibrate")
    per = _divisions(case.get("t_max", 200.0 if kind == "batch" else 168.0), cap, relaxed)
    units = sets * case["cells"] * (1.0 + per) * (max(1, case.get("prolif") or 2) if relaxed else 1.0)
    ops = {"forward": 234.0, "adjoint": 268.0, "autograd": 276.0, "jacobian": 276.0, "calibrate": 276.0}.get(kind, 180.0)
    words = {"forward": 1, "adjoint": 1, "autograd": 6, "jacobian": 3, "calibrate": 3}.get(kind, 2)
    steps = case.get("steps", 1) * (2.0 / case["stride"] if case.get("stride", 1) > 1 else 1.0)
    return {"bytes": 8.0 * entries * words * case.get("steps", 1) + 16.0 * sets * bins, "flops": ops * units * steps}


# ---------------------------------------------------------------------------
# The relaxed estimator in plain torch: all walks of a generation at once.
# ---------------------------------------------------------------------------
_M = 0xFFFFFFFF
_LANES = 32  # partial sums of each tally entry: neighbouring walks share entries


def _philox(c, k):
    c0, c1, c2, c3 = c
    k0, k1 = k
    for _ in range(10):
        a, b = c0 * 0xD2511F53, c2 * 0xCD9E8D57
        c0, c1, c2, c3 = ((b >> 32) & _M) ^ c1 ^ k0, b & _M, ((a >> 32) & _M) ^ c3 ^ k1, a & _M
        k0, k1 = (k0 + 0x9E3779B9) & _M, (k1 + 0xBB67AE85) & _M
    return c0, c1, c2, c3


def _pair(w0, w1, w2, w3):
    u = ((w0 << 21) + (w1 >> 11) + 1).to(torch.float64) * 2.0 ** -53
    a = ((w2 << 21) + (w3 >> 11)).to(torch.float64) * (2.0 ** -53 * 2.0 * math.pi)
    rho = torch.sqrt(-2.0 * torch.log(u))
    return rho * torch.cos(a), rho * torch.sin(a)


def _block(w, node, att):
    return _philox((node & _M, node >> 32, w["cell"], torch.full_like(node, att << 16)), (w["k0"], w["k1"]))


def _timer(w, z, node):
    """z where mean + sd z > 0, else the first such candidate of the node's redraw stream."""
    z, att = z.clone(), 1
    todo = torch.nonzero(~(w["mean"] + w["sd"] * z > 0)).flatten()
    while len(todo):
        sub = {k: v[todo] for k, v in w.items()}
        y0, y1 = _pair(*_block(sub, node[todo], att))
        ok0, ok1 = sub["mean"] + sub["sd"] * y0 > 0, sub["mean"] + sub["sd"] * y1 > 0
        z[todo] = torch.where(ok0, y0, torch.where(ok1, y1, torch.zeros_like(y0)))
        todo, att = todo[~(ok0 | ok1)], att + 1
    return z


def _walk(sets, theta, beta, stride=1, phase=0, chunk=1 << 22):
    """h, dh/dmean and dh/dsd of every set, flat [rows][generations][types] per
    set: a [3, total] tensor, and the sets' offsets."""
    dev = "cuda"
    rows, base, total, parts = [], [], 0, []
    for s, th in zip(sets, theta):
        v, n, phi, cap = _nonzero(s)
        T, K = th.shape[1], int(cap.max()) + 1
        base.append(total)
        rows.append((v, n, phi, cap, T, K))
        total += len(v) * K * T
    out = torch.zeros((3, total * _LANES), dtype=torch.float64, device=dev)
    for i, (s, th) in enumerate(zip(sets, theta)):
        v, n, phi, cap, T, K = rows[i]
        start = np.concatenate([[0], np.cumsum(n)])
        cells = np.arange((-phase) % stride, start[-1], stride)
        row = np.searchsorted(start, cells, side="right") - 1
        for j in range(T):
            at = base[i] + np.arange(len(v)) * (K * T) + j
            if s["mean"][j] < 0:
                cnt = np.bincount(row, minlength=len(v)) * (v >= phi) * th[2, j]
                out[0].index_add_(0, torch.tensor(at * _LANES, device=dev), torch.tensor(cnt, device=dev))
                continue
            parts.append((cells, row, at, cap, v >= phi, th[:, j], s, T))
    # walks of many (set, type) pairs in one batch of about `chunk`
    group, size = [], 0
    for n, part in enumerate(parts):
        group.append(part)
        size += len(part[0])
        if size >= chunk or n + 1 == len(parts):
            _generations(group, beta, out)
            group, size = [], 0
    return out.reshape(3, total, _LANES).sum(-1), base, [(r[4], r[5], len(r[0])) for r in rows]


def _generations(group, beta, out):
    dev = "cuda"

    def per_walk(f, dtype):
        lens = torch.tensor([len(g[0]) for g in group], device=dev)
        return torch.repeat_interleave(torch.tensor([f(g) for g in group], dtype=dtype, device=dev), lens)

    def of_row(f, dtype):
        return torch.cat([torch.tensor(f(g), device=dev)[torch.tensor(g[1], device=dev)] for g in group]).to(dtype)

    f64, i64 = torch.float64, torch.int64
    w = {"cell": torch.cat([torch.tensor(g[0], device=dev) for g in group]),
         "k0": per_walk(lambda g: g[6]["seed"] & _M, i64), "k1": per_walk(lambda g: g[6]["seed"] >> 32, i64),
         "mean": per_walk(lambda g: g[5][0], f64), "sd": per_walk(lambda g: g[5][1], f64),
         "p": per_walk(lambda g: g[5][2], f64), "t": per_walk(lambda g: g[6]["t_max"], f64),
         "T": per_walk(lambda g: g[7], i64), "cap": of_row(lambda g: g[3], i64), "at": of_row(lambda g: g[2], i64)}
    ge = of_row(lambda g: g[4], torch.bool)
    node = torch.zeros_like(w["cell"])
    w0, w1, w2, w3 = _block(w, node, 0)
    u1 = 1.0 + ((w1 << 21) + 1).to(f64) * 2.0 ** -53
    z, zb = _pair(w2, node, w3, node)
    z = torch.where(w["mean"] + w["sd"] * z > 0, z, zb)
    node = node + 1
    z = _timer(w, z, node)
    w["u1"] = u1
    s, b = (w["mean"] + w["sd"] * z) * u1, z * u1
    W, gm, gs = torch.ones_like(s), torch.zeros_like(s), torch.zeros_like(s)
    k = 0
    while len(node):
        x = (w["t"] - s) / beta
        d, e = torch.sigmoid(x), torch.sigmoid(-x)
        a, q = w["u1"] + k, d * e / beta
        e1 = 1.0 - d
        at = (w["at"] + k * w["T"]) * _LANES + torch.arange(len(node), device=dev) % _LANES
        pW = w["p"] * W * ge
        for c, v in enumerate((e1, e1 * gm + q * a, e1 * gs + q * b)):
            out[c].index_add_(0, at, pW * v)
        go = torch.nonzero((k < w["cap"]) & (W * d >= 1e-15)).flatten()
        w = {n: v[go] for n, v in w.items()}
        node, s, b, d = node[go], s[go], b[go], d[go]
        f = (1.0 - d) / beta
        W, gm, gs = W[go] * d, gm[go] - f * a[go], gs[go] - f * b
        z0, z1 = _pair(*_block(w, node, 0))
        z0, z1 = _timer(w, z0, 2 * node), _timer(w, z1, 2 * node + 1)
        s = torch.cat([s + (w["mean"] + w["sd"] * z0), s + (w["mean"] + w["sd"] * z1)])
        b = torch.cat([b + z0, b + z1])
        node = torch.cat([2 * node, 2 * node + 1])
        W, gm, gs = W.repeat(2), gm.repeat(2), gs.repeat(2)
        w = {n: v.repeat(2) for n, v in w.items()}
        ge = torch.ones_like(node, dtype=torch.bool)
        k += 1


def _loss(h, s, target):
    """Loss of one set's h [rows, generations, types], and dL/dh of every (row, generation)."""
    bins, at = _bins(s)
    q = torch.zeros(len(bins), dtype=torch.float64, device=h.device)
    q[torch.tensor(np.searchsorted(bins, target[0]), device=h.device)] = torch.tensor(target[1], device=h.device).double()
    q = q / q.sum()
    at = torch.tensor(at, device=h.device)
    ok = at >= 0
    hb = torch.zeros_like(q).index_add_(0, at[ok], h.sum(-1)[ok])
    S = hb.sum()
    r = hb / S - q
    gb = 2.0 / S * (r - (r * hb).sum() / S)
    return (r * r).sum(), torch.where(ok, gb[at.clamp_min(0)], torch.zeros_like(gb[:1]))


def _gradient(s, th, h, jm, js, g):
    p = torch.tensor(th[2], device=h.device)
    return torch.stack([(g * jm).sum((0, 1)), (g * js).sum((0, 1)), (g * h).sum((0, 1)) / p])


def _split(flat, base, shapes, i):
    T, K, R = shapes[i]
    return flat[:, base[i]:base[i] + R * K * T].reshape(3, R, K, T)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("simulate", "plan", "batch"):
        return None
    if kind in ("autograd", "calibrate"):
        sets, targets = _fit(case, seed)
    else:
        sets = _inputs(case, seed)
    theta = [np.stack([s["mean"], s["sd"], s["proportion"]]) for s in sets]
    if kind != "calibrate":
        flat, base, shapes = _walk(sets, theta, case["beta"])
        if kind == "jacobian":
            return {"h": flat[0], "jac": flat[1:]}
        h, jm, js = _split(flat, base, shapes, 0)
        if kind == "forward":
            return h
        if kind == "adjoint":
            return _gradient(sets[0], theta[0], h, jm, js, _cotangent(tuple(h.shape), seed).to(h.device))
        loss, g = _loss(h, sets[0], targets[0])
        return {"loss": loss, "grad": _gradient(sets[0], theta[0], h, jm, js, g.unsqueeze(-1))}
    # Adam (Kingma & Ba) on log mean, log sd and proportion logits; with a
    # stride the gradient walks the class of cells after the loss's
    stride, x, losses = case["stride"], [], []
    for th in theta:
        x.append(np.stack([np.log(np.where(th[0] < 0, 1.0, th[0])), np.log(np.where(th[0] < 0, 1.0, th[1])), np.log(th[2])]))
    m1, m2 = [np.zeros_like(a) for a in x], [np.zeros_like(a) for a in x]
    for t in range(case["steps"]):
        flat, base, shapes = _walk(sets, theta, case["beta"], stride, t)
        grad_flat = flat if stride == 1 else _walk(sets, theta, case["beta"], stride, t + 1)[0]
        losses = []
        for i, s in enumerate(sets):
            loss, g = _loss(_split(flat, base, shapes, i)[0], s, targets[i])
            h, jm, js = _split(grad_flat, base, shapes, i)
            gr = _gradient(s, theta[i], h, jm, js, g.unsqueeze(-1)).cpu().numpy()
            losses.append(float(loss))
            th, move = theta[i], theta[i][0] >= 0
            gx = np.stack([gr[0] * th[0] * move, gr[1] * th[1] * move, th[2] * (gr[2] - (th[2] * gr[2]).sum())])
            m1[i] = 0.9 * m1[i] + 0.1 * gx
            m2[i] = 0.999 * m2[i] + 0.001 * gx * gx
            x[i] = x[i] - LR / (1 - 0.9 ** (t + 1)) * m1[i] / (np.sqrt(m2[i]) / math.sqrt(1 - 0.999 ** (t + 1)) + 1e-8)
            x[i][1] = np.where(move, np.minimum(x[i][1], x[i][0] + math.log(0.8)), x[i][1])
            p = np.exp(x[i][2] - x[i][2].max())
            theta[i] = np.stack([np.where(move, np.exp(x[i][0]), -1.0), np.where(move, np.exp(x[i][1]), -1.0), p / p.sum()])
    return {"theta": np.concatenate([th.reshape(-1) for th in theta]), "loss": np.array(losses)}
