"""The framework's main paths as timed cases, each with its work, tolerance and an
independent 64-bit result.

A case is a dict of plain values; ``kind`` picks the path:

  step     the closed loop of an interactive program on ball-and-stick cells: write the
           injected currents through variable handles, one ``fadvance``, read the somas;
  run      a whole simulation: ``finitialize``, ``run``, the monitored traces and the final
           voltages (configurations 1-4 of ``heliox_amd.synth``);
  train    one training step: taped forward run, adjoint, gradients, Adam (configurations
           3 and 5);
  replay   the learning-rule replay over host signals, dw and dx;
  learn    signal capture on a running model, then the cached replay.

Morphologies come from ``build_config`` (seeded there); what varies from seed to seed are
the conductances, the synaptic weights, the injected currents, the initial voltage, the
targets, the signals and the kernels.
"""
from __future__ import annotations

import copy
import functools
import math

import numpy as np
import torch

from heliox_amd import Sim, build_config, learn
from heliox_amd.spec import VecPlaySpec

DT = 0.025
DEV = "cuda" if torch.cuda.is_available() else "cpu"


# ------------------------------------------------------------------------------- cases
def listed():
    return [
        # an agent stepping a handful of small cells one step at a time: pure latency
        {"name": "step_ball_stick", "kind": "step", "config": 1, "cells": 8},
        # the first benchmark configuration at its own size: 1000 unbranched cells
        {"name": "run_ball_stick", "kind": "run", "config": 1, "cells": 1000, "steps": 400},
        # branched cells of 500 compartments, synapses driven by spike trains
        {"name": "run_tree", "kind": "run", "config": 2, "cells": 1500, "steps": 200},
        # a few detailed pyramidal cells, conductances varying per compartment (fitted models)
        {"name": "run_pyramidal_few", "kind": "run", "config": 3, "cells": 21, "steps": 200, "varied": True},
        # many pyramidal cells: the benchmark's workload, bandwidth bound
        {"name": "run_pyramidal", "kind": "run", "config": 3, "cells": 1000, "steps": 200},
        # recurrent network: detector-driven netcons, gap junctions, VecPlay currents
        {"name": "run_network", "kind": "run", "config": 4, "cells": 4000, "steps": 300},
        # fitting 500-compartment cells: taped forward, adjoint, Adam
        {"name": "train_tree", "kind": "train", "config": 5, "cells": 200, "steps": 200},
        # fitting detailed cells, calcium and Ih conductances among the parameters
        {"name": "train_pyramidal", "kind": "train", "config": 3, "cells": 12, "steps": 100},
        # a small circuit's replay: two dense blocks, few ticks
        {"name": "replay_small", "kind": "replay", "n": 96, "block": 64, "klen": 8, "ticks": 64, "precise": True,
         "inputs": 4, "outputs": 9, "thr": 1e6},
        # odd block sizes that fill no tile, the norm clip active
        {"name": "replay_ragged", "kind": "replay", "n": 701, "block": 121, "klen": 24, "ticks": 160, "precise": True,
         "inputs": 7, "outputs": 33, "thr": 2.0},
        # the learn surface's benchmark shape
        {"name": "replay_large", "kind": "replay", "n": 2048, "block": 128, "klen": 64, "ticks": 128, "precise": True,
         "inputs": 16, "outputs": 64, "thr": 1e6},
        # forward run with captured signals, then their replay
        {"name": "learn_tree", "kind": "learn", "config": 2, "cells": 40, "steps": 400, "k_mul": 4, "klen": 16,
         "block": 100},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "run", "run", "run", "train", "replay", "replay", "learn"])
    if kind == "step":
        return {"kind": "step", "config": 1, "cells": _log(rng, 1, 200)}
    if kind == "run":
        config = rng.choice([1, 2, 3, 4])
        cells = {1: (2, 1000), 2: (3, 1500), 3: (1, 500), 4: (20, 4000)}[config]
        case = {"kind": "run", "config": config, "cells": _log(rng, *cells), "steps": rng.randint(40, 200)}
        if config == 3:
            case["varied"] = rng.random() < 0.5
        return case
    if kind == "train":
        config = rng.choice([3, 5])
        cells = (1, 12) if config == 3 else (2, 200)
        return {"kind": "train", "config": config, "cells": _log(rng, *cells), "steps": rng.randint(30, 100)}
    if kind == "replay":
        n = _log(rng, 5, 1600)
        return {"kind": "replay", "n": n, "block": _log(rng, min(n, 5), min(n, 200)), "klen": _log(rng, 1, 64),
                "ticks": _log(rng, 8, 128), "precise": rng.random() < 0.8, "inputs": rng.randint(1, min(n, 16)),
                "outputs": rng.randint(1, min(n, 64)), "thr": rng.choice([1e6, 0.5])}
    return {"kind": "learn", "config": 2, "cells": _log(rng, 2, 60), "steps": rng.randint(80, 400),
            "k_mul": rng.randint(1, 5), "klen": _log(rng, 1, 32), "block": rng.randint(7, 128)}


# ------------------------------------------------------------------------------ inputs
@functools.lru_cache(maxsize=2)
def _base(config, cells, tstop):
    return build_config(config, cells, tstop)


def _spec(case, seed):
    """The model of a case: the configuration's morphology with the seed's conductances,
    weights and currents.  Returns (spec, v_init)."""
    steps = case.get("steps", 0)
    spec = copy.deepcopy(_base(case["config"], case["cells"], max(1.0, math.ceil(steps * DT))))
    rng = np.random.default_rng([seed, case["config"], case["cells"]])
    cell = spec.cell_of_node()
    per_cell = lambda nodes, lo=0.9, hi=1.1: rng.uniform(lo, hi, spec.ncell)[cell[nodes]]   # noqa: E731
    for mech, var in (("hh", "gnabar"), ("hh", "gkbar"), ("pas", "g_pas")):
        if mech in spec.mechs and not (case["config"] == 3 and mech == "pas" and not case.get("varied")):
            m = spec.mechs[mech]
            m.params[var] = m.params[var] * per_cell(m.nodes)
    if case.get("varied"):
        for mech, var in (("pas", "g_pas"), ("Ca_HVA", "gbar"), ("hd_la", "ghdbar"), ("CaDynamics_E2", "decay")):
            m = spec.mechs[mech]
            m.params[var] = m.params[var] * rng.uniform(0.8, 1.25, m.n)
        spec.cm = spec.cm * rng.uniform(0.9, 1.1, spec.nnode)
    for nc in spec.netcons.values():
        nc.weight = nc.weight * rng.uniform(2.0, 6.0, nc.weight.size)
    if "IClamp" in spec.mechs and case["config"] == 1:
        ic = spec.mechs["IClamp"]
        ic.params["delay"] = np.full(ic.n, 0.0 if case["kind"] == "step" else 1.0)
        ic.params["amp"] = rng.uniform(0.1, 0.5, ic.n)
    if case["config"] == 4:
        # currents strong enough that the driven cells fire within the window
        amp = rng.uniform(2.0, 3.0, len(spec.vecplay))
        spec.vecplay = [VecPlaySpec(p.mech, p.var, p.idx, p.tvec, a * np.sin(2 * math.pi * p.tvec / 25.0))
                        for p, a in zip(spec.vecplay, amp)]
    if case["config"] in (2, 3, 5):
        # the trains of the benchmark, six times as fast, so that a short window sees them
        spec.vecstim_times = spec.vecstim_times / 6.0
    return spec, float(rng.uniform(-68.0, -62.0))


def _tstop(case):
    """A stop time that is the case's number of steps (``run`` truncates tstop / dt)."""
    return (case["steps"] + 0.25) * DT


def _trainable(config):
    tied = (("hh", "gnabar"), ("hh", "gkbar"), ("pas", "g_pas"))
    if config == 3:
        return tied + (("Ca_HVA", "gbar"), ("hd_la", "ghdbar")), ("Exp2Syn", "weight")
    return tied, ("ExpSyn", "weight")


LR = 1e-7


def _target(case, seed, ncell):
    rng = np.random.default_rng([seed, 77])
    t = np.arange(1, case["steps"] + 1)[:, None] * DT
    phase = rng.uniform(0, 2 * math.pi, ncell)
    return -64.0 + 3.0 * np.sin(2 * math.pi * t / 20.0 + phase) + rng.normal(0, 0.2, (case["steps"], ncell))


def _blocks(total, block, klen, seed, gain):
    rng = np.random.default_rng([seed, 5])
    sizes = [block] * (total // block) + ([total % block] if total % block else [])
    return [(rng.standard_normal((b, b, klen), dtype=np.float32) * np.float32(gain / math.sqrt(b))) for b in sizes]


def _signals(case, seed):
    """Host signals, kernels and index maps of a replay."""
    rng = np.random.default_rng([seed, case["n"], case["ticks"]])
    n, T = case["n"], case["ticks"] + 1
    it = rng.standard_normal((n, T), dtype=np.float32)
    dv = rng.standard_normal((n, T), dtype=np.float32) * np.float32(0.3)
    dp = rng.standard_normal((n, T), dtype=np.float32) * np.float32(0.3)
    it[:, 0] = dv[:, 0] = dp[:, 0] = 0
    pre = np.where(rng.random(n) < 0.6, rng.integers(0, n, n), -1).astype(np.int32)
    po = np.sort(rng.choice(n, case["outputs"], replace=False)).astype(np.int32)
    pin = np.sort(rng.choice(n, case["inputs"], replace=False)).astype(np.int32)
    dl = rng.standard_normal((case["ticks"], case["outputs"]), dtype=np.float32)
    return {"it": it, "dv": dv, "dp": dp, "pre": pre, "po": po, "pin": pin, "dl": dl,
            "blocks": _blocks(n, case["block"], case["klen"], seed, 0.5), "dt": 0.05, "eps": 4.0}


def _learn_inputs(case, seed):
    spec, v_init = _spec(case, seed)
    n = spec.mechs["ExpSyn"].n
    rng = np.random.default_rng([seed, 9])
    ticks = case["steps"] // case["k_mul"]
    return {"spec": spec, "v_init": v_init, "n": n, "ticks": ticks,
            "blocks": _blocks(n, min(case["block"], n), case["klen"], seed, 0.5),
            "scale": (rng.uniform(0.5, 1.5, n) * 50.0).astype(np.float32),
            "po": np.arange(0, n, 3, dtype=np.int32), "pin": np.array([1, n - 2], np.int32),
            "pre": np.where(rng.random(n) < 0.5, rng.integers(0, n, n), -1).astype(np.int32),
            "dl": rng.standard_normal((ticks, len(range(0, n, 3))), dtype=np.float32), "dt": 0.1, "eps": 4.0}


def prepare(case, seed):
    kind = case["kind"]
    g = Sim()
    if kind == "replay":
        s = _signals(case, seed)
        g.load_model_from_spec(_base(1, 1, 1.0), add_monitors=False)
        if g.set_dense_blocks_f32(s["blocks"]) != case["klen"]:
            raise RuntimeError(g.last_error())
        return {"case": case, "sim": g, **s}
    if kind == "learn":
        s = _learn_inputs(case, seed)
        spec = s["spec"]
        g.load_model_from_spec(spec, add_monitors=False)
        es = spec.mechs["ExpSyn"]
        cell = spec.cell_of_node()[es.nodes]
        handles = lambda vs: [g.get_variable_handle(*v) for v in vs]   # noqa: E731
        dest, n = np.arange(s["n"], dtype=np.int32), s["n"]
        sig = {"pure_i": learn.MappedSignal("pure_i", handles([("ExpSyn", "i", k) for k in range(n)]), dest, s["scale"]),
               "didv": learn.MappedSignal("didv", handles([("ExpSyn", "g", k) for k in range(n)]), dest, s["scale"]),
               "didvpre": learn.MappedSignal("didvpre", handles([("global", "v", int(c)) for c in cell]), dest,
                                             np.full(n, 4e-3, np.float32))}
        if g.set_dense_blocks_f32(s["blocks"]) != case["klen"]:
            raise RuntimeError(g.last_error())
        cap = learn.CaptureSpec(output_v_handles=handles([("global", "v", c) for c in range(spec.ncell)]), signals=sig,
                                tstop_ms=case["steps"] * DT, k_mul=case["k_mul"], percise=True, v_init=s["v_init"])
        return {"case": case, "sim": g, "cap": cap, **s}
    spec, v_init = _spec(case, seed)
    if kind == "train":
        g.load_model_from_spec(spec, add_monitors=False)
        g.tape_begin(case["steps"])
        opt = g.adam_create(0.9, 0.999, 1e-8)
        tied, syn = _trainable(case["config"])
        cell = spec.cell_of_node()
        for mech, var in tied:
            cn = cell[spec.mechs[mech].nodes]
            order = np.argsort(cn, kind="stable")
            for idx in np.split(order, np.flatnonzero(np.diff(cn[order])) + 1):
                g.adam_add_group(opt, mech, var, idx)
        for k in range(spec.mechs[syn[0]].n):
            g.adam_add_group(opt, syn[0], syn[1], [k])
        return {"case": case, "sim": g, "opt": opt, "v_init": v_init, "somas": np.arange(spec.ncell),
                "target": _target(case, seed, spec.ncell)}
    g.load_model_from_spec(spec, add_monitors=kind == "run")
    state = {"case": case, "sim": g, "v_init": v_init}
    if kind == "step":
        g.finitialize(v_init)
        state["amp_handles"] = [g.get_variable_handle("IClamp", "amp", k) for k in range(spec.ncell)]
        state["v_handles"] = [g.get_variable_handle("global", "v", k) for k in range(spec.ncell)]
        state["amps"] = np.random.default_rng([seed, 3]).uniform(0.0, 1.0, spec.ncell).tolist()
    return state


# --------------------------------------------------------------------------------- run
def run(state):
    case, g = state["case"], state["sim"]
    kind = case["kind"]
    if kind == "step":
        g.set_variables_by_handles(state["amp_handles"], state["amps"])
        g.fadvance()
        return np.array(g.get_variables_by_handles(state["v_handles"]))
    if kind == "run":
        g.finitialize(state["v_init"])
        g.run(_tstop(case))
        return {"traces": g.traces(), "v": g.get_array("global", "v")}
    if kind == "train":
        g.finitialize(state["v_init"])
        g.run(_tstop(case))
        loss = g.adjoint(state["somas"], state["target"])
        tied, syn = _trainable(case["config"])
        out = {"loss": loss}
        for mech, var in tied + (syn,):
            out[f"grad {mech} {var}"] = g.gradient(mech, var)
        g.adam_step(state["opt"], LR, 1.0)
        for mech, var in tied:
            out[f"new {mech} {var}"] = g.get_array(mech, var)
        return out
    if kind == "replay":
        dw = np.zeros(case["n"], np.float32)
        dx = np.zeros((state["pin"].size, case["ticks"]), np.float32)
        rc = g.replay_compute_dw_dx_from_signals_into(
            state["it"], state["dv"], state["dp"], state["dl"], state["po"], state["pin"], state["pre"], dw, dx,
            state["dt"], case["precise"], eps=state["eps"], grad_l2norm_threshold=case["thr"])
        if rc != 0:
            raise RuntimeError(g.last_error())
        return {"dw": dw, "dx": dx}
    pack = learn.capture_signals_cached(g, state["cap"], total_steps=case["steps"])
    grads = learn.replay_grads_from_cached_signals(
        g, dLtdv_lr_ot=state["dl"], poutput=state["po"], pre_of_col=state["pre"], dt_ms=state["dt"], percise=True,
        pinput=state["pin"], eps=state["eps"])
    return {"v": pack.output_vs_tn, "dw": grads.dw_out_n, "dx": grads.dx_lr_it}


# -------------------------------------------------------------------------------- work
# Per compartment and step: bytes of every array that influences the results read once and
# every state written once (8 B each), and flops with an exponential counted as 20.
_NODE = {1: 101, 2: 500, 3: 5000, 4: 200, 5: 500}
# node arrays v (read, written), a, b, cm; then mechanism data.  Configurations 1, 2, 4, 5
# carry pas everywhere and hh on 1, 50, 50, 50 of the compartments.
_HH_SHARE = {1: 1 / 101, 2: 0.1, 4: 0.25, 5: 0.1}
_SYN = {1: 0, 2: 10, 3: 200, 4: 100, 5: 10}


def _step_work(config, cells):
    n = cells * _NODE[config]
    if config == 3:
        bytes_ = n * (40 + 8 + 16 + 32 + 16 + 40)     # node, pas g, hh, Ca_HVA m h, Ih, calcium
        flops = n * 420.0
    else:
        bytes_ = n * (40 + 8 + 64 * _HH_SHARE[config])
        flops = n * (30 + 150 * _HH_SHARE[config])
    return bytes_ + cells * _SYN[config] * 32, flops + cells * _SYN[config] * 40


def _replay_work(n, sizes, klen, ticks, precise, inputs, outputs):
    area = sum(b * b for b in sizes)
    taps = sum(min(t, klen) for t in range(1, ticks + 1))
    flops = 2.0 * area * taps + (2.0 * n * area * taps if precise else 0.0)
    bytes_ = 4.0 * (n * (ticks + 1) * (3 if precise else 1) + area * klen + ticks * outputs + n + inputs * ticks)
    return bytes_, flops


def _sizes(n, block):
    return [block] * (n // block) + ([n % block] if n % block else [])


def work(case):
    kind = case["kind"]
    if kind == "replay":
        b, f = _replay_work(case["n"], _sizes(case["n"], case["block"]), case["klen"], case["ticks"], case["precise"],
                            case["inputs"], case["outputs"])
        return {"bytes": b, "flops": f}
    b, f = _step_work(case["config"], case["cells"])
    if kind == "step":
        return {"bytes": b, "flops": f}
    n = case["cells"] * _NODE[case["config"]]
    if kind == "run":
        return {"bytes": b * case["steps"] + 8.0 * n, "flops": f * case["steps"]}
    if kind == "train":
        # the tape is written and read once (v and the gates), the backward step costs about two forward ones
        tape = 16.0 * n * (7 if case["config"] == 3 else 1.3)
        return {"bytes": (3 * b + tape) * case["steps"], "flops": 3.0 * f * case["steps"]}
    ncol, ticks = 10 * case["cells"], case["steps"] // case["k_mul"]
    rb, rf = _replay_work(ncol, _sizes(ncol, min(case["block"], ncol)), case["klen"], ticks, True, 2, ncol // 3)
    return {"bytes": b * case["steps"] + rb, "flops": f * case["steps"] + rf}


def tolerance(case):
    """About four times what the paths differ from ``exact`` (measured over listed and drawn cases)."""
    kind = case["kind"]
    if kind in ("step", "run"):
        # 64 bits throughout: rounding of 1e-16 a step, grown along a spike's upstroke
        return {"rel": 5e-13, "max": 5e-11}
    if kind == "train":
        # 64 bits; gradients are sums of cancelling terms over the steps
        return {"rel": 5e-12, "max": 1e-9}
    # 32-bit sums over blocks and taps, fed back through the history
    return {"rel": 1.2e-6, "max": 5e-5}


# ------------------------------------------------------------------------------- exact
class _Tree:
    """x of the tree system, level by level, on all cells at once; differentiable."""

    def __init__(self, spec):
        self.n = n = spec.nnode
        parent = np.asarray(spec.parent, np.int64)
        depth = np.zeros(n, np.int64)
        for i in range(spec.ncell, n):
            depth[i] = depth[parent[i]] + 1
        order = np.argsort(depth, kind="stable")
        bounds = np.flatnonzero(np.diff(depth[order])) + 1
        self.levels = []
        for idx in np.split(order, bounds):
            par = parent[idx]
            by_par = np.argsort(par, kind="stable")
            idx, par = idx[by_par], par[by_par]
            self.levels.append((torch.from_numpy(idx).to(DEV), torch.from_numpy(np.maximum(par, 0)).to(DEV)))
        self.a = torch.from_numpy(np.array(spec.a, np.float64)).to(DEV)
        self.b = torch.from_numpy(np.array(spec.b, np.float64)).to(DEV)
        par = torch.from_numpy(np.maximum(parent, 0)).to(DEV)
        self.par = par
        self.nonroot = torch.from_numpy(parent >= 0).to(DEV)
        ax = torch.zeros(n, dtype=torch.float64, device=DEV)
        ax -= torch.where(self.nonroot, self.b, 0.0)
        ax.index_add_(0, par, torch.where(self.nonroot, -self.a, 0.0))
        self.axial = ax                                   # what the couplings add to the diagonal

    def coupling(self, v):
        """Axial current into every node: the right-hand side's axial terms."""
        dv = torch.where(self.nonroot, v[self.par] - v, torch.zeros_like(v))
        out = -self.b * dv
        return out.index_add(0, self.par, self.a * dv)

    def eliminate(self, d, r, up, down):
        """Solves with the couplings `up` (row parent, column child) and `down` (row child, column parent)."""
        d, r = d.clone(), r.clone()
        for idx, par in reversed(self.levels[1:]):
            f = up[idx] / d[idx]
            d.index_add_(0, par, -f * down[idx])
            r.index_add_(0, par, -f * r[idx])
        x = r / d
        for idx, par in self.levels[1:]:
            x[idx] = (r[idx] - down[idx] * x[par]) / d[idx]
        return x

    def solve(self, d, r):
        return _Solve.apply(self, d + self.axial, r)


class _Solve(torch.autograd.Function):
    @staticmethod
    def forward(ctx, tree, d, r):
        x = tree.eliminate(d, r, tree.a, tree.b)
        ctx.tree = tree
        ctx.save_for_backward(d, x)
        return x

    @staticmethod
    def backward(ctx, gx):
        d, x = ctx.saved_tensors
        gr = ctx.tree.eliminate(d, gx, ctx.tree.b, ctx.tree.a)
        return None, -gr * x, gr


def _vtrap(x, y):
    r = x / y
    small = r.abs() < 1e-6
    safe = torch.where(small, torch.ones_like(r), r)
    return torch.where(small, y * (1 - r / 2), y * safe / (torch.exp(safe) - 1))


def _hh_rates(v):
    am, bm = 0.1 * _vtrap(-(v + 40), 10.0), 4 * torch.exp(-(v + 65) / 18)
    ah, bh = 0.07 * torch.exp(-(v + 65) / 20), 1 / (torch.exp(-(v + 35) / 10) + 1)
    an, bn = 0.01 * _vtrap(-(v + 55), 10.0), 0.125 * torch.exp(-(v + 65) / 80)
    return ((am, bm), (ah, bh), (an, bn))


def _cahva_rates(v):
    ma, mb = 0.055 * _vtrap(-27.0 - v, 3.8), 0.94 * torch.exp((-75.0 - v) / 17.0)
    ha, hb = 0.000457 * torch.exp((-13.0 - v) / 50.0), 0.0065 / (torch.exp((-v - 15.0) / 28.0) + 1.0)
    return ((ma, mb), (ha, hb))


def _step_gates(x, rates, q10=1.0):
    return [g + (1 - torch.exp(-DT * q10 * (a + b))) * (a / (a + b) - g) for g, (a, b) in zip(x, rates)]


class _Model64:
    """The step loop of the benchmark configurations in torch, 64 bits."""

    def __init__(self, spec, v_init):
        self.spec, self.v_init = spec, v_init
        self.tree = _Tree(spec)
        t = lambda x: torch.from_numpy(np.ascontiguousarray(x, np.float64)).to(DEV)   # noqa: E731
        ix = lambda x: torch.from_numpy(np.ascontiguousarray(x, np.int64)).to(DEV)    # noqa: E731
        self.cm, self.area = t(spec.cm), t(spec.area)
        self.node = {k: ix(m.nodes) for k, m in spec.mechs.items()}
        self.p = {(k, c): t(v) for k, m in spec.mechs.items() for c, v in m.params.items()}
        for k, nc in spec.netcons.items():
            w = np.zeros(spec.mechs[k].n)
            w[nc.inst] = nc.weight
            self.p[(k, "weight")] = t(w)
        self.q10 = 3.0 ** ((spec.celsius - 6.3) / 10.0)
        self.qt = 4.5 ** ((spec.celsius - 33.0) / 10.0)

    def trains(self, steps):
        """Per step, the synapses that get an event of a spike train: (mech, instances)."""
        spec = self.spec
        ttab = [0.0]
        for _ in range(steps):
            ttab.append((ttab[-1] + DT / 2) + DT / 2)
        ttab = np.array(ttab)
        due = ttab + DT / 2
        out = {k: [] for k in range(steps)}
        for mech, nc in spec.netcons.items():
            stim = np.flatnonzero(nc.src_kind == 1)
            for k in stim:
                times = spec.vecstim_train(int(nc.src[k]))
                emit = np.searchsorted(due, times, side="left")
                for m in emit[emit < steps]:
                    at = int(np.searchsorted(due, ttab[m] + nc.delay[k], side="left"))
                    if max(at, m) < steps:
                        out[max(at, m)].append((mech, int(nc.inst[k])))
        self.ttab, self.due = ttab, due
        return {k: {mech: np.array([i for q, i in v if q == mech], np.int64) for mech in {q for q, _ in v}}
                for k, v in out.items() if v}

    def run(self, steps, sample=None):
        """Voltages after finitialize and after every step at the somas, and the final v; `sample(state)` is
        called at the same points."""
        spec, p, node, tree = self.spec, self.p, self.node, self.tree
        has = lambda m: m in spec.mechs and spec.mechs[m].n > 0      # noqa: E731
        zeros = lambda m: torch.zeros(spec.mechs[m].n, dtype=torch.float64, device=DEV)   # noqa: E731
        events = self.trains(steps)
        v = torch.full((spec.nnode,), self.v_init, dtype=torch.float64, device=DEV)
        S = {"v": v}
        if has("hh"):
            S["hh"] = [a / (a + b) for a, b in _hh_rates(v[node["hh"]])]
            S["ena"], S["ek"] = float(spec.mechs["na_ion"].params["erev"][0]), float(spec.mechs["k_ion"].params["erev"][0])
        if has("Ca_HVA"):
            S["ca"] = [a / (a + b) for a, b in _cahva_rates(v)]
            S["cai"] = torch.full_like(v, 5e-5)
            S["l"] = 1 / (1 + torch.exp(-(v - p["hd_la", "vhalfl"]) / -8.0))
            ktf = 1000.0 * 1.380649e-23 * (spec.celsius + 273.15) / 1.602176634e-19
        if has("ExpSyn"):
            S["g"], S["i"] = zeros("ExpSyn"), zeros("ExpSyn")
        if has("Exp2Syn"):
            S["A"], S["B"] = zeros("Exp2Syn"), zeros("Exp2Syn")
            t1, t2 = p["Exp2Syn", "tau1"], p["Exp2Syn", "tau2"]
            tp = t1 * t2 / (t2 - t1) * torch.log(t2 / t1)
            factor = 1 / (-torch.exp(-tp / t1) + torch.exp(-tp / t2))
        if has("HalfGap"):
            src = np.zeros(spec.mechs["HalfGap"].n, np.int64)
            src[spec.gap_halfgap] = spec.gap_src_node
            src = torch.from_numpy(src).to(DEV)
            vgap = v[src]
        det = {m: nc for m, nc in spec.netcons.items() if (nc.src_kind == 0).any()}
        above = np.zeros(len(spec.presyn_gid), bool)
        somas = torch.arange(spec.ncell, device=DEV)
        point = lambda m: 1e2 / self.area[node[m]]                   # noqa: E731
        trace = [v[somas]]
        if sample:
            sample(S)
        for k in range(steps):
            tk = self.ttab[k]
            if det:
                vv = v[torch.from_numpy(np.asarray(spec.presyn_node, np.int64)).to(DEV)].cpu().numpy()
                fire = np.flatnonzero((vv > spec.presyn_thr) & ~above)
                above = vv > spec.presyn_thr
                for m, nc in det.items():
                    for e in np.flatnonzero(np.isin(nc.src, fire)):
                        at = int(np.searchsorted(self.due, tk + nc.delay[e], side="left"))
                        if max(at, k) < steps:
                            slot = events.setdefault(max(at, k), {})
                            slot[m] = np.append(slot.get(m, np.zeros(0, np.int64)), int(nc.inst[e]))
            for m, inst in events.get(k, {}).items():
                at = torch.from_numpy(inst).to(DEV)
                w = p[m, "weight"][at]
                if m == "ExpSyn":
                    S["g"] = S["g"].index_add(0, at, w)
                else:
                    S["A"], S["B"] = (S[q].index_add(0, at, w * factor[at]) for q in "AB")
            tm = tk + DT / 2
            d = 1e-3 / DT * self.cm
            r = torch.zeros_like(v)
            if has("pas"):
                n, g = node["pas"], p["pas", "g_pas"]
                d, r = d.index_add(0, n, g), r.index_add(0, n, -g * (v[n] - p["pas", "e_pas"]))
            if has("hh"):
                n, (m_, h_, n_) = node["hh"], S["hh"]
                gna, gk, gl = p["hh", "gnabar"] * m_**3 * h_, p["hh", "gkbar"] * n_**4, p["hh", "gl"]
                vh = v[n]
                d = d.index_add(0, n, gna + gk + gl)
                r = r.index_add(0, n, -(gna * (vh - S["ena"]) + gk * (vh - S["ek"]) + gl * (vh - p["hh", "el"])))
            if has("IClamp"):
                ic, n = spec.mechs["IClamp"].params, node["IClamp"]
                amp = p["IClamp", "amp"]
                if spec.vecplay:
                    amp = amp.clone()
                    for q in spec.vecplay:
                        amp[q.idx] = float(np.interp(tm, q.tvec, q.yvec))
                on = torch.from_numpy((tm >= ic["delay"]) & (tm < ic["delay"] + ic["dur"])).to(DEV)
                r = r.index_add(0, n, torch.where(on, amp, 0.0) * point("IClamp"))
            if has("ExpSyn"):
                n, f = node["ExpSyn"], point("ExpSyn")
                S["i"] = S["g"] * (v[n] - p["ExpSyn", "e"])
                d, r = d.index_add(0, n, S["g"] * f), r.index_add(0, n, -S["i"] * f)
            if has("Exp2Syn"):
                n, f, g = node["Exp2Syn"], point("Exp2Syn"), S["B"] - S["A"]
                d, r = d.index_add(0, n, g * f), r.index_add(0, n, -g * (v[n] - p["Exp2Syn", "e"]) * f)
            if has("Ca_HVA"):
                eca = ktf / 2 * torch.log(2.0 / S["cai"])
                g = p["Ca_HVA", "gbar"] * S["ca"][0]**2 * S["ca"][1]
                ica, gl_ = g * (v - eca), p["hd_la", "ghdbar"] * S["l"]
                d, r = d + g + gl_, r - ica - gl_ * (v + 30.0)
            if has("HalfGap"):
                n, f, g = node["HalfGap"], point("HalfGap"), p["HalfGap", "g"]
                d, r = d.index_add(0, n, g * f), r.index_add(0, n, g * (vgap - v[n]) * f)
            v = v + tree.solve(d, r + tree.coupling(v))
            if has("HalfGap"):
                vgap = v[src]
            if has("Ca_HVA"):
                decay = p["CaDynamics_E2", "decay"]
                drive = -1e4 * ica * p["CaDynamics_E2", "gamma"] / (2 * 96485.3321233100184 * p["CaDynamics_E2", "depth"])
                S["cai"] = S["cai"] + (1 - torch.exp(-DT / decay)) * (drive * decay + p["CaDynamics_E2", "minCai"] - S["cai"])
                S["ca"] = _step_gates(S["ca"], _cahva_rates(v))
                a, bett = torch.exp(0.0378 * 2.2 * (v + 75.0)), torch.exp(0.0378 * 2.2 * 0.4 * (v + 75.0))
                taul = p["hd_la", "tau"] * bett / (self.qt * 0.011 * (1 + a))
                linf = 1 / (1 + torch.exp(-(v - p["hd_la", "vhalfl"]) / -8.0))
                S["l"] = S["l"] + (1 - torch.exp(-DT / taul)) * (linf - S["l"])
            if has("hh"):
                S["hh"] = _step_gates(S["hh"], _hh_rates(v[node["hh"]]), self.q10)
            if has("ExpSyn"):
                S["g"] = S["g"] * torch.exp(-DT / p["ExpSyn", "tau"])
            if has("Exp2Syn"):
                S["A"], S["B"] = S["A"] * torch.exp(-DT / t1), S["B"] * torch.exp(-DT / t2)
            S["v"] = v
            trace.append(v[somas])
            if sample:
                sample(S)
        return torch.stack(trace, 1), v


def _exact_replay(s, it, dv, dp, blocks, ticks, klen, precise, thr):
    """dw, dx of the replay; it, dv, dp are (T, n)."""
    t64 = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV).double()   # noqa: E731
    it, dv, dp, dl = t64(it), t64(dv), t64(dp), t64(s["dl"])
    n = it.shape[1]
    kern = [t64(b) for b in blocks]
    starts = np.concatenate([[0], np.cumsum([b.shape[0] for b in blocks])[:-1]])
    pre = torch.from_numpy(np.maximum(s["pre"], 0).astype(np.int64)).to(DEV)
    has_pre = torch.from_numpy(s["pre"] >= 0).to(DEV).double()
    po, pin = (torch.from_numpy(s[q].astype(np.int64)).to(DEV) for q in ("po", "pin"))
    dt, eps = float(np.float32(s["dt"])), float(np.float32(s["eps"]))
    hist = torch.zeros((klen, n, n), dtype=torch.float64, device=DEV)     # slot t % klen holds X of tick t
    dw, dx, gs = torch.zeros(n, dtype=torch.float64, device=DEV), [], 1.0
    for t in range(1, ticks + 1):
        tw = min(t, klen)
        taus = torch.arange(t - tw, t, device=DEV)
        d = torch.zeros((n, n), dtype=torch.float64, device=DEV)
        for K, s0 in zip(kern, starts):
            e0 = s0 + K.shape[0]
            d[s0:e0, s0:e0] = torch.einsum("iju,ui->ij", K[:, :, klen - tw:], it[taus + 1, s0:e0]) * dt * gs
            if precise:
                X = hist[taus % klen][:, :, s0:e0]
                W = K[:, :, klen - tw:]
                d[:, s0:e0] += dt * torch.matmul(X.permute(1, 0, 2).reshape(n, -1), W.permute(2, 1, 0).reshape(-1, K.shape[0]))
        l2 = float(d.norm())
        if l2 > thr:
            sc = thr / l2
            d, hist, dw, gs = d * sc, hist * sc, dw * sc, gs * sc
            dx = [c * sc for c in dx]
        w = d[:, po] @ dl[t - 1]
        dw = dw + w
        c = d[:, pin]
        dx.append((w[:, None] / (c + eps)).sum(0) * c.sum(0))
        if precise and t < ticks:
            hist[t % klen] = d * dv[t + 1] + d[:, pre] * has_pre * dp[t + 1]
    return {"dw": (dw / ticks).cpu().numpy(), "dx": torch.stack(dx, 1).cpu().numpy()}


def exact(case, seed):
    kind = case["kind"]
    if kind == "replay":
        s = _signals(case, seed)
        return _exact_replay(s, s["it"].T, s["dv"].T, s["dp"].T, s["blocks"], case["ticks"], case["klen"],
                             case["precise"], float(np.float32(case["thr"])))
    if kind == "learn":
        s = _learn_inputs(case, seed)
        model = _Model64(s["spec"], s["v_init"])
        cell = torch.from_numpy(s["spec"].cell_of_node()[s["spec"].mechs["ExpSyn"].nodes]).to(DEV)
        rows = []
        model_trace, _ = model.run(case["steps"], lambda S: rows.append(
            [x.float().cpu().numpy() for x in (S["i"], S["g"], S["v"][cell])]))
        T = s["ticks"] + 1
        sig = [np.zeros((T, s["n"]), np.float32) for _ in range(3)]
        for q, scale in enumerate((s["scale"], s["scale"], np.full(s["n"], 4e-3, np.float32))):
            for t in range(1, T):
                sig[q][t] = rows[t * case["k_mul"]][q] * scale
        out = _exact_replay(s, *sig, s["blocks"], s["ticks"], case["klen"], True, 1e6)
        return {"v": model_trace.T.cpu().numpy(), **out}
    if kind == "run" and case["config"] == 3 and case["steps"] * case["cells"] > 60000:
        return None                                       # over 20 s of level-by-level solves
    spec, v_init = _spec(case, seed)
    if kind == "step":
        amps = np.random.default_rng([seed, 3]).uniform(0.0, 1.0, spec.ncell)
        spec.mechs["IClamp"].params["amp"] = amps
        trace, _ = _Model64(spec, v_init).run(1)
        return trace[:, 1].cpu().numpy()
    model = _Model64(spec, v_init)
    if kind == "run":
        trace, v = model.run(case["steps"])
        return {"traces": trace[[m[2] for m in spec.monitors]].cpu().numpy(), "v": v.cpu().numpy()}
    tied, syn = _trainable(case["config"])
    for key in tied + (syn,):
        model.p[key].requires_grad_(True)
    trace, _ = model.run(case["steps"])
    target = torch.from_numpy(_target(case, seed, spec.ncell)).to(DEV)
    loss = ((trace[:, 1:].T - target) ** 2).mean()
    loss.backward()
    out = {"loss": float(loss)}
    for key in tied + (syn,):
        out["grad %s %s" % key] = model.p[key].grad.cpu().numpy()
    cell = torch.from_numpy(spec.cell_of_node()).to(DEV)
    for mech, var in tied:
        w, cn = model.p[mech, var].detach(), cell[model.node[mech]]
        mean = torch.zeros(spec.ncell, dtype=torch.float64, device=DEV).index_add_(0, cn, model.p[mech, var].grad)
        mean /= torch.bincount(cn, minlength=spec.ncell)
        # a tied group steps from its first instance's value and writes it to all of them
        at = np.unique(cn.cpu().numpy(), return_index=True)[1]
        new = w[torch.from_numpy(at).to(DEV)] - LR * mean / (mean.abs() + 1e-8)
        out[f"new {mech} {var}"] = new[cn].cpu().numpy()
    return out
