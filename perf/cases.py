"""The chemistry step's timed cases: what a program using maxichem_amd has the GPU do, through its public entry points.

A case is a dict of plain values. Its "path" says which entry point it stands for:

- call: CudaSolver.launch, one call of dt per cell (the whole result with its flags);
- graph: CudaSolver.capture, one replay of the captured call, as a time loop that calls on fixed tensors does;
- jvp: ADSolver.jvp, the call and its tangents along random directions (the step control differentiated);
- vjp: ADSolver.vjp, the call and every input's cotangent, the rate multipliers and the rate table among them;
- coupling: the GCM's conversions around a call (mass to mole, mole to mass, element moles, tracer totals);
- predict: Surrogate.predict, the learned warm start's inference on cold cells;
- gradients: one MLP forward, loss and backward on a training batch.

"start" is the state of the cells: "settled" ones come from a dark relaxation of 1e8 s and one lit call (a GCM's
steady time loop, dt = 300 s, a quarter of the cells lit); "cold" ones are a solar gas that has not been stepped, half
of them lit, dt log-uniform (a first call, or a spin-up). The networks are the stand-ins of standin.py: 69 species and
438 reactions (NCHO), 91 and 593 (SNCHO).
"""

from __future__ import annotations

import functools
import math
import random

import numpy as np
import torch

from maxichem_amd import standin
from maxichem_amd.coupling import composition
from maxichem_amd.kincuda import CudaSolver
from maxichem_amd.kincuda_ad import ADSolver
from maxichem_amd.learned import MLP, Surrogate, pad
from maxichem_amd.workloads import START_PER_H

DEVICE = "cuda"
# Per network: species, reactions, photolysis branches, elements, flops of a try and of a cell's rate coefficients
SIZES = {"NCHO": (69, 438, 48, 5, 163698, 9090), "SNCHO": (91, 593, 61, 6, 295529, 12306)}
# Mean tries per cell of a call: settled cells of dt = 300 s, cold ones of dt up to 1e4 s
TRIES = {"settled": 2.1, "cold": 100.0}


def listed() -> list[dict]:
    return [
        # a handful of cells, as a box model or one column of a coarse model calls every step: launches and host work
        {"name": "call_ncho_16", "path": "call", "network": "NCHO", "cells": 16, "start": "settled"},
        # a column model's first call: few cells with many tries each, as long as its costliest cell
        {"name": "call_ncho_256_cold", "path": "call", "network": "NCHO", "cells": 256, "start": "cold"},
        # one GPU's share of a small GCM grid in its time loop, replayed as a graph
        {"name": "graph_ncho_4096", "path": "graph", "network": "NCHO", "cells": 4096, "start": "settled"},
        # the whole GCM grid of the bench's call sequence
        {"name": "call_ncho_65536", "path": "call", "network": "NCHO", "cells": 65536, "start": "settled"},
        # the sulfur network (its lead rows and LDS footprint take other paths), an odd number of cells
        {"name": "call_sncho_8191", "path": "call", "network": "SNCHO", "cells": 8191, "start": "settled"},
        # a spin-up: cold cells of uneven stiffness that fill the GPU
        {"name": "call_ncho_8192_cold", "path": "call", "network": "NCHO", "cells": 8192, "start": "cold"},
        # a bounded call budget: the cells that do not finish in it go through the pivoting recovery
        {"name": "recover_ncho_500", "path": "call", "network": "NCHO", "cells": 500, "start": "cold",
         "max_steps": 40},
        # sensitivities along a few directions (an ensemble's perturbations) on a GCM's share
        {"name": "jvp_ncho_1024x8", "path": "jvp", "network": "NCHO", "cells": 1024, "start": "settled",
         "directions": 8},
        # gradients of a loss over a column's cells with respect to every input
        {"name": "vjp_ncho_64", "path": "vjp", "network": "NCHO", "cells": 64, "start": "settled"},
        # the conversions of one GCM step over the whole grid
        {"name": "coupling_65536_f64", "path": "coupling", "network": "NCHO", "cells": 65536, "dtype": "float64"},
        # the learned warm start of a grid's first call
        {"name": "predict_ncho_65536", "path": "predict", "network": "NCHO", "cells": 65536},
        # one training step's gradients at the surrogate's own batch size
        {"name": "gradients_ncho_8192", "path": "gradients", "network": "NCHO", "cells": 8192},
    ]  # fmt: skip


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random) -> dict:
    path = rng.choice(("call", "call", "call", "graph", "recover", "jvp", "vjp", "coupling", "predict", "gradients"))
    case = {"path": path, "network": rng.choice(("NCHO", "NCHO", "SNCHO"))}
    if path in ("call", "graph"):
        case["start"] = rng.choice(("settled", "settled", "cold"))
        case["cells"] = _log_int(rng, 1, {"settled": 32768, "cold": 3000}[case["start"]])
    elif path == "recover":  # a call whose budget is short
        case.update(path="call", network="NCHO", start="cold", cells=_log_int(rng, 16, 500),
                    max_steps=rng.randint(30, 60))  # fmt: skip
    elif path == "jvp":
        case.update(network="NCHO", start="settled", cells=_log_int(rng, 1, 1000), directions=rng.randint(1, 8))
    elif path == "vjp":
        case.update(network="NCHO", start="settled", cells=_log_int(rng, 1, 60))
    elif path == "coupling":
        case.update(cells=_log_int(rng, 16, 60000), dtype=rng.choice(("float64", "float32")))
    else:
        case["cells"] = _log_int(rng, 64, 60000 if path == "predict" else 8000)
    return case


# ---- inputs ----


@functools.lru_cache(maxsize=None)
def _network(name: str):
    return standin.load(name)


def _generator(seed: int) -> torch.Generator:
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _uniform(g, *shape):
    return torch.rand(*shape, generator=g, device=DEVICE, dtype=torch.float64)


def _log_uniform(g, lo: float, hi: float, *shape):
    return 10.0 ** (math.log10(lo) + (math.log10(hi) - math.log10(lo)) * _uniform(g, *shape))


def _solar_gas(net, g, cells: int) -> torch.Tensor:
    """Solar elements in H2, He, H2O, CH4, CO, CO2, NH3, N2 (and H2S) with each cell's own C and N splits, the other
    species at 1e-30, rows summing to 1 (the gas of workloads.solar_gas)."""
    idx = {q: i for i, q in enumerate(net.species)}
    u, w = _uniform(g, cells), _uniform(g, cells)
    c, o, n = START_PER_H["C"], START_PER_H["O"], START_PER_H["N"]
    s = START_PER_H["S"] if "H2S" in idx else 0.0
    co, co2 = c * 0.9 * (1.0 - u), c * 0.1 * (1.0 - u)
    moles = {"CH4": c * u, "CO": co, "CO2": co2, "H2O": o - co - 2.0 * co2, "NH3": n * w, "N2": n * (1.0 - w) / 2.0,
             "He": torch.full_like(u, START_PER_H["He"])}  # fmt: skip
    moles["H2"] = (1.0 - 2.0 * moles["H2O"] - 4.0 * moles["CH4"] - 3.0 * moles["NH3"] - 2.0 * s) / 2.0
    if s:
        moles["H2S"] = torch.full_like(u, s)
    x = torch.full((cells, len(net.species)), 1e-30, dtype=torch.float64, device=DEVICE)
    for q, m in moles.items():
        x[:, idx[q]] = m
    return x / x.sum(1, keepdim=True)


def _forcing(g, cells: int):
    return _log_uniform(g, 300.0, 3000.0, cells).clamp(300.0, 3000.0), _log_uniform(g, 1e2, 1e9, cells)


def _inputs(case: dict, seed: int, net, solver) -> dict:
    """x, T, P, dt, h, J of the timed call."""
    g = _generator(seed)
    B, nj = case["cells"], len(net.photo)
    T, P = _forcing(g, B)
    x = _solar_gas(net, g, B)
    h = torch.full_like(T, 1e-8)
    J = _log_uniform(g, 1e-9, 1e-3, B, nj)
    if case["start"] == "cold":
        J[_uniform(g, B) < 0.5] = 0.0
        return {"x": x, "T": T, "P": P, "dt": _log_uniform(g, 1e1, 1e4, B), "h": h, "J": J}
    lit = torch.zeros(B, dtype=torch.bool, device=DEVICE)
    lit[torch.argsort(P)[: max(1, B // 4)]] = True  # the quarter of the lowest pressures
    J[~lit] = 0.0
    r = solver(x, T, P, torch.full_like(T, 1e8), h, J=torch.zeros_like(J))
    dt = torch.full_like(T, 300.0)
    r = solver(r.x, T, P, dt, r.h, J=J)
    return {"x": r.x, "T": T, "P": P, "dt": dt, "h": r.h, "J": J}


def prepare(case: dict, seed: int) -> dict:
    net = _network(case["network"])
    path, B = case["path"], case["cells"]
    state = {"path": path}
    if path in ("call", "graph"):
        solver = CudaSolver(net, DEVICE, photo=True)
        d = _inputs(case, seed, net, solver)
        state.update(solver=solver, inputs=[d[k] for k in ("x", "T", "P", "dt", "h")], options={"J": d["J"]})
        if "max_steps" in case:
            state["options"]["max_steps"] = case["max_steps"]
        if path == "graph":
            state["graph"] = solver.capture(*state["inputs"], **state["options"])
    elif path in ("jvp", "vjp"):
        solver = ADSolver(net, DEVICE, photo=True)
        d = _inputs(case, seed, net, solver)
        g = _generator(seed + 1000003)

        def normal(*shape):
            return torch.randn(*shape, generator=g, device=DEVICE, dtype=torch.float64)

        state.update(solver=solver, inputs=[d[k] for k in ("x", "T", "P", "dt", "h")], J=d["J"])
        if path == "jvp":  # relative perturbations of every input
            D = case["directions"]
            state["tangents"] = [normal(D, B, net_x.shape[1]) * net_x if net_x.dim() == 2 else normal(D, B) * net_x
                                 for net_x in state["inputs"]]  # fmt: skip
            state["dJ"] = normal(D, *d["J"].shape) * d["J"]
        else:
            state["gx"], state["gh"] = normal(B, len(net.species)), normal(B)
    elif path == "coupling":
        dtype = getattr(torch, case["dtype"])
        g = _generator(seed)
        mw = composition.molar_masses(net.atoms, net.elements).to(DEVICE)
        x = _solar_gas(net, g, B) * (0.5 + _uniform(g, B, len(net.species)))  # transported: not summing to 1
        q = x * mw
        q = q / q.sum(1, keepdim=True) * (0.9 + 0.1 * _uniform(g, B))[:, None]
        atoms = torch.from_numpy(np.ascontiguousarray(net.atoms, np.float64)).to(DEVICE)
        state.update(q=q.to(dtype), mw=mw.to(dtype), atoms=atoms.to(dtype), mass=q.to(dtype).sum(1),
                     cell_mass=_log_uniform(g, 1e10, 1e14, B).to(dtype))  # fmt: skip
    elif path == "predict":
        g = _generator(seed)
        T, P = _forcing(g, B)
        x = _solar_gas(net, g, B)
        J = _log_uniform(g, 1e-9, 1e-3, B, len(net.photo))
        J[_uniform(g, B) < 0.5] = 0.0
        dt = _log_uniform(g, 1e1, 1e6, B)
        sur = Surrogate(net, DEVICE, seed=seed)
        # the standardisation of calls that move each species by about a factor of three
        x1 = x * 10.0 ** (_uniform(g, *x.shape) - 0.5)
        sur.standardise({"x0": x, "T": T, "P": P, "dt": dt, "J": J, "x1": x1 / x1.sum(1, keepdim=True),
                         "h1": dt * _log_uniform(g, 1e-4, 1.0, B), "steps": torch.round(200.0 * _uniform(g, B))})  # fmt: skip
        state.update(surrogate=sur, inputs=[x, T, P, dt, J])
    else:  # gradients: standardised features and targets
        g = _generator(seed)
        n_in, n_out = len(net.species) + 3 + len(net.photo), len(net.species) + 2
        mlp = MLP(n_in, n_out, DEVICE, seed=seed)
        X = torch.zeros(pad(B), mlp.dims[0], dtype=torch.float32, device=DEVICE)
        X[:B, :n_in] = torch.randn(B, n_in, generator=g, device=DEVICE)
        T = torch.randn(B, n_out, generator=g, device=DEVICE)
        state.update(mlp=mlp, X=mlp.to_bf16(X), T=T, w=torch.ones(n_out, device=DEVICE), rows=B)
    return state


def run(state: dict):
    path = state["path"]
    if path == "call":
        return state["solver"].launch(*state["inputs"], **state["options"])
    if path == "graph":
        return state["graph"].replay()
    if path == "jvp":
        return state["solver"].jvp(*state["inputs"], *state["tangents"], J=state["J"], dJ=state["dJ"])
    if path == "vjp":
        return state["solver"].vjp(*state["inputs"], state["gx"], gh=state["gh"], J=state["J"])
    if path == "coupling":
        q, mw, atoms = state["q"], state["mw"], state["atoms"]
        x = composition.mass_to_mole(q, mw)
        q1 = composition.mole_to_mass(x, mw, state["mass"])
        return (x, q1, composition.element_moles(q1, mw, atoms),
                composition.tracer_totals(q1, state["cell_mass"], mw, atoms))  # fmt: skip
    if path == "predict":
        h0, cost, _ = state["surrogate"].predict(*state["inputs"], 1e-12, proposals=False)
        return h0, cost
    mlp = state["mlp"]
    Y = mlp.forward(state["X"], keep=True)
    mlp.backward(mlp.loss_grad(Y, state["T"], state["w"], state["rows"]))
    return Y, [ly.gw for ly in mlp.layers], [ly.gb for ly in mlp.layers]


def _layer_dims(case: dict) -> list[int]:
    ns, _, nj, _, _, _ = SIZES[case["network"]]
    return [ns + 3 + nj, 256, 256, 256, 256, ns + 2]


def work(case: dict) -> dict:
    ns, nr, nj, ne, per_try, per_rates = SIZES[case["network"]]
    path, B = case["path"], case["cells"]
    if path in ("call", "graph", "jvp", "vjp"):
        row = 8 * (2 * ns + nj + 6) + 8  # x in and out, J, T, P, dt, h in and out, steps; done and flag
        tries = TRIES[case["start"]]
        flops = B * (tries * per_try + per_rates)
        if path in ("call", "graph"):
            return {"bytes": B * row, "flops": flops}
        # a direction's tangent of a try: six dual evaluations of the right-hand side and four solves, about two tries
        D = case["directions"] if path == "jvp" else ns + 4 + nr
        io = 8 * (2 * ns + nj + 6) * D if path == "jvp" else 8 * (2 * ns + nj + nr + 6)
        return {"bytes": B * (row + io), "flops": flops + D * B * tries * 2 * per_try}
    if path == "coupling":
        size = {"float64": 8, "float32": 4}[case["dtype"]]
        # q in, x and the new q out (its moles and totals can come from the same pass), the elements' moles
        return {"bytes": B * size * (3 * ns + ne + 2), "flops": B * ns * (8 + 4 * ne)}
    dims = _layer_dims(case)
    products = sum(a * b for a, b in zip(dims, dims[1:]))
    if path == "predict":
        return {"bytes": 8 * B * (ns + nj + 5) + 2 * products, "flops": 2 * B * products}
    return {"bytes": B * (2 * dims[0] + 8 * dims[-1]) + 6 * products,
            "flops": 2 * B * (3 * products - dims[0] * dims[1])}  # fmt: skip


# ---- the same outputs in 64 bits ----


def _mlp64(mlp: MLP, X: torch.Tensor, keep: list | None = None) -> torch.Tensor:
    a = X
    for l, ly in enumerate(mlp.layers):
        z = a @ ly.w.double().T + ly.b.double()
        if keep is not None:
            keep.append((a, z))
        a = torch.nn.functional.gelu(z) if l < mlp.depth else z
    return a


def exact(case: dict, seed: int):
    """The coupling's and the network's outputs in float64. A call's have none: its step control's decisions make the
    result what it is (a step accepted or not at the margin is another trajectory), so there is no value apart from
    the method's own."""
    path = case["path"]
    if path in ("call", "graph", "jvp", "vjp"):
        return None
    state = prepare(case, seed)
    if path == "coupling":
        q, mw, atoms, mass, cm = (state[k].double() for k in ("q", "mw", "atoms", "mass", "cell_mass"))
        n = q / mw
        x = n / n.sum(1, keepdim=True)
        m = x * mw
        q1 = m * (mass / m.sum(1))[:, None]
        e = (q1 / mw) @ atoms
        return x, q1, e, torch.cat([(q1.sum(1) * cm).sum()[None], (e * cm[:, None]).sum(0)])
    if path == "predict":
        sur, (x, T, P, dt, J) = state["surrogate"], state["inputs"]
        f = (sur.raw_features(x, T, P, dt, J) - sur.mu_in.double()) / sur.sd_in.double()
        X = torch.zeros(x.shape[0], sur.mlp.dims[0], dtype=torch.float64, device=DEVICE)
        X[:, : f.shape[1]] = f
        y = _mlp64(sur.mlp, X)[:, : sur.n_out] * sur.sd_out.double() + sur.mu_out.double()
        return torch.minimum(torch.exp(y[:, 0]).clamp(min=1e-12), dt), torch.expm1(y[:, 1].clamp(min=0.0))
    mlp, rows = state["mlp"], state["rows"]
    X = state["X"].view(torch.bfloat16).double()
    kept: list = []
    Y = _mlp64(mlp, X, kept)
    d = torch.zeros_like(Y)
    n_out = state["T"].shape[1]
    d[:rows, :n_out] = 2.0 * state["w"].double() * (Y[:rows, :n_out] - state["T"].double()) / (rows * n_out)
    gw, gb = [None] * len(mlp.layers), [None] * len(mlp.layers)
    for l in range(mlp.depth, -1, -1):
        a, _ = kept[l]
        gw[l], gb[l] = d.T @ a, d.sum(0)
        if l > 0:
            z = kept[l - 1][1]
            cdf = 0.5 * (1.0 + torch.erf(z / math.sqrt(2.0)))
            d = (d @ mlp.layers[l].w.double()) * (cdf + z * torch.exp(-0.5 * z * z) / math.sqrt(2.0 * math.pi))
    return Y, gw, gb
