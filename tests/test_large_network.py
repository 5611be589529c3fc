"""Networks of more species than the register LU takes: whole calls, a recovery and tangents by rows, against the oracle
(GPU)."""

import numpy as np
import oracle
import pytest
import test_jvp
import torch
from test_lu import network
from test_parity import compare, run_gpu, t

from maxichem_amd import _kernels, _tables
from maxichem_amd.kincuda import CudaSolver

CELLS = 48


def rated(species: int, seed: int = 0):
    """test_lu's network with rate coefficients of eight decades, so that steps are stiff, and an inert last species."""
    net = network(species, seed)
    rng = np.random.default_rng(seed)
    for r in net.reac:
        r["A"] = float(10.0 ** rng.uniform(-18.0, -10.0))
    return net


def inputs(species: int, cells: int, seed: int = 1):
    rng = np.random.default_rng(seed)
    x = 10.0 ** rng.uniform(-12.0, 0.0, (cells, species))
    return {"x": x / x.sum(1, keepdims=True), "T": rng.uniform(400.0, 2900.0, cells),
            "P": 10.0 ** rng.uniform(2.0, 7.0, cells), "dt": 10.0 ** rng.uniform(-2.0, 4.0, cells),
            "h": np.full(cells, 1e-8)}  # fmt: skip


def tangent_case(species: int):
    """inputs and directions as test_jvp's: x moved relatively with its sum kept, T and P by up to 0.5 %."""
    rng = np.random.default_rng(3)
    inp = {**inputs(species, CELLS), "J": np.zeros((CELLS, 0))}
    dx = inp["x"] * rng.uniform(-1.0, 1.0, inp["x"].shape)
    dx -= inp["x"] * dx.sum(1, keepdims=True)
    return inp, {"dx": 1e-2 * dx, "dT": 0.005 * inp["T"] * rng.uniform(-1, 1, CELLS),
                 "dP": 0.005 * inp["P"] * rng.uniform(-1, 1, CELLS), "dJ": np.zeros((CELLS, 0))}  # fmt: skip


@pytest.mark.gpu
@pytest.mark.parametrize("species", [93, 100])
def test_calls_and_recoveries_match_the_oracle(gpu, species):
    net = rated(species)
    tab = _tables.build(net)
    assert not _kernels.lu_layout(tab)["use"]
    inp = inputs(species, CELLS)
    orc = oracle.Oracle(tab)
    with CudaSolver(net, "cuda") as solver:
        want = orc.call(*(inp[k] for k in ("x", "T", "P", "dt", "h")))
        compare(f"{species} species", run_gpu(solver, inp, J=False), want, inp["x"], net.atoms)
        assert want["tries"].max() > 20
        budget = int(np.median(want["tries"]))  # about half of the cells go to the recovery
        want = orc.call(*(inp[k] for k in ("x", "T", "P", "dt", "h")), max_steps=budget)
        r = solver.launch(*(t(inp[k]) for k in ("x", "T", "P", "dt", "h")), max_steps=budget)
        assert int((r.flag == 1).sum()) > 8
        got = {**{k: v.cpu().numpy() for k, v in r._asdict().items()}, "tries": solver.tries.cpu().numpy()}
        compare(f"{species} species, {budget} tries", got, want, inp["x"], net.atoms)


@pytest.mark.gpu
def test_the_tangent_matches_the_frozen_differences(gpu, monkeypatch):
    from maxichem_amd.kincuda_ad import ADSolver

    net = rated(93)
    orc = oracle.Oracle(_tables.build(net))
    inp, d = tangent_case(93)
    with CudaSolver(net, "cuda") as solver:
        want = solver.launch(*(t(inp[k]) for k in ("x", "T", "P", "dt", "h")))
    zero = t(np.zeros(CELLS))
    with ADSolver(net, "cuda") as ad:
        r = ad.jvp(*(t(inp[k]) for k in ("x", "T", "P", "dt", "h")), t(d["dx"]), t(d["dT"]), t(d["dP"]), zero, zero,
                   adapt=False)  # fmt: skip
    for name in ("x", "h", "steps"):
        assert torch.equal(getattr(r, name), getattr(want, name)), name
    worst, compared = 0.0, 0
    for b in range(CELLS):
        fd, n = test_jvp.frozen_differences(orc, inp, d, b)
        with monkeypatch.context() as m:
            m.setattr(test_jvp, "EPS", 10.0 * test_jvp.EPS)
            coarse, _ = test_jvp.frozen_differences(orc, inp, d, b)
        if fd is None or coarse is None or n != int(want.steps[b]) or int(want.flag[b]) != 0:
            continue
        if np.abs(coarse - fd).max() > 2e-6 * np.abs(fd).max():
            continue  # a cell near its equilibrium: its tangent is as small as the differences' rounding
        worst = max(worst, float(np.abs(r.dx[b].cpu().numpy() - fd).max() / np.abs(fd).max()))
        compared += 1
    print(f"{compared} cells compared; largest tangent error against the differences {worst:.2e}")
    assert compared >= CELLS // 4 and worst <= test_jvp.TANGENT_TOLERANCE
