"""The tangent kernels' queue of (direction, cell) pairs and the adjoint's division of its columns, where they can go
wrong: one, two and an odd number of directions with recomputed cells among them, and launches that end inside a
kind of column, at its edges and after one column. Every comparison is bit for bit: a pair's arithmetic does not depend
on the launch it is in, and a cotangent taken with a one-hot gx is one product and zeros."""

import numpy as np
import pytest
import torch

from maxichem_amd import standin, workloads

CELLS = 12
MAX_STEPS = 30  # cells that have not settled need more tries: some go to the recovery, some pass


def case(seed: int):
    """Cells not yet relaxed (the tries vary from cell to cell), a quarter lit."""
    net = standin.load("NCHO")
    inp = workloads.config1(net.species, len(net.photo), cells=CELLS, seed=seed)
    cold = [torch.tensor(np.ascontiguousarray(inp[k]), device="cuda") for k in ("x", "T", "P", "dt_relax", "h")]
    return net, cold, torch.tensor(inp["J"], device="cuda")


def same(a, b):
    return torch.equal(torch.nan_to_num(a, nan=-7.0), torch.nan_to_num(b, nan=-7.0))


@pytest.mark.gpu
@pytest.mark.parametrize("D", [1, 2, 5])
@pytest.mark.parametrize("adapt", [False, True], ids=["frozen", "adaptive"])
def test_recomputed_cells_directions_are_each_alone(gpu, D, adapt):
    from maxichem_amd.kincuda_ad import ADSolver

    net, args, J = case(11)
    gen = torch.Generator().manual_seed(3)
    x = args[0]
    scale = [x, args[1], args[2], args[3], args[4]]
    tangents = [(1e-2 * (torch.rand((D, *s.shape), generator=gen, dtype=torch.float64) - 0.5)).cuda() * s for s in scale]
    with ADSolver(net, "cuda", photo=True) as ad:
        dlm = (torch.rand((D, CELLS, ad.nr), generator=gen, dtype=torch.float64) - 0.5).cuda()
        drc = (1e-3 * (torch.rand((D, ad.nr, 9), generator=gen, dtype=torch.float64) - 0.5)).cuda()
        dJ = (torch.rand((D, *J.shape), generator=gen, dtype=torch.float64) - 0.5).cuda() * J
        kw = dict(adapt=adapt, J=J, max_steps=MAX_STEPS)
        both = ad.jvp(*args, *tangents, dlm=dlm, drc=drc, dJ=dJ, **kw)
        flag, counts, tries = ad.flag.clone(), ad.fallback, ad.tries.clone()
        assert int((flag != 0).sum()) > 0
        for d in range(D):
            one = ad.jvp(*args, *[v[d] for v in tangents], dlm=dlm[d], drc=drc[d], dJ=dJ[d], **kw)
            assert same(both.dx[d], one.dx) and same(both.dh[d], one.dh)
            assert same(both.x, one.x) and same(both.h, one.h) and torch.equal(both.steps, one.steps)
            assert torch.equal(both.done, one.done) and torch.equal(flag, ad.flag) and torch.equal(tries, ad.tries)
            assert ad.fallback == counts  # the last call's: each cell counted once


@pytest.mark.gpu
@pytest.mark.parametrize("size", [1, 23, 69, 70, 71])
def test_adjoint_columns_do_not_depend_on_the_launches(gpu, monkeypatch, size):
    from maxichem_amd import kincuda_ad

    net, args, J = case(13)
    rates = size != 1  # one column a launch: without the reactions' hundreds
    hot = torch.arange(CELLS, device="cuda") * 5 % len(net.species)
    gx = torch.zeros_like(args[0]).scatter_(1, hot[:, None], 1.0)
    gh = torch.linspace(0.5, 1.5, CELLS, dtype=torch.float64, device="cuda")
    with kincuda_ad.ADSolver(net, "cuda", photo=True) as ad:
        run = lambda: ad.vjp(*args, gx, gh=gh, J=J, max_steps=MAX_STEPS, rates=rates)  # noqa: E731
        whole = run()
        per = 8 * CELLS * (2 * ad.ns + 4 + ad.nj + ad.nr)
        monkeypatch.setattr(kincuda_ad, "COLUMN_BYTES", size * per)
        parts = run()
        assert torch.equal(whole.x, parts.x) and torch.equal(whole.steps, parts.steps)
        for a, b in zip(whole.cotangents, parts.cotangents, strict=True):
            assert (a is None and b is None) or same(a, b)
