"""The two-dimensional LU of M0 against the LU by rows, and the solves by blocks against those by rows: the same bits, at
the edges of the slots (16 rows by 4 columns) and of the lead part (64 trailing rows), on random patterns (GPU)."""

import types
from pathlib import Path

import numpy as np
import pytest
import torch

from maxichem_amd import _hip, _kernels, _tables

pytestmark = pytest.mark.gpu
PROBE = Path(__file__).resolve().parent / "lu_probe.hip"


def network(species: int, seed: int):
    """Two-body reactions A + B -> C + D over so many species, between near ones and with a hub (the last species), as
    a network's sparse pattern with its dense end."""
    rng = np.random.default_rng(seed)
    reac, S = [], np.zeros((species, 2 * species))
    for r in range(2 * species):
        a = r % species
        b, c = (int(q) for q in np.clip(a + rng.integers(-4, 5, 2), 0, species - 1))
        d = species - 1 if r % 3 == 0 else int(np.clip(a + rng.integers(-4, 5), 0, species - 1))
        reac.append({"re": [a, b], "pr": [c, d], "kind": 2, "A": 1e-12, "B": 0.0, "C": 0.0, "eq": "A + B -> C + D"})
        for s, n in ((a, -1), (b, -1), (c, 1), (d, 1)):
            S[s, r] += n
    return types.SimpleNamespace(reac=reac, photo=[], photo_missing=[], elements=["H"], atoms=np.ones((species, 1)),
                                 species=[f"s{i}" for i in range(species)], S=S, Sp=np.zeros((species, 0)),
                                 lo=np.zeros((species, 9)), hi=np.zeros((species, 9)))  # fmt: skip


@pytest.mark.parametrize("species", [3, 16, 17, 63, 64, 65, 80, 81, 92])
def test_both_layouts_give_the_same_factors_and_solutions(species):
    tab = _tables.build(network(species, species))
    assert _kernels.lu_layout(tab)["use"] and tab.k0 == max(0, species - 64)
    src = (_kernels.header(tab, 1, 1e-6) + (_kernels.KERNEL_DIR / "common.hip").read_text() + PROBE.read_text())
    module = _hip.Module(_hip.compile_source(src, "lu_probe.hip"), torch.cuda.current_device())
    fn = module.function("mxc_lu_probe")
    rng = np.random.default_rng(7)
    n = tab.ns
    for spread in (0.0, 8.0):  # entries of one size; of sizes 1e-8 to 1e8 by row and column
        scale = 10.0 ** rng.uniform(-spread, spread, (2, n))
        W = np.where(tab.fill, rng.standard_normal((n, n)), 0.0) + 4.0 * np.eye(n)
        W = W * scale[0][:, None] * scale[1][None, :]
        w = torch.tensor(np.ascontiguousarray(W), device="cuda")
        b = torch.tensor(scale[0] * rng.standard_normal((3, n)), device="cuda")
        out = torch.full((2, n * n + 4 * n), float("nan"), dtype=torch.float64, device="cuda")
        _hip.launch(fn, 1, 64, 8 * tab.layout()["SIZE"], torch.cuda.current_stream().cuda_stream,
                    [_hip.ptr(w), _hip.ptr(b), _hip.ptr(out)])  # fmt: skip
        torch.cuda.synchronize()
        got, want = out.cpu().numpy()
        assert np.isfinite(want).all()
        assert np.array_equal(got, want)
    module.unload()


@pytest.mark.parametrize("stem", ["synthetic", "NCHO"])
def test_the_register_lu_takes_the_matrices_without_exchanges(read_network, stem):
    # the recovery's fast LU gives dense_lu's factors bit for bit where the threshold rule exchanges no row, and leaves
    # every other matrix, and one with a NaN, as it is
    import helpers
    from probes import Probes

    from maxichem_amd import standin

    net = standin.load(stem) if stem == "NCHO" else read_network(stem)
    probes = Probes(net)
    tab = probes.tab
    n = tab.ns
    rng = np.random.default_rng(5)
    mats = [rng.standard_normal((n, n)) + d * np.eye(n) for d in (4.0 * n, 2.0 * n, n, 3.0, 0.5) for _ in range(3)]
    edge = 10.0 * np.eye(n)
    edge[1:, 0] = 100.0  # |W_00| is PIVTAU times the column's largest: kept; a bit more exchanges
    more = edge.copy()
    more[n - 1, 0] = np.nextafter(100.0, 200.0)
    nan = mats[0].copy()
    nan[n - 1, 3] = np.nan
    mats = [*mats, edge, more, np.eye(n), *helpers.adversarial_matrices(n, rng), nan]
    want, rows, dinv, _ = probes.run_dense(np.array(mats), np.zeros((len(mats), n)))
    src = (_kernels.header(tab, 1, 1e-6) + "".join((_kernels.KERNEL_DIR / f).read_text()
           for f in ("common.hip", "guard.hip", "recover.hip")) + PROBE.with_name("dense_2d_probe.hip").read_text())  # fmt: skip
    module = _hip.Module(_hip.compile_source(src, "dense_2d_probe.hip"), torch.cuda.current_device())
    W = torch.tensor(np.array(mats), device="cuda")
    d = torch.zeros(len(mats), n, dtype=torch.float64, device="cuda")
    took = torch.zeros(len(mats), dtype=torch.int32, device="cuda")
    lds = 8 * (tab.layout()["SIZE"] + n * n + 2 * n) + 4 * n
    _hip.launch(module.function("mxc_dense_2d_probe"), len(mats), 64, lds, torch.cuda.current_stream().cuda_stream,
                [_hip.ptr(W), _hip.ptr(d), _hip.ptr(took)])  # fmt: skip
    torch.cuda.synchronize()
    got, d, took = W.cpu().numpy(), d.cpu().numpy(), took.cpu().numpy()
    kept = [list(r) == list(range(n)) for r in rows]
    assert kept[:3] == [True] * 3 and took[15] == 1 and took[16] == 0 and sum(took) < len(mats)
    for m, a in enumerate(mats):
        assert bool(took[m]) == (kept[m] and bool(np.isfinite(a).all())), m
        if took[m]:
            assert np.array_equal(got[m], want[m]) and np.array_equal(d[m], dinv[m])
        else:
            assert np.array_equal(got[m], a, equal_nan=True)
    module.unload()
    probes.close()
