"""A try's own path from the derivative terms to M0's factors and solutions (the register slots' assembly and LU, and the
solves by blocks) against the rows': the same bits, at the edges of the slots and of the lead part (GPU)."""

import ctypes
from pathlib import Path

import numpy as np
import pytest
import torch
from test_lu import network

from maxichem_amd import _hip, _kernels, _tables

pytestmark = pytest.mark.gpu
PROBE = Path(__file__).resolve().parent / "assembly_probe.hip"


@pytest.mark.parametrize("species", [3, 16, 17, 63, 64, 65, 80, 81, 92])
def test_a_trys_factors_are_the_rows(species):
    tab = _tables.build(network(species, species))
    assert _kernels.lu_layout(tab)["use"] and tab.k0 == max(0, species - 64)
    src = _kernels.header(tab, 1, 1e-6) + (_kernels.KERNEL_DIR / "common.hip").read_text() + PROBE.read_text()
    module = _hip.Module(_hip.compile_source(src, "assembly_probe.hip"), torch.cuda.current_device())
    fn = module.function("mxc_assembly_probe")
    host = _kernels.host_tables(tab)
    tables = [torch.from_numpy(host[k]).cuda() for k in _kernels.NET_FIELDS]
    net = torch.tensor([a.data_ptr() for a in tables], dtype=torch.int64, device="cuda")
    rng = np.random.default_rng(species)
    n, nr = tab.ns, tab.nr
    nd = 1e18
    for h in (1e-8, 1.0):  # a diagonal of 1 / (gamma h) alone, and one of the rates' own size
        k = 10.0 ** rng.uniform(-18.0, -10.0, 2 * nr)
        x = 10.0 ** rng.uniform(-8.0, 0.0, n)
        args = [torch.tensor(a, device="cuda") for a in (k, x / x.sum(), rng.standard_normal((3, n)))]
        out = torch.full((2, n * n + 5 * n), float("nan"), dtype=torch.float64, device="cuda")
        _hip.launch(fn, 1, 64, 8 * tab.layout()["SIZE"], torch.cuda.current_stream().cuda_stream,
                    [_hip.ptr(net), *map(_hip.ptr, args), ctypes.c_double(nd), ctypes.c_double(2.0 / h),
                     _hip.ptr(out)])  # fmt: skip
        torch.cuda.synchronize()
        got, want = (dict(zip(("w", "factors", "dinv", "y"), np.split(o, np.cumsum([n, n * n, n]))))
                     for o in out.cpu().numpy())  # fmt: skip
        assert all(np.isfinite(v).all() for v in want.values())
        assert np.count_nonzero(want["factors"]) > 2 * n
        factors, rows = got["factors"].reshape(n, n), want["factors"].reshape(n, n).copy()
        if n >= 64:  # the trailing diagonal is 0 where the solves go by blocks
            at = np.arange(tab.k0, n)
            assert (factors[at, at] == 0.0).all() and (rows[at, at] != 0.0).all()
            rows[at, at] = 0.0
        assert np.array_equal(factors, rows)
        for name in ("w", "dinv", "y"):
            assert np.array_equal(got[name], want[name]), name
    module.unload()
