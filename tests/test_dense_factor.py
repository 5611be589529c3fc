"""The recovery's choice between its two LUs over a cell's tries: registers first, the wavefronts' alone while the tries
exchange rows, registers again once one does not; the same factors either way, and no time for a try in registers that
the exchanges would only undo (GPU)."""

import ctypes
from pathlib import Path

import numpy as np
import pytest
import torch

from maxichem_amd import _hip, _kernels, _tables, standin

pytestmark = pytest.mark.gpu
PROBE = Path(__file__).resolve().parent / "dense_factor_probe.hip"


def test_exchanging_tries_leave_the_registers_out(gpu):
    tab = _tables.build(standin.load("NCHO"), True)
    n = tab.ns
    rng = np.random.default_rng(11)
    kept = rng.standard_normal((n, n)) + 4.0 * n * np.eye(n)
    moved = kept[rng.permutation(n)]
    order = "kmmmmmmmkkm"
    want = [0, 1, 2, 3, 4, 5, 6, 7, 0, 0, 1]
    src = _kernels.header(tab, 1, 1e-6) + "".join(
        (_kernels.KERNEL_DIR / f).read_text() for f in ("common.hip", "guard.hip", "recover.hip")) + PROBE.read_text()
    module = _hip.Module(_hip.compile_source(src, "dense_factor_probe.hip"), torch.cuda.current_device())
    fn = module.function("mxc_factor_probe")
    for _ in range(2):  # the first launch pays for loading
        W = torch.tensor(np.array([{"k": kept, "m": moved}[c] for c in order]), device="cuda")
        rows = torch.zeros(len(order), n, dtype=torch.int32, device="cuda")
        state = torch.zeros(len(order), dtype=torch.int32, device="cuda")
        cycles = torch.zeros(len(order), dtype=torch.int64, device="cuda")
        _hip.launch(fn, 1, 64 * _kernels.REC_WAVES, _kernels.lds_bytes(tab, 1)[1],
                    torch.cuda.current_stream().cuda_stream,
                    [_hip.ptr(W), _hip.ptr(rows), _hip.ptr(state), _hip.ptr(cycles), ctypes.c_int(len(order))])  # fmt: skip
        torch.cuda.synchronize()
    assert state.tolist() == want
    for b, c in enumerate(order):  # the same factors, whichever LU gave them
        first = order.index(c)
        assert torch.equal(W[b], W[first]) and torch.equal(rows[b], rows[first])
    assert rows[0].tolist() == list(range(n)) and rows[1].tolist() != list(range(n))
    took = cycles.tolist()
    tried, alone = min(took[1:5]), max(took[5:8])
    print(f"cycles: registers {took[9]}, tried in vain first {took[1:5]}, alone {took[5:8]}")
    assert alone < 0.95 * tried and took[9] < 0.5 * alone
    module.unload()
