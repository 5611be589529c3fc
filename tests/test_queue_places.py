"""The tangent queue's places: two passes where there are more pairs than wavefronts, and one where two would not fit an
int (more than 2^30 pairs of a small network still fit the device's memory; GPU)."""

import ctypes

import pytest
import torch

from maxichem_amd import _hip, _kernels, _tables

pytestmark = pytest.mark.gpu
PROBE = """
extern "C" __global__ void mxc_queue_probe(const int* pairs, int waves, int* places) {
  places[threadIdx.x] = queue_places(pairs[threadIdx.x], waves);
}
"""


def test_the_places_fit_an_int(gpu, read_network):
    tab = _tables.build(read_network("synthetic_small"))
    src = _kernels.header(tab, 1, 1e-6) + (_kernels.KERNEL_DIR / "common.hip").read_text() + PROBE
    module = _hip.Module(_hip.compile_source(src, "queue_probe.hip"), torch.cuda.current_device())
    waves, top = 1024, 2**31 - 1
    half = (top - waves) // 2
    pairs = [0, 1, waves, waves + 1, 65536, half, half + 1, 2**30, top - waves]
    want = [0, 1, waves, 2 * waves + 2, 131072, 2 * half, half + 1, 2**30, top - waves]
    p = torch.tensor(pairs, dtype=torch.int32, device="cuda")
    got = torch.empty_like(p)
    _hip.launch(module.function("mxc_queue_probe"), 1, len(pairs), 0, torch.cuda.current_stream().cuda_stream,
                [_hip.ptr(p), ctypes.c_int(waves), _hip.ptr(got)])  # fmt: skip
    torch.cuda.synchronize()
    assert got.tolist() == want
    module.unload()
