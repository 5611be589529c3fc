"""The call kernel's autotuner: cells (wavefronts) per workgroup, the stream batch, the register budget (wavefronts
per SIMD) and the rate coefficients' place (LDS or global scratch), per network, device and workload.

Each candidate is compiled, loaded and timed by HIP events around the call kernel on a sample of the workload:
"uneven", one synthetic call from cold (solar gas, dt log-uniform 1e1-1e4 s, half of the cells lit), or "settled",
calls of dt = 300 s after a dark relaxation (the GPU FP64 case's sequence, a quarter of the cells lit). The fastest
is stored in the code cache (tune.json) under the network's table digest, the photolysis switch, the device name, the
kernels it was timed on, the precision and the workload, and later solvers of that network on that device take the
uneven choice unless told the workload.
"""

from __future__ import annotations

import hashlib
import json
import os
from pathlib import Path

import numpy as np
import torch

from . import _hip, _kernels, _tables, workloads

VARIANTS = ((1, 16, 1, 0), (1, 8, 1, 0), (2, 16, 1, 0), (4, 16, 1, 0), (1, 16, 2, 0), (1, 16, 1, 1), (1, 16, 2, 1))
DEFAULT = (1, _kernels.DEFAULT_BATCH, 1, 0)
STORE: Path | None = None  # where the choices are kept; None: tune.json in the code cache
CU_LDS = 160 * 1024  # LDS per compute unit (gfx950)
CU_WAVES = 4  # call wavefronts per compute unit at one per SIMD


def default_variant(tab, mixed: bool = False) -> tuple[int, int, int, int]:
    """The variant without a stored choice, with the same bits as every other. Two wavefronts per SIMD where a compute
    unit's LDS holds eight cells (with the rates in LDS, else in global scratch): each waits for its LDS reads and
    chains of broadcasts while the other issues, which outweighs the few registers it spills (NCHO, ms a call against
    (4, 16, 1, 0), two draws each: 65,536 settled cells 11.5 -> 7.2 and 11.6 -> 11.1, 256 cold cells 18.7 -> 16.5 and
    22.0 -> 19.9, 8,192 cold cells 41.0 -> 28.9 and, where one cell's 1,439 tries are the call, 51.5 -> 52.3). Else, and
    in the mixed form: four cells per workgroup when the stream words then fit in the workgroup's LDS at as many cells per compute
    unit; else two when that keeps as many cells per compute unit as one; else one."""
    if not mixed and _kernels.lu_layout(tab)["use"]:
        for rates_global in (0, 1):
            if CU_LDS // _kernels.lds_bytes(tab, 1, False, bool(rates_global), 2)[0] >= 2 * CU_WAVES:
                return (1, _kernels.DEFAULT_BATCH, 2, rates_global)

    def cells(cpw: int) -> int:
        return min(CU_WAVES, CU_LDS // _kernels.lds_bytes(tab, cpw, mixed)[0] * cpw)

    best = max(cells(c) for c in (1, 2, 4))
    if _kernels.words_in_lds(tab, 4, mixed) and cells(4) >= best:
        return (4, _kernels.DEFAULT_BATCH, 1, 0)
    return (2 if cells(2) >= cells(1) else 1, _kernels.DEFAULT_BATCH, 1, 0)


def _store() -> Path:
    return STORE if STORE is not None else _hip.CACHE / "tune.json"


WORKLOADS = ("uneven", "settled")


def kernels_digest() -> str:
    """What a choice was timed on: the kernel files, the modules that write their header and tables, the compiler and its
    options. A choice outlives none of them: other kernels have another best variant."""
    files = [_kernels.KERNEL_DIR / name for name in (*_kernels.KERNEL_FILES, "mixed.hip")]
    parts = [f.read_bytes() for f in (*files, Path(_kernels.__file__), Path(_tables.__file__))]
    options = repr((_kernels.OPTIONS, _hip.compiler_version())).encode()
    return hashlib.sha256(b"\0".join([*parts, options])).hexdigest()[:16]


def _key(net, photo: bool, device: torch.device, workload: str = "uneven", mixed: bool = False) -> str:
    key = f"{_tables.build(net, photo).digest()}|{int(photo)}|{torch.cuda.get_device_name(device)}|{kernels_digest()}"
    return key + ("|mixed" if mixed else "") + ("" if workload == "uneven" else f"|{workload}")


def stored(net, device, photo: bool, workload: str = "uneven", mixed: bool = False) -> dict | None:
    try:
        return json.loads(_store().read_text()).get(_key(net, photo, device, workload, mixed))
    except (OSError, ValueError):
        return None


def choose(net, device, photo: bool, drift: float, run: bool = False, workload: str = "uneven",
           mixed: bool = False) -> tuple[int, ...]:  # fmt: skip
    """The variant for this network, device, workload and form (FP64 or mixed): tuned now when run, else the stored
    choice, else default_variant."""
    if run:
        return tuple(tune(net, device, photo, drift, workload=workload, mixed=mixed)["best"])
    s = stored(net, device, photo, workload, mixed)
    return tuple(s["best"]) if s else default_variant(_tables.build(net, photo), mixed)


def tune(net, device, photo: bool, drift: float, cells: int = 8192, seed: int = 7, repeats: int = 2,
         workload: str = "uneven", mixed: bool = False) -> dict:  # fmt: skip
    """Time every variant of the FP64 or the mixed form on the workload's sample; store and return {"best", "ms":
    {variant: ms}, "private_bytes": {variant: bytes per lane the variant spills}}."""
    from .kincuda import CudaSolver

    if workload not in WORKLOADS:
        raise ValueError(f"workload: one of {WORKLOADS} expected, got {workload!r}")
    dev = torch.device(device)
    nj = len(net.photo) if photo else 0

    def g(a):
        return torch.from_numpy(np.ascontiguousarray(a)).to(dev)

    if workload == "uneven":
        d = workloads.config3(net.species, len(net.photo), cells=cells, seed=seed)
        rng = np.random.default_rng(seed)
        dt = 10.0 ** rng.uniform(1.0, 4.0, cells)
        x, T, P, h, dtt = g(d["x"]), g(d["T"]), g(d["P"]), g(d["h"]), g(dt)
        J = g(d["J"][:, :nj]) if photo else None
    else:
        d = workloads.config1(net.species, len(net.photo), cells=cells, seed=seed)
        T, P = g(d["T"]), g(d["P"])
        J = g(d["J"][:, :nj]) if photo else None
        with CudaSolver(net, dev, photo=photo, drift=drift, variant=DEFAULT) as s:
            r = s(g(d["x"]), T, P, g(d["dt_relax"]), g(d["h"]), J=None if J is None else torch.zeros_like(J))
            x, h, dtt = r.x, r.h, g(d["dt"])
    ms, spills = {}, {}
    for v in VARIANTS:
        with CudaSolver(net, dev, photo=photo, drift=drift, variant=v, precision="mixed" if mixed else "fp64") as s:
            s(x, T, P, dtt, h, J=J)  # the first call pays for loading
            s.timing = []
            for _ in range(repeats):
                s(x, T, P, dtt, h, J=J)
            torch.cuda.synchronize(dev)
            key = ",".join(map(str, v))
            ms[key] = float(np.median([a.elapsed_time(b) for a, b in s.timing]))
            spills[key] = int(s.info["private_bytes"])
            s.timing = None
    best = min(ms, key=ms.get)
    out = {"best": [int(q) for q in best.split(",")], "ms": ms, "private_bytes": spills, "cells": cells,
           "workload": workload}  # fmt: skip
    path = _store()
    try:
        data = json.loads(path.read_text()) if path.exists() else {}
    except ValueError:
        data = {}
    data[_key(net, photo, dev, workload, mixed)] = out
    try:
        path.parent.mkdir(parents=True, exist_ok=True)
        tmp = path.with_suffix(f".tmp{os.getpid()}")
        tmp.write_text(json.dumps(data, indent=1, sort_keys=True))
        os.replace(tmp, path)
    except OSError:
        pass
    return out
