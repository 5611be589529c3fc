"""The recovery kernel's code object: the register LU is apart from the tries, so their registers are not spilled around its
block (inlined into them, SNCHO's recovery spills 211 registers and takes the compiler a minute more; CPU)."""

import re
import subprocess
from pathlib import Path

import pytest

from maxichem_amd import _hip, _kernels, _tables, standin
from maxichem_amd._constants import DRIFT
from maxichem_amd.tune import default_variant

READELF = Path("/opt/rocm/llvm/bin/llvm-readelf")


def notes(code: bytes, folder: Path) -> dict[str, dict[str, int]]:
    """Each kernel's metadata in a code object's notes."""
    (folder / "code.hsaco").write_bytes(code)
    text = subprocess.run([READELF, "--notes", folder / "code.hsaco"], check=True, capture_output=True, text=True).stdout
    kernels = {}
    for part in re.split(r"\n\s+- \.agpr_count:", text)[1:]:
        values = dict(re.findall(r"\.(\w+):\s+(\S+)", part))
        kernels[values["name"]] = {k: int(values[k]) for k in ("vgpr_spill_count", "private_segment_fixed_size")}
    return kernels


@pytest.mark.skipif(not READELF.exists(), reason="needs ROCm's llvm-readelf")
@pytest.mark.parametrize("shape", ["NCHO", "SNCHO"])
def test_the_recovery_does_not_spill_around_its_factorization(shape, tmp_path):
    tab = _tables.build(standin.load(shape), True)
    assert _kernels.lu_layout(tab)["use"]
    cpw, batch, wps, rates_global = default_variant(tab)
    code = _hip.compile_source(_kernels.source(tab, cpw, DRIFT, batch, wps=wps, rates_global=bool(rates_global)))
    recover = notes(code, tmp_path)["mxc_recover"]
    assert recover["vgpr_spill_count"] <= 64, recover
