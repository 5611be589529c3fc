"""The kernels' scratch memory, from the code objects' notes (CPU). A kernel that spills needs it, and the runtime sets it aside
for the whole device at the kernel's first launch on a queue: the recovery, which every call launches, needs none, nor does
the export's default variant, whose static call may not allocate. (With its register LU among the tries SNCHO's recovery
spilled 211 registers, took 430 MB and a minute more of the compiler's time.)"""

import re
import subprocess
from pathlib import Path

import pytest

from maxichem_amd import _hip, _kernels, _tables, standin
from maxichem_amd._constants import DRIFT
from maxichem_amd.tune import default_variant

READELF = Path("/opt/rocm/llvm/bin/llvm-readelf")


def scratch(code: bytes, folder: Path) -> dict[str, int]:
    """Each kernel's scratch bytes a lane."""
    (folder / "code.hsaco").write_bytes(code)
    text = subprocess.run([READELF, "--notes", folder / "code.hsaco"], check=True, capture_output=True, text=True).stdout
    values = [dict(re.findall(r"\.(\w+):\s+(\S+)", part)) for part in re.split(r"\n\s+- \.agpr_count:", text)[1:]]
    return {v["name"]: int(v["private_segment_fixed_size"]) for v in values}


@pytest.mark.skipif(not READELF.exists(), reason="needs ROCm's llvm-readelf")
@pytest.mark.parametrize("shape", ["NCHO", "SNCHO"])
def test_no_call_needs_scratch_for_the_recovery(shape, tmp_path):
    tab = _tables.build(standin.load(shape), True)
    for variant in {default_variant(tab), (1, _kernels.DEFAULT_BATCH, 1, 0)}:
        cpw, batch, wps, rates_global = variant
        code = _hip.compile_source(_kernels.source(tab, cpw, DRIFT, batch, wps=wps, rates_global=bool(rates_global)))
        need = scratch(code, tmp_path)
        assert need["mxc_recover"] == 0, (variant, need)
        if wps == 1:
            assert need["mxc_call"] == 0, (variant, need)


def test_the_registers_take_the_recovery_only_where_they_fit():
    takes = {shape: _kernels.lu_layout(_tables.build(standin.load(shape), True)) for shape in ("NCHO", "SNCHO")}
    assert all(lu["use"] for lu in takes.values())
    assert takes["NCHO"]["dense"] and not takes["SNCHO"]["dense"]
