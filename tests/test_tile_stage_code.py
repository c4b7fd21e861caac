"""The stage code of spmm.h and of decode_rows.hip holds 120 and 98 of a wavefront's 128 registers by number: the kernels around it must
not spill, or every stage pays for it.  That of decode_rows.hip also takes the tiles to begin at LDS address 0: no static LDS."""
import os
import re
import shutil
import subprocess

import pytest

from crosslayer_coding_amd import build as clt_build


@pytest.mark.parametrize("source,kernels,count", [
    ("spmm.hip", r"k_(?:decode|grad)_tiles", 5),            # two 16-bit types; with the step, as rows and as parameters
    ("decode_rows.hip", r"k_(?:decode|grad)_rows", 2),
])
def test_tile_kernels_spill_nothing(tmp_path, source, kernels, count):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not found")
    out = tmp_path / "stages.s"
    flags = [f for f in clt_build.HIP_FLAGS if f != "-fPIC"]
    proc = subprocess.run([hipcc, *flags, "--cuda-device-only", "-S", "-o", str(out), os.path.join(clt_build.CSRC, source)],
                          stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert proc.returncode == 0, proc.stdout[-2000:]
    text = open(out).read()
    found = re.findall(r"^(_Z\w*" + kernels + r"\w*):.*?^; NumVgprs: (\d+).*?^; ScratchSize: (\d+).*?^; LDSByteSize: (\d+)", text, re.S | re.M)
    assert len(found) == count, found
    for name, registers, scratch, lds in found:
        assert int(scratch) == 0 and int(registers) <= 128 and int(lds) == 0, (name, registers, scratch, lds)
