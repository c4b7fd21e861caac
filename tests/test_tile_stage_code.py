"""The stage code of spmm.h holds 120 of a wavefront's 128 registers by number: the kernels around it must not spill, or every stage
pays for it."""
import os
import re
import shutil
import subprocess

import pytest

from crosslayer_coding_amd import build as clt_build


def test_tile_kernels_spill_nothing(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not found")
    out = tmp_path / "spmm.s"
    flags = [f for f in clt_build.HIP_FLAGS if f != "-fPIC"]
    proc = subprocess.run([hipcc, *flags, "--cuda-device-only", "-S", "-o", str(out), os.path.join(clt_build.CSRC, "spmm.hip")],
                          stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert proc.returncode == 0, proc.stdout[-2000:]
    text = open(out).read()
    scratch = re.findall(r"^(_Z\w*k_(?:decode|grad)_tiles\w*):.*?^; ScratchSize: (\d+)", text, re.S | re.M)
    assert len(scratch) == 5, scratch               # two 16-bit types; with the step, as rows and as parameters
    assert all(int(size) == 0 for _, size in scratch), scratch
