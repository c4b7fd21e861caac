"""The benchmark's traffic figures are of the kernels that run, or left out."""
import os
import re

import pytest

import bench


@pytest.mark.parametrize("workload", ["c1", "c2", "c3"])
def test_kept_traffic_is_of_these_kernels(workload):
    table, forwards = bench.profiled_traffic(workload)
    if not forwards:
        pytest.skip("the kept counters are of other kernels: the figures are left out")
    csrc = os.path.join(bench.ROOT, "crosslayer-coding_amd", "csrc")
    source = "".join(open(os.path.join(csrc, n)).read() for n in os.listdir(csrc) if n.endswith((".hip", ".h")))
    for name in table:
        assert re.search(rf"\b{re.split('[< ]', name)[0]}\b", source), name


def test_traffic_of_other_kernels_is_left_out(tmp_path, monkeypatch):
    (tmp_path / "profiles").mkdir()
    csrc = tmp_path / "crosslayer-coding_amd" / "csrc"
    csrc.mkdir(parents=True)
    (csrc / "a.hip").write_text("int a;  // one\n")
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    table = "k_a<float>   3   1   2   3   4   5.5\n"
    kept = tmp_path / "profiles" / "forward_c1_hbm_traffic.txt"

    kept.write_text("forwards profiled: 3\n" + table)                       # of unknown kernels
    assert bench.profiled_traffic("c1") == ({}, 0)
    kept.write_text(f"forwards profiled: 3\nkernel sources: {bench.kernel_sources_digest()}\n" + table)
    assert bench.profiled_traffic("c1") == ({"k_a<float>": (3, 5.5e6)}, 3)
    (csrc / "a.hip").write_text("int  a;  // a comment changes nothing\n")
    assert bench.profiled_traffic("c1") == ({"k_a<float>": (3, 5.5e6)}, 3)
    (csrc / "a.hip").write_text("int b;\n")
    assert bench.profiled_traffic("c1") == ({}, 0)
