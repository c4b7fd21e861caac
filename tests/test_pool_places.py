"""Places in the candidate pool of the selection's streaming pass, where they come near 2^32: the arithmetic of the kernel
(select_state.h) in a host program."""
import os
import shutil
import subprocess

import pytest

from crosslayer_coding_amd import build as clt_build

PROGRAM = r"""
#include <cstdio>
#include "select_state.h"

int main() {
  const uint32_t slot = 1u << 18, waves = 4096;                     // parts of 2^30 entries together
  for (unsigned long long cap : {1ull << 31, POOL_MOST}) {
    static PoolPart part[4096];
    for (uint32_t w = 0; w < waves; ++w) part[w] = {w * slot, (w + 1) * slot, (unsigned long long)waves * slot, cap, false};
    unsigned long long counter = 0, refused = 0;
    // the counter handed out almost everything before; then every wavefront goes through far more rows than fit
    counter = cap - (unsigned long long)waves * slot - 513 * 1000;
    unsigned long long last = counter;
    for (int round = 0; round < 64; ++round)
      for (uint32_t w = 0; w < waves; ++w) {
        const uint32_t n = round < 2 ? slot / 2 : 513;
        const uint32_t at = part[w].take(n, [&](uint32_t k) { const uint32_t was = (uint32_t)counter; counter += k; return was; });
        if (at == POOL_FULL) { ++refused; continue; }
        const bool own = at >= w * slot && at + n <= (w + 1) * slot;
        const bool shared = at >= (unsigned long long)waves * slot && at + (unsigned long long)n <= cap && at == waves * slot + last;
        if (!own && !shared) { printf("wavefront %u got %u\n", w, at); return 1; }
        if (shared) last = at - waves * slot + n;
      }
    if (counter >= 1ull << 32) { printf("the counter came round: %llu\n", counter); return 1; }
    if (refused != 62ull * waves - 1000) { printf("%llu refused\n", refused); return 1; }
  }
  return 0;
}
"""


def test_places_near_the_end_of_32_bits(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not found")
    src, exe = tmp_path / "places.hip", tmp_path / "places"
    src.write_text(PROGRAM)
    proc = subprocess.run([hipcc, "-O1", "-std=c++17", "--cuda-host-only", "-I", clt_build.CSRC, str(src), "-o", str(exe)],
                          stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert proc.returncode == 0, proc.stdout[-2000:]
    run = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True, timeout=60)
    assert run.returncode == 0, run.stdout
