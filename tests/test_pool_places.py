"""The candidate pool of the selection's streaming pass: places where they come near 2^32, by the arithmetic of the kernel
(select_state.h) in a host program, and the pool's size."""
import os
import shutil
import subprocess

import pytest
import torch

from crosslayer_coding_amd import _native as nat
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


@pytest.mark.parametrize("L,T,F,k", [(16, 8192, 8192, 2000), (12, 4096, 24576, 200), (24, 4096, 32768, 256), (16, 2048, 8192, 3000),
                                     (16, 2048, 8192, 8000)])
def test_the_pool_holds_four_times_what_is_kept_or_all_elements(L, T, F, k):
    """The largest part of a selection's workspace: 8 bytes for each of 4 K candidates of a layer, or for all its elements, and one
    header per extent; 2^25 bytes hold the rest (sample, statistics of rows, ends of the wavefronts' parts)."""
    lib = nat.load()
    K, N, rest = k * T, T * F, 20 * L * T + 2 ** 25
    room = L * 8 * (min(4 * K, N) + 2 * T + 4096)
    assert room <= lib.clt_batchtopk_workspace_bytes(T, F, L, k, nat.TOPK_PER_LAYER, nat.dtype_code(torch.bfloat16)) <= room + rest
    # where the encoder collects the candidates this pool is for repeated passes, its own one beside it has fixed slots for
    # 4.5 times the share of a tile, 64 each, and 2 K behind them
    tiles = (T + 255) // 256 * 4 * ((F + 255) // 256 * 2)
    slot = min(int(4.5 * k / F * 64 * 128) + 64, 64 * 128)
    own = L * 8 * (tiles * slot + min(2 * K + 4096, N)) + L * (8 * tiles + 12 * T * (F // 256 + 2))
    assert lib.clt_encode_collect_workspace_bytes(T, 768, F, L, k, nat.dtype_code(torch.bfloat16)) <= room + own + rest
