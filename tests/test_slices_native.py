"""The cutting of a launch below HIP's limit of 2^32 work-items
(cuspx_amd/csrc/slices.hpp), built with g++: every request belongs to exactly
one slice, in order, and no slice's launch reaches the limit, for the chain
launches of batches just below and above the one at which a single launch
would, and for small ones (one slice)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "cuspx_amd", "csrc")

HARNESS = r"""
#include <cstdio>
#include <cstdlib>
#include "slices.hpp"

// lanes of a chain launch: a wave per chain and 64 leaves, whole workgroups
static uint64_t lanes(uint64_t n, uint64_t leaves, uint64_t len) {
    const uint64_t waves = (n * leaves + 63) / 64 * len;
    return (waves + 3) / 4 * 256;
}

int main(int, char** argv) {
    const uint32_t n = (uint32_t)strtoul(argv[1], nullptr, 10);
    const uint64_t leaves = strtoull(argv[2], nullptr, 10), len = strtoull(argv[3], nullptr, 10);
    uint64_t next = 0;
    int slices = 0;
    bool ok = true;
    spx::for_slices(n, lanes(n, leaves, len), [&](uint32_t a, uint32_t m) {
        ok = ok && a == next && m > 0 && lanes(m, leaves, len) < (1ull << 32);
        next = (uint64_t)a + m;
        slices++;
    });
    std::printf("%d %d\n", ok && next == n, slices);
    return 0;
}
"""

# requests, leaves per request, chains per leaf, slices
BATCHES = [(0, 3584, 35, 0), (1, 8, 35, 1), (4096, 176, 35, 1), (17119, 3584, 35, 1),
           (17120, 3584, 35, 2), (34239, 3584, 35, 2), (34240, 3584, 35, 3),  # 128s signing
           (23497, 3584, 51, 2), (23498, 3584, 51, 3), (31300, 2048, 67, 2), (31301, 2048, 67, 3),
           (697234, 176, 35, 2), (697235, 176, 35, 3),                        # 128f signing
           (239674, 512, 35, 2), (239675, 512, 35, 3), (4000000, 8, 35, 1)]   # key generation


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_slices_cover_the_batch_below_the_limit(tmp_path):
    src = tmp_path / "slices.cpp"
    src.write_text(HARNESS)
    exe = tmp_path / "slices"
    b = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-I" + CSRC, str(src),
                        "-o", str(exe)], capture_output=True, text=True, timeout=120)
    assert b.returncode == 0 and b.stderr == "", b.stderr
    for n, leaves, ln, slices in BATCHES:
        r = subprocess.run([str(exe), str(n), str(leaves), str(ln)], capture_output=True,
                           text=True, timeout=60)
        assert r.stdout.split() == ["1", str(slices)], (n, leaves, ln, r.stdout)
