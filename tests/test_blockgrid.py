"""Host-side test of the grid dimensions of launches of very many blocks
(csrc/blockgrid.hpp): compiled with g++ into a small driver, no GPU.  Every
dimension stays below 2^32 threads, every block has a place, and fewer blocks
than a row holds keep one row of exactly their number."""
import os
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "mrfingerprintingrecon.jl_amd", "csrc")

DRIVER = r"""
#include <cstdio>
#include <initializer_list>
#include "blockgrid.hpp"
using namespace msr;

static int fails = 0;
#define EXPECT(c) do { if (!(c)) { std::printf("FAIL line %d: %s\n", __LINE__, #c); ++fails; } } while (0)

int main() {
    const int64_t ns[] = {1, 7, 8, 1000, (1 << 23) - 1, 1 << 23, (1 << 23) + 1, 256LL * 256 * 256,
                          320LL * 320 * 176, 512LL * 512 * 512};
    for (int64_t n : ns)
        for (int threads : {64, 256, 1024}) {
            const BlockGrid g = split_blocks(n, threads);
            EXPECT(g.x >= 1 && g.y >= 1 && g.y <= 65535);
            EXPECT((int64_t)g.x * threads < (int64_t)1 << 32);
            EXPECT((int64_t)g.x * g.y >= n && (int64_t)g.x * g.y - n < g.y);
            if (n * threads <= (int64_t)1 << 31) EXPECT(g.y == 1 && g.x == n);
        }
    std::printf("%s\n", fails ? "FAILED" : "OK");
    return fails ? 1 : 0;
}
"""


def test_split_blocks(tmp_path):
    src = tmp_path / "blocks.cpp"
    src.write_text(DRIVER)
    exe = tmp_path / "blocks"
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-I" + CSRC, str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    if r.returncode != 0 and "not found" in r.stderr:
        pytest.skip("g++ unavailable")
    assert r.returncode == 0, r.stderr
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.strip().endswith("OK"), out.stdout
