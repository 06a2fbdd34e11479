"""Host-side test of the binary search behind the sort bounds (csrc/search.hpp):
compiled with g++ into a small driver, no GPU.  Key sequences of up to 2^31 - 1
entries are given by a formula, so that no memory is needed; every position read
lies inside the sequence, also above 2^30 entries, where the sum of two
positions no longer fits an int."""
import os
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "mrfingerprintingrecon.jl_amd", "csrc")

DRIVER = r"""
#include <climits>
#include <cstdio>
#include <vector>
#include "search.hpp"
using namespace msr;

static int fails = 0;
#define EXPECT(c) do { if (!(c)) { std::printf("FAIL line %d: %s\n", __LINE__, #c); ++fails; } } while (0)

// n keys, key(i) = i / per: the first position >= v is min(v * per, n)
static void blocks(int n, int per) {
    bool inside = true;
    auto at = [&](int i) {
        if (i < 0 || i >= n) { inside = false; return INT_MAX; }
        return i / per;
    };
    const int last = n ? (n - 1) / per : 0;
    const int vs[] = {0, 1, last / 3, last / 2, last - 1, last};
    for (int v : vs) {
        if (v < 0) continue;
        const long long want = (long long)v * per;
        EXPECT(lower_bound_at(n, v, at) == (int)(want < n ? want : n));
    }
    if (last < INT_MAX) EXPECT(lower_bound_at(n, last + 1, at) == n);
    EXPECT(inside);
}

int main() {
    const int ns[] = {0, 1, 2, 3, 64, 1000, (1 << 30) - 1, 1 << 30, (1 << 30) + 1, 1700000000, INT_MAX};
    for (int n : ns)
        for (int per : {1, 7, 1 << 20}) blocks(n, per);
    // gaps and repeats
    const std::vector<int> k{0, 0, 0, 2, 2, 5, 9, 9};
    auto at = [&](int i) { return k.at(i); };
    const int want[] = {0, 3, 3, 5, 5, 5, 6, 6, 6, 6, 8};
    for (int v = 0; v <= 10; ++v) EXPECT(lower_bound_at((int)k.size(), v, at) == want[v]);
    std::printf("%s\n", fails ? "FAILED" : "OK");
    return fails ? 1 : 0;
}
"""


def test_lower_bound_stays_inside(tmp_path):
    src = tmp_path / "search.cpp"
    src.write_text(DRIVER)
    exe = tmp_path / "search"
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-fwrapv", "-I" + CSRC, str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    if r.returncode != 0 and "not found" in r.stderr:
        pytest.skip("g++ unavailable")
    assert r.returncode == 0, r.stderr
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.strip().endswith("OK"), out.stdout
