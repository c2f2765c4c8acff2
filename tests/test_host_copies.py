"""Runs of adjacent arrays that one host-device copy takes together (CPU: the header compiled by itself)."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "psi4_amd", "csrc", "dfjk")

# arrays as (allocation, first double, doubles) -> runs as (first double, offset in the staging, doubles)
CASES = [
    ([], []),
    ([(0, 0, 5)], [(0, 0, 5)]),
    ([(0, 0, 5), (0, 5, 7), (0, 12, 1)], [(0, 0, 13)]),
    ([(0, 0, 5), (0, 6, 7)], [(0, 0, 5), (6, 5, 7)]),
    # two allocations side by side: C fills its buffer, the results' buffer begins where it ends
    ([(0, 0, 8), (0, 8, 8), (1, 16, 4), (1, 20, 4)], [(0, 0, 16), (16, 16, 8)]),
    ([(1, 16, 4), (0, 8, 8)], [(16, 0, 4), (8, 4, 8)]),
]


@pytest.fixture(scope="module")
def runs(tmp_path_factory):
    d = tmp_path_factory.mktemp("copies")
    (d / "runs.cpp").write_text("""
#include "host_copies.hpp"
#include <cstdint>
#include <cstdio>
int main() {
    static double mem[64];
    static int bufs[4];
    std::vector<p4a::HostCopy> x;
    int b, o, n;
    while (std::scanf("%d %d %d", &b, &o, &n) == 3) x.push_back({mem + o, nullptr, static_cast<size_t>(n), bufs + b});
    p4a::for_runs(x, [&](double* dev, size_t off, size_t bytes) {
        std::printf("%d %d %d\\n", int(dev - mem), int(off / 8), int(bytes / 8));
    });
}
""")
    exe = str(d / "runs")
    subprocess.run(["g++", "-std=c++17", f"-I{CSRC}", str(d / "runs.cpp"), "-o", exe], check=True)

    def call(arrays):
        text = "".join("%d %d %d\n" % a for a in arrays)
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True, timeout=20).stdout
        return [tuple(int(v) for v in line.split()) for line in out.splitlines()]

    return call


@pytest.mark.parametrize("arrays,want", CASES)
def test_runs_stay_in_one_allocation(runs, arrays, want):
    assert runs(arrays) == want
