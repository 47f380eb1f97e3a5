"""The light stream's state from its number of draws (pcg_at and its table, csrc/tr_device.h): the table
is evaluated on the CPU from the header's own source and compared with stepping the stream."""
import os
import re
import subprocess

from tests.conftest import ROOT

HEADER = os.path.join(ROOT, "jarabotransientrendering_amd", "csrc", "tr_device.h")

PROG = r"""
#include <cstdint>
#include <cstdio>
%s
int main() {
    static constexpr PcgJumps t = pcg_jumps();
    for (uint32_t n = 0; n < kPcgJumps; ++n) std::printf("%%llu %%llu\n", (unsigned long long)t.ac[n][0], (unsigned long long)t.ac[n][1]);
    return 0;
}
"""


def test_jumps_equal_stepping(tmp_path):
    src = open(HEADER).read()
    part = re.search(r"constexpr uint32_t kPcgJumps.*?\n}\n(?=__device__ __constant__)", src, re.S).group(0)
    (tmp_path / "t.cpp").write_text(PROG % part)
    subprocess.check_call(["g++", "-std=c++17", "-fconstexpr-loop-limit=10000", str(tmp_path / "t.cpp"), "-o", str(tmp_path / "t")])
    table = [tuple(map(int, l.split())) for l in subprocess.check_output([str(tmp_path / "t")], text=True).splitlines()]
    assert len(table) > 3 * 254  # three draws per vertex before the last of at most 255
    m, a = (1 << 64) - 1, 6364136223846793005
    for seed, seq in ((0, 1), (5, 2 * 12345 + 1), (m, 2 * ((1 << 61) - 1) + 1)):
        inc = ((seq << 1) | 1) & m
        state = ((inc + seed) * a + inc) & m  # pcg_seed
        for big_a, big_c in table:
            assert (big_a * (inc + seed) + big_c * inc) & m == state
            state = (state * a + inc) & m
