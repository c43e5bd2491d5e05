"""Sizes of the sampler's and calibrator's class tables (hbfsim_amd/csrc/class_table.hpp), compiled
on the CPU: a table whose probes have no limit always keeps an empty slot, and kernels over its
slots are launches that the GPU accepts."""
from __future__ import annotations

import pathlib
import subprocess

CSRC = pathlib.Path(__file__).resolve().parent.parent / "hbfsim_amd" / "csrc"

MAIN = """
#include "class_table.hpp"
#include <cstdio>
using namespace hbfamd;
#define CHECK(x) do { if (!(x)) { std::printf("n %llu seen %llu: %s\\n", \\
    (unsigned long long)n, (unsigned long long)seen, #x); return 1; } } while (0)
int main()
{
    const std::size_t top = 0xffffffffull;  // the most requests a call takes
    const std::size_t sizes[] = {1, 511, 512, 513, 65536, 4000037, (1ull << 30) + 1, 1ull << 31,
                                 (1ull << 31) + 1, top};
    const std::size_t held[] = {0, 1, 16385, 1ull << 29, (1ull << 29) + 1, 1ull << 31, top,
                                1ull << 33};
    for (std::size_t n : sizes) {
        for (std::size_t seen : held) {
            const std::uint64_t most = most_slots(n, seen);
            CHECK(most >= 2 * (n + seen) && (most & (most - 1)) == 0);
            for (std::uint32_t sampled : {0u, 16384u}) {
                std::uint64_t cap = first_slots(seen, most);
                int steps = 0;
                for (; cap != most; cap = next_slots(cap, most, sampled)) {
                    CHECK((cap & (cap - 1)) == 0 && cap > seen);
                    CHECK(++steps < 10);
                }
                CHECK(sample_limit(cap, most) >= kSample);  // the last table is always tried
            }
            CHECK(std::uint64_t{walk_blocks(most)} * 256 < 1ull << 32);
            CHECK(walk_blocks(most) != 0);
        }
        const std::size_t seen = 0;
        const std::uint64_t numbered = most_slots(n, 0, 1ull << 32);
        CHECK(numbered > n && numbered <= 1ull << 32);  // 32-bit slot numbers, one slot empty
    }
    return 0;
}
"""


def test_class_table_sizes(tmp_path):
    src = tmp_path / "sizes.cpp"
    src.write_text(MAIN)
    exe = tmp_path / "sizes"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-I", str(CSRC), str(src), "-o", str(exe)],
                   check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
