"""The scratch pool (hbfsim_amd/csrc/scratch.cpp) on the CPU: compiled with g++ against a stand-in
for the HIP runtime that counts allocations, frees and waits."""
from __future__ import annotations

import pathlib
import subprocess
import textwrap

import pytest

CSRC = pathlib.Path(__file__).resolve().parent.parent / "hbfsim_amd" / "csrc"

RUNTIME = """
#pragma once
#include <cstddef>
#include <cstdlib>
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
using hipStream_t = void*;
struct Fake {
    int device = 0, waits = 0, mallocs = 0, frees = 0;
    std::size_t held = 0, limit = ~std::size_t{0};
};
inline Fake fake;
struct FakeBlock { std::size_t bytes; };
inline hipError_t hipGetDevice(int* d) { *d = fake.device; return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { ++fake.waits; return hipSuccess; }
inline hipError_t hipMalloc(void** p, std::size_t bytes)
{
    if (bytes > fake.limit - fake.held) { return hipErrorOutOfMemory; }
    ++fake.mallocs;
    fake.held += bytes;
    *p = new FakeBlock{bytes};
    return hipSuccess;
}
inline hipError_t hipFree(void* p)
{
    if (p != nullptr) {
        ++fake.frees;
        fake.held -= static_cast<FakeBlock*>(p)->bytes;
        delete static_cast<FakeBlock*>(p);
    }
    return hipSuccess;
}
"""

MAIN = """
#include "scratch.cpp"
#include <cstdio>
#define CHECK(x) do { if (!(x)) { std::printf("line %%d: %%s\\n", __LINE__, #x); return 1; } } while (0)
using namespace hbfamd;
constexpr std::size_t MiB = std::size_t{1} << 20;
int main()
{
    scratch_hold();
%s
    return 0;
}
"""


def run(tmp_path, body):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(RUNTIME)
    src = tmp_path / "pool.cpp"
    src.write_text(MAIN % textwrap.indent(textwrap.dedent(body), "    "))
    exe = tmp_path / "pool"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", str(tmp_path), "-I", str(CSRC),
                    str(src), "-o", str(exe), "-pthread"], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout


@pytest.mark.parametrize("waited,waits", [("hipSuccess", 0), ("hipErrorUnknown", 1)])
def test_block_goes_back_only_after_a_wait(tmp_path, waited, waits):
    """A lease whose wait failed, or was skipped for an earlier error, waits again before its
    block can have another user."""
    run(tmp_path, f"""
        {{
            ScratchLease lease(1, nullptr);
            CHECK(lease.ok());
            lease.synced({waited});
        }}
        CHECK(fake.waits == {waits});
        {{
            ScratchLease lease(1, nullptr);  // never marked
        }}
        CHECK(fake.waits == {waits} + 1);
    """)


def test_a_block_past_the_limit_leaves_the_others(tmp_path):
    """A block larger than the pool keeps at all is freed by itself when it comes back; below the
    limit the oldest idle blocks make room."""
    run(tmp_path, """
        void* small[3];
        for (void*& p : small) { p = scratch_take(8 * MiB); }
        void* large = scratch_take(kScratchKeep + MiB);
        for (void* p : small) { scratch_give(p); }
        CHECK(fake.frees == 0);
        scratch_give(large);
        CHECK(fake.frees == 1 && fake.held == 24 * MiB);
        CHECK(scratch_take(8 * MiB) == small[0]);
        CHECK(fake.mallocs == 4);
        scratch_give(small[0]);
        void* wide = scratch_take(kScratchKeep - 8 * MiB);
        scratch_give(wide);  // small[0] came back last: it stays with this one
        CHECK(fake.held == kScratchKeep);
        CHECK(scratch_take(8 * MiB) == small[0]);
        scratch_give(small[0]);
        scratch_drop();  // the last holder
        CHECK(fake.held == 0);
    """)


def test_a_small_request_leaves_a_large_block(tmp_path):
    run(tmp_path, """
        void* large = scratch_take(256 * MiB);
        scratch_give(large);
        void* tiny = scratch_take(1000);
        CHECK(tiny != large && fake.mallocs == 2);
        void* again = scratch_take(200 * MiB);  // at least half of it
        CHECK(again == large && fake.mallocs == 2);
        scratch_give(tiny);
        scratch_give(again);
        CHECK(scratch_take(2000) == tiny);
    """)


def test_idle_blocks_go_before_an_allocation_fails(tmp_path):
    run(tmp_path, """
        fake.limit = 100 * MiB;
        void* a = scratch_take(60 * MiB);
        CHECK(scratch_take(60 * MiB) == nullptr);  // a is in use
        scratch_give(a);
        void* b = scratch_take(90 * MiB);  // a is idle, too small, and freed for it
        CHECK(b != nullptr && fake.frees == 1);
    """)
