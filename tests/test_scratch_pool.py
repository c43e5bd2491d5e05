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
