"""The device memory pool (csrc/device_pool.cpp) on the host: its source built
against a hipMalloc and hipFree that hand out addresses from a bounded count,
and driven by small C++ programs."""
import os
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "kodama_amd", "csrc")
ROCM = os.environ.get("ROCM", "/opt/rocm")

PRELUDE = r"""
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include "device.h"
// A device of `g_room` bytes; addresses are never dereferenced.
static std::map<void*, size_t> g_live;
static size_t g_used = 0, g_room = size_t(64) << 30, g_next = 4096;
static int g_mallocs = 0, g_frees = 0;
extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  ++g_mallocs;
  if (g_used + n > g_room) return hipErrorOutOfMemory;
  *p = reinterpret_cast<void*>(g_next);
  g_next += n;
  g_live[*p] = n;
  g_used += n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  ++g_frees;
  if (!g_live.count(p)) { std::printf("freed twice\n"); std::exit(2); }
  g_used -= g_live[p];
  g_live.erase(p);
  return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stub"; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
}
using namespace kodama_hip;
namespace kodama_hip {
hipStream_t take_stream(int) { return reinterpret_cast<hipStream_t>(8); }
void give_stream(int, hipStream_t) {}
}
static hipStream_t tag(size_t i) { return reinterpret_cast<hipStream_t>(16 * (i + 1)); }
constexpr size_t MiB = size_t(1) << 20;
#define EXPECT(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)
"""


@pytest.fixture
def run(tmp_path):
    def go(body):
        src, exe = tmp_path / "pool.cpp", tmp_path / "pool"
        src.write_text(PRELUDE + "int main() {\n" + body + "\nreturn 0;\n}\n")
        subprocess.run(["g++", "-std=gnu++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"),
                        "-I", CSRC, str(src), os.path.join(CSRC, "device_pool.cpp"), "-o", str(exe), "-pthread"],
                       check=True, capture_output=True, text=True)
        out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
        assert out.returncode == 0, out.stdout + out.stderr
    return go


def test_a_full_pool_takes_blocks_of_another_size(run):
    """A call that leaves the pool full of large blocks, then calls with small
    ones: from the second of these on nothing is allocated or freed."""
    run(r"""
    PoolBlock big[4];
    for (auto& b : big) b = pool_take(512 * MiB, 0, tag(0));
    for (auto& b : big) pool_give(b);
    pool_settle(0, tag(0));
    EXPECT(g_used == 2048 * MiB);
    int mallocs = 0, frees = 0;
    for (int call = 0; call < 5; ++call) {
      if (call == 1) { mallocs = g_mallocs; frees = g_frees; }
      PoolBlock small[8];
      for (auto& b : small) b = pool_take(40 * MiB, 0, tag(1));
      for (auto& b : small) pool_give(b);
      pool_settle(0, tag(1));
    }
    EXPECT(g_mallocs == mallocs && g_frees == frees);
    EXPECT(g_used <= kPoolBytes);
    """)


def test_the_longest_unused_block_goes_first(run):
    run(r"""
    PoolBlock a = pool_take(600 * MiB, 0, tag(0)), b = pool_take(700 * MiB, 0, tag(0)), c = pool_take(500 * MiB, 0, tag(0));
    void* const pb = b.p; void* const pc = c.p;
    pool_give(a); pool_give(b); pool_give(c);
    pool_settle(0, tag(0));
    pool_give(pool_take(840 * MiB, 0, tag(1)));  // beside 1800 kept: the oldest leaves
    pool_settle(0, tag(1));
    EXPECT(g_frees == 1 && g_live.count(a.p) == 0);
    PoolBlock b2 = pool_take(700 * MiB, 0, tag(2)), c2 = pool_take(500 * MiB, 0, tag(2));
    EXPECT(b2.p == pb && c2.p == pc);
    pool_give(b2); pool_give(c2);
    """)


def test_blocks_of_unfinished_work_are_not_evicted(run):
    """Blocks whose stream may still be using them stay; what comes back over
    the bound is freed (hipFree waits for its work)."""
    run(r"""
    PoolBlock held[4];
    for (auto& b : held) b = pool_take(500 * MiB, 0, tag(0));
    for (auto& b : held) pool_give(b);           // not settled
    PoolBlock other = pool_take(400 * MiB, 0, tag(1));
    void* const p = other.p;
    pool_give(other);
    EXPECT(g_frees == 1 && g_live.count(p) == 0);
    for (auto& b : held) EXPECT(g_live.count(b.p) == 1);
    """)


def test_a_block_larger_than_the_pool_evicts_nothing(run):
    run(r"""
    PoolBlock keep = pool_take(100 * MiB, 0, tag(0)), huge = pool_take(kPoolBytes + MiB, 0, tag(0));
    pool_give(keep);
    pool_settle(0, tag(0));
    pool_give(huge);
    EXPECT(g_live.count(keep.p) == 1 && g_live.count(huge.p) == 0);
    """)


def test_an_allocation_outside_a_call_gets_the_kept_memory(run):
    """A buffer without a stream scope (the arrays of a resident graph) on a
    device whose free memory is what the pool keeps."""
    run(r"""
    g_room = 1024 * MiB;
    PoolBlock b = pool_take(800 * MiB, 0, tag(0));
    pool_give(b);
    pool_settle(0, tag(0));
    DeviceBuffer<float> plain(600 * MiB / sizeof(float));
    EXPECT(plain.get() != nullptr && g_live.size() == 1 && g_used == 600 * MiB);
    plain.release();
    EXPECT(g_used == 0);
    bool threw = false;
    try { DeviceBuffer<float> much(1025 * MiB / sizeof(float)); } catch (const DeviceError&) { threw = true; }
    EXPECT(threw);
    """)


def test_everything_kept_can_be_given_back(run):
    """Settled blocks and those of unfinished work (hipFree waits for it), on
    one device only; blocks in use stay."""
    run(r"""
    PoolBlock a = pool_take(10 * MiB, 0, tag(0)), b = pool_take(20 * MiB, 0, tag(1)), c = pool_take(30 * MiB, 0, tag(1));
    PoolBlock other = pool_take(40 * MiB, 1, tag(2));
    pool_give(a); pool_give(b); pool_give(other);
    pool_settle(0, tag(0));
    pool_empty(0);
    EXPECT(g_live.size() == 2 && g_live.count(c.p) && g_live.count(other.p));
    pool_give(c);
    EXPECT(pool_take(30 * MiB, 0, tag(1)).p == c.p);
    """)
