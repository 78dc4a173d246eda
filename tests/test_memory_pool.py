"""The library's pool of device memory, compiled from its own header with g++ against stand-ins for the HIP calls it
makes (no GPU): which calls a release makes and in which capture mode, when a block that comes back is waited for before
it is handed on, what happens where the device cannot be waited for or has no memory left, and the bound on idle memory."""

import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]
CSRC = ROOT / "alpha-fly_amd" / "csrc"
HIP_INCLUDE = pathlib.Path("/opt/rocm/include")

PROGRAM = r"""
#include "common.hpp"
#include <cstdio>
#include <cstdlib>
#include <set>

// stand-ins: every call is noted, memory is an address
static int waits = 0, mallocs = 0, frees = 0, unsafe = 0;
static bool wait_fails = false;
static size_t held = 0, limit = (size_t)1 << 40;
static std::map<void *, size_t> blocks;
static thread_local hipStreamCaptureMode mode = hipStreamCaptureModeGlobal;
static uintptr_t next_address = 1 << 20;

hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stand-in"; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *m) { std::swap(*m, mode); return hipSuccess; }
hipError_t hipDeviceSynchronize() { ++unsafe; return hipSuccess; }   // spoils a capture in any mode
hipError_t hipMalloc(void **p, size_t n) {
  if (held + n > limit) return hipErrorOutOfMemory;
  if (n > 4096) ++mallocs;
  *p = reinterpret_cast<void *>(next_address);
  next_address += n + 4096;
  blocks[*p] = n;
  held += n;
  return hipSuccess;
}
hipError_t hipFree(void *p) {                 // waits for the device; the pool waits with a block of 4 KiB
  if (blocks.at(p) > 4096) ++frees;
  else ++waits;
  if (mode != hipStreamCaptureModeRelaxed) ++unsafe;
  held -= blocks.at(p);
  const bool fails = blocks.at(p) == 4096 && wait_fails;
  blocks.erase(p);
  return fails ? hipErrorUnknown : hipSuccess;
}
namespace fly { void set_error(const std::string &) {} }

using fly::DevArray;
using fly::DevicePool;
#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); exit(1); } } while (0)
static void reset() { waits = mallocs = frees = 0; }

int main() {
  const size_t MB = 1 << 20;
  DevArray<char> keep(10 * MB);                 // a live object throughout
  CHECK(mallocs == 1);

  // a release frees nothing and waits for nothing; the block is handed on after one wait
  { DevArray<char> a(20 * MB); }
  CHECK(frees == 0 && waits == 0 && mallocs == 2);
  reset();
  { DevArray<char> a(20 * MB); CHECK(waits == 1 && mallocs == 0); }

  // one wait covers every block that came back before it, and none that came back after
  { DevArray<char> a(20 * MB), b(40 * MB); }
  reset();
  {
    DevArray<char> a(20 * MB);
    CHECK(waits == 1);
    DevArray<char> b(40 * MB);
    CHECK(waits == 1 && mallocs == 0);
    b.release();
    DevArray<char> c(40 * MB);
    CHECK(waits == 2 && mallocs == 0);
  }

  // a block released as idle already needs no wait
  DevicePool::get().trim(-1);
  { DevArray<char> a(20 * MB); fly::QuietRelease quiet; a.release(); }
  reset();
  { DevArray<char> a(20 * MB); CHECK(waits == 0 && mallocs == 0); }

  // where the device cannot be waited for, new memory is taken and the block stays idle until it can be
  wait_fails = true;
  reset();
  {
    DevArray<char> a(20 * MB);
    CHECK(waits == 1 && mallocs == 1);
    wait_fails = false;
    DevArray<char> b(20 * MB);
    CHECK(waits == 2 && mallocs == 1);
  }

  // no more than 512 MiB stay idle
  DevicePool::get().trim(-1);
  CHECK(held == 10 * MB);
  { DevArray<char> a(300 * MB), b(200 * MB), c(100 * MB); }
  CHECK(held <= (10 + 512) * MB && held >= 300 * MB);

  // an allocation that fails gets the idle blocks' memory
  limit = held;
  reset();
  { DevArray<char> a(250 * MB); CHECK(mallocs == 1 && frees == 2); }
  limit = (size_t)1 << 40;

  // trimming, and the last release, give all of it back
  DevicePool::get().trim(-1);
  CHECK(held == 10 * MB);
  { DevArray<char> a(20 * MB); }
  keep.release();
  CHECK(held == 0 && blocks.empty());

  // no free outside the relaxed capture mode, which is the thread's own again, and no hipDeviceSynchronize
  CHECK(unsafe == 0 && mode == hipStreamCaptureModeGlobal);
  printf("ok\n");
  return 0;
}
"""


def test_pool_against_stand_ins(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None or not (HIP_INCLUDE / "hip" / "hip_runtime.h").exists():
        pytest.skip("g++ or the HIP headers are not installed")
    (tmp_path / "pool.cpp").write_text(PROGRAM)
    subprocess.run([gxx, "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{HIP_INCLUDE}", f"-I{CSRC}", f"-I{ROOT / 'include'}",
                    str(tmp_path / "pool.cpp"), "-o", str(tmp_path / "pool")], check=True)
    out = subprocess.run([str(tmp_path / "pool")], capture_output=True, text=True)
    assert out.stdout == "ok\n", out.stdout
