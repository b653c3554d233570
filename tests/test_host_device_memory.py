"""Device memory that the library keeps between calls (votca_amd/csrc/xtpgpu_internal.h): the kept blocks, the
contexts' kept scratch and what becomes of both before an allocation is refused. Compiled with g++ against a card of
1 GiB that the driver plays itself: the HIP calls are its own and hand out addresses that nothing reads."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include "xtpgpu_internal.h"
#include <cstdlib>
#include <map>
namespace {
std::map<void*, size_t> live;
size_t used = 0;
const size_t kCard = (size_t)1 << 30, MB = (size_t)1 << 20;
}
extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  if (used + n > kCard) { *p = nullptr; return hipErrorOutOfMemory; }
  static size_t at = 0x1000000;
  *p = reinterpret_cast<void*>(at);
  at += n + 256;
  used += n;
  live[*p] = n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (!live.count(p)) std::abort();
  used -= live[p];
  live.erase(p);
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) { *f = kCard - used; *t = kCard; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipEventCreate(hipEvent_t*) { return hipSuccess; }
hipError_t hipEventElapsedTime(float*, hipEvent_t, hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
}
using namespace xg;
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s (used %zu MiB)\n", __LINE__, #c, used / MB); return 1; } } while (0)
bool fits(size_t n) {
  try { DevBuf b(n); return b.p != nullptr; } catch (const Error& e) { if (e.code != XTPGPU_ERR_OOM) std::abort(); return false; }
}
int main() {
  {
    xtpgpu_ctx_s a, b;
    for (xtpgpu_ctx_s* c : {&a, &b})
      for (KeptBuf* k : c->kept()) KeptList::get().add(0, k);
    { Scratch s(a.adjoint_ws), t(b.sum_ws); s.get(200 * MB); t.get(100 * MB); }
    { DevBuf x(300 * MB); }
    CHECK(used == 600 * MB);            // 300 in the contexts' scratch, 300 in the kept block
    CHECK(fits(1000 * MB));             // all of it goes back first
    DevBuf::drain_current();
    CHECK(used == 0);
    {
      Scratch s(a.adjoint_ws);
      s.get(200 * MB);
      { Scratch t(b.host_ws); t.get(100 * MB); }
      CHECK(!fits(900 * MB));           // a call's own scratch stays
      CHECK(fits(800 * MB));
      DevBuf::drain_current();
      CHECK(used == 200 * MB);
      Scratch again(a.adjoint_ws);      // held: a buffer of its own
      again.get(8 * MB);
      CHECK(used == 208 * MB);
      CHECK(a.adjoint_ws.buf.bytes == 200 * MB);
    }
    CHECK(used == 200 * MB);
    { Scratch s(a.adjoint_ws); s.get(KeptBuf::kKeepBytes + MB); }
    CHECK(a.adjoint_ws.buf.bytes == 200 * MB);  // more than is kept is not
    int calls = 0;
    const int r = with_reclaim(5, [&] { return ++calls == 1 ? 5 : (used == 0 ? 0 : 5); });
    CHECK(r == 0 && calls == 2);
    CHECK(with_reclaim(5, [&] { return 3; }) == 3);
  }
  KeptList::get().release(0);           // the contexts are gone from the list
  CHECK(used == 0 && live.empty());
  std::printf("ok\n");
  return 0;
}
"""


def test_kept_memory_is_given_back(tmp_path):
    if shutil.which("g++") is None or not os.path.exists("/opt/rocm/include/hip/hip_runtime.h"):
        pytest.skip("needs g++ and the HIP headers")
    src, exe = tmp_path / "driver.cpp", tmp_path / "driver"
    src.write_text(DRIVER)
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                        "-I", os.path.join(ROOT, "votca_amd", "csrc"), str(src), "-o", str(exe), "-pthread"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout + out.stderr
