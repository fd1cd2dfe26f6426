"""The staged host copies (flusi_amd/csrc/hostcopy.cpp) built for the host
against a stand-in for the HIP runtime, whose copies happen at once and whose
calls can be made to fail.  CPU only."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "flusi_amd", "csrc")

HIP = r"""
#pragma once
#include <atomic>
#include <cstddef>
#include <cstdio>
#include <cstdlib>
#include <cstring>
enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
struct Event { int device; };
using hipEvent_t = Event*;
using hipStream_t = int*;  // its device
constexpr unsigned hipEventDisableTiming = 2, hipHostMallocDefault = 0;
inline thread_local int cur_device = 0;
inline thread_local hipError_t last_error = hipSuccess;
inline std::atomic<int> allocs{0}, frees{0}, fail_alloc_from{1 << 30}, events{0}, fail_event_from{1 << 30}, faults{0};
inline std::atomic<int> fail_copies{0};
inline hipError_t hip_ret(hipError_t e) { if (e) last_error = e; return e; }
inline hipError_t hipGetLastError() { hipError_t e = last_error; last_error = hipSuccess; return e; }
inline hipError_t hipSetDevice(int d) { cur_device = d; return hipSuccess; }
inline hipError_t hipGetDevice(int* d) { *d = cur_device; return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (allocs++ >= fail_alloc_from) return hip_ret(hipErrorOutOfMemory);
  *p = std::malloc(n);
  return hipSuccess;
}
inline hipError_t hipHostFree(void* p) { std::free(p); ++frees; return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  if (events++ >= fail_event_from) return hip_ret(hipErrorOutOfMemory);
  *e = new Event{cur_device};
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (e->device != *s) ++faults;  // an event of another device
  return hipSuccess;
}
enum hipMemoryType { hipMemoryTypeHost, hipMemoryTypeDevice, hipMemoryTypeManaged, hipMemoryTypeUnregistered };
struct hipPointerAttribute_t { hipMemoryType type; };
inline int pointer_type = -1;  // -1: the call knows nothing of the address
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) {
  if (pointer_type < 0) return hip_ret(hipErrorInvalidValue);
  a->type = (hipMemoryType)pointer_type;
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  if (fail_copies) return hip_ret(hipErrorInvalidValue);
  std::memcpy(d, s, n);
  return hipSuccess;
}
"""

MAIN = r"""
#include "hostcopy.h"
#include <vector>
using namespace flusi;
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
// with slots made by a copy out: a pool's first small copy in makes none
template <typename T> int round_trip(HostCopyPool& pool, int* stream) {
  const long n = 13000003;  // 48 MB on the wire and a remainder
  std::vector<double> a(n), b(n);
  std::vector<T> dev(n);
  for (long i = 0; i < n; ++i) a[i] = 1.0 / (double)(i + 1);
  hipError_t e = hipErrorInvalidValue;
  CHECK(host_copy_out<T>(pool, dev.data(), b.data(), n, stream, e) && e == hipSuccess);
  e = hipErrorInvalidValue;
  CHECK(host_copy_in<T>(pool, a.data(), dev.data(), n, stream, e) && e == hipSuccess);
  CHECK(host_copy_out<T>(pool, dev.data(), b.data(), n, stream, e) && e == hipSuccess);
  for (long i = 0; i < n; ++i) CHECK(dev[i] == (T)a[i] && b[i] == (double)dev[i]);
  return 0;
}
"""


def _run(tmp_path, body):
    os.makedirs(tmp_path / "hip")
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    main = tmp_path / "main.cpp"
    main.write_text(MAIN + "int main() {\n" + body + "\n  std::printf(\"ok\\n\");\n  return 0;\n}\n")
    exe = str(tmp_path / "a.out")
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-I", str(tmp_path), "-I", CSRC, str(main),
                    os.path.join(CSRC, "hostcopy.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr


def test_round_trips(tmp_path):
    _run(tmp_path, """
  int s = 0;
  auto pool = host_copy_pool(0);
  if (round_trip<double>(*pool, &s) || round_trip<float>(*pool, &s)) return 1;
  pool.reset();
  CHECK(allocs == frees);""")


@pytest.mark.parametrize("what", ["alloc", "event"])
def test_no_staging_memory_is_not_an_error(tmp_path, what):
    """Nothing is copied, no error is left behind, and the caller is told to
    copy plainly; a transfer that fails is an error."""
    _run(tmp_path, f"""
  int s = 0;
  auto pool = host_copy_pool(0);
  const long n = 7000000;
  std::vector<double> a(n, 1.0), dev(n, 0.0);
  hipError_t e = hipSuccess;
  fail_{what}_from = {"0" if what == "alloc" else "5"};
  CHECK(!host_copy_in<double>(*pool, a.data(), dev.data(), n, &s, e));
  CHECK(hipGetLastError() == hipSuccess && dev[0] == 0.0 && dev[n - 1] == 0.0);
  CHECK(!host_copy_out<double>(*pool, dev.data(), a.data(), n, &s, e));
  CHECK(hipGetLastError() == hipSuccess && a[0] == 1.0 && a[n - 1] == 1.0);
  fail_{what}_from = 1 << 30;
  CHECK(host_copy_in<double>(*pool, a.data(), dev.data(), n, &s, e) && e == hipSuccess && dev[n - 1] == 1.0);
  fail_copies = 1;
  CHECK(host_copy_in<double>(*pool, a.data(), dev.data(), n, &s, e) && e != hipSuccess);""")


def test_device_of_the_context(tmp_path):
    """The events are made and recorded on the pool's device, and the caller's
    current device is left as it was."""
    _run(tmp_path, """
  int s = 1;
  cur_device = 0;
  auto pool = host_copy_pool(1);
  if (round_trip<double>(*pool, &s) || round_trip<float>(*pool, &s)) return 1;
  CHECK(faults == 0 && cur_device == 0);""")


def test_memory_the_runtime_knows(tmp_path):
    """Pinned arrays of FP64 fields, managed and device memory are copied
    plainly, as everything below the threshold is."""
    _run(tmp_path, """
  const void* p = &events;
  const long n = 7000000, m = 2 * n;
  for (int t : {-1, (int)hipMemoryTypeUnregistered}) {
    pointer_type = t;
    CHECK(host_copy_pays(p, n, 8) && host_copy_pays(p, m, 4) && hipGetLastError() == hipSuccess);
    CHECK(!host_copy_pays(p, n / 2, 8) && !host_copy_pays(p, n, 4));
  }
  pointer_type = hipMemoryTypeHost;
  CHECK(!host_copy_pays(p, n, 8) && host_copy_pays(p, m, 4));
  for (int t : {(int)hipMemoryTypeDevice, (int)hipMemoryTypeManaged}) {
    pointer_type = t;
    CHECK(!host_copy_pays(p, n, 8) && !host_copy_pays(p, m, 4));
  }""")


def test_when_slots_are_made(tmp_path):
    """A small copy in makes none at first; a copy out, a second one in and a
    large one in do, and a larger copy's replace smaller slots."""
    _run(tmp_path, """
  int s = 0;
  const long n = 7000000, big = 45000000;  // 56 and 360 MB of FP64
  std::vector<double> a(big, 2.0), dev(big, 0.0);
  hipError_t e = hipSuccess;
  auto pool = host_copy_pool(0);
  CHECK(!host_copy_in<double>(*pool, a.data(), dev.data(), n, &s, e) && allocs == 0 && dev[0] == 0.0);
  CHECK(host_copy_in<double>(*pool, a.data(), dev.data(), n, &s, e) && allocs == 1 && dev[n - 1] == 2.0);
  CHECK(host_copy_in<double>(*pool, a.data(), dev.data(), big / 2, &s, e) && allocs == 1 && dev[big / 2 - 1] == 2.0);
  CHECK(host_copy_in<double>(*pool, a.data(), dev.data(), big, &s, e) && allocs == 2 && frees == 1 && dev[big - 1] == 2.0);
  CHECK(host_copy_out<double>(*pool, dev.data(), a.data(), n, &s, e) && allocs == 2);
  pool.reset();
  CHECK(frees == 2);
  pool = host_copy_pool(0);
  CHECK(host_copy_out<double>(*pool, dev.data(), a.data(), n, &s, e) && allocs == 3);
  pool.reset();
  pool = host_copy_pool(0);
  CHECK(host_copy_in<double>(*pool, a.data(), dev.data(), big, &s, e) && allocs == 4);""")
