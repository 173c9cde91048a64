"""The copies of whole fields to the host (ilbm_host_copy.h) without a GPU:
the header compiled for the host against a model of the HIP calls it makes.
The model's copies run when something waits for them, its last error stays
until it is read, and its events belong to the device they were created on."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ilbmrex_amd", "csrc")

HIP = r"""
#pragma once
#include <unistd.h>
#include <cstdlib>
#include <cstring>
#include <mutex>
enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorInvalidHandle = 400 };
enum { hipMemcpyDeviceToHost, hipEventDisableTiming, hipHostMallocDefault };
struct Op { void* dst; const void* src; size_t n; };
struct Stream { int dev; std::mutex m; Op q[4096]; int head, tail; };
struct Event { int dev; Stream* s; int tail; };
typedef Stream* hipStream_t;
typedef Event* hipEvent_t;
inline thread_local int model_device = 0;
inline thread_local hipError_t model_last = hipSuccess;
inline bool model_no_pinned = false;
inline hipError_t model(hipError_t e) { if (e != hipSuccess) model_last = e; return e; }
inline hipError_t hipGetLastError() { hipError_t e = model_last; model_last = hipSuccess; return e; }
inline hipError_t hipGetDevice(int* d) { *d = model_device; return hipSuccess; }
inline hipError_t hipSetDevice(int d) { model_device = d; return hipSuccess; }
inline hipError_t hipStreamGetDevice(hipStream_t s, int* d) { *d = s->dev; return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = (Event*)calloc(1, sizeof(Event));
  (*e)->dev = model_device;
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (model_no_pinned) return model(hipErrorOutOfMemory);
  *p = malloc(n);
  return hipSuccess;
}
inline hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t st) {
  std::lock_guard<std::mutex> l(st->m);
  if (st->tail - st->head >= 4096) return model(hipErrorInvalidValue);
  st->q[st->tail++ % 4096] = Op{d, s, n};
  return hipSuccess;
}
inline void model_run(Stream* s, int until) {
  usleep(200);
  std::lock_guard<std::mutex> l(s->m);
  for (; s->head < until; ++s->head) { Op& o = s->q[s->head % 4096]; memcpy(o.dst, o.src, o.n); }
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (e->dev != s->dev) return model(hipErrorInvalidHandle);
  std::lock_guard<std::mutex> l(s->m);
  e->s = s;
  e->tail = s->tail;
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) { model_run(e->s, e->tail); return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t s) {
  int t;
  { std::lock_guard<std::mutex> l(s->m); t = s->tail; }
  model_run(s, t);
  return hipSuccess;
}
"""

MAIN = r"""
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <string>
#include <vector>
#include "ilbm_host_copy.h"
static thread_local bool no_host_memory = false;
void* operator new(size_t n) {
  void* p = no_host_memory ? nullptr : malloc(n);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }
using ilbm::HostCopy;
static const size_t kBytes = HostCopy::kDirect + 3 * HostCopy::kSlice + 40;
static std::vector<uint32_t> field(uint32_t seed) {
  std::vector<uint32_t> v(kBytes / 4);
  for (size_t i = 0; i < v.size(); ++i) v[i] = (uint32_t)i * 2654435761u + seed;
  return v;
}
int main(int, char** argv) {
  const std::string what = argv[1];
  static Stream s;
  s.dev = (what == "device") ? 1 : 0;
  const std::vector<uint32_t> a = field(1), b = field(2);
  std::vector<uint32_t> x(a.size()), y(b.size());
  HostCopy c;
  if (what == "threads") {
    for (int rep = 0; rep < 3; ++rep) {
      std::thread t([&] { c.copy(x.data(), a.data(), kBytes, &s); });
      c.copy(y.data(), b.data(), kBytes, &s);
      t.join();
      if (x != a || y != b) return 1;
      std::fill(x.begin(), x.end(), 0);
      std::fill(y.begin(), y.end(), 0);
    }
    return 0;
  }
  model_no_pinned = what == "pinned";
  no_host_memory = what == "memory";
  try {
    c.copy(x.data(), a.data(), kBytes, &s);
  } catch (const ilbm::HipError& e) {
    printf("error %d\n", (int)e.e);
    return 2;
  }
  no_host_memory = false;
  if (x != a) return 1;
  if (hipGetLastError() != hipSuccess) return 3;   // nothing failed for the caller
  return model_device == 0 ? 0 : 4;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("host_copy")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(HIP)
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", str(d), "-I", CSRC, str(d / "main.cpp"), "-o",
                    str(d / "prog")], check=True)
    return str(d / "prog")


def _run(program, what):
    return subprocess.run([program, what], timeout=60).returncode


def test_one_copy(program):
    assert _run(program, "plain") == 0


def test_two_threads_read_one_level(program):
    assert _run(program, "threads") == 0


def test_no_pinned_memory_leaves_no_error_behind(program):
    assert _run(program, "pinned") == 0


def test_level_of_another_device_than_the_current_one(program):
    assert _run(program, "device") == 0


def test_no_host_memory_for_a_thread(program):
    assert _run(program, "memory") == 0
