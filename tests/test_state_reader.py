"""StateReader (csrc/state_reader.hpp) on the CPU, against a stub of the HIP calls it makes: states of
every size arrive whole whatever size its slots were made for, and pinned memory is taken for those
that go through it alone; a large state arrives whole also where some of its threads cannot be started, for want of memory (the
thread's own record) as for want of threads."""
import shutil
import subprocess

import pytest

from shaderous_amd import build

STUB = r"""
#pragma once
#include <stddef.h>
#include <stdlib.h>
#include <string.h>
typedef void* hipStream_t;
typedef void* hipEvent_t;
typedef int hipError_t;
enum { hipSuccess = 0, hipHostMallocDefault = 0, hipEventDisableTiming = 2, hipMemcpyDeviceToHost = 2 };
enum { hipMemoryTypeUnregistered = 0 };
struct hipPointerAttribute_t { int type; };
static size_t pinned = 0;
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) { pinned = n; *p = malloc(n); return *p ? 0 : 2; }
inline hipError_t hipHostFree(void* p) { free(p); return 0; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = nullptr; return 0; }
inline hipError_t hipEventDestroy(hipEvent_t) { return 0; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return 0; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return 0; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return 0; }
inline hipError_t hipSetDevice(int) { return 0; }
inline hipError_t hipGetLastError() { return 0; }
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) { a->type = 0; return 0; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t) { memcpy(d, s, n); return 0; }
"""

MAIN = r"""
#include "state_reader.hpp"
#include <new>
#include <stdio.h>
#include <vector>
static thread_local bool counting = false;
static int left = -1;      // allocations of the reading thread until one fails
void* operator new(size_t n) {
  if (counting && left >= 0 && left-- == 0) throw std::bad_alloc();
  void* p = malloc(n);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }
int main() {
  const size_t n = ((size_t)20 << 20) + 48;
  std::vector<char> a(n), b(n), x(n), y(n);
  for (size_t i = 0; i < n; i++) { a[i] = (char)(i * 7 + i / 4099); b[i] = (char)(i * 5 + 1); }
  shx::StateReader r;
  r.fit(2 * n, 2 * n);
  for (int fail = -1; fail < 6; fail++) {
    std::fill(x.begin(), x.end(), 0);
    std::fill(y.begin(), y.end(), 0);
    left = fail;
    counting = true;
    const int rc = r.read(nullptr, 0, x.data(), a.data(), y.data(), b.data(), n);
    counting = false;
    if (rc != 0 || x != a || y != b) return 1;
    printf("allocation %d failed: read whole\n", fail);
  }
  // readers made for states of one size, or of a range as an ensemble's, read any other
  const size_t K = 1024, M = K * K;
  const size_t fits[][3] = {{3000, 3000, 4096}, {512 * K, 512 * K, 512 * K}, {512 * K + 16, 512 * K + 16, 0},
                            {8 * M - 16, 8 * M - 16, 0}, {128 * K, 2 * M, 512 * K}, {4 * K, 96 * K, 96 * K}};
  for (auto& f : fits) {
    pinned = 0;
    shx::StateReader s;
    s.fit(f[0], f[1]);
    if (pinned != f[2]) return 2;
    for (size_t each : {(size_t)16, 64 * K, 256 * K, 256 * K + 16, M, 4 * M, 9 * M + 16}) {
      std::fill(x.begin(), x.end(), 0);
      std::fill(y.begin(), y.end(), 0);
      if (s.read(nullptr, 0, x.data(), a.data(), y.data(), b.data(), each) != 0) return 3;
      if (memcmp(x.data(), a.data(), each) || memcmp(y.data(), b.data(), each) || x[each] || y[each]) return 4;
      s.fit(2 * each, 2 * each);   // as after a re-mesh
    }
  }
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_reads_arrive_whole_when_threads_cannot_start(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(STUB)
    (tmp_path / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", f"-I{tmp_path}", f"-I{build.CSRC}", "main.cpp", "-o", "main"],
                   cwd=tmp_path, check=True)
    r = subprocess.run(["./main"], cwd=tmp_path, capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
