"""The device block cache (cheese_amd/csrc/host.h, built here with g++ over a HIP stub that counts): a full cache frees its
oldest blocks, not the one that comes in; a request takes a cached block of up to twice its size.  CPU only."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

STUB = r"""
#pragma once
#include <cstddef>
#include <cstdint>
#include <cstdlib>
typedef int hipError_t; typedef void *hipStream_t; typedef void *hipEvent_t;
enum { hipSuccess = 0, hipHostMallocDefault = 0 };
enum hipStreamCaptureMode { hipStreamCaptureModeRelaxed };
enum hipMemcpyKind { hipMemcpyDefault };
extern long n_malloc, n_free, live;
inline hipError_t hipMalloc(void **p, size_t) { *p = (void *)(uintptr_t)(++n_malloc * 4096); live++; return 0; }
inline hipError_t hipFree(void *) { n_free++; live--; return 0; }
inline hipError_t hipGetDevice(int *d) { *d = 0; return 0; }
inline hipError_t hipGetLastError() { return 0; }
inline const char *hipGetErrorString(hipError_t) { return ""; }
inline hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *) { return 0; }
inline hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t) { return 0; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return 0; }
inline hipError_t hipDeviceSynchronize() { return 0; }
inline hipError_t hipHostMalloc(void **, size_t, int) { return 0; }
inline hipError_t hipHostFree(void *) { return 0; }
inline hipError_t hipEventCreate(hipEvent_t *) { return 0; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return 0; }
inline hipError_t hipEventElapsedTime(float *, hipEvent_t, hipEvent_t) { return 0; }
inline hipError_t hipEventDestroy(hipEvent_t) { return 0; }
"""

MAIN = r"""
#include <cstdio>
#include "host.h"
long n_malloc, n_free, live;
#define CHECK(c) do { if (!(c)) { std::printf("%d: %s\n", __LINE__, #c); return 1; } } while (0)
int main() {
  chz::DevPool pool;
  const size_t G = (size_t)1 << 30;
  size_t got = 0, big = 0;
  // 16 blocks of 1 GiB fill the cache; a small block given back after them stays and is found again
  void *a[16];
  for (int i = 0; i < 16; i++) a[i] = pool.get(G, got);
  for (int i = 0; i < 16; i++) pool.put(a[i], got);
  CHECK(pool.cached == 16 * G && n_free == 0);
  void *s = pool.get(G / 64, got);
  CHECK(got == G / 64 && n_malloc == 17);
  pool.put(s, got);
  CHECK(n_free == 1 && pool.cached == 15 * G + G / 64);
  CHECK(pool.get(G / 64, got) == s && n_malloc == 17);
  // the oldest went: the second one is still there
  CHECK(pool.get(G, got) == a[1] && n_malloc == 17);
  pool.put(a[1], got);
  // up to twice the size, with the block's own size reported, and no further
  void *h = pool.get(G / 2, got);
  CHECK(n_malloc == 17 && got == G);
  pool.put(h, got);
  pool.get(G / 2 - 1024 * 1024, got);
  CHECK(n_malloc == 17 && got == G);
  pool.get(G / 4, got);
  CHECK(n_malloc == 18 && got == G / 4);
  // a block above the bound is never cached, one of exactly the bound replaces everything
  void *b = pool.get(20 * G, big);
  const long before = n_free;
  const size_t kept = pool.cached;
  pool.put(b, big);
  CHECK(n_free == before + 1 && pool.cached == kept);
  b = pool.get(16 * G, big);
  pool.put(b, big);
  CHECK(pool.cached == 16 * G && pool.free_blocks.size() == 1);
  pool.trim();
  CHECK(pool.cached == 0 && pool.free_blocks.empty());
  return 0;
}
"""


def test_a_full_cache_frees_its_oldest_blocks(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(STUB)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = tmp_path / "main"
    subprocess.run(["g++", "-O1", "-std=c++17", f"-I{tmp_path}", f"-I{ROOT}/cheese_amd/csrc", "-o", str(exe),
                    str(tmp_path / "main.cpp"), "-pthread"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
