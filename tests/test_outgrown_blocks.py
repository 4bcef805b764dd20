"""Blocks that a context's buffers outgrew (cheese_amd/csrc/host.h, built here with g++ over a HIP stub with a limited
amount of device memory) are memory too: whatever asks for a block when the device has none left, be it a growing buffer or
an untyped block, waits for the stream, gives them back and asks again.  CPU only."""
import re
import subprocess

from test_block_cache import ROOT, STUB

LIMIT = r"""
#include <map>
extern size_t device_left; extern long n_sync;
inline std::map<void *, size_t> &device_blocks() { static std::map<void *, size_t> m; return m; }
inline hipError_t hipMalloc(void **p, size_t n) {
  if (n > device_left) return 2;
  device_left -= n;
  *p = (void *)(uintptr_t)(++n_malloc * 4096);
  device_blocks()[*p] = n;
  return 0;
}
inline hipError_t hipFree(void *p) { n_free++; device_left += device_blocks()[p]; device_blocks().erase(p); return 0; }
inline hipError_t hipStreamSynchronize(hipStream_t) { n_sync++; return 0; }
"""

MAIN = r"""
#include <cstdio>
#include "host.h"
long n_malloc, n_free, live, n_sync;
size_t device_left;
#define CHECK(c) do { if (!(c)) { std::printf("%d: %s\n", __LINE__, #c); return 1; } } while (0)
// a buffer of 4 MiB that has grown to 8 leaves its first block with the context, 12 MiB in use of `total`
static void grown(chz::DBuf<char> &b, size_t total) {
  chz::dev_pool().trim();
  device_left = total;
  b.need(4 << 20);
  b.need(8 << 20);
}
int main() {
  const size_t M = 1 << 20;
  const hipStream_t stream = (hipStream_t)1;
  for (int how = 0; how < 3; how++) {
    chz::Retired retired;
    chz::StreamScope scope(stream, &retired);
    chz::DBuf<char> b, o;
    grown(b, 14 * M);
    CHECK(retired.size() == 1 && device_left == 2 * M);
    const long syncs = n_sync;
    void *p = nullptr;
    size_t got = 0;
    // 5 MiB: more than is left, less than with the outgrown block given back
    if (how == 0) { o.need(5 * M); p = o.p; }
    else if (how == 1) p = chz::dev_alloc(5 * M);
    else p = chz::block_get(5 * M, got);
    CHECK(p && retired.empty() && n_sync == syncs + 1);
    // 9 MiB: not there at all, an error as ever
    bool failed = false;
    try { chz::dev_alloc(9 * M); } catch (chz::DeviceError &) { failed = true; }
    CHECK(failed && n_sync == syncs + 1);
    if (how == 0) o.release();
    else if (how == 1) chz::dev_free(p);
    else chz::dev_pool().put(p, got);
    b.release();
  }
  {   // without a context's list an outgrown block goes back at once, after a synchronisation
    chz::StreamScope scope(stream);
    chz::DBuf<char> b;
    grown(b, 14 * M);
    CHECK(chz::dev_pool().cached == 4 * M);
    b.release();
  }
  return 0;
}
"""


def test_a_full_device_gives_outgrown_blocks_back(tmp_path):
    stub = STUB
    for name in ("hipMalloc", "hipFree", "hipStreamSynchronize"):
        stub = re.sub(rf"inline hipError_t {name}\(.*\n", "", stub)
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(stub + LIMIT)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = tmp_path / "main"
    subprocess.run(["g++", "-O1", "-std=c++17", f"-I{tmp_path}", f"-I{ROOT}/cheese_amd/csrc", "-o", str(exe),
                    str(tmp_path / "main.cpp"), "-pthread"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
