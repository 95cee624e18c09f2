"""Device memory of the library: blocks of closed contexts are kept for the next one, but never at the cost of an
allocation that fails. devmem.cpp is built here against a stand-in for the HIP runtime's allocator with a
fixed capacity, and the sources are checked to allocate device memory through it alone. On the GPU: what a context gives
back while it lives goes back to the device."""
import glob
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = glob.glob(os.path.join(ROOT, "*_amd", "csrc"))[0]

DRIVER = r"""
#include "devmem.h"
#include <cstdio>
#include <cstdlib>
#include <unordered_map>
static size_t capacity = 0, used = 0;
static std::unordered_map<void*, size_t> blocks;
static int mallocs = 0, frees = 0;
extern "C" hipError_t hipMalloc(void** p, size_t n) {
  *p = nullptr;
  if (used + n > capacity) return hipErrorOutOfMemory;
  *p = std::malloc(1);
  blocks[*p] = n;
  used += n;
  ++mallocs;
  return hipSuccess;
}
extern "C" hipError_t hipFree(void* p) {
  auto it = blocks.find(p);
  if (it == blocks.end()) return hipErrorInvalidValue;
  used -= it->second;
  blocks.erase(it);
  std::free(p);
  ++frees;
  return hipSuccess;
}
extern "C" hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
extern "C" hipError_t hipGetLastError() { return hipSuccess; }
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
using namespace mmsb;
int main() {
  const size_t M = 1 << 20;
  void *a, *b, *c;
  capacity = 100 * M;
  // a block given back is kept, and serves the next allocation of about its size
  CHECK(dev_alloc(&a, 40 * M) == hipSuccess && used == 40 * M);
  dev_free(a);
  CHECK(used == 40 * M && dev_cached_bytes() == 40 * M);
  CHECK(dev_alloc(&b, 39 * M) == hipSuccess && b == a && mallocs == 1 && dev_cached_bytes() == 0);
  dev_free(b);
  // either kind of allocation takes the kept memory rather than fail
  CHECK(dev_malloc(&c, 80 * M) == hipSuccess && used == 80 * M && dev_cached_bytes() == 0 && frees == 1);
  CHECK(hipFree(c) == hipSuccess && used == 0);
  CHECK(dev_alloc(&a, 40 * M) == hipSuccess);
  dev_free(a);
  CHECK(dev_alloc(&c, 80 * M) == hipSuccess && used == 80 * M && dev_cached_bytes() == 0);
  // and fails when nothing is left to give
  CHECK(dev_malloc(&b, 40 * M) == hipErrorOutOfMemory && !b);
  CHECK(dev_alloc(&b, 40 * M) == hipErrorOutOfMemory && !b);
  // a block released goes back to the device at once
  dev_release(c);
  CHECK(used == 0 && dev_cached_bytes() == 0);
  dev_release(nullptr);
  dev_free(nullptr);
  // no more than kDevCacheBytes are kept
  capacity = 4 * kDevCacheBytes;
  CHECK(dev_alloc(&a, kDevCacheBytes / 2 + M) == hipSuccess && dev_alloc(&b, kDevCacheBytes / 2 + M) == hipSuccess);
  dev_free(a);
  dev_free(b);
  CHECK(dev_cached_bytes() == kDevCacheBytes / 2 + M && used == dev_cached_bytes());
  release_device_cache();
  CHECK(used == 0 && blocks.empty());
  std::puts("ok");
  return 0;
}
"""


def test_kept_blocks_never_fail_an_allocation(tmp_path):
    src = tmp_path / "driver.cpp"
    src.write_text(DRIVER)
    exe = str(tmp_path / "driver")
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + CSRC, str(src),
                    os.path.join(CSRC, "devmem.cpp"), "-o", exe, "-lpthread"], check=True)
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout


def test_device_memory_comes_from_one_place():
    for path in sorted(glob.glob(os.path.join(CSRC, "*"))):
        if os.path.basename(path) == "devmem.cpp":
            continue
        with open(path) as f:
            code = re.sub(r"//.*|\"[^\"\n]*\"", "", f.read())
        assert not re.search(r"\bhipMalloc\w*\s*\(", code), os.path.basename(path)


@pytest.mark.gpu
def test_sketches_go_back_to_the_device(mmsb):
    """Recomputing contexts release the whitening sketches and V (here about 130 MB) while they live, so nothing of that
    size is left for mmsb_release to give back."""
    import torch
    n, k = 100000, 10
    g = mmsb.generate(n, n, n, n, k, 1.0, 40.0 * k / n, 10.0 / n, seed=3)
    p = mmsb.Pipeline(mmsb.config(nx=n, na=n, nb=n, nc=n, ncom=k, alpha_0=1.0, seed=1, minibatch=1024, y_mode="recompute"))
    p.set_graph(g)
    mmsb.lib.mmsb_release()
    p.whiten()
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    mmsb.lib.mmsb_release()
    assert torch.cuda.mem_get_info()[0] - free0 < (32 << 20)
    p.close()
