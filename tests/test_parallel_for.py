"""ParallelFor (octlb_amd/csrc/parallel_for.h), which builds the adjoint's
tables: every index once whatever the count, what a body throws is thrown in the
caller, and an allocation that fails while its threads are started costs threads,
not the process.  Compiled for the host."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "octlb_amd" / "csrc"

PROGRAM = r'''
#include "parallel_for.h"
#include <cstdio>
#include <cstdlib>
#include <new>
#include <stdexcept>

static std::atomic<long> allocations{0};
static std::atomic<long> fail_at{-1};  // this allocation and all after it fail

void* operator new(std::size_t size) {
  const long at = allocations.fetch_add(1);
  if (fail_at >= 0 && at >= fail_at) throw std::bad_alloc();
  if (void* p = std::malloc(size ? size : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

static std::atomic<int> done[5000];

static bool EveryIndexOnce(int count, int each) {
  for (auto& d : done) d = 0;
  octlb::ParallelFor(count, each, [](int k) { ++done[k]; });
  for (int k = 0; k < 5000; ++k)
    if (done[k] != (k < count ? 1 : 0)) return false;
  return true;
}

int main() {
  for (int count : {0, 1, 2, 3, 15, 16, 17, 31, 32, 33, 256, 1000, 4097})
    for (int each : {1, 2, 16})
      if (!EveryIndexOnce(count, each)) {
        std::printf("count %d each %d\n", count, each);
        return 1;
      }
  for (int bad : {0, 17, 999}) {
    bool thrown = false;
    try {
      octlb::ParallelFor(1000, 1, [&](int k) {
        if (k == bad) throw std::invalid_argument("body");
      });
    } catch (const std::invalid_argument&) {
      thrown = true;
    }
    if (!thrown) {
      std::printf("lost the exception of %d\n", bad);
      return 1;
    }
  }
  for (long k = 0; k < 24; ++k) {
    fail_at = allocations + k;
    const bool good = EveryIndexOnce(4097, 1);
    fail_at = -1;
    if (!good) {
      std::printf("allocation %ld\n", k);
      return 1;
    }
  }
  return 0;
}
'''


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_parallel_for(tmp_path):
    src, exe = tmp_path / "parallel.cpp", tmp_path / "parallel"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread", f"-I{CSRC}", str(src), "-o", str(exe)],
                   check=True)
    done = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0, done.stdout + done.stderr
