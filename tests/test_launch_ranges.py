"""ForLaunches (octlb_amd/csrc/launch.h) covers its workgroups in order by
launches of fewer than 2^32 threads each; compiled for the host."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "octlb_amd" / "csrc"

PROGRAM = r'''
#include "launch.h"
#include <cstdio>
int main() {
  for (int threads : {64, 256, 512, 1024})
    for (int64_t groups : {int64_t{0}, int64_t{1}, octlb::kMaxLaunchThreads / threads,
                           octlb::kMaxLaunchThreads / threads + 1, int64_t{3} << 32}) {
      int64_t at = 0;
      int launches = 0;
      octlb::ForLaunches(groups, threads, [&](int64_t first, int64_t count) {
        if (first != at || count <= 0 || count * threads >= (int64_t{1} << 32)) launches += 1000000;
        at = first + count;
        ++launches;
      });
      const int64_t most = octlb::kMaxLaunchThreads / threads;
      if (at != groups || launches != (groups + most - 1) / most) {
        std::printf("threads %d groups %lld: %d launches up to %lld\n", threads, static_cast<long long>(groups),
                    launches, static_cast<long long>(at));
        return 1;
      }
    }
  return 0;
}
'''


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_ranges(tmp_path):
    src, exe = tmp_path / "ranges.cpp", tmp_path / "ranges"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    done = subprocess.run([str(exe)], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout
