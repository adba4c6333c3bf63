"""The voxelizer's candidate queue entry (octlb_amd/csrc/voxelize_queue.h)
holds every triangle index a call may have, up to 2^31 - 2, beside its list;
compiled for the host."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "octlb_amd" / "csrc"

PROGRAM = r'''
#include "voxelize_queue.h"
#include <cstdio>
#include <initializer_list>
int main() {
  for (int64_t t : {int64_t{0}, int64_t{1}, (int64_t{1} << 30) - 1, int64_t{1} << 30, (int64_t{1} << 31) - 2})
    for (int l = 0; l < 4; ++l) {
      const octlb::VoxEntry e = octlb::MakeVoxEntry(t, l);
      if (octlb::VoxTriangle(e) != t || octlb::VoxList(e) != l) {
        std::printf("triangle %lld list %d came back as %lld, %d\n", static_cast<long long>(t), l,
                    static_cast<long long>(octlb::VoxTriangle(e)), octlb::VoxList(e));
        return 1;
      }
    }
  return 0;
}
'''


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_every_index_round_trips(tmp_path):
    src, exe = tmp_path / "queue.cpp", tmp_path / "queue"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    done = subprocess.run([str(exe)], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout
