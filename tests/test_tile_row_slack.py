"""The row list of the back projection by image tiles of short images
(stir_amd/csrc/pmrt_tile.hip, bp_tile_short_kernel) ends in tile_row_slack rows
for the copy waves' read-ahead. The furthest row that any lane of any copy wave
asks for, from the same ShortCopyWalk as the kernel's, in tables of one to
three phases of 1 to 700 rows and of every stride, is inside the list. CPU only.
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROBE = r"""
#include <algorithm>
#include <cstdio>
#include <vector>
#include "pmrt_device.hpp"
using namespace mi;

// the furthest row of the list that the copies of a table's phases ask for
static int furthest(const std::vector<int>& rows, int stride) {
  const uint32_t div = static_cast<uint32_t>(((uint64_t{1} << 32) + stride - 1) / stride);
  int far = 0;
  for (int wave = 0; wave < kShortCopyWaves; ++wave)
    for (int lane = 0; lane < 64; ++lane) {
      const ShortCopyWalk walk(wave, lane, stride, div);
      int base = 0;
      for (size_t p = 0; p <= rows.size(); ++p) {  // the last: the phase after the table's last
        const int n = p < rows.size() ? rows[p] * stride : 0;
        int row = walk.row_first, at = walk.at_first;
        for (int first = 0; first == 0 || (wave + kShortCopyWaves * first) * 64 < n; first += kShortBatch)
          for (int j = 0; j < kShortBatch; ++j) {
            const int f = (wave + kShortCopyWaves * (first + j)) * 64 + lane;
            if (row != f / stride || at != f % stride) return -1;
            far = std::max(far, base + row);
            row += walk.row_step;
            row += walk.carry(at);
          }
        if (p < rows.size()) base += rows[p];
      }
    }
  return far;
}

int main() {
  const std::vector<std::vector<int>> tables = {{1}, {2}, {63}, {64, 1}, {700}, {1, 700}, {341, 342, 5}, {512, 511, 1}};
  for (int stride = 2; stride <= 128; ++stride) {
    int over = -(1 << 30);  // rows asked for past the last one
    for (const auto& t : tables) {
      int total = 0;
      for (int r : t) total += r;
      const int far = furthest(t, stride);
      if (far < 0) {
        std::printf("stride %d: a row or place that is not the float's\n", stride);
        return 1;
      }
      over = std::max(over, far + 1 - total);
    }
    std::printf("%d %d %d\n", stride, over, tile_row_slack(stride));
  }
  return 0;
}
"""


def test_copies_of_short_images_stay_inside_the_row_list(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not available")
    src, exe = tmp_path / "reach.cpp", tmp_path / "reach"
    src.write_text(PROBE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", os.path.join(ROOT, "stir_amd", "csrc"), "-I",
                    os.path.join(ROOT, "include"), "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", str(src), "-o",
                    str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[-300:]
    got = {int(s): (int(over), int(slack)) for s, over, slack in (line.split() for line in r.stdout.splitlines())}
    assert sorted(got) == list(range(2, 129))
    assert got[2][0] == 1024  # 2048 floats of two to a row
    for stride, (over, slack) in got.items():
        assert over <= slack, stride
        assert slack >= 512  # the tall images' read-ahead
