"""The general z pass runs in place over columns dealt to workgroups: on the CPU,
every column has exactly one live lane, that lane's component is the column's,
and no lane, live or not, reads a column of another workgroup."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "voxel-lmfem_amd" / "csrc"
PROGRAM = r"""
#include <cstdio>
#include <vector>
#define __host__
#define __device__
#include "vxl_zlanes.h"
using namespace vxl;
int main() {
  long bad = 0;
  for (int P : {4, 8, 16, 32, 64})
    for (int cols = 3; cols <= 400; cols += 3) {
      const int units = z_units(P);
      std::vector<int> lanes(cols, 0);
      for (int b = 0; b * units < cols; ++b)
        for (int p = 0; p < P; ++p) {
          const ZLane l = z_lane(P, p, b, cols);
          bad += l.col < b * units || l.col >= (b + 1) * units || l.col >= cols;
          if (l.live) {
            ++lanes[l.col];
            bad += l.comp != l.col % 3;
          }
        }
      for (int n : lanes) bad += n != 1;
    }
  std::printf("%ld\n", bad);
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_lanes_stay_in_their_workgroup(tmp_path):
    (tmp_path / "lanes.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", str(CSRC), "-o", str(tmp_path / "lanes"), str(tmp_path / "lanes.cpp")],
                   check=True)
    out = subprocess.run([str(tmp_path / "lanes")], check=True, capture_output=True, text=True).stdout
    assert out.strip() == "0"
