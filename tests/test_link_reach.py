"""The extent that bounds the solid test's shortcut (csrc/link_reach.h), compiled
for the host: a level of one box reaches to its far corner or to the triangles;
a level of many boxes as far as its boxes and the triangles, however many nodes
it stores (its flat node count is no length: taken for one, the shortcut would
never answer)."""
import os
import subprocess

import pytest

from conftest import PKG_DIR

SOURCE = r"""
#include <cstdio>
#include "link_reach.h"
int main() {
  const double origin[3] = {1.0, -2.0, 0.5}, gbb[6] = {9.0, 3.0, 4.0, -30.0, 2.0, 1.0};
  const int one[3] = {11, 21, 31}, flat[3] = {12000000, 1, 1};
  const int32_t blo[6] = {4, 4, 4, 20, 4, 8}, bhi[6] = {19, 11, 11, 35, 19, 15};
  printf("%.17g %.17g %.17g %.17g\n", uclbs::link_reach(origin, 0.5, one, 0, nullptr, nullptr, nullptr),
         uclbs::link_reach(origin, 0.5, one, 0, nullptr, nullptr, gbb),
         uclbs::link_reach(origin, 0.5, flat, 2, blo, bhi, nullptr),
         uclbs::link_reach(origin, 0.5, flat, 2, blo, bhi, gbb));
}
"""


def test_reach(tmp_path):
    (tmp_path / "reach.cpp").write_text(SOURCE)
    exe = str(tmp_path / "reach")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(PKG_DIR, "csrc"),
                    str(tmp_path / "reach.cpp"), "-o", exe], check=True)
    got = [float(v) for v in subprocess.run([exe], check=True, capture_output=True, text=True).stdout.split()]
    # one box: x 1..6, y -2..8, z 0.5..15.5; triangles out to 9, -30, 2
    # boxes with shell: x 3..36 -> 2.5..19, y 3..20 -> -0.5..8, z 3..16 -> 2..8.5
    assert got == pytest.approx([6 + 8 + 15.5, 9 + 30 + 15.5, 19 + 8 + 8.5, 19 + 30 + 8.5], abs=1e-12)
