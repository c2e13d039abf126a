"""The search that places an entry's DoFs among a leaf's sorted columns
(find_sorted in pbfmm_impl.h, which the device code uses too) finds every
column and says where there is none, so that a malformed plan is refused."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pi-bem_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include "pbfmm_impl.h"
using pbfmm::find_sorted;
int main() {
  int bad = 0;
  for (int n = 0; n <= 40; ++n) {
    // columns 3, 5, 7, ... between guards that hold looked-for values
    std::vector<int32_t> v(n + 4, -7);
    v[0] = v[1] = 4, v[n + 2] = v[n + 3] = 2 * n + 3;
    for (int i = 0; i < n; ++i) v[2 + i] = 2 * i + 3;
    for (int d = 0; d <= 2 * n + 6; ++d) {
      const int at = find_sorted(v.data(), 2, 2 + n, d);
      const bool is = d >= 3 && d % 2 == 1 && d < 2 * n + 3;
      if (at != (is ? 2 + (d - 3) / 2 : -1)) ++bad, std::printf("n %d d %d at %d\n", n, d, at);
    }
  }
  return bad != 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_find_sorted(tmp_path):
    src, exe = tmp_path / "find.cpp", tmp_path / "find"
    src.write_text(PROGRAM)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, "-I", os.path.join(rocm, "include"),
                    "-D__HIP_PLATFORM_AMD__", "-o", str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
