"""launch_p2p refuses arguments whose kernel would not write the output they
name.  A host program calls it with no device memory behind them: the refusal
comes before any launch."""
import os
import subprocess

import pytest

from bbfmmongpu_amd import _build

PROGRAM = r"""
#include "kernels.h"
#include <cstdio>
using namespace bb;
int main()
{
  static real out[1];
  static int ints[1];
  static real4 pos[1];
  static int2 seg[1];
  static float qt[1];
  P2PArgs a{};
  a.N = a.nleaf = 1;
  a.nrhs = 1;
  a.out = out;
  a.perm = ints;
  a.leafof = ints;  // a lane per target particle
  printf("%d", launch_p2p(a, nullptr));
  a.leafof = nullptr;
  a.nrhs = 17;  // 16 vectors on the matrix unit, then one
  a.use_mfma = 1;
  a.qt = qt;
  a.ppos = pos;
  a.seg = seg;
  printf(" %d\n", sizeof(real) == 4 ? launch_p2p(a, nullptr) : BBFMM_E_ARG);
  printf("%d\n", BBFMM_E_ARG);
}
"""


@pytest.mark.parametrize("prec", ["s", "d"])
def test_near_field_output_is_written_or_refused(prec, tmp_path):
    src, exe = tmp_path / "p.hip", tmp_path / "p"
    src.write_text(PROGRAM)
    lib = _build.lib_path(prec)
    if not os.path.exists(lib):
        pytest.skip("libraries not built")
    cmd = [_build.HIPCC, "-x", "hip", "--cuda-host-only", "-std=c++17", "-w", "-I", os.path.join(_build.ROOT, "include"), "-I",
           _build.CSRC, *(["-DSINGLE"] if prec == "s" else []), str(src), "-x", "none", lib,
           f"-Wl,-rpath,{os.path.dirname(lib)}", "-o", str(exe)]
    subprocess.run(cmd, check=True, capture_output=True, text=True)
    got = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=60).stdout.split()
    assert got[:2] == [got[2]] * 2
