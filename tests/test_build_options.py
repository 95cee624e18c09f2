"""The build options that the kernel sources offer beside their defaults still compile: eight waves per STGD tile, narrower
Jacobi column blocks."""
import glob
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = glob.glob(os.path.join(ROOT, "*_amd"))[0]
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.parametrize("source,option", [("stgd.hip", "MMSB_STGD_WAVES=8"), ("jacobi.hip", "MMSB_JACOBI_BMAX=4"),
                                           ("jacobi.hip", "MMSB_JACOBI_BMAX=2")])
def test_option_compiles(source, option):
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-std=c++17",
                    "-Wno-everything", "-D" + option, "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(PKG, "csrc"),
                    "-fsyntax-only", os.path.join(PKG, "csrc", source)], check=True)
