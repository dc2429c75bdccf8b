"""The build-time choices of csrc/hdog_internal.hpp (tile height, the region pass's tile group)
within the limits that its comments and static_asserts name.  Compiler only, no GPU."""
import os
import shutil
import subprocess

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                   "cubic-informatics_amd")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="no HIP compiler")


def compile_with(unit, choices, *args):
    return subprocess.run([HIPCC, "-std=c++17", "--offload-arch=gfx950", "--cuda-device-only",
                           "-I../include", "-Icsrc", *choices, *args, f"csrc/{unit}.hip"],
                          cwd=PKG, capture_output=True, text=True)


# labels: bitmaps of more words than threads, LDS of a taller tile; the soft adjoint: rows in
# three tile rows, or in two
@pytest.mark.parametrize("unit,choices", [("ccl", ["-DHDOG_HESS_TY=12"]),
                                          ("ccl", ["-DHDOG_HESS_TY=16", "-DHDOG_ACC_GZ=1"]),
                                          ("soft", ["-DHDOG_HESS_TY=4"]),
                                          ("soft", ["-DHDOG_HESS_TY=12"])])
def test_tile_heights_compile(unit, choices):
    r = compile_with(unit, choices, "-fsyntax-only")
    assert r.returncode == 0, r.stderr[-2000:]
