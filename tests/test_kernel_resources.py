"""Registers of kernels whose speed hangs on the waves per SIMD they leave room for (from the
compiler's own report; no GPU): 128 vector registers for four."""
import os
import re
import shutil
import subprocess

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                   "cubic-informatics_amd")


def report(tmp, unit):
    """{mangled kernel name: (vector registers, scratch bytes)} of one source file"""
    r = subprocess.run(["make", "-s", "-C", PKG, f"BUILD={tmp}", f"{tmp}/{unit}.o",
                        "EXTRA_HIPFLAGS=-Rpass-analysis=kernel-resource-usage"],
                       capture_output=True, text=True, check=True)
    out, name = {}, None
    for line in r.stderr.splitlines():
        if m := re.search(r"Function Name: (\S+)", line):
            name = m.group(1)
            out[name] = {}
        elif m := re.search(r" (VGPRs|ScratchSize \[bytes/lane\]): (\d+)", line):
            out[name].setdefault(m.group(1)[0], int(m.group(2)))
    return {n: (v["V"], v["S"]) for n, v in out.items()}


# records-only Hessian, four rows per wave: of the FP32 form, and of FP32 DoG with 16-bit elements
@pytest.mark.skipif(not shutil.which("hipcc") and not os.path.exists("/opt/rocm/bin/hipcc"),
                    reason="no HIP compiler")
def test_records_hessian_leaves_room_for_four_waves(tmp_path):
    kernels = {n: v for n, v in report(tmp_path, "hessian").items()
               if re.search(r"k_hessian_recIf(f|6__half|14__hip_bfloat16)Lb.ELi0ELi4EE", n)}
    assert len(kernels) == 3, sorted(kernels)
    for name, (vgprs, scratch) in kernels.items():
        assert vgprs <= 128 and scratch == 0, (name, vgprs, scratch)
