"""The small-matrix kernel keeps a whole matrix in the registers of one workgroup: up to 128 registers of X a lane beside
the operands of the products.  What does not fit goes through scratch memory, once per iteration, and the point of the kernel is
gone.  This test compiles ns_small.hip for gfx950 and reads the compiler's own account of every instantiation: 32 bytes a
lane (addresses put aside over the iterations, six registers) is what it may use.  Needs hipcc, no GPU."""
import os
import re
import shutil
import subprocess

import pytest

from dion_amd import _build

SRC = os.path.join(_build.CSRC, "ns_small.hip")


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc not on PATH")
def test_no_form_of_the_small_matrix_kernel_keeps_its_matrix_in_scratch_memory(tmp_path):
    cmd = ["hipcc", *[f for f in _build.HIPCC_FLAGS if f != "-fPIC"], "-S", "--cuda-device-only", SRC, "-o",
           str(tmp_path / "ns_small.s"), "-Rpass-analysis=kernel-resource-usage"]
    out = subprocess.run(cmd, check=True, capture_output=True, text=True, timeout=900).stderr
    scratch, name = {}, None
    for line in out.split("\n"):
        m = re.search(r"Function Name: (\S+)", line)
        if m:
            name = m.group(1)
        m = re.search(r"ScratchSize \[bytes/lane\]: (\d+)", line)
        if m:
            scratch[name] = int(m.group(1))
    forms = {k: v for k, v in scratch.items() if "ns_reg_kernel" in k}
    assert len(forms) >= 40, sorted(scratch)
    assert not {k: v for k, v in forms.items() if v > 32}
