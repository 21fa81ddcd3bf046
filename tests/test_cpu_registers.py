"""What the compiler reports of kernels that hold their data in registers."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "slepc_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_slot_kernels_do_not_spill(tmp_path):
    """The Gram-Schmidt slots (sa_gw.hip) keep a chunk of the basis in registers
    while the next is loaded; with scratch memory instead they take twice the
    time.  No instantiation uses any."""
    r = subprocess.run([HIPCC, "-O3", "-std=c++17", "-fPIC", "--offload-arch=gfx950", "-Xclang", "-target-feature",
                        "-Xclang", "-packed-fp32-ops", "--cuda-device-only", "-Rpass-analysis=kernel-resource-usage",
                        "-c", os.path.join(CSRC, "sa_gw.hip"), "-o", str(tmp_path / "gw.o")],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    names = re.findall(r"remark:.*Function Name: (\S+)", r.stderr)
    scratch = [int(x) for x in re.findall(r"remark:.*ScratchSize \[bytes/lane\]: (\d+)", r.stderr)]
    assert len(names) == len(scratch) >= 24
    assert not [n for n, b in zip(names, scratch) if b]
