"""Kernels that wait until at most N loads are in flight, where ordinary loads are among the N, hold only while the compiler
leaves those loads between the assembly statements that the source has around them.  A memory clobber keeps them there,
unless the pointer is known to be unaliased: then assembly that was not given it cannot have written what it points to."""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "optimus-lm_amd", "csrc")


@pytest.mark.parametrize("source,kernel,parameter", [("gate_bwd.hip", "gate_wgrad_wide_kernel", 1),      # dlogits
                                                     ("gate_bwd.hip", "gate_dgrad_wide_kernel", 2)])     # base
def test_counted_loads_keep_their_place(source, kernel, parameter, tmp_path):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    out = str(tmp_path / "device.ll")
    subprocess.run([hipcc, "--offload-arch=gfx950", "-O1", "-std=c++17", "--cuda-device-only", "-emit-llvm", "-S", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops", os.path.join(CSRC, source), "-o", out],
                   check=True, capture_output=True)
    found = [l for l in open(out) if l.startswith("define amdgpu_kernel") and kernel in l]
    assert found
    for line in found:
        parameters = re.search(r"\((ptr.*?)\) local_unnamed_addr", line).group(1)
        parameters = re.split(r",(?=\s*(?:ptr|i\d+)\b)", parameters)
        assert parameters[parameter].strip().startswith("ptr") and "noalias" not in parameters[parameter], line
