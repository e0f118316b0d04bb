"""The ghost-cell rules checked on the CPU: tests/fill_rules_check.hip compiles
fill_value and its adjoint for the host and compares them, for every
combination of boundary codes and for domains from one cell up, with the rules
written out as a recursion and with central differences."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_ghost_rules_of_every_boundary_combination(tmp_path):
    exe = str(tmp_path / "fill_rules_check")
    cmd = [HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-ffp-contract=off", "-Wno-unused-value",
           "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "mesoflow_amd", "csrc"),
           os.path.join(ROOT, "tests", "fill_rules_check.hip"), "-o", exe]
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0 and "PASSED" in r.stdout, r.stdout[-4000:]
