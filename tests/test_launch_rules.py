"""Host-side rules of the library's launch sequences (no GPU), compiled from the
library's own source (tests/launch_rules_check.hip)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("rules") / "launch_rules_check")
    subprocess.check_call(["/opt/rocm/bin/hipcc", "-O1", "-std=c++17", "--offload-arch=gfx950", "-Xclang",
                           "-target-feature", "-Xclang", "-packed-fp32-ops", "-I" + os.path.join(ROOT, "include"),
                           os.path.join(HERE, "launch_rules_check.hip"),
                           os.path.join(ROOT, "solids4foam_amd", "csrc", "s4f_polymesh.cpp"), "-o", out], timeout=600)
    return out


@pytest.mark.parametrize("rule", ["passRule", "progressWatch", "lduSlots"])
def test_rule(harness, rule):
    r = subprocess.run([harness, rule], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
