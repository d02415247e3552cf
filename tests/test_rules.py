"""The launch rules shared by the schedule builder and the launchers
(tests/rules_check.cpp against ollipticid_amd/csrc/kernels.hpp)."""
import os
import subprocess

import pytest

from tests.test_layout import HERE, HIPCC


@pytest.mark.skipif(HIPCC is None, reason="hipcc not available")
def test_launch_rules(tmp_path):
    exe = tmp_path / "rules_check"
    subprocess.run([HIPCC, "-O1", "-std=c++17", "-I" + os.path.join(os.path.dirname(HERE), "include"),
                    "-o", str(exe), os.path.join(HERE, "rules_check.cpp")],
                   check=True, capture_output=True, timeout=300)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout
