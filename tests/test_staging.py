"""The pinned-staging pool and its threaded copy on the host
(tests/staging_check.cpp against ollipticid_amd/csrc/staging.cpp)."""
import os
import shutil
import subprocess

import pytest

from tests.test_layout import HERE

ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir(os.path.join(ROCM, "include", "hip")),
                    reason="g++ or the HIP headers not available")
def test_staging_pool_and_copy(tmp_path):
    exe = tmp_path / "staging_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-D__HIP_PLATFORM_AMD__",
                    "-I" + os.path.join(ROCM, "include"), "-o", str(exe),
                    os.path.join(HERE, "staging_check.cpp")],
                   check=True, capture_output=True, timeout=300)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr
