"""The threads that copy out of staging slots (fallingsand3d_amd/csrc/copy_job.h) on the
CPU, with and without ThreadSanitizer: bytes, errors, processor time while the device is
busy with something else, and no thread left behind."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("flags", [["-O2"], ["-O1", "-g", "-fsanitize=thread"]], ids=["plain", "tsan"])
def test_copy_job(tmp_path, flags):
    exe = tmp_path / "copy_job_check"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-pthread", *flags, "-o", str(exe),
                    os.path.join(ROOT, "tests", "cpp", "copy_job_check.cpp")], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "copy job checks passed" in r.stdout, r.stdout + r.stderr
