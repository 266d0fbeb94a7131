"""Host arrays of 16 MiB and more travel through pinned slices, unless the runtime knows their memory (pinned,
managed): that it copies by itself, at the link's full rate.  Checked on the CPU against a host stand-in of the
runtime calls, up and down, with arrays of each kind, of two kinds in one call, without slices, and with every host
allocation failing."""
import os
import shutil
import subprocess

import pytest

TESTS = os.path.dirname(os.path.abspath(__file__))
CXX = shutil.which("g++")


@pytest.mark.skipif(CXX is None, reason="needs g++")
def test_routes(tmp_path):
    exe = str(tmp_path / "transfer_check")
    subprocess.run([CXX, "-O2", "-std=c++17", "-pthread", "-I", os.path.join(TESTS, "host_hip"),
                    os.path.join(TESTS, "transfer_check.cpp"), "-o", exe], check=True, capture_output=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.count("ok ") == 32
