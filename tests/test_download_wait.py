"""The wait for results on their way to the host (qwanto_amd/csrc/
qwn_download.h, as qwn_runtime.hip uses it), on the CPU: a stream that has
finished without raising the piece's flag is an error, never the window's
earlier contents; a caller's buffer holds what it held until results come."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def test_wait_for_a_piece(tmp_path):
    cxx = shutil.which(os.environ.get("CXX", "g++"))
    if not cxx:
        pytest.skip("no C++ compiler")
    exe = str(tmp_path / "probe")
    subprocess.run([cxx, "-O2", "-std=c++17", "-Wall", "-I" + os.path.join(ROOT, "qwanto_amd", "csrc"),
                    os.path.join(HERE, "download_wait_probe.cpp"), "-o", exe], check=True)
    res = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout
