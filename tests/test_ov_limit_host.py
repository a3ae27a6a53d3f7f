"""The overlaps' row chunks under a fixed partial-sum buffer (host only: the
geometry header compiled with g++ into tests/cpp/ov_limit_check.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_capped_chunks(tmp_path):
    exe = str(tmp_path / "ov_limit_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-o", exe, os.path.join(HERE, "cpp", "ov_limit_check.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    assert ", 0 wrong" in r.stdout
