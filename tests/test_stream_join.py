"""The order of a dispatcher's launch behind the caller's streams, on a
stand-in runtime: tests/stream_join_check.cpp, built here with the host
compiler."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.mark.skipif(not shutil.which("g++"), reason="no host compiler")
def test_launch_order(tmp_path):
    out = str(tmp_path / "stream_join_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-Wextra", "-I",
                    os.path.join(ROOT, "include"), "-I",
                    os.path.join(ROOT, "powersparse_amd", "host"),
                    os.path.join(HERE, "stream_join_check.cpp"), "-o", out], check=True)
    r = subprocess.run([out], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
