"""The kept-block pool behind ps_malloc / ps_free, on a stand-in driver:
tests/block_pool_check.cpp, built here with the host compiler."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "powersparse_amd", "csrc")

pytestmark = pytest.mark.skipif(not shutil.which("g++"), reason="no host compiler")


CHECKS = ["huge", "double_free", "freed_elsewhere", "idle", "idle_reuse", "refused", "trim_to",
          "threads"]


@pytest.fixture(scope="module", params=["address", "thread"])
def program(request, tmp_path_factory):
    out = str(tmp_path_factory.mktemp("pool") / "block_pool_check")
    build = ["g++", "-std=c++17", "-O1", "-g", "-Wall", "-Wextra", "-pthread", "-I", CSRC,
             os.path.join(HERE, "block_pool_check.cpp"), "-o", out]
    build.insert(1, "-fsanitize=" + request.param)
    subprocess.run(build, check=True)
    return out


@pytest.mark.parametrize("check", CHECKS)
def test_pool(program, check):
    r = subprocess.run([program, check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
