"""Matrix construction under the sanitizers: the host library's sources on a
stand-in runtime (tests/host_build_check.cpp), repeated builds from several
threads."""
import os
import re
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
PKG = os.path.join(ROOT, "powersparse_amd")

pytestmark = pytest.mark.skipif(not shutil.which("g++"), reason="no host compiler")

# OpenMP's barriers are invisible to the thread sanitizer: that build runs the
# sort and the copies of each thread without a team
BUILDS = {"address": ["-fsanitize=address,undefined", "-fopenmp"], "thread": ["-fsanitize=thread"]}


@pytest.fixture(scope="module", params=sorted(BUILDS))
def program(request, tmp_path_factory):
    d = str(tmp_path_factory.mktemp("host"))
    flags = ["-std=c++17", "-O1", "-g", "-pthread", "-Wno-unknown-pragmas", "-I",
             os.path.join(ROOT, "include"), "-I", os.path.join(PKG, "host"), "-I",
             os.path.join(PKG, "csrc")] + BUILDS[request.param]
    objs, jobs = [], []
    for src in (os.path.join(PKG, "host", "matrix_utils.cpp"),
                os.path.join(PKG, "host", "staged_upload.cpp"),
                os.path.join(HERE, "host_build_check.cpp")):
        objs.append(os.path.join(d, os.path.basename(src)[:-4] + ".o"))
        jobs.append(subprocess.Popen(["g++"] + flags + ["-c", src, "-o", objs[-1]]))
    assert all(j.wait() == 0 for j in jobs)
    # the stages whose results the host does not read: empty functions
    names = [subprocess.run(["nm"] + opt + objs, check=True, capture_output=True, text=True).stdout
             for opt in (["-u"], ["--defined-only"])]
    need, have = (set(re.findall(r"\b(ps_[a-z0-9_]+)$", n, re.M)) for n in names)
    stub = os.path.join(d, "stages.c")
    with open(stub, "w") as f:
        f.writelines(f"unsigned long {n}(void) {{ return 0; }}\n" for n in sorted(need - have))
    out = os.path.join(d, "host_build_check")
    subprocess.run(["gcc", "-c", stub, "-o", stub + ".o"], check=True)
    subprocess.run(["g++"] + flags + objs + [stub + ".o", "-o", out], check=True)
    return request.param, out


@pytest.mark.parametrize("blocks", ["pool", "direct"])
@pytest.mark.parametrize("size,threads,rounds", [("small", 3, 6), ("large", 1, 2)])
def test_repeated_builds(program, blocks, size, threads, rounds):
    kind, out = program
    if size == "large" and (kind == "thread" or blocks == "direct"):
        pytest.skip("one large run is enough")
    r = subprocess.run([out, blocks, str(threads), str(rounds), size], capture_output=True,
                       text=True, timeout=300)
    print(r.stdout, r.stderr[-3000:])
    assert r.returncode == 0, r.stdout + r.stderr[-3000:]
