"""The copy pool's jobs and parts (libsais_amd/csrc/copy_pool.h) on the CPU, under sanitizers.

tests/pool_check.cpp includes the pool and the shapes of the staged copies, so that what no
entry point shows can be checked: the room of a job against the parts that each form of a
copy grants, a grant that does not fit, callers with different thread counts at once, the threads that may
work on a job, and a copy for which there is no memory.
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CXX = shutil.which("g++")

pytestmark = pytest.mark.skipif(CXX is None, reason="no host C++ compiler")


@pytest.fixture(scope="module", params=["address", "thread"])
def program(request, tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("pool") / ("pool_" + request.param))
    subprocess.run([CXX, "-std=c++17", "-O2", "-g", "-Wall", "-Werror",
                    "-Wno-mismatched-new-delete", "-fsanitize=" + request.param,
                    os.path.join(ROOT, "tests", "pool_check.cpp"), "-o", exe, "-pthread"], check=True, timeout=300)
    return exe


def _run(program, check):
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0", TSAN_OPTIONS="halt_on_error=1")
    r = subprocess.run([program, check], env=env, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout[-2000:] + r.stderr[-4000:]


@pytest.mark.parametrize("check", ["forms", "refused", "counts", "limits", "no_memory"])
def test_parts(program, check):
    _run(program, check)
