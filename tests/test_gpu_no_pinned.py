"""Calls of a process that gets no large block of pinned memory.

Short texts then take the general engine, which needs no block of its own, and copies go
directly.  The calls run in a child process, in which tests/no_pinned_shim.c stands before
the HIP runtime and refuses pinned blocks of 700,000 bytes and more.
"""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CC = shutil.which("gcc")

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(CC is None, reason="no C compiler")]

CHILD = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import numpy as np
import libsais_amd as la
from libsais_amd import serving
from tests import oracle_lib as ol
from tests.test_gpu_parity import fused
refused = ctypes.c_int.in_dll(shim, "no_pinned_refused")
for n in (2, 4001, 24576, 1200007):
    rng = np.random.default_rng(n)
    T = rng.integers(97, 101, n).astype(np.uint8)
    rc, SA = ol.sa(T)
    U, p = ol.bwt(T, SA)
    P = ol.plcp(T, SA)
    A, B, V = np.zeros(n, np.int32), np.zeros(n, np.int32), np.zeros(n, np.uint8)
    A64, f = np.zeros(n, np.int64), np.zeros(256, np.int32)
    assert la.libsais(T, A, n, 0, f) == 0 and np.array_equal(A, SA), la.last_error()
    assert np.array_equal(f, np.bincount(T, minlength=256))
    assert la.libsais64(T, A64, n, 0, None) == 0 and np.array_equal(A64, SA), la.last_error()
    assert la.libsais_bwt(T, V, B, n, 0, None) == p and np.array_equal(V, U), la.last_error()
    I = np.zeros((n - 1) // 2 + 1, np.int32)
    assert la.libsais_bwt_aux(T, V, B, n, 0, None, 2, I) == 0 and np.array_equal(V, U), la.last_error()
    assert I[0] == p
    assert la.libsais_plcp(T, SA, B, n) == 0 and np.array_equal(B, P), la.last_error()
    gSA, gU, gp, gP, gL, _ = fused(T)
    assert np.array_equal(gSA, SA) and np.array_equal(gU, U) and gp == p and np.array_equal(gP, P)
    for kind in (serving.JOB_SA, serving.JOB_BWT, serving.JOB_LCP):
        r = serving.Request(T, kind)
        assert serving.run_alone(r) == 0 and np.array_equal(r.SA[:n], SA), la.last_error()
        assert kind != serving.JOB_BWT or r.job.primary == p
    print("n", n, "refused", refused.value, flush=True)
assert refused.value > 0
print("ok")
"""


def test_short_texts_without_pinned_memory(tmp_path):
    shim = str(tmp_path / "no_pinned_shim.so")
    subprocess.run([CC, "-O1", "-fPIC", "-shared", "-Wall", "-Werror", os.path.join(ROOT, "tests", "no_pinned_shim.c"),
                    "-o", shim, "-ldl"], check=True, timeout=100)
    print("[no pinned] child process", flush=True)
    env = dict(os.environ, NO_PINNED_FROM="700000")
    r = subprocess.run([sys.executable, "-c", CHILD, shim], cwd=ROOT, env=env, capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout[-2000:] + r.stderr[-3000:]
