"""Sizes where single kernels and dispatch rules of the engine can go wrong: edges of
tiles, remainders, the smallest and largest of a range.  Every comparison is exact
(the outputs are whole numbers)."""
import numpy as np
import pytest

import libsais_amd as la
from libsais_amd import workloads
from tests import oracle_lib as ol

pytestmark = pytest.mark.gpu

H16_TILE = 16384   # symbols a workgroup of the 16-bit histogram counts between flushes


def _freq16(T):
    n = len(T)
    SA, f = np.zeros(n, np.int32), np.zeros(65536, np.int32)
    assert la.libsais16(T, SA, n, 0, f) == 0, la.last_error()
    return SA, f


@pytest.mark.parametrize("n", [2, 65, H16_TILE - 1, H16_TILE, H16_TILE + 1, 2 * H16_TILE + 1, 1024 * H16_TILE + 5])
def test_hist16(n):
    """freq of the 16-bit API: one, several and more tiles than workgroups; both halves
    of a counter word, the extreme symbols, and runs of one symbol a whole tile long."""
    print(f"[hist16] n={n}", flush=True)
    rng = np.random.default_rng(n)
    T = rng.integers(0, 65536, n).astype(np.uint16)
    T[::3] = 65535
    T[1::7] = 0
    SA, f = _freq16(T)
    assert np.array_equal(f, np.bincount(T, minlength=65536))
    if n < 100000:
        rc, ref = ol.sa16(T)
        assert rc == 0 and np.array_equal(SA, ref)
        T[:] = 40001
        SA, f = _freq16(T)
        assert f[40001] == n and f.sum() == n and np.array_equal(SA, np.arange(n)[::-1])


@pytest.mark.parametrize("n", [2, 5, 20001])
@pytest.mark.parametrize("wide", [False, True])
def test_int_value_table(n, wide):
    """Alphabets ranked through a table of the values (largest value below 4 n) and, one
    above, through the sort; both from the first value past 16 bits on."""
    for largest in (65536, 4 * n - 1, 4 * n):
        print(f"[int table] n={n} largest={largest} wide={wide}", flush=True)
        rng = np.random.default_rng(largest)
        T = rng.integers(0, max(2, largest // 3), n).astype(np.int64 if wide else np.int32)
        T[0], T[n // 2] = largest, largest
        ref = ol.sa_int(T)
        SA = np.zeros(n, T.dtype)
        f = la.libsais64_long if wide else la.libsais_int
        assert f(T, SA, n, largest + 1, 0) == 0, la.last_error()
        assert np.array_equal(SA, ref)
