"""Staged copies of several calls at once, beside which a download takes its shared form.

Each thread makes calls with 32- and 64-bit index arrays of its own and checks every output
against the oracle.
"""
import threading

import numpy as np
import pytest

import libsais_amd as la
from libsais_amd import workloads
from tests import oracle_lib as ol

pytestmark = pytest.mark.gpu

THREADS = 6


def _set(mode, threads):
    lib = la.load()
    assert lib.sagpu_set_option(b"host_staging", mode) == 0
    assert lib.sagpu_set_option(b"copy_threads", threads) == 0


@pytest.fixture
def reset_staging():
    yield
    _set(1, 0)


def _texts(n):
    out = []
    for k in range(THREADS):
        T = workloads.dna_like(n + 211 * k, seed=300 + k)
        rc, SA = ol.sa(T)
        assert rc == 0
        P = ol.plcp(T, SA)
        out.append((T, SA, P, ol.lcp(P, SA)))
    return out


def _calls(T, SA, P, L):
    """What differs from the oracle, if anything does."""
    n = len(T)
    for t, sa, plcp, lcp in ((np.int32, la.libsais, la.libsais_plcp, la.libsais_lcp),
                             (np.int64, la.libsais64, la.libsais64_plcp, la.libsais64_lcp)):
        A, B, C = (np.full(n, -1, t) for _ in range(3))
        if sa(T, A, n, 0, None) != 0 or not np.array_equal(A, SA):
            return sa.__name__
        if plcp(T, A, B, n) != 0 or not np.array_equal(B, P):
            return plcp.__name__
        if lcp(B, A, C, n) != 0 or not np.array_equal(C, L):
            return lcp.__name__
    return None


def _at_once(texts, rounds):
    wrong = []

    def work(k):
        try:
            for _ in range(rounds):
                w = _calls(*texts[k])
                if w:
                    wrong.append((k, w, la.last_error()))
        except Exception as e:  # pragma: no cover - reported below
            wrong.append((k, repr(e)))

    ts = [threading.Thread(target=work, args=(k,)) for k in range(THREADS)]
    for t in ts:
        t.start()
    for t in ts:
        t.join(100)
    assert not any(t.is_alive() for t in ts) and wrong == []


@pytest.mark.parametrize("mode,threads", [(2, 0), (2, 1), (2, 3), (1, 1)])
@pytest.mark.parametrize("n", [100_003, 300_007])
def test_calls_at_once(n, mode, threads, reset_staging):
    """Every copy in 64 KiB chunks (mode 2), and the 64-bit arrays' copies of the default
    mode, which start at 2^18 entries."""
    print(f"[copies] n={n} host_staging={mode} copy_threads={threads}", flush=True)
    texts = _texts(n)
    _set(mode, threads)
    _at_once(texts, 2)


def test_form_settled_at_the_start(reset_staging):
    """host_staging and copy_threads change while copies run: each copy keeps the form that
    it started with."""
    print("[copies] options changed under the calls", flush=True)
    texts = _texts(300_007)
    stop = threading.Event()

    def change():
        k = 0
        while not stop.is_set():
            _set((1, 2, 2, 0)[k % 4], (0, 1, 3)[k % 3])
            k += 1
            stop.wait(0.0005)

    t = threading.Thread(target=change)
    t.start()
    try:
        _at_once(texts, 2)
    finally:
        stop.set()
        t.join(30)


@pytest.mark.parametrize("n", [(10 << 20) - 1, 10 << 20, (16 << 20) + 1, (40 << 20) + 4099])
def test_large_arrays(n, reset_staging):
    """32-bit arrays on both sides of 40 MiB, from where copies take a larger ring: uploads
    that wrap in it, downloads by DMA slot, and smaller and converted copies between them,
    on one context and after another that never grew."""
    print(f"[copies] large arrays, n={n}", flush=True)
    rng = np.random.default_rng(n)
    SA = rng.integers(0, n, n, dtype=np.int32)
    P = rng.integers(0, 1 << 30, n, dtype=np.int32)
    ref = P[SA]
    m = 3_000_001
    sa64, p64 = rng.integers(0, m, m), rng.integers(0, 1 << 30, m)
    for _ in range(2):
        L = np.full(n, -1, np.int32)
        assert la.libsais_lcp(P, SA, L, n) == 0 and np.array_equal(L, ref), la.last_error()
        L64 = np.full(m, -1, np.int64)
        assert la.libsais64_lcp(p64, sa64, L64, m) == 0 and np.array_equal(L64, p64[sa64])
        A = SA.copy()
        assert la.libsais_lcp(P, A, A, n) == 0 and np.array_equal(A, ref)   # over its input
        k = m // 2
        L = np.full(k, -1, np.int32)
        small = SA[:k] % k
        assert la.libsais_lcp(P[:k].copy(), small, L, k) == 0 and np.array_equal(L, P[:k][small])


@pytest.mark.parametrize("n,callers", [((2 << 20) - 1, 4), (2 << 20, 4), ((5 << 20) + 3, 4), ((12 << 20) + 1, 4),
                                       ((8 << 20) - 9, 2), (8 << 20, 2), ((12 << 20) + 1, 2)])
def test_large_arrays_at_once(n, callers, reset_staging):
    """Callers with 32- and 64-bit arrays on both sides of 8 MiB, from where copies beside other
    calls take the larger ring, and of several slots and chunks; two of them on both sides of
    32 MiB, from where their downloads take the kernel instead of DMAs."""
    print(f"[copies] large arrays at once, n={n}, callers={callers}", flush=True)
    wrong = []

    def work(k):
        try:
            rng = np.random.default_rng(n + k)
            m = n + 7 * k
            SA = rng.integers(0, m, m, dtype=np.int32)
            P = rng.integers(0, 1 << 30, m, dtype=np.int32)
            ref = P[SA]
            for t, lcp in ((np.int32, la.libsais_lcp), (np.int64, la.libsais64_lcp)):
                A, B = SA.astype(t), P.astype(t)
                for _ in range(2):
                    L = np.full(m, -1, t)
                    if lcp(B, A, L, m) != 0 or not np.array_equal(L, ref):
                        wrong.append((k, lcp.__name__, la.last_error()))
        except Exception as e:  # pragma: no cover - reported below
            wrong.append((k, repr(e)))

    ts = [threading.Thread(target=work, args=(k,)) for k in range(callers)]
    for t in ts:
        t.start()
    for t in ts:
        t.join(100)
    assert not any(t.is_alive() for t in ts) and wrong == []
