"""Sizes where single kernels and dispatch rules of the engine can go wrong: edges of
tiles, remainders, the smallest and largest of a range.  Every comparison is exact
(the outputs are whole numbers)."""
import numpy as np
import pytest

import libsais_amd as la
from libsais_amd import batch, workloads
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


@pytest.mark.parametrize("n", [2, 3, 15, 16, 17, 31, 32, 33, 47, 49, 255, 256, 257, 4095, 4096, 4097, 65537])
def test_unbwt_edges(n):
    """Inverse BWT around the sample spacing, the words a walk keeps, powers of two (the
    width of the position hash) and the decode table; every text form whose walks
    run differently (one symbol, two, all 256, 16-bit symbols), plain and with samples
    closer than an output word."""
    rng = np.random.default_rng(n)
    for name, T in (("one", np.full(n, 7, np.uint8)), ("two", rng.integers(0, 2, n).astype(np.uint8) * 255),
                    ("bytes", rng.integers(0, 256, n).astype(np.uint8)), ("period", np.arange(n, dtype=np.uint8) % 5)):
        print(f"[unbwt] n={n} {name}", flush=True)
        rc, SA = ol.sa(T)
        U, p = ol.bwt(T, SA)
        out, A = np.zeros(n, np.uint8), np.zeros(n + 1, np.int32)
        assert la.libsais_unbwt(U, out, A, n, None, p) == 0, la.last_error()
        assert np.array_equal(out, T), name
        for r in (2, 4, 16):
            U, I = ol.bwt_aux(T, SA, r)
            out[:] = 9
            assert la.libsais_unbwt_aux(U, out, A, n, None, r, I.astype(np.int32)) == 0, la.last_error()
            assert np.array_equal(out, T), (name, r)
    T = rng.integers(0, 65536, n).astype(np.uint16)
    rc, SA = ol.sa16(T)
    U, p = ol.bwt16(T, SA)
    out, A = np.zeros(n, np.uint16), np.zeros(n + 1, np.int32)
    assert la.libsais16_unbwt(U, out, A, n, None, p) == 0, la.last_error()
    assert np.array_equal(out, T)


@pytest.mark.parametrize("n,r", [(1 << 22, 0), ((1 << 22) + 1, 0), ((1 << 24) - 1, 0), ((1 << 24) + 3, 0),
                                 (100003, 2), ((1 << 22) + 5, 64), ((1 << 22) + 5, 2048)])
def test_unbwt_spacing(n, r):
    """The sizes where the sample spacing changes, and both decoders of auxiliary samples
    (many chunks of odd total length; few)."""
    print(f"[unbwt] n={n} r={r}", flush=True)
    T = workloads.dna_like(n, seed=n)
    U, out, A = np.zeros(n, np.uint8), np.zeros(n, np.uint8), np.zeros(n + 1, np.int32)
    if r:
        I = np.zeros((n - 1) // r + 1, np.int32)
        assert la.libsais_bwt_aux(T, U, A, n, 0, None, r, I) == 0, la.last_error()
        assert la.libsais_unbwt_aux(U, out, A, n, None, r, I) == 0, la.last_error()
    else:
        p = la.libsais_bwt(T, U, A, n, 0, None)
        assert p > 0
        assert la.libsais_unbwt(U, out, A, n, None, p) == 0, la.last_error()
    assert np.array_equal(out, T)


def test_unbwt_short_of_memory():
    """Under a falling memory cap the walks get less room (shorter chunks, pages that run
    out, gaps walked twice): the call returns the text or -2, nothing else."""
    n = 65537
    T = workloads.dna_like(n, seed=5)
    rc, SA = ol.sa(T)
    U, p = ol.bwt(T, SA)
    lib = la.load()
    out, A = np.zeros(n, np.uint8), np.zeros(n + 1, np.int32)

    def capped(limit):
        lib.sagpu_set_memory_limit(limit)
        out[:] = 0
        rc = la.libsais_unbwt(U, out, A, n, None, p)
        assert rc in (0, -2), rc
        assert rc == -2 or np.array_equal(out, T), limit
        return rc == 0

    try:
        low, high = 1, 1 << 36   # the context keeps scratch of earlier calls: look for the least cap
        while high - low > (16 << 10):
            mid = (low + high) // 2
            low, high = (low, mid) if capped(mid) else (mid, high)
        for step in range(64):
            capped(low + (step << 14))
    finally:
        lib.sagpu_set_memory_limit(0)
    assert la.libsais_unbwt(U, out, A, n, None, p) == 0 and np.array_equal(out, T)


SMALL_MAX = 24 * 1024   # the longest text one workgroup builds


def _small_texts(n, rng):
    yield "one", np.full(n, 65, np.uint8)
    yield "two", rng.integers(0, 2, n).astype(np.uint8)
    yield "bytes", rng.integers(0, 256, n).astype(np.uint8)
    yield "acgt", workloads.iid(n, seed=n, alphabet=b"ACGT")
    yield "period", workloads.periodic(n, 17, 3)
    yield "fibonacci", workloads.fibonacci(n)
    copies = np.tile(workloads.iid(max(2, n // 3), seed=n, alphabet=b"abcdefghijklmnopqrstuvwxyz"), 4)[:n].copy()
    yield "copies", copies
    runs = copies.copy()
    runs[n // 4: n // 4 + 300] = 97   # one group on either side of what is ranked by counting
    runs[n // 2: n // 2 + 90] = 97
    yield "runs", runs


@pytest.mark.parametrize("n", [2, 3, 17, 63, 64, 65, 1023, 1024, 1025, 2049, 4096, 4097, 8192, 8193, 16384, 16385,
                               SMALL_MAX - 1, SMALL_MAX, SMALL_MAX + 1])
def test_small_build(n):
    """Texts built by one workgroup, at the edges of its rows and of its range, and the
    first size past it: every output of the device and the host entry points (both
    index widths) against the oracle, and the general engine on the same text."""
    from tests.test_gpu_parity import fused
    lib = la.load()
    rng = np.random.default_rng(n)
    for name, T in _small_texts(n, rng):
        print(f"[small] n={n} {name}", flush=True)
        rc, SA = ol.sa(T)
        U, p = ol.bwt(T, SA)
        P = ol.plcp(T, SA)
        L, f = ol.lcp(P, SA), ol.freq(T)
        for small in (1, 0):
            assert lib.sagpu_set_option(b"small_build", small) == 0
            try:
                gSA, gU, gp, gP, gL, gf = fused(T)
            finally:
                assert lib.sagpu_set_option(b"small_build", 1) == 0
            assert np.array_equal(gSA, SA), (name, small)
            assert gp == p and np.array_equal(gU, U), (name, small)
            assert np.array_equal(gP, P) and np.array_equal(gL, L) and np.array_equal(gf, f), (name, small)
        for dt, sa, bwt, plcp, aux in ((np.int32, la.libsais, la.libsais_bwt, la.libsais_plcp, la.libsais_bwt_aux),
                                       (np.int64, la.libsais64, la.libsais64_bwt, la.libsais64_plcp,
                                        la.libsais64_bwt_aux)):
            out, fr, hU, A = np.zeros(n, dt), np.zeros(256, dt), T.copy(), np.zeros(n, dt)
            assert sa(T, out, n, 0, fr) == 0 and np.array_equal(out, SA) and np.array_equal(fr, f), name
            assert bwt(hU, hU, A, n, 0, fr) == p and np.array_equal(hU, U) and np.array_equal(fr, f), name
            out[:] = 0
            assert plcp(T, np.ascontiguousarray(SA, dt), out, n) == 0 and np.array_equal(out, P), name
            for r in (2, 64, 1 << 30):
                I = np.zeros((n - 1) // r + 1, dt)
                rU, rI = ol.bwt_aux(T, SA, r)
                assert aux(T, hU, A, n, 0, None, r, I) == 0 and np.array_equal(hU, rU), (name, r)
                assert np.array_equal(I, rI), (name, r)


@pytest.mark.parametrize("n", [2, 65, 1025, 4097, 16385, SMALL_MAX, SMALL_MAX + 1])
def test_small_gsa(n):
    """String sets built by one workgroup: SA, PLCP and LCP against the oracle; invalid
    sets refused."""
    from tests.test_gpu_parity import fused
    rng = np.random.default_rng(n)
    unit = rng.integers(1, 4, 200).astype(np.uint8)
    for name, every in (("single", 0), ("many", 23), ("alike", 201)):
        T = np.tile(unit, n // 200 + 1)[:n].copy() if every == 201 else rng.integers(1, 5, n).astype(np.uint8)
        if every:
            T[every - 1::every] = 0
        if n > 1:
            T[-2:] = (1, 0)
        print(f"[small gsa] n={n} {name}", flush=True)
        rc, SA = ol.sa(T, gsa=True)
        assert rc == 0
        P = ol.plcp(T, SA, gsa=True)
        gSA, _, _, gP, gL, _ = fused(T, gsa=True)
        assert np.array_equal(gSA, SA) and np.array_equal(gP, P) and np.array_equal(gL, ol.lcp(P, SA)), name
        out = np.zeros(n, np.int32)
        assert la.libsais_gsa(T, out, n, 0, None) == 0 and np.array_equal(out, SA)
        assert la.libsais_plcp_gsa(T, out, out, n) == 0 and np.array_equal(out, P)
        bad = T.copy()
        bad[0] = 0
        assert la.libsais_gsa(bad, out, n, 0, None) == -1
        if n > 64:
            bad = T.copy()
            bad[30:32] = 0
            assert la.libsais_gsa(bad, out, n, 0, None) == -1


def _chain_texts(n, rng):
    """Repeats whose groups continue into one another: two and nine copies (the most a
    chain takes is eight), copies up to the text's last symbol, and copies that change
    how many they are along the way."""
    base = rng.integers(97, 101, n).astype(np.uint8)
    two = base.copy()
    two[n // 2 + 7:] = two[:n - n // 2 - 7]
    yield "two, to the end", two
    mixed = base.copy()
    k = n // 16
    for c, size in ((3, k), (6, k - 1), (9, k // 2), (12, k // 3), (14, 2 * k)):
        mixed[c * k:c * k + size] = mixed[:size]
    yield "two to six", mixed
    yield "eight", np.tile(base[:n // 8], 9)[:n].copy()
    nine = np.tile(base[:n // 10], 10)[:n].copy()
    nine[n // 10 * 9:] = base[n // 10 * 9:][:len(nine) - n // 10 * 9]
    yield "nine", nine


@pytest.mark.parametrize("n", [40, 1000, 4097, 65535 * 2 + 3, 300007])
def test_round_chains(n):
    """Groups compared at the end of their chains (from lists of 2 entries on, and never),
    over words, tiles and the text's last positions: plain texts and string sets, with
    codes and marks, against the oracle."""
    from tests.test_gpu_parity import fused
    lib = la.load()
    rng = np.random.default_rng(n)
    for name, T in _chain_texts(n, rng):
        for gsa in (False, True):
            if gsa:
                T = T.copy()
                T[n // 5::n // 3 + 1] = 0
                T[-2:] = (98, 0)
            rc, SA = ol.sa(T, gsa=gsa)
            assert rc == 0
            P = ol.plcp(T, SA, gsa=gsa)
            L = ol.lcp(P, SA)
            for least in (2, 0):
                assert lib.sagpu_set_option(b"chain_min", least) == 0
                try:
                    gSA, gU, gp, gP, gL, _ = fused(T, gsa=gsa)
                    print(f"[chains] n={n} {name} gsa={gsa} from {least}: {la.stats().rounds} rounds", flush=True)
                finally:
                    assert lib.sagpu_set_option(b"chain_min", 4096) == 0
                assert np.array_equal(gSA, SA) and np.array_equal(gP, P) and np.array_equal(gL, L), (name, least)
                if not gsa:
                    U, p = ol.bwt(T, SA)
                    assert gp == p and np.array_equal(gU, U), (name, least)
    S = rng.integers(0, 40000, n).astype(np.uint16)
    S[n // 2:] = S[:n - n // 2]
    rc, SA = ol.sa16(S)
    assert rc == 0
    for least in (2, 0):
        assert lib.sagpu_set_option(b"chain_min", least) == 0
        try:
            out = np.zeros(n, np.int32)
            assert la.libsais16(S, out, n, 0, None) == 0 and np.array_equal(out, SA), least
        finally:
            assert lib.sagpu_set_option(b"chain_min", 4096) == 0


@pytest.mark.parametrize("n", [(1 << 28) - 1, (1 << 28) + 1, (1 << 28) + 12345])
def test_isa_windows(n):
    """Texts on both sides of 2^28 suffixes, above which the ISA's buckets grow: windowed
    and direct scatter give one suffix array, and the BWT of both is the text's."""
    lib = la.load()
    T = workloads.iid(n, seed=n & 255, alphabet=b"ACGT")
    from tests.test_gpu_parity import fused
    out = []
    for on in (1, 0):
        print(f"[isa windows] n={n} windowed_scatter={on}", flush=True)
        assert lib.sagpu_set_option(b"windowed_scatter", on) == 0
        try:
            out.append(fused(T)[:3])
        finally:
            assert lib.sagpu_set_option(b"windowed_scatter", 1) == 0
    (SA, U, p), (SA0, U0, p0) = out
    assert np.array_equal(SA, SA0) and p == p0 and np.array_equal(U, U0)
    rng = np.random.default_rng(n)
    j = rng.integers(1, n, 20000)
    a, b = SA[j - 1].astype(np.int64), SA[j].astype(np.int64)
    keys = [[T[q:q + 64].tobytes() for q in (x, y)] for x, y in zip(a, b)]
    assert all(x <= y for x, y in keys)


SEG_KEYS = 16384   # keys of a tile of a segmented sort


def _string_sets():
    """(name, string lengths, symbols): sets of at least 2^22 symbols, whose strings are
    sorted four to a segment (5 codes: 30-bit keys), one (16 and 256 codes: no bits left),
    sixteen (100 codes) and more with fewer symbols; lengths around whole tiles, one string,
    a few long ones."""
    rng = np.random.default_rng(7)
    n = 1 << 22
    edges = [SEG_KEYS - 1, SEG_KEYS, SEG_KEYS + 1, 4 * SEG_KEYS, 2, 3, 65]
    around = [edges[i % 7] for i in range(7 * (n // sum(edges) + 1))]
    mixed = rng.integers(2, 60000, 160)
    yield "around tiles", around, 4
    yield "one string", [n], 4
    yield "two strings", [n // 2, n // 2 + 5], 15
    yield "long and short", [n - 100, 2, 2, 50, 70001], 255
    yield "mixed, 4 bits", list(mixed) + [3], 15
    yield "mixed, 7 bits", list(mixed) + [5, 2], 99
    yield "alike", [40000] * 106, 4
    yield "short", [90] * (n // 90 + 1), 4   # fewer symbols, 256 strings to a segment
    yield "reads", list(rng.integers(30, 400, n // 200)), 4
    yield "tiny", [4] * (n // 4 + 1), 4      # too short: the 64-bit sort


@pytest.mark.parametrize("name,lengths,sigma", list(_string_sets()), ids=lambda v: v if isinstance(v, str) else "")
def test_segmented_sort(name, lengths, sigma):
    """Sets sorted string by string against the sort by (string, symbols) of the same set
    (the form that other tiles take), and sampled strings against the oracle."""
    lib = la.load()
    rng = np.random.default_rng(len(lengths))
    n = int(np.sum(lengths))
    offs = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    T = rng.integers(1, sigma + 1, n).astype(np.uint8)
    if name == "alike":
        T[:] = np.tile(T[:40000], len(lengths))
    T[offs[1:] - 1] = 0
    out = []
    for items in (32, 16):
        print(f"[segments] {name}: n={n} strings={len(lengths)} radix_items={items}", flush=True)
        assert lib.sagpu_set_option(b"radix_items", items) == 0
        try:
            out.append(batch.batched(T, offs))
            print(f"[segments] bytes sorted per symbol: {la.stats().sorted_bytes / n:.0f}", flush=True)
        finally:
            assert lib.sagpu_set_option(b"radix_items", 32) == 0
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    SA, L = out[0]
    for k in sorted({0, len(lengths) // 2, len(lengths) - 1}):
        o, e = int(offs[k]), int(offs[k + 1])
        if e - o > 100000:
            continue
        rc, ref = ol.sa(T[o:e].copy(), gsa=True)
        assert rc == 0 and np.array_equal(SA[o:e], ref), k
        assert np.array_equal(L[o:e], ol.lcp(ol.plcp(T[o:e].copy(), ref, gsa=True), ref)), k


@pytest.mark.parametrize("n", [2, 5, 1023, 1025, 4095, 4096, 4097, 8193, 12290])
def test_string_ids(n):
    """Sets whose separators fall on every position of a tile's words and steps."""
    rng = np.random.default_rng(n)
    T = rng.integers(1, 4, n).astype(np.uint8)
    at = np.flatnonzero(rng.random(n) < 0.3)
    T[at[at > 0]] = 0
    T[1:][(T[1:] == 0) & (T[:-1] == 0)] = 3   # no empty strings
    T[-2:] = (1, 0)
    ends = np.flatnonzero(T == 0) + 1
    offs = np.concatenate([[0], ends]).astype(np.int64)
    print(f"[string ids] n={n} strings={len(offs) - 1}", flush=True)
    SA, L = batch.batched(T, offs)
    for k in range(len(offs) - 1):
        S = T[offs[k]:offs[k + 1]].copy()
        rc, ref = ol.sa(S, gsa=True)
        assert rc == 0 and np.array_equal(SA[offs[k]:offs[k + 1]], ref), k
        assert np.array_equal(L[offs[k]:offs[k + 1]], ol.lcp(ol.plcp(S, ref, gsa=True), ref)), k


def _check_lcp(T, SA, L, n, rng):
    j = rng.integers(1, n, 5000)
    for a, b, l in zip(SA[j - 1], SA[j], L[j]):
        assert np.array_equal(T[a:a + l], T[b:b + l])
        assert max(a, b) + l == n or T[a + l] != T[b + l]


@pytest.mark.parametrize("n", [1 << 28, (1 << 28) + 1, (1 << 29) + 1])
def test_plcp_hint_ranges(n):
    """PLCP hints on both sides of the sizes where the bits for them get fewer: the same
    LCP and PLCP with hints and without, and sampled lcps of the text."""
    from tests.test_gpu_parity import fused
    lib = la.load()
    T = workloads.iid(n, seed=n & 255, alphabet=b"ACGT")
    T[n // 2: n // 2 + 3000] = T[:3000]
    out = []
    for on in (1, 0):
        print(f"[hints] n={n} plcp_hint={on}", flush=True)
        assert lib.sagpu_set_option(b"plcp_hint", on) == 0
        try:
            SA, _, _, P, L, _ = fused(T)
        finally:
            assert lib.sagpu_set_option(b"plcp_hint", 1) == 0
        out.append((SA, P, L))
    assert all(np.array_equal(a, b) for a, b in zip(*out))
    _check_lcp(T, out[0][0], out[0][2], n, np.random.default_rng(n))


@pytest.mark.parametrize("n", [1 << 23, (1 << 28) + 5])
def test_plcp_hint_sets(n):
    """The same for string sets sorted string by string."""
    lib = la.load()
    rng = np.random.default_rng(n)
    T = workloads.iid(n, seed=n & 255, alphabet=b"ACGT")
    T[np.cumsum(rng.integers(3, 90000, n // 45000 - 100))] = 0
    T[-1] = 0
    T[(n - 50):(n - 1)] = 67
    ends = np.flatnonzero(T == 0) + 1
    offs = np.concatenate([[0], ends]).astype(np.int64)
    out = []
    for on in (1, 0):
        print(f"[hint sets] n={n} strings={len(offs) - 1} plcp_hint={on}", flush=True)
        assert lib.sagpu_set_option(b"plcp_hint", on) == 0
        try:
            out.append(batch.batched(T, offs))
        finally:
            assert lib.sagpu_set_option(b"plcp_hint", 1) == 0
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    for k in (0, len(offs) // 2, len(offs) - 2):
        S = T[offs[k]:offs[k + 1]].copy()
        rc, ref = ol.sa(S, gsa=True)
        assert rc == 0 and np.array_equal(out[0][0][offs[k]:offs[k + 1]], ref), k
        assert np.array_equal(out[0][1][offs[k]:offs[k + 1]], ol.lcp(ol.plcp(S, ref, gsa=True), ref)), k


RADIX_SIZES = [1, 2, 255, 2047, 2049, 8191, 8193, (1 << 18) - 1, (1 << 18) + 1, (1 << 20) - 1, (1 << 20) + 1,
               (3 << 19) - 1, (3 << 19) + 1, (1 << 22) - 1, (1 << 22) + 1]


@pytest.mark.parametrize("n", RADIX_SIZES)
def test_radix_tile_rules(n):
    """Sorted pairs at the sizes where tiles, the skipped wait for the histograms and
    generated keys change; digits all alike, and key bits that end inside a digit."""
    from tests.test_gpu_parity import fused
    T = workloads.iid(max(n, 2), seed=n & 255, alphabet=b"ACGT")
    print(f"[radix] n={n}", flush=True)
    SA, U, p, P, L, f = fused(T)
    rc, ref = ol.sa(T)
    assert rc == 0 and np.array_equal(SA, ref)
    rU, rp = ol.bwt(T, ref)
    assert p == rp and np.array_equal(U, rU)
    S = np.full(max(n, 2), 7, np.int32)   # 3-bit symbols, most digits alike
    S[::97] = 1
    out = np.zeros(len(S), np.int32)
    assert la.libsais_int(S.copy(), out, len(S), 8, 0) == 0
    assert np.array_equal(out, ol.sa_int(S))


@pytest.mark.parametrize("n", [(1 << 20) - 1, (1 << 20) + 1, (1 << 22) - 1, (1 << 22) + 1])
def test_round_rules(n):
    """Rounds at the sizes where the first list's length is left on the device, the next
    round is queued ahead and the round's end takes the big groups along: lists of small
    groups, of big ones (pivots and not), both, and empty ones; plain and string sets."""
    from tests.test_gpu_parity import fused
    rng = np.random.default_rng(n)
    words = workloads.iid(n, seed=3, alphabet=b"ab")
    words[n // 3:n // 3 + n // 4] = words[:n // 4]
    big = np.tile(rng.integers(97, 123, 601).astype(np.uint8), n // 601 + 1)[:n].copy()
    runs = np.full(n, 97, np.uint8)
    runs[::1000] = 98
    for name, T in (("unique", rng.integers(0, 256, n).astype(np.uint8)), ("small", words), ("big", big), ("runs", runs)):
        for gsa in (False, True):
            if gsa:
                T = np.where(T == 0, 1, T).astype(np.uint8)
                T[5000::70001] = 0
                T[-2:] = (98, 0)
            rc, SA = ol.sa(T, gsa=gsa)
            assert rc == 0
            P = ol.plcp(T, SA, gsa=gsa)
            gSA, gU, gp, gP, gL, _ = fused(T, gsa=gsa)
            print(f"[rounds] n={n} {name} gsa={gsa}: {la.stats().rounds} rounds", flush=True)
            assert np.array_equal(gSA, SA) and np.array_equal(gP, P) and np.array_equal(gL, ol.lcp(P, SA)), (name, gsa)
            if not gsa:
                U, p = ol.bwt(T, SA)
                assert gp == p and np.array_equal(gU, U), name


@pytest.mark.parametrize("n", [131071, 131073, 1048575, 1048577, 4194303, 4194305, 8388609, 12582913])
def test_staged_copies(n):
    """Host arrays of both index widths around the sizes where their copies are staged, the
    chunk and ring sizes, in calls that carry several arrays up and down."""
    T = workloads.iid(n, seed=n & 255, alphabet=b"ACGT")
    rc, SA = ol.sa(T)
    assert rc == 0
    U, p = ol.bwt(T, SA)
    P = ol.plcp(T, SA)
    L = ol.lcp(P, SA)
    for dt, sa, bwt, unbwt, plcp, lcp in (
            (np.int32, la.libsais, la.libsais_bwt, la.libsais_unbwt, la.libsais_plcp, la.libsais_lcp),
            (np.int64, la.libsais64, la.libsais64_bwt, la.libsais64_unbwt, la.libsais64_plcp, la.libsais64_lcp)):
        print(f"[staged] n={n} {dt.__name__}", flush=True)
        out, hU, A = np.zeros(n, dt), np.zeros(n, np.uint8), np.zeros(n + 1, dt)
        assert sa(T, out, n, 0, None) == 0 and np.array_equal(out, SA)
        assert bwt(T, hU, A, n, 0, None) == p and np.array_equal(hU, U)
        back = np.zeros(n, np.uint8)
        assert unbwt(hU, back, A, n, None, p) == 0 and np.array_equal(back, T)
        S, PL = SA.astype(dt), np.zeros(n, dt)
        assert plcp(T, S, PL, n) == 0 and np.array_equal(PL, P)
        out[:] = 0
        assert lcp(PL, S, out, n) == 0 and np.array_equal(out, L)


@pytest.mark.parametrize("n", [24577, 65536, 65537, (1 << 20) + 3])
def test_alphabet_kernel(n):
    """Symbol counts and codes: one, two and 256 symbols, and symbols that occur once, at
    the text's ends and around its words."""
    from tests.test_gpu_parity import fused
    rng = np.random.default_rng(n)
    for name, T in (("one", np.full(n, 255, np.uint8)), ("all", rng.integers(0, 256, n).astype(np.uint8)),
                    ("two", rng.integers(0, 2, n).astype(np.uint8) * 255)):
        T[0], T[-1], T[n // 2] = 3, 9, 250
        print(f"[alphabet] n={n} {name}", flush=True)
        SA, _, _, _, _, f = fused(T)
        rc, ref = ol.sa(T)
        assert rc == 0 and np.array_equal(SA, ref) and np.array_equal(f, np.bincount(T, minlength=256)), name


@pytest.mark.parametrize("n", [1048577, 6000001, 8388608])
def test_concurrent_staged_copies(n):
    """Downloads of several calls at once, which take turns on the bus a half ring at a
    time: both index widths, lengths around the half."""
    from concurrent.futures import ThreadPoolExecutor
    T = [workloads.iid(n, seed=k, alphabet=b"ACGT") for k in range(2)]
    ref = [ol.sa(t)[1] for t in T]

    def one(k):
        dt, sa = (np.int32, la.libsais) if k % 2 else (np.int64, la.libsais64)
        out = np.zeros(n, dt)
        for _ in range(3):
            out[:] = 0
            if sa(T[k // 2 % 2], out, n, 0, None) != 0 or not np.array_equal(out, ref[k // 2 % 2]):
                return False
        return True

    print(f"[concurrent copies] n={n}", flush=True)
    with ThreadPoolExecutor(6) as ex:
        assert all(ex.map(one, range(6)))


@pytest.mark.parametrize("n", [30000, 1 << 20, (1 << 22) - 1])
def test_build_under_a_memory_limit(n):
    """Under a limit, texts below 2^22 wait for the first list's length: the same results."""
    print(f"[limit] n={n}", flush=True)
    T = workloads.iid_acgt(n, seed=n)
    lib = la.load()
    SA0 = np.zeros(n, np.int32)
    assert la.libsais(T, SA0, n, 0, None) == 0, la.last_error()
    rc, ref = ol.sa(T)
    assert rc == 0 and np.array_equal(SA0, ref)
    try:
        lib.sagpu_set_memory_limit(1 << 36)   # (the context keeps scratch of earlier calls)
        SA = np.zeros(n, np.int32)
        assert la.libsais(T, SA, n, 0, None) == 0, la.last_error()
        U = np.zeros(n, np.uint8)
        p = la.libsais_bwt(T, U, np.zeros(n, np.int32), n, 0, None)
    finally:
        lib.sagpu_set_memory_limit(0)
    U_r, p_r = ol.bwt(T, ref)
    assert np.array_equal(SA, ref)
    assert p == p_r and np.array_equal(U, U_r)


@pytest.mark.parametrize("length,sigma,segmented,fewer", [(90, 4, True, True), (1 << 22, 4, True, False),
                                                          (60000, 255, True, False), (4, 4, False, False)])
def test_string_set_route(length, sigma, segmented, fewer):
    """Which sort a set takes, and the symbols in its keys, from the statistics: 32-bit keys by
    segment move 16 bytes a symbol and pass, the others 24; short strings' keys hold fewer
    symbols than 32 bits do.  One more pass of 16 bytes groups the ranks into windows, unless
    they go straight to the ISA (segmented sets of strings below 3 * 2^18 symbols)."""
    count = (1 << 22) // length + 1
    lengths = [length] * count
    offs = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    n = int(offs[-1])
    T = np.random.default_rng(length).integers(1, sigma + 1, n).astype(np.uint8)
    T[offs[1:] - 1] = 0
    print(f"[set route] {count} strings of {length}", flush=True)
    batch.batched(T, offs)
    st = la.stats()
    most = 32 // st.bits_per_symbol
    per_symbol = st.sorted_bytes / n
    print(f"[set route] bytes per symbol {per_symbol:.1f}, symbols {st.initial_symbols} of {most}", flush=True)
    if not segmented or length > 3 << 18:
        per_symbol -= 16
    if segmented:
        assert per_symbol % 16 == 0 and per_symbol <= 4 * 16
    else:
        assert per_symbol % 24 == 0
    assert st.initial_symbols < most if fewer else st.initial_symbols == most


@pytest.mark.parametrize("n", [1 << 16, 300007])
def test_round_chains_save_rounds(n):
    """Two copies of one random text: every group continues in one group up to the copies'
    end, so with chains the build ends within a round or two of the first that uses them."""
    from tests.test_gpu_parity import fused
    lib = la.load()
    T = np.random.default_rng(n).integers(97, 101, n).astype(np.uint8)
    T[n // 2:] = T[:n - n // 2]
    rounds = []
    for least in (2, 0):
        assert lib.sagpu_set_option(b"chain_min", least) == 0
        try:
            out = fused(T)
            rounds.append(la.stats().rounds)
        finally:
            assert lib.sagpu_set_option(b"chain_min", 4096) == 0
    print(f"[chains] n={n}: {rounds} rounds", flush=True)
    rc, SA = ol.sa(T)
    assert rc == 0 and np.array_equal(out[0], SA)
    assert rounds[0] + 3 < rounds[1]


@pytest.mark.parametrize("length", [8, 16, 32, 64])
@pytest.mark.parametrize("n", [30011, 70000])
def test_plcp_bound_at_the_end(n, length):
    """The text's last `length` symbols stand earlier, before zero bytes: the known bound of
    their lcp is all that is left of the text, and the bytes past both places agree (the
    padding is zero).  Byte comparisons (plain and with separators) and the code stream."""
    from tests.test_gpu_parity import fused
    lib = la.load()
    rng = np.random.default_rng(n + length)
    T = rng.integers(1, 5, n).astype(np.uint8)
    for at in (101, n // 2):
        T[at:at + length] = T[n - length:]
        T[at + length:at + length + 40] = 0
    rc, SA = ol.sa(T)
    assert rc == 0
    P = ol.plcp(T, SA)
    for compare in (1, 0):
        print(f"[plcp end] n={n} length={length} stream_compare={compare}", flush=True)
        assert lib.sagpu_set_option(b"stream_compare", compare) == 0
        try:
            gSA, _, _, gP, gL, _ = fused(T)
        finally:
            assert lib.sagpu_set_option(b"stream_compare", 1) == 0
        assert np.array_equal(gSA, SA) and np.array_equal(gP, P) and np.array_equal(gL, ol.lcp(P, SA))
    for at in (101, n // 2):
        T[at + length + 1:at + length + 40] = 1
    T[-1] = 0
    rc, SA = ol.sa(T, gsa=True)
    assert rc == 0
    P = ol.plcp(T, SA, gsa=True)
    gSA, _, _, gP, gL, _ = fused(T, gsa=True)
    assert np.array_equal(gSA, SA) and np.array_equal(gP, P) and np.array_equal(gL, ol.lcp(P, SA))


@pytest.mark.parametrize("n", [30000, 1 << 18, (1 << 22) - 1, (1 << 22) + 1])
def test_timed_bytes(n):
    """Timing mode counts the gathers' and tile kernels' bytes for the lists that the rounds
    had: 12 and 28 bytes an entry, and 4 more where the first round reads the groups."""
    from tests.test_gpu_parity import fused
    lib = la.load()
    T = workloads.dna_like(n, seed=n & 255)
    print(f"[timed bytes] n={n}", flush=True)
    lib.sagpu_set_timing(1)
    try:
        fused(T)
        st = la.stats()
    finally:
        lib.sagpu_set_timing(0)
    entries = sum(st.active[:st.rounds])
    assert st.rounds > 1 and st.active[0] < n
    assert st.kernel_bytes[5] == 12 * entries + 4 * st.active[0]
    assert st.kernel_bytes[6] == 28 * entries


@pytest.mark.parametrize("n", [70001, 300007])
def test_round_chains_mixed_groups(n):
    """Lists of mostly pairs, which take chains, with groups of 3 to 12 among them: some small
    enough to be marked, some not, some ending inside another's copies."""
    from tests.test_gpu_parity import fused
    lib = la.load()
    rng = np.random.default_rng(n)
    T = rng.integers(97, 101, n).astype(np.uint8)
    k = n // 40
    T[20 * k:36 * k] = T[:16 * k]   # pairs
    for c, (copies, size) in enumerate(((3, k), (4, k // 2), (7, k // 8), (8, k // 9), (9, k // 10), (12, k // 13))):
        at = 36 * k + c * (k // 2) + np.arange(copies) * size // 2   # overlapping
        for q in at:
            T[q:q + size // 2] = T[c * k:c * k + size // 2]
    rc, SA = ol.sa(T)
    assert rc == 0
    P = ol.plcp(T, SA)
    rounds = []
    for least in (2, 0):
        assert lib.sagpu_set_option(b"chain_min", least) == 0
        try:
            gSA, gU, gp, gP, gL, _ = fused(T)
            rounds.append(la.stats().rounds)
        finally:
            assert lib.sagpu_set_option(b"chain_min", 4096) == 0
        assert np.array_equal(gSA, SA) and np.array_equal(gP, P) and np.array_equal(gL, ol.lcp(P, SA)), least
    print(f"[chains] n={n}: {rounds} rounds", flush=True)
    assert rounds[0] < rounds[1]


@pytest.mark.parametrize("copies", [3, 5, 7])
@pytest.mark.parametrize("length", [9001, 40000])
def test_round_chains_exact_copies(length, copies):
    """Exact copies of one block in a random text: their groups of up to seven all end in one
    place, and chains take them there."""
    from tests.test_gpu_parity import fused
    lib = la.load()
    T = np.random.default_rng(length + copies).integers(97, 101, (length + 300) * copies).astype(np.uint8)
    block = T[:length].copy()
    for k in range(copies):
        at = k * (length + 300) + 7 * k
        T[at:at + length] = block
    rounds = []
    for least in (2, 0):
        assert lib.sagpu_set_option(b"chain_min", least) == 0
        try:
            out = fused(T)
            rounds.append(la.stats().rounds)
        finally:
            assert lib.sagpu_set_option(b"chain_min", 4096) == 0
    print(f"[chains] {copies} copies of {length}: {rounds} rounds", flush=True)
    rc, SA = ol.sa(T)
    assert rc == 0
    P = ol.plcp(T, SA)
    assert np.array_equal(out[0], SA) and np.array_equal(out[3], P) and np.array_equal(out[4], ol.lcp(P, SA))
    assert rounds[0] + 3 < rounds[1]
