"""The calls that users of the engine make, as measurable cases.

Every case is one pass through public entry points: the device ABI (``sagpu_*``) on torch
tensors that already live in HBM, or the libsais API on host arrays, which copies to the
GPU and back inside the call.  A case holds its ``kind`` (the entry points), its ``text``
(the inputs' distribution) and its sizes:

  fused    sagpu_build32: SA + BWT + PLCP + LCP of a resident text
  string   sagpu_build32 with SAGPU_FLAG_GSA: SA + LCP of one separator-terminated string
  batch    sagpu_gsa_batch32: SA + LCP of a set of strings in one call
  bwt      libsais_bwt on host buffers (block compressors, BWT encode)
  unbwt    libsais_unbwt, or libsais_unbwt_aux with a sample every `r` rows (BWT decode)
  salcp    libsais, libsais_plcp and libsais_lcp on host buffers
  salcp64  the same three calls of the 64-bit API
  bwt16    libsais16_bwt on a 16-bit alphabet
  int      libsais_int on an integer alphabet of `k` symbols
"""
from __future__ import annotations

import numpy as np
import torch

import libsais_amd as la
from libsais_amd import workloads

KIB, MIB = 1 << 10, 1 << 20


def listed():
    return [
        # One small block of a stream of text blocks through the host API: latency and launches.
        {"name": "bwt_words_4k", "kind": "bwt", "text": "words", "n": 4001},
        # One read or contig of a string set built by itself: the mean string of the batched workload.
        {"name": "string_acgt_22k", "kind": "string", "text": "acgt", "n": 22347},
        # One 900 KB compressor block of natural-language-like text.
        {"name": "bwt_words_900k", "kind": "bwt", "text": "words", "n": 900_000},
        # The 1 MiB i.i.d. ACGT configuration.
        {"name": "fused_acgt_1m", "kind": "fused", "text": "acgt", "n": 1 * MIB},
        # A resident corpus of natural-language-like bytes, odd size.
        {"name": "fused_words_48m", "kind": "fused", "text": "words", "n": 48 * MIB + 13},
        # The benchmark's genome-like text.
        {"name": "fused_dna_256m", "kind": "fused", "text": "dna", "n": 256 * MIB},
        # Highly repetitive text (long common prefixes), a degenerate configuration of the benchmark.
        {"name": "fused_fibonacci_64m", "kind": "fused", "text": "fibonacci", "n": 64 * MIB},
        # The benchmark's string set: 20,000 strings, 512 MiB.
        {"name": "batch_acgt_512m", "kind": "batch", "text": "strings", "n": 512 * MIB, "count": 20000},
        # A libsais user's index construction on host buffers, 64-bit index width.
        {"name": "salcp64_dna_12m", "kind": "salcp64", "text": "dna", "n": 12_000_001},
        # BWT decode of a large block.
        {"name": "unbwt_words_32m", "kind": "unbwt", "text": "words", "n": 32 * MIB, "r": 0},
        # 16-bit symbols (token ids) encoded through the 16-bit API.
        {"name": "bwt16_tokens_4m", "kind": "bwt16", "text": "tokens", "n": 4 * MIB + 3, "k": 50_000},
        # Token ids of a vocabulary beyond 16 bits.
        {"name": "int_tokens_6m", "kind": "int", "text": "tokens", "n": 6_000_003, "k": 100_000},
    ]


def _size(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["fused", "fused", "fused", "string", "batch", "bwt", "bwt", "unbwt", "unbwt", "salcp",
                       "salcp64", "bwt16", "int"])
    if kind == "fused":
        text, hi = rng.choice([("acgt", 128 * MIB), ("dna", 256 * MIB), ("words", 48 * MIB), ("bytes", 64 * MIB),
                               ("protein", 64 * MIB), ("periodic", 64 * MIB), ("fibonacci", 64 * MIB)])
        return {"kind": kind, "text": text, "n": _size(rng, 2 * KIB, hi)}
    if kind == "string":
        return {"kind": kind, "text": "acgt", "n": _size(rng, 257, 4 * MIB)}
    if kind == "batch":
        n = _size(rng, 1 * MIB, 512 * MIB)
        return {"kind": kind, "text": "strings", "n": n, "count": max(16, n // _size(rng, 8 * KIB, 64 * KIB))}
    if kind == "bwt":
        return {"kind": kind, "text": rng.choice(["words", "words", "bytes", "dna"]), "n": _size(rng, 500, 32 * MIB)}
    if kind == "unbwt":
        return {"kind": kind, "text": rng.choice(["words", "dna"]), "n": _size(rng, 4 * KIB, 32 * MIB),
                "r": rng.choice([0, 0, 64, 1024])}
    if kind in ("salcp", "salcp64"):
        return {"kind": kind, "text": rng.choice(["dna", "words"]), "n": _size(rng, 4 * KIB, 12_000_001)}
    if kind == "bwt16":
        return {"kind": kind, "text": "tokens", "n": _size(rng, 2 * KIB, 4 * MIB), "k": _size(rng, 300, 65_536)}
    return {"kind": "int", "text": "tokens", "n": _size(rng, 2 * KIB, 6_000_003), "k": _size(rng, 300, 1_000_000)}


# ---------------------------------------------------------------- inputs

def _zipf(n, k, gen, shift=2.7, power=1.07):
    """n ids in [0, k), Zipf-Mandelbrot distributed, as token and word frequencies are."""
    w = (torch.arange(k, device="cuda", dtype=torch.float64) + shift).pow(-power)
    c = torch.cumsum(w, 0)
    return torch.searchsorted(c / c[-1], torch.rand(n, device="cuda", dtype=torch.float64, generator=gen)).clamp_(max=k - 1)


def _passages(t, gen):
    """Quotes: up to 48 passages (about 5% of the text) repeat an earlier stretch of it."""
    n = t.numel()
    count = min(48, n // 512)
    if count:
        most = max(2, 2 * n // (20 * count))
        p = torch.rand(count, 3, device="cuda", generator=gen).cpu().numpy()
        for a, b, c in p:
            size = 1 + int(c * (most - 1))
            src, dst = int(a * (n - size)), int(b * (n - size))
            t[dst:dst + size] = t[src:src + size].clone()
    return t


def _words(n, gen):
    """Words of a 20,000-word vocabulary with letter frequencies of English, separated by blanks."""
    vocab, longest = 20_000, 13
    letters = torch.tensor(list(b"etaoinshrdlcumwfgypbvkjxqz"), device="cuda", dtype=torch.uint8)
    table = letters[_zipf(vocab * longest, 26, gen, 4.0, 1.2)].view(vocab, longest)
    size = torch.randint(2, longest, (vocab,), device="cuda", generator=gen)
    table.scatter_(1, size[:, None], ord(" "))
    size += 1
    ids = _zipf(n // 3 + 8, vocab, gen)
    start = torch.cumsum(size[ids], 0)
    ids = ids[: int(torch.searchsorted(start, n)) + 1]
    take = size[ids]
    word = torch.repeat_interleave(ids, take)
    first = torch.repeat_interleave(torch.cumsum(take, 0) - take, take)
    at = torch.arange(word.numel(), device="cuda") - first
    return _passages(table[word, at][:n].contiguous(), gen)


def _text(case, seed):
    """The case's byte text as a tensor on the GPU."""
    n, kind = case["n"], case["text"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if kind == "words":
        return _words(n, gen)
    if kind == "bytes":
        return torch.randint(0, 256, (n,), device="cuda", dtype=torch.uint8, generator=gen)
    if kind == "dna":
        t = workloads.dna_like(n, seed)
    elif kind == "acgt":
        t = workloads.iid_acgt(n, seed)
    elif kind == "protein":
        t = workloads.iid(n, seed, b"ACDEFGHIKLMNPQRSTVWY")
    elif kind == "periodic":
        t = workloads.periodic(n, 17, seed)
    elif kind == "fibonacci":  # a factor of the Fibonacci word, its place taken from the seed
        skip = (seed * 2654435761) % 9973
        t = workloads.fibonacci(n + skip)[skip:]
    else:
        raise ValueError(kind)
    return torch.from_numpy(np.ascontiguousarray(t)).cuda()


def _strings(case, seed):
    """A set of about `count` separator-terminated strings, n bytes in all, and their offsets."""
    n = case["n"]
    t, offsets = workloads.gsa_batch(case["count"], seed, median=min(4096.0, n / case["count"] / 2),
                                     target_total=float(n))
    if len(t) < n + 2:  # one more string fills the set up (and is cut to size with the rest)
        t = np.concatenate([t, workloads.iid_acgt(n + 2 - len(t), seed + 1)])
    t = t[:n].copy()
    if t[n - 2] == 0:
        t[n - 2] = ord("A")
    t[n - 1] = 0
    ends = np.flatnonzero(t == 0) + 1
    return t, np.concatenate([[0], ends]).astype(np.int64)


def _tokens(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    order = torch.randperm(case["k"], device="cuda", generator=gen)  # ids are not sorted by frequency
    return _passages(order[_zipf(case["n"], case["k"], gen)], gen)


def prepare(case, seed):
    kind, n = case["kind"], case["n"]
    s = {"kind": kind, "n": n}

    def out(count, dtype):
        return torch.empty(count, device="cuda", dtype=dtype)

    if kind == "fused":
        s |= {"T": _text(case, seed), "SA": out(n, torch.int32), "U": out(n, torch.uint8),
              "PLCP": out(n, torch.int32), "LCP": out(n, torch.int32)}
    elif kind == "string":
        t = _text(case, seed)
        t[-1] = 0
        s |= {"T": t, "SA": out(n, torch.int32), "LCP": out(n, torch.int32)}
    elif kind == "batch":
        t, offsets = _strings(case, seed)
        s |= {"T": torch.from_numpy(t).cuda(), "offsets": offsets, "SA": out(n, torch.int32), "LCP": out(n, torch.int32)}
    elif kind in ("bwt", "salcp", "salcp64", "unbwt"):
        t = _text(case, seed).cpu().numpy()
        index = np.int64 if kind == "salcp64" else np.int32
        s |= {"T": t}
        if kind in ("salcp", "salcp64"):
            s |= {"SA": np.empty(n, index), "PLCP": np.empty(n, index), "LCP": np.empty(n, index)}
        else:
            s |= {"U": np.empty(n, np.uint8), "A": np.empty(n + 1, np.int32)}
        if kind == "unbwt":
            r = case["r"]
            s["r"] = r
            s["L"] = np.empty(n, np.uint8)
            if r:
                s["I"] = np.empty((n - 1) // r + 1, np.int32)
                _ok(la.libsais_bwt_aux(t, s["L"], s["A"], n, 0, None, r, s["I"]))
            else:
                s["primary"] = _ok(la.libsais_bwt(t, s["L"], s["A"], n, 0, None))
            del s["T"]
    elif kind == "bwt16":
        s |= {"T": _tokens(case, seed).to(torch.int32).cpu().numpy().astype(np.uint16), "U": np.empty(n, np.uint16),
              "A": np.empty(n, np.int32)}
    elif kind == "int":
        s |= {"T": _tokens(case, seed).to(torch.int32).cpu().numpy(), "k": case["k"], "SA": np.empty(n, np.int32)}
    else:
        raise ValueError(kind)
    torch.cuda.synchronize()
    la.load()
    return s


# ---------------------------------------------------------------- passes

def _ok(rc):
    if rc < 0:
        raise RuntimeError(f"returned {rc}: {la.last_error()}")
    return rc


def run(s):
    kind, n = s["kind"], s["n"]
    if kind == "fused":
        primary = _ok(la.load().sagpu_build32(s["T"].data_ptr(), n, 0, s["SA"].data_ptr(), s["U"].data_ptr(),
                                              s["PLCP"].data_ptr(), s["LCP"].data_ptr(), None))
        return {"primary": primary, "SA": s["SA"], "U": s["U"], "PLCP": s["PLCP"], "LCP": s["LCP"]}
    if kind == "string":
        _ok(la.load().sagpu_build32(s["T"].data_ptr(), n, la.SAGPU_FLAG_GSA, s["SA"].data_ptr(), None, None,
                                    s["LCP"].data_ptr(), None))
        return {"SA": s["SA"], "LCP": s["LCP"]}
    if kind == "batch":
        _ok(la.load().sagpu_gsa_batch32(s["T"].data_ptr(), n, s["offsets"].ctypes.data, len(s["offsets"]) - 1,
                                        s["SA"].data_ptr(), s["LCP"].data_ptr()))
        return {"SA": s["SA"], "LCP": s["LCP"]}
    if kind == "bwt":
        return {"primary": _ok(la.libsais_bwt(s["T"], s["U"], s["A"], n, 0, None)), "U": s["U"]}
    if kind == "unbwt":
        if s["r"]:
            _ok(la.libsais_unbwt_aux(s["L"], s["U"], s["A"], n, None, s["r"], s["I"]))
        else:
            _ok(la.libsais_unbwt(s["L"], s["U"], s["A"], n, None, s["primary"]))
        return {"T": s["U"]}
    if kind in ("salcp", "salcp64"):
        wide = kind == "salcp64"
        _ok((la.libsais64 if wide else la.libsais)(s["T"], s["SA"], n, 0, None))
        _ok((la.libsais64_plcp if wide else la.libsais_plcp)(s["T"], s["SA"], s["PLCP"], n))
        _ok((la.libsais64_lcp if wide else la.libsais_lcp)(s["PLCP"], s["SA"], s["LCP"], n))
        return {"SA": s["SA"], "PLCP": s["PLCP"], "LCP": s["LCP"]}
    if kind == "bwt16":
        return {"primary": _ok(la.libsais16_bwt(s["T"], s["U"], s["A"], n, 0, None)), "U": s["U"]}
    _ok(la.libsais_int(s["T"], s["SA"], n, s["k"], 0))
    return {"SA": s["SA"]}


def work(case):
    """The bytes of one pass (each input read once, each output written once); all of it is integer work."""
    n = case["n"]
    per = {"fused": 1 + 4 + 1 + 4 + 4, "string": 1 + 4 + 4, "batch": 1 + 4 + 4, "bwt": 2, "unbwt": 2,
           "salcp": 1 + 4 + 4 + 4, "salcp64": 1 + 8 + 8 + 8, "bwt16": 4, "int": 8}[case["kind"]]
    return {"bytes": per * n, "flops": 0}


# ---------------------------------------------------------------- exact results, plain numpy

def _suffixes(t):
    """Suffix array of an array of symbols by prefix doubling."""
    n = len(t)
    rank, h = np.unique(t, return_inverse=True)[1].astype(np.int64) + 1, 1
    while True:
        key = rank * (n + 2)
        key[:n - h] += rank[h:]
        sa = np.argsort(key, kind="stable")
        new = np.concatenate([[1], 1 + np.cumsum(key[sa][1:] != key[sa][:-1])])
        if new[-1] == n or h >= n:
            return sa
        rank[sa] = new
        h *= 2


def _plcp(t, sa):
    """PLCP: the lcp of every suffix with its predecessor in the suffix array, all suffixes a step at a time."""
    n = len(t)
    before = np.full(n, n, np.int64)
    before[sa[1:]] = sa[:-1]
    padded = np.concatenate([t.astype(np.int64), [-1]])
    lcp, live = np.zeros(n, np.int64), np.arange(n)
    while len(live):
        a, b = live + lcp[live], before[live] + lcp[live]
        fine = (a < n) & (b < n)
        live = live[fine]
        live = live[padded[a[fine]] == padded[b[fine]]]
        lcp[live] += 1
    return lcp


def exact(case, seed):
    kind, n = case["kind"], case["n"]
    if kind == "unbwt":  # the text that was transformed
        return {"T": _text(case, seed).cpu().numpy()}
    if n > 64 * KIB or kind == "batch" or case["text"] in ("periodic", "fibonacci"):
        return None
    if kind in ("bwt16", "int"):
        t = _tokens(case, seed).cpu().numpy()
    else:
        t = _text(case, seed).cpu().numpy()
        if kind == "string":
            t[-1] = 0
    sa = _suffixes(t)
    row = int(np.nonzero(sa == 0)[0][0])
    last = np.concatenate([t[-1:], np.delete(t[sa - 1], row)])
    if kind == "int":
        return {"SA": sa}
    if kind in ("bwt", "bwt16"):
        return {"primary": row + 1, "U": last}
    plcp = _plcp(t, sa)
    lcp = plcp[sa]
    if kind == "string":
        return {"SA": sa, "LCP": lcp}
    out = {"SA": sa, "PLCP": plcp, "LCP": lcp}
    return out | {"primary": row + 1, "U": last} if kind == "fused" else out
