"""Workloads of the search pipeline, as its users call it.

Every case is one call of a stage through the C ABI (include/golay_gpu.h) on host
records in buffers that the caller keeps, as the command line tool and a C
program make it, or, for the two batched PSD filters, on host rows and on device
rows.  Configurations are those of the tests and of bench.py: the searches of
order 50 (compression 5 -> 1), 45 (3 -> 1), 90 (10 -> 5), 40 (4 -> 2) and 34
(2 -> 1), whole or in part.

listed() is what is timed, draw() gives further sizes of the same ranges.
"""
import ctypes
import functools
import math

import numpy as np
import torch

import golaypair_amd as g

# (order, coarse compression, fine compression, paf): matched pairs of the level,
# leaves per pair (mean over the level), output pairs per pair to make room for
UNC = {
    (50, 5, 1, 0): (4691, 1.964e8, 400),
    (45, 3, 1, -2): (7577, 3.88e5, 64),
    (90, 10, 5, 0): (156, 1.22e6, 400),
}
# (order, compression, paf) of the generated candidate sets
GEN = [(50, 5, 0), (45, 3, -2), (90, 10, 0), (34, 2, 0)]
# (order, compression, letters of the pairs) of the equivalence filter
FILTER = [(50, 1, (-1, 1)), (45, 1, (-1, 1)), (34, 1, (-1, 1)), (90, 5, (-5, -3, -1, 1, 3, 5))]
# word length, compression, order, paf, share of the mixed-length PSD batch
MIX = [(9, 10, 90, 0, 32), (10, 5, 50, 0, 16), (15, 3, 45, -2, 8), (17, 3, 51, -2, 4), (18, 5, 90, 0, 2),
       (25, 2, 50, 0, 2)]


def listed():
    return [
        # One shard (-j/-n) of a level's candidate generation: the first stage of every search.
        {"name": "gen v45 c3 shard", "stage": "gen", "order": 45, "compress": 3, "paf": -2, "jobs": 8},
        # The candidate files of a level, several shards with repeats, into line order.
        {"name": "sort v45 c3 61k", "stage": "sort", "order": 45, "compress": 3, "paf": -2, "records": 61003},
        # The same for a search whose candidate files are large.
        {"name": "sort n15 4M", "stage": "sort", "order": 45, "compress": 3, "paf": -2, "records": 4000037},
        # The merge-join of a level's two sorted files.
        {"name": "match v45 c3", "stage": "match", "order": 45, "compress": 3, "paf": -2, "records": 53000},
        # Uncompression: a handful of pairs (a slice of a shared job), where latency counts ...
        {"name": "uncompress v90 7 pairs", "stage": "uncompress", "order": 90, "compress": 10, "fine": 5, "paf": 0,
         "pairs": 7},
        # ... an ordinary level of many small expansions ...
        {"name": "uncompress v45 2500 pairs", "stage": "uncompress", "order": 45, "compress": 3, "fine": 1,
         "paf": -2, "pairs": 2500},
        # ... and a slice of the exhaustive order-50 search, 2e8 words a pair.
        {"name": "uncompress v50 401 pairs", "stage": "uncompress", "order": 50, "compress": 5, "fine": 1, "paf": 0,
         "pairs": 401},
        # Equivalence classes of a finished search: odd length, the group without altnegative ...
        {"name": "filter v45 18645 pairs", "stage": "filter", "order": 45, "compress": 1, "pairs": 18645},
        # ... and length 50 with altnegative, the largest group.
        {"name": "filter v50 120k pairs", "stage": "filter", "order": 50, "compress": 1, "pairs": 120011},
        # A caller's own words of many lengths through the PSD filter, with the PSD maxima.
        {"name": "psd host mixed 100k", "stage": "psd", "rows": 100003},
        # The device-resident PSD filter in a serving loop: a small block of rows ...
        {"name": "psd device n10 4k", "stage": "static", "n": 10, "compress": 5, "order": 50, "paf": 0, "rows": 4099},
        # ... and a large one.
        {"name": "psd device n25 8M", "stage": "static", "n": 25, "compress": 2, "order": 50, "paf": 0,
         "rows": 8000009},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    stage = rng.choice(["gen", "sort", "match", "uncompress", "uncompress", "filter", "psd", "static"])
    if stage == "gen":
        order, compress, paf = rng.choice(GEN)
        return {"stage": stage, "order": order, "compress": compress, "paf": paf, "jobs": rng.randint(2, 40)}
    if stage == "sort":
        order, compress, paf = rng.choice(GEN)
        return {"stage": stage, "order": order, "compress": compress, "paf": paf,
                "records": _log_int(rng, 50, 4000000)}
    if stage == "match":
        order, compress, paf = rng.choice(GEN)
        return {"stage": stage, "order": order, "compress": compress, "paf": paf, "records": _log_int(rng, 200, 60000)}
    if stage == "uncompress":
        order, compress, fine, paf = rng.choice(sorted(UNC))
        top = {50: 400, 45: 7500, 90: 156}[order]
        return {"stage": stage, "order": order, "compress": compress, "fine": fine, "paf": paf,
                "pairs": _log_int(rng, 1 if order != 45 else 20, top)}
    if stage == "filter":
        order, compress, _ = rng.choice(FILTER)
        return {"stage": stage, "order": order, "compress": compress, "pairs": _log_int(rng, 100, 120000)}
    if stage == "psd":
        return {"stage": stage, "rows": _log_int(rng, 100, 200000)}
    n, compress, order, paf, _ = rng.choice(MIX)
    return {"stage": stage, "n": n, "compress": compress, "order": order, "paf": paf,
            "rows": _log_int(rng, 500, 16000000)}


# ---------------------------------------------------------------------------
# inputs


@functools.lru_cache(maxsize=None)
def _ctx():
    """The program's one context."""
    return g.Context(0)


@functools.lru_cache(maxsize=None)
def _level(order, compress, paf):
    """The candidate sets of a level, sorted, and its matched pairs (empty where the level is only generated)."""
    ctx = _ctx()
    a, b, _ = ctx.generate(order, compress, paf)
    a, b = ctx.sort_candidates(a), ctx.sort_candidates(b)
    _, pa, pb, _ = ctx.match(order, compress, paf, a, b)
    return a, b, pa, pb


def _rng(seed):
    return np.random.default_rng(int(seed))


def _ptr(a, t):
    return a.ctypes.data_as(ctypes.POINTER(t))


def _cands_buf(cap, n):
    return np.zeros((cap, n), np.int8), np.zeros((cap, n // 2), np.uint8)


def _cands(words, keys, count):
    return g.GpCands(words.shape[1], keys.shape[1], count, words.shape[0], _ptr(words, ctypes.c_int8),
                     _ptr(keys, ctypes.c_uint8))


def _pairs(a, b, count):
    return g.GpPairs(a.shape[1], count, a.shape[0], _ptr(a, ctypes.c_int8), _ptr(b, ctypes.c_int8))


def _images(rng, n, letters, pairs, alt):
    """Pairs of length n as a finished search leaves them: about 15 members of each equivalence class."""
    base = max(1, pairs // 15)
    ba, bb = (rng.choice(np.array(letters, np.int8), size=(base, n)) for _ in range(2))
    pick = rng.integers(0, base, size=pairs)
    units = np.array([u for u in range(1, n) if math.gcd(u, n) == 1])
    u, e = rng.choice(units, size=pairs), rng.choice([1, -1], size=pairs)
    i = np.arange(n)
    rows = np.arange(pairs)[:, None]
    a = ba[pick][rows, (u[:, None] * i + rng.integers(0, n, size=(pairs, 1))) % n]
    b = bb[pick][rows, (e[:, None] * u[:, None] * i + rng.integers(0, n, size=(pairs, 1))) % n]
    if alt:
        flip = rng.integers(0, 2, size=(pairs, 1)) * (i % 2)
        a = np.where(flip, -a, a) * rng.choice(np.array([1, -1], np.int8), size=(pairs, 1))
        b = np.where(flip, -b, b) * rng.choice(np.array([1, -1], np.int8), size=(pairs, 1))
    swap = rng.integers(0, 2, size=(pairs, 1)) == 1
    return (np.ascontiguousarray(np.where(swap, b, a), dtype=np.int8),
            np.ascontiguousarray(np.where(swap, a, b), dtype=np.int8))


def _mixed_rows(seed, rows):
    rng = _rng(seed)
    share = np.array([m[4] for m in MIX], float)
    kind = rng.choice(len(MIX), size=rows, p=share / share.sum())
    words = np.zeros((rows, 32), np.int8)
    for k, (n, c, _, _, _) in enumerate(MIX):
        at = np.flatnonzero(kind == k)
        words[at, :n] = -c + 2 * rng.integers(0, c + 1, size=(len(at), n))
    lens, orders, pafs = (np.array([m[j] for m in MIX], np.int32)[kind] for j in (0, 2, 3))
    return words, lens, orders, pafs


def prepare(case, seed):
    ctx, stage = _ctx(), case["stage"]
    s = dict(case, ctx=ctx)
    if stage == "gen":
        # job seed mod jobs of the level; room for the whole level
        a, b, _, _ = _level(case["order"], case["compress"], case["paf"])
        n = case["order"] // case["compress"]
        s["job"] = seed % case["jobs"]
        s["a"], s["b"] = _cands_buf(len(a) + 1, n), _cands_buf(len(b) + 1, n)
    elif stage == "sort":
        # records of the level's files, repeats among them, in no order
        a, b, _, _ = _level(case["order"], case["compress"], case["paf"])
        rng, m = _rng(seed), case["records"]
        if m <= len(a) + len(b):
            words, keys = np.concatenate([a.words, b.words]), np.concatenate([a.keys, b.keys])
            at = rng.integers(0, len(words), size=m)
            s["in"] = (np.ascontiguousarray(words[at]), np.ascontiguousarray(keys[at]))
        else:  # more records than the level has: random ones of its letters and key range
            n, letters = a.n, np.unique(b.words)
            top = int(max(a.keys.max(initial=1), b.keys.max(initial=1)))
            s["in"] = (rng.choice(letters, size=(m, n)).astype(np.int8),
                       rng.integers(0, top + 1, size=(m, n // 2)).astype(np.uint8))
        s["out"] = tuple(np.zeros_like(x) for x in s["in"])
    elif stage == "match":
        # a subset of the level's sorted A and B files
        a, b, _, _ = _level(case["order"], case["compress"], case["paf"])
        rng = _rng(seed)
        ia, ib = (np.sort(rng.permutation(len(x))[: case["records"]]) for x in (a, b))
        s["a"], s["b"] = g.Cands(a.words[ia], a.keys[ia]), g.Cands(b.words[ib], b.keys[ib])
        cap = 4 * (len(ia) + len(ib)) + 1024
        s["pa"], s["pb"] = (np.zeros((cap, a.n), np.int8) for _ in range(2))
    elif stage == "uncompress":
        order, fine = case["order"], case["fine"]
        _, _, pa, pb = _level(order, case["compress"], case["paf"])
        at = np.sort(_rng(seed).permutation(len(pa))[: case["pairs"]])
        s["ia"], s["ib"] = np.ascontiguousarray(pa[at]), np.ascontiguousarray(pb[at])
        cap = UNC[order, case["compress"], fine, case["paf"]][2] * len(at) + 4096
        s["pa"], s["pb"] = (np.zeros((cap, order // fine), np.int8) for _ in range(2))
    elif stage == "filter":
        order, compress = case["order"], case["compress"]
        n = order // compress
        letters = next(x for o, c, x in FILTER if (o, c) == (order, compress))
        s["ia"], s["ib"] = _images(_rng(seed), n, letters, case["pairs"], compress == 1 and n % 2 == 0)
        s["pa"], s["pb"] = np.zeros_like(s["ia"]), np.zeros_like(s["ib"])
    elif stage == "psd":
        s["rows"] = _mixed_rows(seed, case["rows"])
    else:  # device rows at the stride the filter takes: 16 bytes per 16 letters
        n, c, m = case["n"], case["compress"], case["rows"]
        gen = torch.Generator(device="cuda").manual_seed(int(seed))
        w = torch.zeros((m, 16 * -(-n // 16)), dtype=torch.int8, device="cuda")
        w[:, :n] = torch.randint(0, c + 1, (m, n), dtype=torch.int8, device="cuda", generator=gen) * 2 - c
        s["words"], s["pass"] = w, torch.zeros(m, dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()  # the filter runs on the context's own stream
    return s


def run(s):
    ctx, lib, stage = s["ctx"], s["ctx"].lib, s["stage"]
    if stage == "gen":
        a, b = _cands(*s["a"], 0), _cands(*s["b"], 0)
        ctx.check(lib.gp_generate(ctx.h, s["order"], s["compress"], s["paf"], s["job"], s["jobs"], ctypes.byref(a),
                                  ctypes.byref(b), None), "gp_generate")
        return {"a": s["a"], "b": s["b"], "count": [a.count, b.count]}
    if stage == "sort":  # in place: the records are loaded into the buffers that are sorted
        for dst, src in zip(s["out"], s["in"]):
            np.copyto(dst, src)
        c = _cands(*s["out"], len(s["in"][0]))
        ctx.check(lib.gp_sort_candidates(ctx.h, ctypes.byref(c)), "gp_sort_candidates")
        return {"records": s["out"], "count": c.count}
    if stage == "match":
        out = _pairs(s["pa"], s["pb"], 0)
        a, b = s["a"].struct(), s["b"].struct()
        ctx.check(lib.gp_match(ctx.h, s["order"], s["compress"], s["paf"], ctypes.byref(a), ctypes.byref(b),
                               ctypes.byref(out), None), "gp_match")
        return {"pairs": (s["pa"], s["pb"]), "count": out.count}
    if stage == "uncompress":
        inp, out = _pairs(s["ia"], s["ib"], len(s["ia"])), _pairs(s["pa"], s["pb"], 0)
        ctx.check(lib.gp_uncompress(ctx.h, s["order"], s["compress"], s["fine"], s["paf"], ctypes.byref(inp),
                                    ctypes.byref(out), None, None, None), "gp_uncompress")
        return {"pairs": (s["pa"], s["pb"]), "count": out.count}
    if stage == "filter":
        inp, out = _pairs(s["ia"], s["ib"], len(s["ia"])), _pairs(s["pa"], s["pb"], 0)
        ctx.check(lib.gp_filter(ctx.h, s["order"], s["compress"], ctypes.byref(inp), ctypes.byref(out), None),
                  "gp_filter")
        return {"pairs": (s["pa"], s["pb"]), "count": out.count}
    if stage == "psd":
        ok, mx, _ = ctx.psd_filter_batch(*s["rows"], want_max=True)
        return {"pass": ok, "max": mx}
    w = s["words"]
    ctx.check(lib.gp_psd_filter_batch_static(ctx.h, w.data_ptr(), w.shape[1], s["n"], s["order"], s["paf"],
                                             w.shape[0], s["pass"].data_ptr(), None), "gp_psd_filter_batch_static")
    return {"pass": s["pass"]}


def work(case):
    """Bytes: records in and out once.  Flops: per word filtered, one complex add per frequency (partial sums of a
    word's prefix are shared between words) and |X|^2."""
    stage = case["stage"]
    if stage == "uncompress":
        key = (case["order"], case["compress"], case["fine"], case["paf"])
        n = case["order"] // case["fine"]
        pairs = min(case["pairs"], UNC[key][0])
        return {"bytes": 2.0 * pairs * (case["order"] // case["compress"]) + 2.0 * pairs * n,
                "flops": pairs * UNC[key][1] * 5 * (n // 2)}
    if stage == "static":
        return {"bytes": case["rows"] * (case["n"] + 1.0), "flops": case["rows"] * 4.0 * case["n"] * (case["n"] // 2)}
    if stage == "psd":
        share = sum(m[4] for m in MIX)
        n = sum(m[0] * m[4] for m in MIX) / share
        return {"bytes": case["rows"] * (n + 12 + 5), "flops": case["rows"] * 2.0 * n * n}
    n = case["order"] // case["compress"]
    if stage == "filter":
        units = sum(math.gcd(u, n) == 1 for u in range(1, n))
        images = 2 * units * (4 if case["compress"] == 1 and n % 2 == 0 else 1)
        return {"bytes": case["pairs"] * 2.0 * n * (1 + 1 / 15), "flops": case["pairs"] * 2.0 * images * n}
    if stage == "gen":  # the words of fixed row sum that start with their least letter: about 1 / n of the sum's
        k = case["compress"] + 1
        words = k ** n / math.sqrt(2 * math.pi * n * (k * k - 1) / 12) * 2
        return {"bytes": words / n / case["jobs"] * 0.02 * (n + n // 2), "flops": words * n / case["jobs"]}
    if stage == "sort":
        return {"bytes": case["records"] * 2.0 * (n + n // 2), "flops": 0}
    return {"bytes": 2.0 * case["records"] * (n + n // 2), "flops": 0}  # match


def exact(case, seed):
    """The PSD maxima in 64 bits; every other output is whole numbers."""
    if case["stage"] != "psd":
        return None
    words, lens, _, _ = _mixed_rows(seed, case["rows"])
    mx = np.zeros(len(words))
    for n in np.unique(lens):
        at = np.flatnonzero(lens == n)
        f = np.fft.fft(words[at, :n].astype(np.float64), axis=1)[:, 1: n // 2 + 1]
        mx[at] = (f.real ** 2 + f.imag ** 2).max(axis=1)
    return {"pass": None, "max": mx}
