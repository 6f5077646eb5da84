"""Device sort + uniq of candidate records (gp_sort_candidates, the GNU_sort seam:
src/core/sort/sort.cpp:7-23 run as `LC_ALL=C sort | uniq` on the lines of
src/utils/io.cpp:14-36).  The sorted records, written as text, must be the
byte-ordered unique lines: against Python's code-point order on ASCII text (the
C locale's byte order) for random record sets, and against coreutils itself on
the gen files."""
import os
import subprocess
import tempfile
import time

import numpy as np
import pytest

import golaypair_amd as g
from tests import _oracle

pytestmark = pytest.mark.gpu


def _random_records(rng, m, n, letters, key_values):
    words = rng.choice(letters, size=(m, n)).astype(np.int8)
    keys = rng.choice(key_values, size=(m, n // 2)).astype(np.uint8)
    if m > 4:  # duplicates: copies of earlier rows, and rows equal but for one key digit
        dup = rng.integers(0, m, size=m // 4)
        words[rng.integers(0, m, size=m // 4)] = words[dup]
        keys[rng.integers(0, m, size=m // 4)] = keys[dup]
    return g.Cands(words, keys)


@pytest.mark.parametrize("n,m,letters,key_values", [
    (2, 50, [-1, 1], [0, 1, 2, 10]),
    (3, 1, [-1, 1], [5]),
    (8, 3000, [-2, 0, 2], list(range(0, 40))),
    (15, 60000, [-3, -1, 1, 3], list(range(0, 93))),                    # 15 radix blocks of 4096
    (18, 20000, list(range(-10, 11, 2)), [0, 1, 9, 10, 11, 99, 100, 101, 180, 255]),
    (25, 5000, list(range(-20, 21, 2)), list(range(0, 256))),           # 21 letters: 5-bit symbols
    (45, 8000, [-1, 1], [1, 12, 2, 23, 3, 123, 31, 231]),               # key texts that collide as prefixes
    (50, 30000, [-1, 1], list(range(0, 101))),
    (64, 2000, [-128, -100, -7, 0, 7, 100, 127], [0, 255, 100, 99, 9, 10]),
])
def test_sort_random_records_byte_order(gpu_ctx, n, m, letters, key_values):
    rng = np.random.default_rng(n * 1000 + m)
    c = _random_records(rng, m, n, letters, key_values)
    want = sorted(set(c.lines()))
    got = gpu_ctx.sort_candidates(c)
    assert got.lines() == want


def test_sort_empty_and_all_equal(gpu_ctx):
    e = g.Cands(np.zeros((0, 10), np.int8), np.zeros((0, 5), np.uint8))
    assert len(gpu_ctx.sort_candidates(e)) == 0
    w = np.tile(np.array([[1, -1, 1, 1, -1, 1, -1, -1, 1, 1]], np.int8), (9000, 1))
    k = np.tile(np.array([[3, 14, 15, 92, 65]], np.uint8), (9000, 1))
    got = gpu_ctx.sort_candidates(g.Cands(w, k))
    assert len(got) == 1 and got.lines() == [g.cand_line(w[0], k[0])]


@pytest.mark.parametrize("order,compress,paf", [(26, 2, 0), (34, 2, 0), (45, 3, -2), (50, 5, 0)])
def test_sort_gen_files_equal_coreutils(gpu_ctx, order, compress, paf):
    """The GPU's gen candidates, shuffled and duplicated, sorted on the GPU: the same
    lines as coreutils `sort | uniq` with LC_ALL=C on the oracle's gen files."""
    with tempfile.TemporaryDirectory() as d:
        subprocess.run([_oracle.CLI, "-d", d, str(order), "-c", str(compress), "--paf", str(paf), "gen"], check=True,
                       capture_output=True)
        wd = os.path.join(d, "order-%d" % order)
        a, b, _ = gpu_ctx.generate(order, compress, paf)
        rng = np.random.default_rng(order)
        for side, cands in (("a", a), ("b", b)):
            path = os.path.join(wd, "%d-filtered-%s#0" % (order, side))
            env = dict(os.environ, LC_ALL="C")
            ref = subprocess.run("sort %s | uniq" % path, shell=True, check=True, capture_output=True, env=env,
                                 text=True).stdout
            perm = rng.permutation(np.concatenate([np.arange(len(cands)), rng.integers(0, len(cands), 100)]))
            mixed = g.Cands(cands.words[perm], cands.keys[perm])
            got = gpu_ctx.sort_candidates(mixed)
            assert "".join(l + "\n" for l in got.lines()) == ref, side


@pytest.mark.parametrize("m", [2047, 2048, 2049, 4097, 10241])
@pytest.mark.parametrize("key_values", [[7], [7, 70, 77]])
def test_sort_runs_and_ties(gpu_ctx, m, key_values):
    """Record counts around the runs of 2048 and their merges, with keys whose first
    words are mostly equal, so that the other words decide."""
    rng = np.random.default_rng(m)
    c = _random_records(rng, m, 15, [-3, -1, 1, 3], key_values)
    assert gpu_ctx.sort_candidates(c).lines() == sorted(set(c.lines()))


@pytest.mark.parametrize("m", [2050, 3073, 32768, 32769, 49153, 65536, 65537])
@pytest.mark.parametrize("key_values", [[7], list(range(0, 93))])
def test_sort_ranked_runs(gpu_ctx, m, key_values):
    """Record counts around the sizes up to which runs are ranked all at once (2^15:
    32 runs of 1024; 2^16: 16 runs and merges), with distinct and equal first words."""
    c = _random_records(np.random.default_rng(m), m, 15, [-3, -1, 1, 3], key_values)
    assert gpu_ctx.sort_candidates(c).lines() == sorted(set(c.lines()))


@pytest.mark.parametrize("letters", [[3], [-1, 1], [-2, 0, 2], [-128, 127, 5, 33, -33], list(range(-128, 128))])
@pytest.mark.parametrize("kind", ["keys", "all but one", "words", "all"])
@pytest.mark.parametrize("n,m", [(2, 300), (15, 5000), (37, 3000)])
def test_sort_shared_digits_and_letters(gpu_ctx, n, m, kind, letters):
    """Records that share their keys (but for the last one), their words or both, over
    letters of 1 to 8 bits."""
    rng = np.random.default_rng(n + len(letters))
    words = rng.choice(letters, size=(m, n)).astype(np.int8)
    keys = rng.choice([0, 7, 12, 123, 255], size=(m, n // 2)).astype(np.uint8)
    if kind != "words":
        keys[:m - (kind == "all but one")] = keys[0]
    if kind in ("words", "all"):
        words[:] = words[0]
    c = g.Cands(words, keys)
    assert gpu_ctx.sort_candidates(c).lines() == sorted(set(c.lines()))


@pytest.mark.parametrize("n,m", [(50, 61000), (25, 400000)])
def test_sort_repeats_cost_no_more_than_distinct_records(gpu_ctx, n, m):
    """Records that share their first digits, or all of them, sort no slower than
    records without ties."""
    rng = np.random.default_rng(n)
    words = rng.choice(np.array([-3, -1, 1, 3], np.int8), size=(m, n))
    keys = rng.integers(0, 100, size=(m, n // 2)).astype(np.uint8)
    best = {}
    for kind, (w, k) in {"distinct": (words, keys), "same keys": (words, np.repeat(keys[:1], m, 0)),
                         "same": (np.repeat(words[:1], m, 0), np.repeat(keys[:1], m, 0))}.items():
        c = g.Cands(w.copy(), k.copy())
        for _ in range(6):
            np.copyto(c.words, w)
            np.copyto(c.keys, k)
            s = c.struct()
            t0 = time.perf_counter()
            gpu_ctx.check(gpu_ctx.lib.gp_sort_candidates(gpu_ctx.h, g.ctypes.byref(s)), "gp_sort_candidates")
            best[kind] = min(best.get(kind, 1e9), time.perf_counter() - t0)
        assert s.count == (1 if kind == "same" else m)
    assert best["same"] < best["distinct"] and best["same keys"] < 1.3 * best["distinct"], best
