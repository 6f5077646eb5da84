"""GPU gen / sort / match vs the oracle, byte-exact on the file text.

gen: generate_hybrid.cpp:107-163 (A/B candidate files in FKM order)
sort: sort.cpp:7-23 under LC_ALL=C (+ uniq)
match: match_pairs.cpp:15-121 (pair lines in emission order)
"""
import hashlib
import json
import os

import numpy as np
import pytest

import golaypair_amd as g
from tests import _device, _oracle

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(__file__), "golden")


def _text(lines):
    return "".join(l + "\n" for l in lines)


SMALL = [  # (order, compress, paf, job, njobs): oracle runs in < ~10 s
    (8, 1, 0, 0, 1),
    (10, 1, 0, 0, 1),
    (16, 2, 0, 0, 1),
    (16, 1, 0, 0, 1),
    (26, 2, 0, 0, 1),
    (26, 2, 0, 1, 3),
    (26, 2, 0, 2, 3),
    (20, 2, 0, 0, 1),
    (18, 3, -2, 0, 1),
    (50, 5, 0, 0, 1),
    (34, 2, 0, 0, 1),
]


@pytest.mark.parametrize("order,compress,paf,job,njobs", SMALL)
def test_gen_matches_oracle(gpu_ctx, order, compress, paf, job, njobs):
    rc, ta, tb, _ = _oracle.generate(order, compress, paf, job, njobs)
    a, b, st = gpu_ctx.generate(order, compress, paf, job, njobs)
    if rc == 1:
        assert a is None
        return
    assert _text(a.lines()) == ta
    assert _text(b.lines()) == tb
    assert st.tie_band == 0


def test_gen_no_decomposition(gpu_ctx):
    # 2*7 = 14 is not a sum of two squares: the reference prints and returns 1
    a, b, st = gpu_ctx.generate(7, 1, 0)
    assert a is None and b is None


@pytest.mark.parametrize("order,compress,paf", [(16, 2, 0), (26, 2, 0), (50, 5, 0), (34, 2, 0)])
def test_sort_and_match_match_oracle(gpu_ctx, order, compress, paf):
    rc, ta, tb, _ = _oracle.generate(order, compress, paf)
    a, b, _ = gpu_ctx.generate(order, compress, paf)
    sa = gpu_ctx.sort_candidates(a)
    sb = gpu_ctx.sort_candidates(b)
    ref_sa = sorted(set(ta.splitlines()))
    ref_sb = sorted(set(tb.splitlines()))
    assert sa.lines() == ref_sa
    assert sb.lines() == ref_sb
    rc, pa, pb, st = gpu_ctx.match(order, compress, paf, sa, sb)
    got = _text(g.pair_line(x, y) for x, y in zip(pa, pb))
    ref = _oracle_match(order, compress, paf, _text(ref_sa), _text(ref_sb))
    assert got == ref
    assert st.pairs == len(pa)


def _oracle_match(order, compress, paf, ta, tb):
    import subprocess
    import tempfile
    with tempfile.TemporaryDirectory() as d:
        wd = os.path.join(d, "order-%d" % order)
        os.makedirs(wd)
        open(os.path.join(wd, "%d-filtered_sorted-a" % order), "w").write(ta)
        open(os.path.join(wd, "%d-filtered_sorted-b" % order), "w").write(tb)
        subprocess.run([_oracle.CLI, str(order), "-c", str(compress), "--paf", str(paf), "-d", d, "match"],
                       check=True, capture_output=True)
        return open(os.path.join(wd, "%d-pairs-%d" % (order, compress))).read()


def test_match_empty_input_returns_1(gpu_ctx):
    a, b, _ = gpu_ctx.generate(16, 2, 0)
    empty = g.Cands(np.zeros((0, 8), np.int8), np.zeros((0, 4), np.uint8))
    rc, pa, pb, st = gpu_ctx.match(16, 2, 0, empty, b)
    assert rc == g.GP_NO_INPUT and len(pa) == 0


def test_psd_keys_match_oracle_lines(gpu_ctx):
    rc, ta, tb, _ = _oracle.generate(26, 2, 0)
    for text, inv in ((ta, False), (tb, True)):
        lines = text.splitlines()
        words = np.array([[int(t) for t in l.split()[1:]] for l in lines], np.int8)
        keys = gpu_ctx.psd_keys(words, 52, inv)
        assert [g.cand_line(w, k) for w, k in zip(words, keys)] == lines


@pytest.mark.parametrize("count", [524287, 524288, 1048577, 1300001])
def test_psd_keys_of_large_buffers(gpu_ctx, count):
    """Caller buffers on both sides of the size from which copies go through pinned
    memory in chunks (8 MiB: 524288 words, the keys of 1048576), against small calls."""
    rng = np.random.default_rng(count)
    words = rng.choice(np.array([-1, 1], np.int8), size=(count, 16))
    words[:, 0] = 0  # every PSD below 256
    got = gpu_ctx.psd_keys(words, 255, False)
    want = np.concatenate([gpu_ctx.psd_keys(words[i:i + 100000], 255, False) for i in range(0, count, 100000)])
    assert (got == want).all()


def _golden(name):
    p = os.path.join(GOLDEN, name)
    if not os.path.exists(p):
        pytest.skip("golden fixture %s not generated" % name)
    return json.load(open(p))


@pytest.mark.parametrize("fixture", ["gen_v45_c3_paf-2.json", "gen_v90_c10.json"])
def test_gen_large_matches_golden_digest(gpu_ctx, fixture):
    fx = _golden(fixture)
    a, b, st = gpu_ctx.generate(fx["order"], fx["compress"], fx["paf"])
    for side, c in (("a", a), ("b", b)):
        text = _text(c.lines())
        assert len(c) == fx[side]["lines"]
        assert hashlib.sha256(text.encode()).hexdigest() == fx[side]["sha256"]
    assert st.tie_band == 0


@pytest.mark.parametrize("n,ma,mb,nkeys", [(6, 300, 300, 4), (8, 1, 700, 1), (18, 257, 64, 3), (21, 90, 1000, 2)])
def test_match_many_equal_keys(gpu_ctx, n, ma, mb, nkeys):
    """Long chains of B records with equal keys (more candidate pairs than the first
    list holds), shifts beyond one per lane, few records on either side."""
    rng = np.random.default_rng(n)
    wa = rng.choice([-1, 1], size=(ma, n)).astype(np.int8)
    wb = rng.choice([-1, 1], size=(mb, n)).astype(np.int8)
    wb[: min(ma, mb) // 2] = wa[: min(ma, mb) // 2]
    kinds = rng.integers(0, 256, size=(nkeys, n // 2)).astype(np.uint8)
    xa, xb = rng.integers(0, nkeys, ma), rng.integers(0, nkeys, mb)
    target = 2 * int(wa[0].astype(int) @ np.roll(wa[0], 1)) if n == 6 else 4
    paf = lambda w: np.stack([(w.astype(int) * np.roll(w, -s, axis=1)).sum(1) for s in range(1, n // 2 + 1)], 1)
    fa, fb = paf(wa), paf(wb)
    want = [(i, j) for i in range(ma) for j in range(mb) if xa[i] == xb[j] and (fa[i] + fb[j] == target).all()]
    rc, pa, pb, st = gpu_ctx.match(n, 1, target, g.Cands(wa, kinds[xa]), g.Cands(wb, kinds[xb]))
    assert st.pair_checks == int((xa[:, None] == xb[None, :]).sum())
    assert [(x.tolist(), y.tolist()) for x, y in zip(pa, pb)] == [(wa[i].tolist(), wb[j].tolist()) for i, j in want]


@pytest.mark.parametrize("order,compress,paf,njobs", [
    (8, 2, 0, 1), (26, 1, 0, 1), (26, 2, 0, 7), (34, 2, 0, 5), (45, 3, -2, 40), (50, 5, 0, 3), (50, 5, 0, 1000),
])
def test_gen_jobs_and_word_widths(gpu_ctx, order, compress, paf, njobs):
    """The shards of a level together are the level (each is the level where the job
    split has no prefix length), and the 2-bit and 4-bit packed words agree (the FP32
    path packs every level in 4 bits)."""
    rows = lambda c: sorted(c.lines())
    a, b, _ = gpu_ctx.generate(order, compress, paf)
    gpu_ctx.set_mode(g.GP_PSD_FP32)
    try:
        fa, fb, _ = gpu_ctx.generate(order, compress, paf)
        ja, jb, _ = gpu_ctx.generate(order, compress, paf, njobs - 1, njobs)
    finally:
        gpu_ctx.set_mode(g.GP_PSD_SPLIT_BF16)
    assert fa.lines() == a.lines() and fb.lines() == b.lines()
    parts = [gpu_ctx.generate(order, compress, paf, j, njobs)[:2] for j in range(min(njobs, 40))]
    if njobs <= 40:
        assert ja.lines() == parts[-1][0].lines() and jb.lines() == parts[-1][1].lines()
    if all(p[0].lines() == a.lines() and p[1].lines() == b.lines() for p in parts):
        return
    assert njobs <= 40
    assert sorted(sum((p[0].lines() for p in parts), [])) == rows(a)
    assert sorted(sum((p[1].lines() for p in parts), [])) == rows(b)


def test_gen_wide_words(gpu_ctx):
    """Words of more than 64 bits (17 letters of an alphabet of 5): one shard of many."""
    a, b, _ = gpu_ctx.generate(68, 4, 0, 7, 1000)
    gpu_ctx.set_mode(g.GP_PSD_FP32)
    try:
        fa, fb, _ = gpu_ctx.generate(68, 4, 0, 7, 1000)
    finally:
        gpu_ctx.set_mode(g.GP_PSD_SPLIT_BF16)
    assert len(a) + len(b) > 0 and a.lines() == fa.lines() and b.lines() == fb.lines()


def test_match_chain_of_equal_keys_beside_other_records(gpu_ctx):
    """2^16 B records of one key: A records of other keys do not walk them all."""
    rng, n, m = np.random.default_rng(3), 16, 1 << 16
    wa, wb = (rng.choice([-1, 1], size=(m, n)).astype(np.int8) for _ in range(2))
    ka = rng.integers(0, 256, size=(m, n // 2)).astype(np.uint8)
    one, other = np.repeat(ka[:1] ^ 255, m, 0), rng.integers(0, 256, size=(m, n // 2)).astype(np.uint8)
    ms = []
    for kb in (other, one):
        runs = [gpu_ctx.match(n, 1, 0, g.Cands(wa, ka), g.Cands(wb, kb))[3] for _ in range(4)]
        assert all(r.pair_checks == 0 for r in runs)
        ms.append(min(r.kernel_ms for r in runs[1:]))
    assert ms[1] < 8 * ms[0]


def test_match_many_candidates_few_pairs(gpu_ctx):
    """20000 x 20000 records of one key: 4e8 candidate pairs are checked without a
    list of them all."""
    rng, n, m = np.random.default_rng(4), 12, 20000
    wa, wb = (rng.choice([-1, 1], size=(m, n)).astype(np.int8) for _ in range(2))
    k = np.full((m, n // 2), 9, np.uint8)
    paf = lambda w: np.stack([(w.astype(int) * np.roll(w, -s, axis=1)).sum(1) for s in range(1, n // 2 + 1)], 1)
    fa, fb = paf(wa), paf(wb)
    target = 24
    by = {}
    for j, f in enumerate(map(tuple, fb)):
        by.setdefault(f, []).append(j)
    want = [(i, j) for i in range(m) for j in by.get(tuple(target - fa[i]), [])]
    assert 0 < len(want) < 100000
    (rc, pa, pb, st), held = _device.held_by(lambda ctx: ctx.match(n, 1, target, g.Cands(wa, k), g.Cands(wb, k)))
    assert st.pair_checks == m * m
    assert (pa == wa[[i for i, _ in want]]).all() and (pb == wb[[j for _, j in want]]).all() and len(pa) == len(want)
    assert held < 1 << 28


@pytest.mark.parametrize("order,compress,paf", [(212, 7, 372), (208, 7, 195)])
def test_gen_refuses_levels_beyond_64_bits(gpu_ctx, order, compress, paf):
    """Levels whose row sums each have fewer than 2^62 words, but together more than 2^63."""
    with pytest.raises(g.GolayError, match="search space too large"):
        gpu_ctx.generate(order, compress, paf, 0, 5)


@pytest.mark.parametrize("mode", [g.GP_PSD_SPLIT_BF16, g.GP_PSD_FP32])
def test_gen_device_times(gpu_ctx, mode):
    """psd_kernel_ms is the time of the kernel with the PSD filter, kernel_ms that of all."""
    gpu_ctx.set_mode(mode)
    try:
        st = gpu_ctx.generate(45, 3, -2, 1, 8)[2]
    finally:
        gpu_ctx.set_mode(g.GP_PSD_SPLIT_BF16)
    assert 0 < st.psd_kernel_ms < st.kernel_ms and st.psd_launches == 1


def _splits(n, k, njobs):
    """Whether njobs jobs share the necklaces of length n (lyndon.cpp:87-106): some prefix
    shorter than the words has 10^4 necklaces per job."""
    count = lambda i: sum(k ** int(np.gcd(i, j)) for j in range(1, i + 1)) // i
    return njobs > 1 and any(count(i) >= 10000 * njobs for i in range(1, n))


@pytest.mark.parametrize("order,compress,paf,njobs,split", [
    (8, 2, 0, 3, False), (26, 2, 0, 7, False), (26, 1, 0, 2, True), (26, 1, 0, 40, True), (34, 2, 0, 5, True),
    (34, 2, 0, 40, True), (45, 3, -2, 8, True), (45, 3, -2, 40, True), (50, 5, 0, 3, True), (50, 5, 0, 200, False),
])
def test_gen_job_split(gpu_ctx, order, compress, paf, njobs, split):
    """Where the level is split, its jobs' records are disjoint and together the level's;
    where it is not, every job has them all."""
    assert _splits(order // compress, compress + 1, njobs) == split
    a, b, _ = gpu_ctx.generate(order, compress, paf)
    parts = [gpu_ctx.generate(order, compress, paf, j, njobs)[:2] for j in range(min(njobs, 40))]
    for side, level in ((0, a.lines()), (1, b.lines())):
        jobs = [p[side].lines() for p in parts]
        if split:
            assert sorted(sum(jobs, [])) == sorted(level) and len(set(level)) == len(level) > 0
            assert len(level) < 100 or max(map(len, jobs)) < len(level)
        else:
            assert all(j == level for j in jobs)
