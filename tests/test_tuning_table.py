"""The committed tuning table (golaypair_amd/tuning.tsv, written by
python -m golaypair_amd.autotune) is well formed: "key value" lines with the
keys the library reads (golaypair_amd/csrc/tuning.hip)."""
import os
import re

import golaypair_amd as g

TABLE = os.path.join(os.path.dirname(g.__file__), "tuning.tsv")
KEYS = [r"unc_waves/\d+", r"unc_leaf_budget/\d+", r"unc_counter_rounds/\d+", r"unc_counter_streams/\d+", r"gen_ranks_per_lane/\d+/\d+"]


def test_tuning_table_format():
    assert os.path.exists(TABLE)
    entries = 0
    for line in open(TABLE):
        line = line.split("#", 1)[0].strip()
        if not line:
            continue
        key, value = line.split()
        assert any(re.fullmatch(p, key) for p in KEYS), key
        assert int(value) >= 0 if key.startswith("unc_counter_rounds/") else int(value) > 0
        entries += 1
    head = open(TABLE).read()
    assert "golaypair_amd.autotune" in head


def test_tuning_choice_is_beyond_the_noise():
    """A candidate is kept only where its runs lie below the default's, not where a few do."""
    from golaypair_amd.autotune import choose
    noisy = [5.37, 5.22, 5.45, 5.31, 5.08, 5.57, 5.40, 5.28]
    assert choose({None: noisy, 2: [4.99, 5.45, 5.36, 5.30, 5.50, 5.21, 5.33, 5.41]}) is None
    assert choose({None: noisy, 2: [x - 0.02 for x in noisy], 4: [x + 0.1 for x in noisy]}) is None
    assert choose({None: noisy, 2: [4.99, 5.45, 5.36, 5.30, 5.50, 5.21, 5.33, 5.41], 3: [4.7] * 7 + [5.9]}) == 3
    assert choose({None: [5.30, 5.31, 5.30, 5.32], 2: [5.27, 5.28, 5.27, 5.28]}) is None
    assert choose({None: noisy}) is None
