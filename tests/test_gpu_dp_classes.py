"""The affine DP classes in one launch against the oracle: query lengths at the
edges of every row class and of a pass, few and many tasks per class (one and
several rounds per queue claim), traced and score-only, with the re-run of a
saturated task."""
import numpy as np
import pytest

from helpers import oracle_params, pairs_of, rand_seq, seqset
from oracle import oracle as orc
from pastis_amd.aligner import Aligner, config_for_cli

pytestmark = pytest.mark.gpu

LENGTHS = [1, 2, 16, 17, 127, 128, 129, 255, 256, 257, 511, 512, 513, 1023,
           1025]


# the last: more than 4 rounds of 8 tasks for every wave (claims of several)
@pytest.mark.parametrize("longest,reps", [(1025, 1), (1025, 120), (129, 8300)])
def test_local_classes(longest, reps):
    rng = np.random.default_rng(6)
    base = rand_seq(rng, 7000)
    lens = [n for n in LENGTHS if n <= longest]
    n = len(lens)
    seqs = [base[i * 31:i * 31 + m].copy() for i, m in enumerate(lens)]
    seqs += [base, base.copy()]   # 7,000 equal residues leave int16
    codes, offs = seqset(seqs)
    rc = [(r, c) for r in range(n) for c in range(n)]
    pairs = pairs_of(rc + [(n, n + 1)], [[0, 0, 0, 0]] * (len(rc) + 1))
    many = np.concatenate([np.tile(pairs[:-1], reps), pairs[-1:]])
    ref = orc.sfa_batch(codes, offs, pairs["r"], pairs["c"],
                        oracle_params("as_documented"))
    al = Aligner(config_for_cli(-11, -2, 6, 0, 2, "as_documented"))
    al.load_seqs(codes, offs)
    print("classes", longest, reps, flush=True)
    got = al.align(many)

    def wanted(x):
        x = x.astype(np.int64)
        return np.concatenate([np.tile(x[:-1], reps), x[-1:]])

    for f in ("score", "matches", "cols", "gap_opens"):
        bad = np.nonzero(got[f].astype(np.int64) != wanted(ref[f]))[0]
        assert bad.size == 0, (f, int(bad[0]), got[bad[0]])
    assert al.stats()["rerun_pairs"] == 1
    names = [k["name"] for k in al.kernel_stats()]
    assert "swt.all.r8.i16" in names and "swt.all.r8.i32" in names
    sc = al.sw_scores(many)
    assert np.array_equal(sc["score"].astype(np.int64), wanted(ref["score"]))
    al.close()
