"""Row edges beyond a pass of their class with the default affine shapes:
tasks of several passes in a lower class beside those of the last class, whose
boundary rows must not be shared, against the oracle."""
import numpy as np
import pytest

from helpers import oracle_params, pairs_of, rand_seq, seqset
from oracle import oracle as orc
from pastis_amd.aligner import Aligner, config_for_cli

pytestmark = pytest.mark.gpu

ROWS = [257, 300, 384, 385, 513, 600, 767, 768, 769, 1025, 1100, 1500, 2049]


@pytest.mark.parametrize("edges", [(128, 256, 768), (128, 384, 768),
                                   (200, 300, 600)])
def test_edges_beyond_a_pass(edges):
    rng = np.random.default_rng(8)
    base = rand_seq(rng, 2200)
    # homologous rows of every length, short columns cut from the same base
    seqs = [base[(7 * i):(7 * i) + m].copy() for i, m in enumerate(ROWS)]
    nr = len(seqs)
    seqs += [base[97 * i:97 * i + 60 + 9 * i].copy() for i in range(12)]
    codes, offs = seqset(seqs)
    rc = [(r, nr + c) for r in range(nr) for c in range(12)]
    pairs = pairs_of(rc, [[20, 20, 30, 30]] * len(rc))
    reps = 40
    many = np.tile(pairs, reps)
    p = oracle_params("as_documented")
    for mode in ("sfa", "sxa"):
        al = Aligner(config_for_cli(-11, -2, 6, 49 if mode == "sxa" else 0, 2,
                                    "as_documented"))
        al.load_seqs(codes, offs)
        al.set_tuning(dp_edge=list(edges), dp_shape=[5, 1, 4, 3])
        print("edges", edges, mode, flush=True)
        got = al.align(many)
        if mode == "sfa":
            ref = orc.sfa_batch(codes, offs, pairs["r"], pairs["c"], p)
        else:
            ref = orc.sxa_batch(codes, offs, pairs["r"], pairs["c"],
                                pairs["seed"], p)
        for f in ("score", "matches", "cols", "gap_opens"):
            want = np.tile(ref[f].astype(np.int64), reps)
            bad = np.nonzero(got[f].astype(np.int64) != want)[0]
            assert bad.size == 0, (f, int(bad[0]), got[bad[0]])
        if mode == "sfa":
            sc = al.sw_scores(many)["score"].astype(np.int64)
            assert np.array_equal(sc, np.tile(ref["score"].astype(np.int64),
                                              reps))
            assert not any(".all." in k["name"] for k in al.kernel_stats())
        al.close()
