"""Batches large enough (more than 65,536 X-drop work items) for the split by
reach: items of 512 residues and more with 16 lanes each beside the sorted
rest with one lane each.  The same pairs in a small batch run with 16 lanes
per item (where the bands fit) and are compared with the oracle; every copy in
the large batch must give the same bytes, at X-drop values and gaps on both
sides of the rule and of the per-lane kernel's cell encodings."""
import numpy as np
import pytest

from helpers import rand_seq, seqset, small_config2
from oracle import oracle as orc
from pastis_amd._lib import PAIR_DTYPE
from pastis_amd.aligner import Aligner, config_for_cli

pytestmark = pytest.mark.gpu


def _workload():
    w = small_config2(n_pairs=500)
    rng = np.random.default_rng(8)
    o = w.offsets.astype(np.int64)
    seqs = [w.codes[o[i]:o[i + 1]] for i in range(len(o) - 1)]
    n0 = len(seqs)
    # homologs with segments on both sides of 512 residues
    extra = []
    for n in (511, 512, 513, 1030, 1500):
        s = rand_seq(rng, n + 6)
        t = s.copy()
        m = rng.random(len(t)) < 0.1
        m[:6] = m[-6:] = False
        t[m] = rng.integers(0, 20, int(m.sum()))
        a = len(seqs)
        seqs += [s, t]
        extra += [(a, a + 1, 0), (a, a + 1, n), (a + 1, a, 0)]
    pairs = np.concatenate([w.pairs, np.zeros(len(extra), PAIR_DTYPE)])
    for k, (r, c, p) in enumerate(extra):
        pairs[len(w.pairs) + k] = (r, c, 2, 0, (p, p, 0, 0))
    assert n0 + 10 == len(seqs)
    codes, offs = seqset(seqs)
    return codes, offs, pairs


@pytest.mark.parametrize("X,gap", [(49, -11), (49, -32), (49, -33),
                                   (160, -32), (161, -33), (49, -1000),
                                   (49, -1001), (65, -11), (66, -11),
                                   (49, -2)])
def test_large_batch_equals_small(X, gap):
    codes, offs, pairs = _workload()
    cfg = config_for_cli(xdrop=X)
    cfg.xdrop_gap = gap
    al = Aligner(cfg)
    al.load_seqs(codes, offs)
    print("X-drop split", X, gap, flush=True)
    small = al.align(pairs)
    ref = orc.sxa_batch(codes, offs, pairs["r"], pairs["c"], pairs["seed"],
                        orc.params(-2, -11, gap, X, 6, 2))
    for f in ("score", "matches", "cols", "gap_opens"):
        assert np.array_equal(small[f].astype(np.int64),
                              ref[f].astype(np.int64)), f
    cells = int(ref["ext"]["cells"].sum())
    assert al.stats()["xdrop_cells"] == cells
    reps = 65536 // (4 * len(pairs)) + 2
    order = np.random.default_rng(1).permutation(np.tile(np.arange(len(pairs)),
                                                         reps))
    al.reset_stats()
    big = al.align(pairs[order])
    assert np.array_equal(big.view(np.uint8).reshape(len(big), -1),
                          small[order].view(np.uint8).reshape(len(big), -1))
    assert al.stats()["xdrop_cells"] == reps * cells
    al.close()
