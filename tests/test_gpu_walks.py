"""Tracebacks through gap runs of every length around a window of the walk (16
residues, two segments of eight steps), in either sequence, at several rows of
a lane, against the oracle: local and global, linear and affine gaps, staged
or not."""
import numpy as np
import pytest

from helpers import oracle_params, pairs_of, rand_seq, seqset
from oracle import oracle as orc
from pastis_amd.aligner import Aligner, config_for_cli

pytestmark = pytest.mark.gpu

GAPS = [1, 2, 7, 8, 9, 15, 16, 17, 31, 32, 33, 70]


def gapped(seed):
    rng = np.random.default_rng(seed)
    a = rand_seq(rng, 700)
    seqs, rc = [a], []
    for g in GAPS:
        for at in (200, 333, 350):   # cut out of, or inserted into, a copy
            seqs.append(np.concatenate([a[:at], a[at + g:]]))
            seqs.append(np.concatenate([a[:at], rand_seq(rng, g), a[at:]]))
    for k in range(1, len(seqs)):
        rc += [(0, k), (k, 0), (k, 1 + (k * 7) % (len(seqs) - 1))]
    codes, offs = seqset(seqs)
    # seeds in the shared prefix and in the shared suffix
    lens = [len(s) for s in seqs]
    return codes, offs, pairs_of(rc, [[50, 50, lens[r] - 60, lens[c] - 60]
                                      for r, c in rc])


@pytest.mark.parametrize("model", ["as_called", "as_documented"])
@pytest.mark.parametrize("xdrop,stage", [(0, 1), (0, 0), (200, 1), (200, 0)])
def test_gap_runs(model, xdrop, stage):
    codes, offs, pairs = gapped(3)
    al = Aligner(config_for_cli(-11, -2, 6, xdrop, 2, model))
    al.set_tuning(tb_stage=stage)
    al.load_seqs(codes, offs)
    print("walks", model, xdrop, stage, flush=True)
    got = al.align(pairs)
    if xdrop:
        ref = orc.sxa_batch(codes, offs, pairs["r"], pairs["c"], pairs["seed"],
                            oracle_params(model, xdrop=xdrop))
    else:
        ref = orc.sfa_batch(codes, offs, pairs["r"], pairs["c"],
                            oracle_params(model))
    assert (ref["cols"] > 600).any()
    for f in ("score", "matches", "cols", "gap_opens"):
        bad = np.nonzero(got[f].astype(np.int64) != ref[f].astype(np.int64))[0]
        assert bad.size == 0, (f, int(bad[0]), got[bad[0]], ref[bad[0]])
    al.close()
