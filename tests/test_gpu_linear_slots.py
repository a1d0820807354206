"""Pipelined passes of long tasks whose items reuse the boundary slots several
times, tasks of few and of many columns mixed so that a slot's owner can be
slower than the items after it: scores against the oracle, with the slots of a
grid and with those of the fixed workspace."""
import numpy as np
import pytest

from helpers import pairs_of, rand_seq, seqset
from oracle import oracle as orc
from pastis_amd._lib import SCORE_DTYPE
from pastis_amd.aligner import Aligner, config_for_cli

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("longest,npairs,noalloc", [(4096, 2500, True),
                                                    (4096, 5000, False),
                                                    (9000, 1500, False)])
def test_slots_are_reused(longest, npairs, noalloc):
    rng = np.random.default_rng(longest)
    # row sequences of two passes and more, column sequences from the fewest
    # columns that are pipelined to the most
    lens = [2049, 2100, 4096, 2500, longest, 2048, 2060, longest, 3000, 2049]
    codes, offs = seqset([rand_seq(rng, n) for n in lens])
    r = rng.choice([0, 1, 2, 3, 4], npairs)
    c = rng.choice([4, 5, 5, 5, 6, 6, 7, 8, 9, 9], npairs)
    pairs = pairs_of(list(zip(r.tolist(), c.tolist())), [[0, 0, 0, 0]] * npairs)
    uniq, inv = np.unique(np.stack([r, c], axis=1), axis=0, return_inverse=True)
    inv = inv.reshape(-1)
    sc, ve, he = orc.sw_batch(codes, offs, uniq[:, 0].astype(np.uint32),
                              uniq[:, 1].astype(np.uint32), -2, -11)
    al = Aligner(config_for_cli(-11, -2, 6, 0, 2, "as_called"))
    al.load_seqs(codes, offs)
    print("slots", longest, npairs, noalloc, flush=True)
    if noalloc:
        d_pairs = al.device_alloc(pairs.nbytes)
        d_out = al.device_alloc(npairs * SCORE_DTYPE.itemsize)
        al.h2d(d_pairs, pairs)
        al.sw_scores_noalloc(d_pairs, npairs, d_out)
        al.synchronize()
        got = np.zeros(npairs, SCORE_DTYPE)
        al.d2h(got, d_out)
    else:
        got = al.sw_scores(pairs)
    assert np.array_equal(got["score"], sc[inv])
    assert np.array_equal(got["r_end"].astype(np.int64), ve[inv])
    assert np.array_equal(got["c_end"].astype(np.int64), he[inv])
    al.close()
