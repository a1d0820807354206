"""The wide-band X-drop kernels (128- and 256-column windows of int16 values)
against the oracle, extents and evaluated cells bit-exact: bands below, at and
above each window, best scores beyond the int16 range, segments that end after
a few residues on either side, and X at the largest value the kernels take."""
import numpy as np
import pytest

from helpers import pairs_of, rand_seq, seqset
from oracle import oracle as orc
from pastis_amd.aligner import Aligner, config_for_cli

pytestmark = pytest.mark.gpu


def mutated(rng, a, every, indel):
    b = a.copy()
    b[::every] = rand_seq(rng, len(b[::every]))
    return np.delete(b, np.arange(indel, len(b), indel)) if indel else b


def sets(seed):
    rng = np.random.default_rng(seed)
    # (7,000 equal residues score more than int16 holds)
    a, big = rand_seq(rng, 900), rand_seq(rng, 7000 if seed == 49 else 1500)
    seqs = [a, mutated(rng, a, 5, 0), mutated(rng, a, 9, 31), rand_seq(rng, 900),
            rand_seq(rng, 6), a[:150].copy(), a[430:].copy(),
            rand_seq(rng, 2500), big, big.copy(), a[:7].copy()]
    rc, seeds = [], []
    lens = [len(s) for s in seqs]
    for r, c in [(0, 1), (1, 0), (0, 2), (2, 0), (0, 3), (3, 7), (7, 0), (4, 0),
                 (0, 4), (5, 0), (0, 5), (6, 0), (0, 6), (8, 9), (10, 0),
                 (0, 10), (4, 4), (10, 7), (8, 7)]:
        for f in (0.0, 0.013, 0.5, 0.97, 1.0):
            vr, vc = int(f * (lens[r] - 6)), int(f * (lens[c] - 6))
            rc.append((r, c))
            seeds.append([vr, vc, lens[r] - 6 - vr, lens[c] - 6 - vc])
    return seqset(seqs), pairs_of(rc, seeds)


# (X, gap): X / -gap sets the band's width, about twice that in columns
@pytest.mark.parametrize("xdrop,gap", [(49, -2), (49, -1), (90, -2), (105, -2),
                                       (120, -1), (208, -2), (300, -1),
                                       (30000, -11), (30001, -11), (160, -11)])
def test_wide_bands(xdrop, gap):
    (codes, offs), pairs = sets(xdrop)
    cfg = config_for_cli(-11, -2, 6, xdrop, 2, "as_called")
    cfg.xdrop_gap = gap
    want = [[], []]
    for s in range(2):
        for p in pairs:
            v = codes[int(offs[p["r"]]):int(offs[p["r"] + 1])]
            h = codes[int(offs[p["c"]]):int(offs[p["c"] + 1])]
            x = orc.xdrop_extend(h, v, int(p["seed"][2 * s + 1]),
                                 int(p["seed"][2 * s]), 6, gap, xdrop)
            want[s].append((x["beg_v"], x["end_v"], x["beg_h"], x["end_h"]))
    for reps in (1, 200):   # fewer and more items than rows of waves
        many = np.tile(pairs, reps)
        for wave in (1, 2):
            print("band", xdrop, gap, reps, wave, flush=True)
            al = Aligner(cfg)
            al.set_tuning(xd_wave=wave)
            al.load_seqs(codes, offs)
            for s in range(2):
                got = al.xdrop_extents(many, s)
                have = np.stack([got[f].astype(np.int64) for f in
                                 ("r_beg", "r_end", "c_beg", "c_end")], axis=1)
                bad = np.nonzero(np.any(have != np.tile(want[s], (reps, 1)),
                                        axis=1))[0]
                assert bad.size == 0, (s, int(bad[0]), have[bad[0]],
                                       want[s][bad[0] % len(pairs)])
            al.close()
