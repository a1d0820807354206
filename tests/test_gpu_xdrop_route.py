"""Batches whose X-drop items start in other kernels than those of their parts:
the same results, and those of the oracle."""
import numpy as np
import pytest

from oracle import oracle as orc
from pastis_amd import synth
from pastis_amd._lib import RESULT_DTYPE
from pastis_amd.aligner import Aligner, config_for_cli

pytestmark = pytest.mark.gpu


# four items a pair: beyond 4 million; bands wider than most rings hold, in
# batches that are too large for the band kernels alone
@pytest.mark.parametrize("n,xdrop,gap", [((1 << 20) + 7, 49, -11),
                                         (70000, 66, -11), (200000, 35, -5)])
def test_large_batches_equal_their_parts(n, xdrop, gap):
    w = synth.make(600, n, model="lognormal", a=60, b=0.8, clip=(12, 1500),
                   fam_size=20, ident=(0.3, 0.95), frac_hom=0.3, seed=31)
    cfg = config_for_cli(-11, -2, 6, xdrop, 2, "as_called")
    cfg.xdrop_gap = gap
    al = Aligner(cfg)
    al.load_seqs(w.codes, w.offsets)
    d_pairs = al.device_alloc(w.pairs.nbytes)
    d_out = al.device_alloc(n * RESULT_DTYPE.itemsize)
    al.h2d(d_pairs, w.pairs)
    print("whole batch", flush=True)
    al.align_dev(d_pairs, n, d_out)
    whole = np.zeros(n, RESULT_DTYPE)
    al.synchronize()
    al.d2h(whole, d_out)
    # a small batch and one whose far-reaching items are split off
    for a, b in [(0, 5000), (5000, min(305000, n - 9)), (n - 20000, n)]:
        print("part", a, b, flush=True)
        part = al.align(w.pairs[a:b])
        assert np.array_equal(part, whole[a:b]), (a, b)
    p = w.pairs[:1500]
    ref = orc.sxa_batch(w.codes, w.offsets, p["r"], p["c"], p["seed"],
                        orc.params(-2, -11, gap, xdrop, 6, 2, 0.7, 30))
    for f in ("score", "matches", "cols", "gap_opens"):
        assert np.array_equal(whole[f][:1500].astype(np.int64),
                              ref[f].astype(np.int64)), f
    al.device_free(d_pairs)
    al.device_free(d_out)
    al.close()
