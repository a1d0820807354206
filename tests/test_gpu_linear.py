"""The linear-gap global kernel (as-called gaps, BLOSUM62) against the oracle
at the sizes where its layout changes: 32 rows per lane, the lane counts per
task (1 .. 10, 12, 16, 21, 32, 64), passes of 2048 rows, blocks of 8 steps
and the shortest spans.  Values are whole numbers: equality."""
import numpy as np
import pytest

from helpers import oracle_params
from oracle import oracle as orc
from pastis_amd._lib import PAIR_DTYPE
from pastis_amd.aligner import Aligner, config_for_cli

pytestmark = pytest.mark.gpu


def _homolog(rng, s, indels):
    """s with a few substitutions and `indels` short insertions/deletions."""
    t = s.copy()
    sub = rng.random(len(t)) < 0.1
    t[sub] = rng.integers(0, 20, int(sub.sum()))
    for _ in range(indels):
        if len(t) < 40:
            break
        p = int(rng.integers(10, len(t) - 10))
        k = int(rng.integers(1, 4))
        if rng.random() < 0.5:
            t = np.delete(t, slice(p, p + k))
        else:
            t = np.insert(t, p, rng.integers(0, 20, k))
    return t.astype(np.uint8)


def _edges(lo, hi):
    """Row counts on both sides of every lane-count edge within lo..hi."""
    lanes = [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 12, 16, 21, 32, 64]
    out = {6, 7, 8, 9, 15, 16, 17}
    for v in lanes:
        out |= {32 * v - 1, 32 * v, 32 * v + 1}
    out |= {2047, 2048, 2049, 2079, 2081, 4096, 4097}
    return sorted(n for n in out if lo <= n <= hi)


@pytest.mark.parametrize("lo,hi", [(6, 353), (354, 1025), (1026, 4097)])
@pytest.mark.parametrize("tail", [False, True])
def test_row_edges(lo, hi, tail):
    """Whole-length infixes of every edge size, alone in a batch order that
    mixes classes; tail: more tasks than one wave of each class holds."""
    rng = np.random.default_rng(lo + tail)
    seqs, pairs = [], []
    for n in _edges(lo, hi):
        for rep in range((70 if n <= 64 else 14 if n <= 353 else 3) if tail
                         else 1):
            s = rng.integers(0, 20, n).astype(np.uint8)
            t = _homolog(rng, s, rep % 4) if n > 40 else s.copy()
            if rep % 5 == 3 and n > 8:   # letters outside the 20
                t[n // 2] = rng.integers(20, 25)
            a, b = len(seqs), len(seqs) + 1
            seqs += [s, t]
            k = 0   # the exact 6-mer nearest the middle, if any
            m = min(len(s), len(t)) - 6
            for d in range(m // 2 + 1):
                for p in (m // 2 - d, m // 2 + d):
                    if 0 <= p <= m and np.array_equal(s[p:p + 6], t[p:p + 6]):
                        k = p
                        break
                else:
                    continue
                break
            pairs.append((a, b, k) if rep % 2 == 0 else (b, a, k))
    pairs = [pairs[i] for i in rng.permutation(len(pairs))]
    arr = np.zeros(len(pairs), PAIR_DTYPE)
    for i, (r, c, k) in enumerate(pairs):
        arr[i] = (r, c, 2, 0, (k, k, 0, 0))
    offs = np.zeros(len(seqs) + 1, np.uint64)
    offs[1:] = np.cumsum([len(s) for s in seqs])
    codes = np.concatenate(seqs)
    al = Aligner(config_for_cli(xdrop=49))
    al.load_seqs(codes, offs)
    print("linear edges", lo, hi, tail, len(arr), flush=True)
    got = al.align(arr)
    names = [k["name"] for k in al.kernel_stats()]
    assert "nwl.r16.i16" in names, names
    ref = orc.sxa_batch(codes, offs, arr["r"], arr["c"], arr["seed"],
                        oracle_params("as_called"))
    for gf, rf in [("score", "score"), ("matches", "matches"),
                   ("cols", "cols"), ("gap_opens", "gap_opens"),
                   ("seed", "seed")]:
        bad = np.nonzero(got[gf].astype(np.int64) !=
                         ref[rf].astype(np.int64))[0]
        assert bad.size == 0, (gf, int(bad[0]), got[bad[0]], arr[bad[0]])
    assert np.array_equal(got["score_aln"], ref["score_aln"])
    al.close()
