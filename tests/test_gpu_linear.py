"""The linear-gap kernels (as-called gaps, BLOSUM62) against the oracle at the
sizes where their layout changes: 32 rows per lane, the lane counts per task
(1 .. 10, 12, 16, 21, 32, 64), passes of 2048 rows, pipelined passes from 2048
columns, blocks of 8 steps, the shortest spans and the bounds of the int16
maxima.  Values are whole numbers: equality."""
import numpy as np
import pytest

from helpers import oracle_params, small_config1
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


SFA = [("score", "score"), ("r_beg", "v_beg"), ("r_end", "v_end"),
       ("c_beg", "h_beg"), ("c_end", "h_end"), ("matches", "matches"),
       ("cols", "cols"), ("gap_opens", "gap_opens")]


def _check_local(seqs, pairs, what):
    """Scores and traced alignments of pairs (r, c) against the oracle;
    returns the results."""
    offs = np.zeros(len(seqs) + 1, np.uint64)
    offs[1:] = np.cumsum([len(s) for s in seqs])
    codes = np.concatenate(seqs).astype(np.uint8)
    arr = np.zeros(len(pairs), PAIR_DTYPE)
    for i, (r, c) in enumerate(pairs):
        arr["r"][i], arr["c"][i] = r, c
    al = Aligner(config_for_cli())
    al.load_seqs(codes, offs)
    print("linear local", what, len(arr), flush=True)
    ref = orc.sfa_batch(codes, offs, arr["r"], arr["c"],
                        oracle_params("as_called"))
    sc = al.sw_scores(arr)
    reruns = al.stats()["rerun_pairs"]
    got = al.align(arr)
    names = [k["name"] for k in al.kernel_stats()]
    assert "swl.r16.i16" in names and "swtl.r16.i16" in names, names
    for gf, rf in SFA:
        bad = np.nonzero(got[gf].astype(np.int64) !=
                         ref[rf].astype(np.int64))[0]
        assert bad.size == 0, (gf, int(bad[0]), got[bad[0]], arr[bad[0]])
    for f in ("score", "r_end", "c_end"):
        assert np.array_equal(sc[f].astype(np.int64),
                              got[f].astype(np.int64)), f
    # re-runs are reported by the scores that leave int16 (score only) and
    # a quarter of it (traced)
    assert reruns == int((ref["score"] >= 32766).sum())
    assert np.array_equal((got["flags"] & 2) != 0, ref["score"] >= 8190)
    al.close()
    return got


@pytest.mark.parametrize("lo,hi", [(1, 353), (354, 1025), (1026, 4097)])
def test_local_row_edges(lo, hi):
    """Local alignment at every edge of the row classes, homologs and
    unrelated sequences, rows and columns of unequal lengths."""
    rng = np.random.default_rng(hi)
    seqs, pairs = [], []
    for n in sorted(set(_edges(lo, hi)) | ({1, 2, 3} if lo == 1 else set())):
        s = rng.integers(0, 20, n).astype(np.uint8)
        t = _homolog(rng, s, n % 4) if n > 40 else s.copy()
        x = rng.integers(0, 25, int(rng.integers(1, 400)))
        a = len(seqs)
        seqs += [s, t, x.astype(np.uint8)]
        pairs += [(a, a + 1), (a + 1, a), (a, a + 2), (a + 2, a)]
    _check_local(seqs, [pairs[i] for i in rng.permutation(len(pairs))],
                 (lo, hi))


def test_pipelined_passes():
    """Tasks of several passes around the column count from which each pass
    is an item of its own (2048), more items than the chip has waves beside
    short tasks, and a task of many passes."""
    rng = np.random.default_rng(9)
    base = rng.integers(0, 20, 9000).astype(np.uint8)
    lens = [2047, 2048, 2049, 2050, 2175, 2176, 4096, 4097, 6145]
    seqs = [_homolog(rng, base[:n + 6], 2)[:n] for n in lens]
    seqs += [rng.integers(0, 20, 150).astype(np.uint8), base]
    pairs = [(i, j) for i in range(len(seqs)) for j in range(len(seqs))]
    _check_local(seqs, pairs, "pipelined")


def test_saturation_bounds():
    """Scores on both sides of the int16 maxima's bounds (half-float order
    ends at 0x7c00) and of the reported ones."""
    W = 17   # scores 11 against itself
    lens = [719, 720, 721, 722, 743, 744, 745, 746, 2883, 2884, 2885, 2886,
            2977, 2978, 2979, 2980]
    seqs = [np.full(n, W, np.uint8) for n in lens]
    got = _check_local(seqs, [(i, i) for i in range(len(seqs))], "saturation")
    assert list(got["score"]) == [11 * n for n in lens]


@pytest.mark.parametrize("go,ge", [(-1, -2), (-2, -2), (-2, -3), (-3, -11),
                                   (-30, -31)])
def test_gap_values(go, ge):
    """Gap costs on both sides of the linear kernels' rule (open > ext; the
    global one also needs -2): local and X-drop runs against the oracle."""
    w = small_config1(n_seq=60, n_pairs=400, seed=3)
    p = orc.params(go, ge, -11, 49, 6, 2)
    for xdrop in (0, 49):
        cfg = config_for_cli(xdrop=xdrop)
        cfg.gap_open, cfg.gap_ext = go, ge
        al = Aligner(cfg)
        al.load_seqs(w.codes, w.offsets)
        print("gaps", go, ge, xdrop, flush=True)
        got = al.align(w.pairs)
        lin = {k["name"] for k in al.kernel_stats()} & {"nwl.r16.i16",
                                                        "swtl.r16.i16"}
        assert bool(lin) == (go > ge and (xdrop == 0 or go == -2))
        if xdrop:
            ref = orc.sxa_batch(w.codes, w.offsets, w.pairs["r"],
                                w.pairs["c"], w.pairs["seed"], p)
        else:
            ref = orc.sfa_batch(w.codes, w.offsets, w.pairs["r"],
                                w.pairs["c"], p)
        for f in ("score", "matches", "cols", "gap_opens"):
            assert np.array_equal(got[f].astype(np.int64),
                                  ref[f].astype(np.int64)), f
        al.close()
