"""Which kernels a call launches, on the CPU emulation of tests/test_emu.py.

The emulation runs workgroups one after the other, so a race between two of
them changes no result here; these tests look at the launches instead.
"""
import os
import subprocess

import numpy as np
import pytest

from helpers import oracle_params, pairs_of, rand_seq, seqset
from oracle import oracle as orc
from pastis_amd._lib import PAIR_DTYPE, RESULT_DTYPE, SCORE_DTYPE
from test_emu import EMU, OUT, driver  # noqa: F401  (driver: a fixture)


def run(driver, tmp_path, codes, offs, pairs, mode=0, xdrop=0, gap_model=0,
        shapes=None, **env):
    """Results (pa_result) and the launches as (kernel, workgroups)."""
    inp, outp, log = (tmp_path / n for n in ("in.bin", "out.bin", "log.txt"))
    log.unlink(missing_ok=True)
    hdr = np.array([mode, -11, -2, 6, xdrop, 2, gap_model, 0], np.int32)
    with open(inp, "wb") as f:
        f.write(hdr.tobytes())
        f.write(np.array([len(offs) - 1, len(pairs)], np.uint64).tobytes())
        f.write(np.ascontiguousarray(offs, np.uint64).tobytes())
        f.write(np.ascontiguousarray(codes, np.uint8).tobytes())
        f.write(np.ascontiguousarray(pairs, PAIR_DTYPE).tobytes())
    e = dict(os.environ, ASAN_OPTIONS="detect_leaks=0:abort_on_error=1",
             UBSAN_OPTIONS="print_stacktrace=1", EMU_LAUNCHES=str(log), **env)
    if shapes is not None:
        e["EMU_SHAPES"] = ",".join(str(v) for v in shapes)
    r = subprocess.run([driver, str(inp), str(outp)], env=e,
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-4000:]
    launches = [(n, int(g)) for n, g, _ in
                (ln.split() for ln in open(log))]
    return outp.read_bytes(), launches


# Default shapes: 128, 256 and 512 rows a pass in the classes below the last.
# A task of several passes keeps a boundary row at workgroup * slots + slot,
# and the classes have 8, 4, 2 and 1 slots a workgroup, so in one launch the
# second workgroup of class 2 (rows 2 and 3) and workgroups 2 and 3 of class 3
# would share rows if both classes held such tasks.
@pytest.mark.parametrize("edges,one", [
    ((128, 256, 512), True), ((64, 200, 400), True),
    ((129, 256, 512), False), ((128, 257, 512), False),
    ((128, 256, 513), False), ((128, 256, 768), False),
    ((128, 384, 768), False)])
def test_affine_one_launch_only_with_one_pass_below_the_last_class(
        driver, tmp_path, edges, one):
    rng = np.random.default_rng(5)
    seqs = [rand_seq(rng, n) for n in (600, 1030, 300, 12)]
    codes, offs = seqset(seqs)
    pairs = pairs_of([(0, 3), (1, 3), (2, 3)])
    raw, launches = run(driver, tmp_path, codes, offs, pairs, gap_model=1,
                        shapes=(5, 1, 4, 3) + edges + (1, 0))
    got = np.frombuffer(raw, RESULT_DTYPE)
    ref = orc.sfa_batch(codes, offs, pairs["r"], pairs["c"],
                        oracle_params("as_documented"))
    for f in ("score", "matches", "cols", "gap_opens"):
        assert np.array_equal(got[f].astype(np.int64),
                              ref[f].astype(np.int64)), f
    names = [n for n, _ in launches]
    assert ("k_dp_all" in names) == one
    assert ("k_traceback_all" in names) == one


# Seeds far past the end of their sequences, and pairs outside the sets, in
# the kernels that take a small batch first: 16 lanes per item as called, the
# band kernels as documented, among good pairs or alone.  The sanitizers report
# a read outside the store.
@pytest.mark.parametrize("alone", [False, True])
@pytest.mark.parametrize("gap_model", [0, 1])
def test_pairs_that_do_not_fit_read_no_residues(driver, tmp_path, gap_model,
                                                alone):
    rng = np.random.default_rng(9)
    codes, offs = seqset([rand_seq(rng, 40) for _ in range(3)])
    far = [1 << k for k in range(15, 11, -1)] + list(range(3000, 40, -61))
    rc = [(2, 2)] * len(far) + [(7, 2), (2, 9), (0, 1), (1, 2)]
    seeds = [[f, f, f, f + 1] for f in far] + [[900, 900, 900, 900]] * 2 + \
        [[10, 12, 10, 12], [3, 4, 3, 4]]
    pairs = pairs_of(rc, seeds)
    if alone:
        pairs = pairs[:-2]
    raw, launches = run(driver, tmp_path, codes, offs, pairs, mode=1,
                        xdrop=49, gap_model=gap_model, EMU_DEV="1")
    assert ("k_xdrop_band" if gap_model else "k_xdrop_coop") in \
        [n for n, _ in launches]
    got = np.frombuffer(raw, RESULT_DTYPE)
    for f in ("score", "matches", "cols", "score_aln"):
        assert not got[f][:len(far) + 2].any(), f
    if alone:
        return
    good = pairs[-2:]
    ref = orc.sxa_batch(codes, offs, good["r"], good["c"], good["seed"],
                        oracle_params(["as_called", "as_documented"]
                                      [gap_model]))
    for f in ("score", "matches", "cols", "gap_opens"):
        assert np.array_equal(got[f][-2:].astype(np.int64),
                              ref[f].astype(np.int64)), f


def _equal_scores(tmp_path, driver, codes, offs, pairs, **env):
    raw, launches = run(driver, tmp_path, codes, offs, pairs, **env)
    got = np.frombuffer(raw, RESULT_DTYPE)
    ref = orc.sfa_batch(codes, offs, pairs["r"], pairs["c"],
                        oracle_params("as_called"))
    for f in ("score", "matches", "cols", "gap_opens"):
        assert np.array_equal(got[f].astype(np.int64),
                              ref[f].astype(np.int64)), f
    return launches


def test_linear_rerun_has_the_grid_of_the_first_run(driver, tmp_path):
    """Every task of a batch may leave int16, and the int32 run of them is
    then the longer one."""
    rng = np.random.default_rng(10)
    codes, offs = seqset([rand_seq(rng, 12) for _ in range(6)])
    pairs = pairs_of([(r, c) for r in range(6) for c in range(6)])
    grids = dict(_equal_scores(tmp_path, driver, codes, offs, pairs))
    assert grids["k_sw_linear_rerun"] == grids["k_sw_linear"] > 2


# X-drop items 16 lanes take beside the one-lane kernel only while they do not
# fill the chip: of 20 million items (5 million pairs) they took 45.2 ms so,
# and 42.7 ms in the one-lane kernel alone.
@pytest.mark.parametrize("items,xdrop,gap,coop,wave,want", [
    (4, 49, -11, 0, 1, "1 0 0 0"), (65536, 49, -11, 0, 1, "1 0 0 0"),
    (65540, 49, -11, 0, 1, "0 1 1 0"), (1 << 22, 49, -11, 0, 1, "0 1 1 0"),
    ((1 << 22) + 4, 49, -11, 0, 1, "0 0 1 0"),
    (20000000, 49, -11, 0, 1, "0 0 1 0"),
    (4, 49, -2, 0, 1, "0 0 1 1"), (20000000, 49, -2, 0, 1, "0 0 1 1"),
    (20000000, 49, -2, 0, 2, "0 0 0 0"), (4, 30001, -2, 0, 1, "0 0 0 0"),
    (4, 2147483647, -2147483648, 0, 1, "1 0 0 0"),
    # bands a little wider: the band kernels for all items took 20.5 ms of
    # 400,000 pairs at X = 66, where one lane per item had taken 9.5
    (240000, 66, -11, 0, 1, "0 0 1 1"), (1600000, 66, -11, 0, 1, "0 1 1 0"),
    (20000000, 66, -11, 0, 1, "0 0 1 0"), (1600000, 100, -11, 0, 1, "0 1 1 0"),
    (1600000, 130, -11, 0, 1, "0 0 1 1"), (1600000, 40, -5, 0, 1, "0 0 1 1"),
    (2100000, 40, -5, 0, 1, "0 1 1 0"), (1600000, 200, -31, 0, 1, "0 1 1 0"),
    (1600000, 66, -11, 0, 0, "0 0 0 0"),
    (4000000000, 30000, -5999, 0, 1, "0 0 1 0"),
    (4, 49, -11, 1, 1, "0 0 0 0"), (20000000, 49, -2, 1, 1, "0 0 0 0")])
def test_xdrop_route(items, xdrop, gap, coop, wave, want):
    rules = os.path.join(OUT, "rules")
    subprocess.run(["make", "-s", "-C", EMU, "OUT=" + OUT, rules], check=True,
                   timeout=300)
    r = subprocess.run([rules, "xdrop"] + [str(v) for v in
                                           (items, xdrop, gap, coop, wave)],
                       capture_output=True, text=True, check=True)
    assert r.stdout.strip() == want


# pa_stats counts the launches of the DP, X-drop and traceback kernels
COUNTED = ("k_dp", "k_nw_", "k_sw_", "k_lin_", "k_xdrop", "k_traceback")


@pytest.mark.parametrize("mode,gap_model,env", [
    (0, 0, {}), (0, 1, {}), (1, 0, {}), (1, 1, {}),
    (0, 0, {"EMU_SCORES": "dev"}), (0, 1, {"EMU_SCORES": "dev"})])
def test_launches_are_counted(driver, tmp_path, mode, gap_model, env):
    rng = np.random.default_rng(11)
    codes, offs = seqset([rand_seq(rng, 14) for _ in range(3)])
    pairs = pairs_of([(0, 1), (1, 2)], [[2, 2, 4, 4]] * 2)
    stats = tmp_path / "stats.txt"
    _, launches = run(driver, tmp_path, codes, offs, pairs, mode=mode,
                      xdrop=49 if mode else 0, gap_model=gap_model,
                      EMU_DEV="1", EMU_STATS=str(stats), **env)
    assert int(stats.read_text()) == sum(n.startswith(COUNTED)
                                         for n, _ in launches)


@pytest.mark.parametrize("entry", ["dev", "noalloc"])
def test_passes_wait_for_one_another_only_on_a_workspace_of_ones_own(
        driver, tmp_path, entry):
    """pa_sw_scores_noalloc calls that overlap race on their common workspace:
    their results may be wrong, but no wave may wait for progress that the
    other call took away, so no task's passes are pipelined there."""
    rng = np.random.default_rng(12)
    seqs = [rand_seq(rng, n) for n in (2049, 2048, 30)]
    seqs[1][500:900] = seqs[0][700:1100]
    codes, offs = seqset(seqs)
    pairs = pairs_of([(0, 1), (0, 2), (2, 1)])
    raw, launches = run(driver, tmp_path, codes, offs, pairs,
                        EMU_SCORES=entry)
    got = np.frombuffer(raw, SCORE_DTYPE)
    sc, ve, he = orc.sw_batch(codes, offs, pairs["r"], pairs["c"], -2, -11)
    assert np.array_equal(got["score"], sc)
    assert np.array_equal(got["r_end"].astype(np.int32), ve)
    assert np.array_equal(got["c_end"].astype(np.int32), he)
    names = [n for n, _ in launches]
    assert "k_sw_linear" in names
    assert ("k_lin_passes" in names) == (entry == "dev")


def _same_as_the_oracle(raw, codes, offs, pairs, gap, xdrop):
    got = np.frombuffer(raw, RESULT_DTYPE)
    ref = orc.sxa_batch(codes, offs, pairs["r"], pairs["c"], pairs["seed"],
                        orc.params(-2, -11, gap, xdrop, 6, 2, 0.7, 30))
    for f in ("score", "matches", "cols", "gap_opens", "seed"):
        assert np.array_equal(got[f].astype(np.int64),
                              ref[f].astype(np.int64)), f
    return got


# Bands of some 250 columns: a few such items took most of a batch's time in
# the kernel that has its rings in global memory, a lane for an item.
def test_wide_bands_stay_in_lds(driver, tmp_path):
    rng = np.random.default_rng(13)
    codes, offs = seqset([rand_seq(rng, 262), rand_seq(rng, 265)])
    # the second seed leaves little to extend
    pairs = pairs_of([(0, 1)], [[0, 0, 256, 258]])
    raw, launches = run(driver, tmp_path, codes, offs, pairs, mode=1,
                        xdrop=250, EMU_XDGAP="-1", EMU_DEV="1")
    names = [n for n, _ in launches]
    assert "k_xdrop_band" in names and "k_xdrop_pl" not in names
    _same_as_the_oracle(raw, codes, offs, pairs, -1, 250)


# An X that leaves 16-bit values room for a best score of 2,000: 16 lanes per
# item to the end all the same, as for homologs of thousands of residues.
def test_high_scores_stay_in_lds(driver, tmp_path):
    rng = np.random.default_rng(14)
    a = rand_seq(rng, 270, "WWWWCP")
    b = a.copy()
    b[::50] = rand_seq(rng, len(b[::50]))
    codes, offs = seqset([a, b])
    pairs = pairs_of([(0, 1)], [[4, 4, 0, 260]])
    raw, launches = run(driver, tmp_path, codes, offs, pairs, mode=1,
                        xdrop=29900, EMU_XDGAP="-1000", EMU_DEV="1")
    assert "k_xdrop_pl" not in [n for n, _ in launches]
    got = _same_as_the_oracle(raw, codes, offs, pairs, -1000, 29900)
    assert got["score"][0] > 2200
