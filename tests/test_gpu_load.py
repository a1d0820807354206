"""Sequence loading on the GPU (encoding of raw bytes, four at a time) and the
per-sequence sketches and residue bounds, a wave per sequence: set sizes and
lengths around the word, the wave and the k-mer length, every byte value."""
import numpy as np
import pytest

from helpers import oracle_params
from oracle import mlp_oracle as M
from oracle import oracle as orc
from pastis_amd import _lib
from pastis_amd.aligner import Aligner, config_for_cli

pytestmark = pytest.mark.gpu

TABLE = np.full(256, 22, np.uint8)
for _i, _ch in enumerate(orc.ALPHABET):
    TABLE[ord(_ch)] = TABLE[ord(_ch.lower())] = _i


@pytest.mark.parametrize("lens", [[1], [3, 2], [5, 6, 7], [63, 64, 65],
                                  [127, 1, 0, 128, 129, 6, 333],
                                  [70000 // 3, 11, 4097]])
@pytest.mark.parametrize("ascii_", [True, False])
def test_load_encodings(lens, ascii_):
    rng = np.random.default_rng(sum(lens) + ascii_)
    total = sum(lens)
    offs = np.zeros(len(lens) + 1, np.uint64)
    offs[1:] = np.cumsum(lens)
    if ascii_:
        # every byte value, then mostly letters
        raw = rng.integers(0, 256, total).astype(np.uint8)
        keep = rng.random(total) < 0.8
        letters = np.frombuffer(b"ARNDCQEGHILKMFPSTWYVBZXJarndc*", np.uint8)
        raw[keep] = letters[rng.integers(0, len(letters), int(keep.sum()))]
        codes = TABLE[raw]
    else:
        raw = codes = rng.integers(0, 25, total).astype(np.uint8)
    o = offs.astype(int)
    seqs = [codes[o[i]:o[i + 1]] for i in range(len(lens))]
    al = Aligner(config_for_cli(xdrop=49))
    al.load_seqs(raw, offs,
                 encoding=_lib.PA_ENC_ASCII if ascii_ else _lib.PA_ENC_CODES)
    n = len(lens)
    pairs = np.zeros(n * n, _lib.PAIR_DTYPE)
    pairs["r"] = np.repeat(np.arange(n), n)
    pairs["c"] = np.tile(np.arange(n), n)
    pairs["count"] = 1
    print("load", lens, ascii_, flush=True)
    assert np.array_equal(al.filter_features(pairs),
                          M.features(pairs, seqs, seqs))
    if ascii_:
        got = al.kmer_candidates(k=3)
        ref = orc.kmer_candidates(raw, offs, k=3)
        assert len(got) == len(ref)
        assert np.array_equal(got["count"], ref["count"])
    small = pairs[[max(lens[p["r"]], lens[p["c"]]) < 5000 for p in pairs]]
    sw = Aligner(config_for_cli())
    sw.load_seqs(raw, offs, encoding=_lib.PA_ENC_ASCII if ascii_
                 else _lib.PA_ENC_CODES)
    ref = orc.sfa_batch(codes, offs, small["r"], small["c"],
                        oracle_params("as_called"))
    assert np.array_equal(sw.align(small)["score"], ref["score"])
    al.close()
    sw.close()


def test_residue_bound_of_affine_infixes():
    """The int16 rule of the affine global kernels reads the bound's sums at
    both ends of a span: infixes that start and end at the sequence ends and
    inside, over sets whose sequences follow each other without a gap."""
    rng = np.random.default_rng(2)
    lens = [64, 65, 1000, 2500, 2500, 63]
    base = rng.integers(0, 20, 2500).astype(np.uint8)
    seqs = [base[:n].copy() for n in lens]
    seqs[4][100:130] = 17
    offs = np.zeros(len(lens) + 1, np.uint64)
    offs[1:] = np.cumsum(lens)
    codes = np.concatenate(seqs)
    pr = [(a, b, k) for a in range(6) for b in range(6)
          for k in (0, min(lens[a], lens[b]) - 6, 30)]
    pairs = np.zeros(len(pr), _lib.PAIR_DTYPE)
    for i, (a, b, k) in enumerate(pr):
        pairs[i] = (a, b, 2, 0, (k, k, 5, 5))
    al = Aligner(config_for_cli(xdrop=49, gap_model="as_documented"))
    al.load_seqs(codes, offs)
    print("residue bound", len(pairs), flush=True)
    got = al.align(pairs)
    ref = orc.sxa_batch(codes, offs, pairs["r"], pairs["c"], pairs["seed"],
                        oracle_params("as_documented"))
    for f in ("score", "matches", "cols", "gap_opens"):
        assert np.array_equal(got[f].astype(np.int64),
                              ref[f].astype(np.int64)), f
    al.close()
