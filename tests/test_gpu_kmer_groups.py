"""k-mer groups of every size class against the oracle.

The products of a k-mer code are counted and emitted by the size of its group
of occurrences (up to 4 of one set; up to 32 column occurrences; up to 64 and
up to 65,536 products; more), so sets are built whose codes occur a chosen
number of times, and all symmetric rules, equal and unequal bases and column
blocks must give the oracle's candidates exactly."""
import numpy as np
import pytest

from oracle import oracle as orc
from pastis_amd import _lib
from pastis_amd.aligner import Aligner, config_for_cli

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 3, 4, 5, 8, 9, 11, 12, 31, 32, 33, 64, 65, 255, 257, 300]


def pack(seqs):
    offs = np.zeros(len(seqs) + 1, np.uint64)
    offs[1:] = np.cumsum([len(s) for s in seqs])
    return np.frombuffer(b"".join(seqs), np.uint8), offs


def family_set(seed):
    """Each 6-mer of SIZES occurs that often, at shuffled places, some twice
    in a sequence."""
    rng = np.random.default_rng(seed)
    aa = np.frombuffer(b"ARNDCQEGHILKMFPSTWYV", np.uint8)
    words = [bytes(rng.choice(aa, 6)) for _ in SIZES]
    seqs = [b"" for _ in range(220)]
    for word, n in zip(words, SIZES):
        for i in rng.integers(0, len(seqs), n):
            seqs[i] += bytes(rng.choice(aa, int(rng.integers(0, 3)))) + word
    return pack(seqs + [b"", b"MKV"])


def same(got, ref):
    assert len(got) == len(ref)
    for f in ("r", "c", "count", "kscore", "seed"):
        assert np.array_equal(got[f], ref[f]), f


@pytest.mark.parametrize("sym", ["none", "upper", "even_odd"])
@pytest.mark.parametrize("bases", [(0, 0), (7, 7), (0, 101), (150, 3)])
def test_group_sizes(sym, bases):
    res, offs = family_set(5)
    n = len(offs) - 1
    al = Aligner(config_for_cli(-11, -2, 6, 49, 2, "as_called"))
    al.load_seqs(res, offs, encoding=_lib.PA_ENC_ASCII)
    roff, coff = bases
    ref = orc.kmer_candidates(res, offs, k=6, sym=sym, roff=roff, coff=coff)
    assert len(ref)
    print("one set", sym, bases, flush=True)
    kw = dict(k=6, symmetric=sym, row_base=roff, col_base=coff)
    same(al.kmer_candidates(**kw), ref)
    same(np.concatenate([al.kmer_candidates(c_begin=a, c_end=b, **kw)
                         for a, b in [(0, 1), (1, 90), (90, n)]]), ref)
    # the same set after another rule's group table
    same(al.kmer_candidates(k=6, symmetric="none"),
         orc.kmer_candidates(res, offs, k=6, sym="none"))
    same(al.kmer_candidates(**kw), ref)
    al.close()


@pytest.mark.parametrize("sym", ["none", "upper", "even_odd"])
def test_group_sizes_of_two_sets(sym):
    rres, roffs = family_set(5)
    cres, coffs = pack([bytes(rres[int(a):int(b)])
                        for a, b in zip(roffs[30:170], roffs[31:171])])
    al = Aligner(config_for_cli(-11, -2, 6, 49, 2, "as_called"))
    al.load_seqs(rres, roffs, encoding=_lib.PA_ENC_ASCII,
                 side=_lib.PA_SIDE_ROW)
    al.load_seqs(cres, coffs, encoding=_lib.PA_ENC_ASCII,
                 side=_lib.PA_SIDE_COL)
    print("two sets", sym, flush=True)
    for roff, coff in [(0, 0), (0, 30)]:
        same(al.kmer_candidates(k=6, symmetric=sym, row_base=roff,
                                col_base=coff),
             orc.kmer_candidates(rres, roffs, cres, coffs, k=6, sym=sym,
                                 roff=roff, coff=coff))
    al.close()
