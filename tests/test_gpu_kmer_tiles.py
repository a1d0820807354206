"""k-mer sets whose groups are joined in the smallest tiles, in tiles of some
size between, and in full ones, against the oracle."""
import numpy as np
import pytest

from oracle import oracle as orc
from pastis_amd import _lib
from pastis_amd.aligner import Aligner, config_for_cli
from test_gpu_kmer_groups import pack, same

pytestmark = pytest.mark.gpu


# about 330 occurrences a sequence, nearly all of a code of their own
@pytest.mark.parametrize("nseq", [770, 2500, 6900])
def test_tiles(nseq):
    rng = np.random.default_rng(nseq)
    aa = np.frombuffer(b"ARNDCQEGHILKMFPSTWYV", np.uint8)
    seqs = [bytes(rng.choice(aa, int(n)))
            for n in rng.integers(300, 370, nseq)]
    for i in range(0, nseq - 50, 50):   # relatives, for runs of several seeds
        seqs[i + 37] = seqs[i][40:300]
    res, offs = pack(seqs)
    al = Aligner(config_for_cli(-11, -2, 6, 49, 2, "as_called"))
    al.load_seqs(res, offs, encoding=_lib.PA_ENC_ASCII)
    for sym, coff in [("upper", 0), ("upper", 3)]:
        print("tiles", nseq, sym, coff, flush=True)
        same(al.kmer_candidates(k=6, symmetric=sym, col_base=coff),
             orc.kmer_candidates(res, offs, k=6, sym=sym, coff=coff))
    al.close()
