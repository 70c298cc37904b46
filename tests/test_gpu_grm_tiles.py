"""The 2-bit-input SYRK's tile sizes (64, 128 and 256) and operand forms, at
sample counts around the tiles and marker counts around the chunks, and the
read-back of blocks of K."""
import numpy as np
import pytest

from fixtures import random_bed
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _load(session, N, M, seed):
    body, _, _ = random_bed(N, M, 0.02, seed=seed, maf_lo=0.02)
    session.setminMAFforGRM(0.01)
    session.setmaxMissingRateforGRM(0.15)
    session.setminMAC_VarianceRatio(20, -1, False)
    session.setgeno_bytes(body, N, M)
    return O.setgeno(body, N, M, min_maf=0.01, max_missing=0.15)


def test_block_read_back(session):
    """Blocks of K at odd offsets equal the whole matrix's; 4200 x 4200 values
    come in more than one piece."""
    print("case: GRM block read-back N=4200", flush=True)
    N = 4200
    _load(session, N, 64, 11)
    session.build_grm("bf16_split")
    K = session.grm_block(0, 0, N, N)
    assert np.array_equal(K, K.T)
    for r0, c0, nr, nc in [(0, 0, 1, 1), (3, 5, 7, 1025), (4093, 1, 107, 4199), (N - 1, N - 3, 1, 3), (17, 0, 0, 5)]:
        assert np.array_equal(session.grm_block(r0, c0, nr, nc), K[r0:r0 + nr, c0:c0 + nc])
    e = np.zeros(N, np.float32)
    e[4099] = 1
    assert np.array_equal(session.getCrossprodMatAndKin(e), K[:, 4099])
