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


@pytest.mark.parametrize("N,M", [(60, 40), (256, 64), (257, 65), (700, 129), (520, 1001)])
@pytest.mark.parametrize("prec", ["bf16", "bf16_split", "fp32"])
def test_tiles_agree(session, monkeypatch, N, M, prec):
    """Every tile size gives the same bits: the whole GRM and one with a range
    of markers taken off it (starting and ending inside chunks)."""
    print(f"case: SYRK tiles {prec} N={N} M={M}", flush=True)
    og = _load(session, N, M, N + M)
    mq = og["Mqc"]
    e = np.zeros(N, np.float32)
    e[N // 3] = 1
    got = {}
    for tile in ("64", "128", "256"):
        monkeypatch.setenv("SAIGE_SYRK_TILE", tile)
        session.build_grm(prec)
        K = session.grm_block(0, 0, N, N)
        session.setStartEndIndex(mq // 5, mq // 2, 0)
        got[tile] = (K, session.getCrossprodMatAndKin_LOCO(e))
        assert np.array_equal(K, K.T)
    for tile in ("64", "128"):
        for a, b in zip(got[tile], got["256"]):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    # against FP64: an FP32 sum of Mqc terms, plus the operands' rounding (BF16
    # z: 2^-8 relative each; the split's storage at 16 bits; FP32: the FP32
    # frequency, 1/sd and z, a few 2^-24 of a value)
    K64 = O.grm_f64(og) / mq
    tol = 4.0 * np.sqrt(mq) * 2.0 ** -24 + {"bf16": 2.0 ** -7, "bf16_split": 2.0 ** -16, "fp32": 8 * 2.0 ** -24}[prec]
    assert np.max(np.abs(got["256"][0] - K64)) <= tol * np.max(np.abs(K64))


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
