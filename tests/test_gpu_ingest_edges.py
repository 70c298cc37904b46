"""Ingest at the edges of the kernels' tiles: sample counts around a
workgroup's 256 samples, a cache line's 512 and a byte's 4, marker counts
around the 128-marker tiles.  Bit-exact against the oracle."""
import numpy as np
import pytest

from fixtures import random_bed
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,M", [(3, 5), (255, 127), (256, 128), (257, 129), (513, 256), (1021, 385), (2049, 130)])
def test_diag_tile_edges(session, N, M):
    print(f"case: diag N={N} M={M}", flush=True)
    body, _, _ = random_bed(N, M, 0.03, seed=7 * N + M, maf_lo=0.05)
    session.setminMAFforGRM(0.0)
    session.setmaxMissingRateforGRM(1.0)
    session.setminMAC_VarianceRatio(20, -1, False)
    session.setgeno_bytes(body, N, M)
    og = O.setgeno(body, N, M)
    assert session.getMsub_MAFge_minMAFtoConstructGRM() == og["Mqc"]
    assert np.array_equal(session.Get_Diagof_StdGeno().view(np.uint32), O.diag_std(og).view(np.uint32))


def _same_genotypes(session, body, N, M, sub):
    session.setminMAFforGRM(0.0)
    session.setmaxMissingRateforGRM(1.0)
    session.setminMAC_VarianceRatio(20, -1, False)
    session.setgeno_bytes(body, N, M, sub)
    og = O.setgeno(body, N, M, subidx=sub)
    assert session.getMsub_MAFge_minMAFtoConstructGRM() == og["Mqc"] == M
    n = len(sub)
    for j in range(M):
        assert np.array_equal(session.Get_OneSNP_Geno(j), O.get_geno(og["packed"][j], n)), j


@pytest.mark.parametrize("N", [1, 4, 15, 16, 17, 63, 64, 65, 255, 257, 1030, 16390])
def test_repack_in_order(session, N):
    """One wave per marker, 16 output bytes (64 samples) per lane and step,
    four steps (16,384 samples) at a time; rows of every alignment."""
    print(f"case: repack in order N={N}", flush=True)
    body, _, _ = random_bed(N, 9, 0.3, seed=N)
    _same_genotypes(session, body, N, 9, np.arange(1, N + 1, dtype=np.int32))


@pytest.mark.parametrize("N,n,M", [(5, 1, 1), (17, 16, 3), (64, 15, 4), (130, 129, 5), (1003, 1003, 6), (8201, 8190, 7),
                                   (163840, 40, 3), (163841, 41, 3)])
def test_repack_listed(session, N, n, M):
    """Samples in an order of their own, four markers per workgroup; the last
    case's rows are too long for LDS."""
    print(f"case: repack listed N={N} n={n} M={M}", flush=True)
    body, _, _ = random_bed(N, M, 0.3, seed=N + n)
    sub = (np.random.default_rng(n).permutation(N)[:n] + 1).astype(np.int32)
    _same_genotypes(session, body, N, M, sub)
