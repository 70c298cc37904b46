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
