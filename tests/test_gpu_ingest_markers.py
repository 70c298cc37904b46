"""More markers than one launch of the listed-order repack can take (2^25: four
markers per workgroup of 512 threads, fewer than 2^32 threads): every marker's
genotypes arrive, those around the passes' ends among them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_many_markers_listed_order(session):
    N, M = 8, (1 << 25) + 4099
    print(f"case: listed-order ingest of {M} markers", flush=True)
    rng = np.random.default_rng(11)
    body = np.frombuffer(rng.bytes(2 * M), np.uint8)
    sub = np.array([5, 1, 8, 2, 7], np.int32)
    session.setminMAFforGRM(0.0)
    session.setmaxMissingRateforGRM(1.0)
    try:
        session.setgeno_bytes(body, N, M, sub)
        q = np.flatnonzero(session.getQCdMarkerIndex())
        assert len(q) > 1 << 25
        for j in (0, (1 << 24) - 1, 1 << 24, (1 << 25) - 1, 1 << 25, len(q) - 1):
            row = body.reshape(M, 2)[q[j]]
            code = (row[(sub - 1) >> 2] >> (2 * ((sub - 1) & 3))) & 3
            g = np.array([2.0, np.nan, 1.0, 0.0])[code]
            seen = g[~np.isnan(g)]
            g[np.isnan(g)] = np.floor(np.mean(seen) + 0.5) if len(seen) else 0.0
            assert np.array_equal(session.Get_OneSNP_Geno(j), g.astype(np.int32)), j
    finally:
        session.setminMAFforGRM(0.01)
        session.setmaxMissingRateforGRM(0.15)
        session.setgeno_bytes(body[:400], N, 200, np.arange(1, 9, dtype=np.int32))
