"""The lower-triangle product at few rows, read from all of S: bitwise the
triangle walk's results for both workgroups, every width, the split and the FP32
GRM, where a last row set is whole or ragged, and on a leave-out range; against
FP64 at the end of its range."""
import numpy as np
import pytest

from fixtures import random_bed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["bf16_split", "fp32"])
@pytest.mark.parametrize("N", [40, 300, 700, 1530, 4700, 11200])
def test_flat_product(session, monkeypatch, N, prec):
    print(f"case: flat lower-triangle product N={N} {prec}", flush=True)
    body, _, _ = random_bed(N, 200, 0.01, seed=N, maf_lo=0.05, maf_hi=0.5)
    session.setminMAFforGRM(0.01)
    session.setmaxMissingRateforGRM(0.15)
    session.setgeno_bytes(body, N, 200)
    session.build_grm(prec)
    session.setStartEndIndex(20, 60, 0)
    rng = np.random.default_rng(N)
    B = rng.standard_normal((N, 64)).astype(np.float32)
    w = rng.uniform(0.05, 0.25, N).astype(np.float32)
    try:
        session.set_gemm_mode("bf16x3_tri")
        for nwv in (1, 2):
            session.set_gemm_config(nwv, 3, 8)
            out = {}
            for limit in ("0", "20000"):
                monkeypatch.setenv("SAIGE_TRI_FLAT_MAX", limit)
                r = [session.grm_matvec(B[:, :k]) for k in (64, 48, 20, 7)]
                session.engine_reserve(64, 1)
                session.engine_use_loco(True)
                session.engine_set_system(0, w, np.array([1.0, 0.3], np.float32))
                slots = list(range(1, 64, 2))
                session.engine_add_products(slots, [0] * len(slots), np.asfortranarray(B[:, slots]))
                done, _ = session.engine_step(1)
                assert all(done[s] for s in slots)
                r.append(session.engine_take_batch(slots))
                session.engine_use_loco(False)
                out[limit] = r
            for a, b in zip(out["0"], out["20000"]):
                assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), nwv
        if N <= 4700:
            K = session.grm_block(0, 0, N, N).astype(np.float64)
            mag = np.abs(K) @ np.abs(B.astype(np.float64))
            # N FP32 products and sums, random signs; K's own rounding when read
            assert np.all(np.abs(r[0] - K @ B.astype(np.float64)) <= (4 * np.sqrt(N) + 2) * 2.0 ** -24 * mag)
    finally:
        monkeypatch.delenv("SAIGE_TRI_FLAT_MAX", raising=False)
        session.engine_use_loco(False)
        session.set_gemm_mode("fp32")
        session.set_gemm_config(1, 1, 4)
