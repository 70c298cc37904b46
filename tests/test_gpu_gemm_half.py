"""The FP32 block product over one 32-column half: bitwise the 64-column
product's columns, for both workgroup shapes (below and above 12,288 rows) and
every slice count, on the first half (grm_matvec) and the second (occupied
slots 32 and up)."""
import numpy as np
import pytest

from fixtures import random_bed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [100, 700, 12200, 12300])
def test_half_product(session, N):
    print(f"case: FP32 half product N={N}", flush=True)
    body, _, _ = random_bed(N, 96, 0.01, seed=N, maf_lo=0.05, maf_hi=0.5)
    session.setminMAFforGRM(0.01)
    session.setmaxMissingRateforGRM(0.15)
    session.setgeno_bytes(body, N, 96)
    session.build_grm("fp32")
    rng = np.random.default_rng(N)
    B = rng.standard_normal((N, 64)).astype(np.float32)
    w = rng.uniform(0.05, 0.25, N).astype(np.float32)
    try:
        session.set_gemm_mode("fp32")
        for rt, pd, nsplit in [(1, 1, 1), (1, 3, 2), (1, 1, 4), (2, 3, 8)]:
            session.set_gemm_config(rt, pd, nsplit)
            full = session.grm_matvec(B)
            y = session.grm_matvec(B[:, :20])
            assert np.array_equal(y.view(np.uint32), full[:, :20].view(np.uint32)), (rt, pd, nsplit)
            session.engine_reserve(64, 1)
            session.engine_set_system(0, w, np.array([1.0, 0.3], np.float32))
            slots = list(range(33, 64, 3))
            session.engine_add_products(slots, [0] * len(slots), np.asfortranarray(B[:, slots]))
            done, _ = session.engine_step(1)
            assert all(done[s] for s in slots)
            y = session.engine_take_batch(slots)
            assert np.array_equal(y.view(np.uint32), full[:, slots].view(np.uint32)), (rt, pd, nsplit)
    finally:
        session.set_gemm_mode("fp32")
        session.set_gemm_config(1, 1, 4)
