"""Engine launch statistics: launches over 48 columns are counted among the full
ones and by themselves, so that the 64-column ones can be told apart."""
import numpy as np
import pytest

from fixtures import random_bed

pytestmark = pytest.mark.gpu


def test_48_column_launches_are_told_apart(session):
    N = 700
    print("case: launch statistics by width", flush=True)
    body, _, _ = random_bed(N, 96, 0.01, seed=4, maf_lo=0.05, maf_hi=0.5)
    session.setminMAFforGRM(0.01)
    session.setmaxMissingRateforGRM(0.15)
    session.setgeno_bytes(body, N, 96)
    session.build_grm("bf16_split")
    B = np.random.default_rng(1).standard_normal((N, 64)).astype(np.float32)
    try:
        session.set_gemm_mode("bf16x3_tri")
        session.engine_reserve(64, 1)
        session.engine_set_system(0, np.full(N, 0.2, np.float32), np.array([1.0, 0.3], np.float32))
        for k, full, wide in ((64, 1, 0), (49, 1, 0), (48, 1, 1), (33, 1, 1), (32, 0, 0)):
            t0 = [session.engine_stats(s) for s in ("gemm_full", "gemm_48")]
            total = session.engine_stats()[1]
            session.engine_add_products(list(range(k)), [0] * k, np.asfortranarray(B[:, :k]))
            session.engine_step(1)
            session.engine_take_batch(list(range(k)))
            t1 = [session.engine_stats(s) for s in ("gemm_full", "gemm_48")]
            assert [b[1] - a[1] for a, b in zip(t0, t1)] == [full, wide], k
            assert session.engine_stats()[1] == total + 1
            assert not wide or t1[1][0] - t0[1][0] == pytest.approx(t1[0][0] - t0[0][0])
    finally:
        session.set_gemm_mode("fp32")
