"""saige_autotune times shapes that run the same kernel once: the one-half shapes
of the FP32 mode, and the depths of the lower-triangle mode at few rows."""
import pytest

from fixtures import random_bed

pytestmark = pytest.mark.gpu


def test_same_kernel_same_time(session, monkeypatch):
    N = 900
    print("case: autotune of shapes without effect", flush=True)
    body, _, _ = random_bed(N, 128, 0.01, seed=9, maf_lo=0.05, maf_hi=0.5)
    session.setminMAFforGRM(0.01)
    session.setmaxMissingRateforGRM(0.15)
    session.setgeno_bytes(body, N, 128)
    session.build_grm("fp32")
    try:
        session.set_gemm_mode("fp32")
        res = session.autotune(reps=2)
        assert len({t for *_, t in res["half_table"]}) == 1
        assert len({t for *_, t in res["table"]}) > 1
        session.set_gemm_mode("bf16x3_tri")
        for limit, times in (("20000", 2), ("0", 4)):           # k_gemm_flat; k_gemm_t16
            monkeypatch.setenv("SAIGE_TRI_FLAT_MAX", limit)
            res = session.autotune(reps=2)
            for tab in ("table", "half_table", "quarter_table"):
                by_rt = {(rt, t) for rt, _, _, t in res[tab]}
                assert len(res[tab]) == 4 and (times == 4 or len(by_rt) == 2), (limit, tab)
    finally:
        monkeypatch.delenv("SAIGE_TRI_FLAT_MAX", raising=False)
        session.set_gemm_mode("fp32")
        session.set_gemm_config(1, 1, 4)
