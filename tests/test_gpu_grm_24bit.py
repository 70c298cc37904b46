"""Products on the split GRM's three-byte triangle, at the sizes where its
strips and row sets change: one row set (no stored strip in use), a few rows of
a second, several; the block product against the FP32 triangle bit by bit, the
single column against the GRM's own values in FP64, before and after a LOCO
range was subtracted in place and added back."""
import numpy as np
import pytest

from fixtures import random_bed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [200, 257, 513, 2305, 7200])
def test_three_byte_triangle(session, monkeypatch, N):
    M = 320
    print(f"case: three-byte triangle N={N}", flush=True)
    body, _, _ = random_bed(N, M, 0.01, seed=N, maf_lo=0.05, maf_hi=0.5)
    session.setminMAFforGRM(0.01)
    session.setmaxMissingRateforGRM(0.15)
    session.setgeno_bytes(body, N, M)
    session.build_grm("bf16_split")
    B = np.random.default_rng(N).standard_normal((N, 64)).astype(np.float32)

    def check():
        K = session.grm_block(0, 0, N, N).astype(np.float64)
        y = session.getCrossprodMatAndKin(B[:, 0])
        # N FP32 products and sums, random signs: 4 sqrt(N) roundings of sum |K b|;
        # and K's own rounding when it was read (a division)
        mag = np.abs(K) @ np.abs(B[:, 0].astype(np.float64))
        assert np.all(np.abs(y - K @ B[:, 0].astype(np.float64)) <= (4 * np.sqrt(N) + 2) * 2.0 ** -24 * mag)
        for nwv in (1, 2):
            session.set_gemm_config(nwv, 3, 8)
            for k in (64, 20, 9):
                monkeypatch.delenv("SAIGE_GEMM_S_PIECES", raising=False)
                a = session.grm_matvec(B[:, :k])
                monkeypatch.setenv("SAIGE_GEMM_S_PIECES", "3")
                b = session.grm_matvec(B[:, :k])
                assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (nwv, k)
        monkeypatch.delenv("SAIGE_GEMM_S_PIECES")

    try:
        session.set_gemm_mode("bf16x3_tri")
        check()
        if N == 2305:
            monkeypatch.setenv("SAIGE_LOCO_INPLACE", "1")
            session.setStartEndIndex(40, 139, 0)
            session.getCrossprodMatAndKin_LOCO(B[:, 0])
            check()
    finally:
        session.set_gemm_mode("fp32")
        session.set_gemm_config(1, 1, 4)
