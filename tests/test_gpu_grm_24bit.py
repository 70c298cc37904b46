"""Lower-triangle products.  On the split GRM's three-byte triangle, at the
sizes where its strips and row sets change: one row set (no stored strip in use), a few rows of
a second, several; the block product against the FP32 triangle bit by bit, the
single column against the GRM's own values in FP64, before and after a LOCO
range was subtracted in place and added back; and launches of every width, for
each depth and workgroup."""
import numpy as np
import pytest

from fixtures import random_bed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,tile", [(200, "64"), (257, "128"), (513, "64"), (513, "256"), (2305, "128"), (7200, "256")])
def test_three_byte_triangle(session, monkeypatch, N, tile):
    M = 320
    monkeypatch.setenv("SAIGE_SYRK_TILE", tile)
    print(f"case: three-byte triangle N={N} tile={tile}", flush=True)
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


@pytest.mark.parametrize("prec", ["bf16_split", "fp32"])
@pytest.mark.parametrize("N", [200, 700, 4700])
def test_launch_widths(session, N, prec):
    """A column's bits do not depend on its launch's width: blocks of 33 and 48
    columns (48-column launches), of 49 (64) and 20 (32), and engine products of
    34 and 48 occupied slots spread over the block, against the 64-column
    launch."""
    print(f"case: launch widths N={N} {prec}", flush=True)
    body, _, _ = random_bed(N, 320, 0.01, seed=N, maf_lo=0.05, maf_hi=0.5)
    session.setminMAFforGRM(0.01)
    session.setmaxMissingRateforGRM(0.15)
    session.setgeno_bytes(body, N, 320)
    session.build_grm(prec)
    rng = np.random.default_rng(N)
    B = rng.standard_normal((N, 64)).astype(np.float32)
    w = rng.uniform(0.05, 0.25, N).astype(np.float32)
    try:
        session.set_gemm_mode("bf16x3_tri")
        for nwv in (1, 2):
            for pd in (1, 3):
                session.set_gemm_config(nwv, pd, 8)
                full = session.grm_matvec(B)
                for k in (20, 33, 48, 49):
                    y = session.grm_matvec(B[:, :k])
                    assert np.array_equal(y.view(np.uint32), full[:, :k].view(np.uint32)), (nwv, pd, k)
                session.engine_reserve(64, 1)
                session.engine_set_system(0, w, np.array([1.0, 0.3], np.float32))
                out = {}
                for slots in (range(64), range(0, 64, 2), sorted(set(range(0, 64, 2)) | {5, 63}),
                              [k for k in range(64) if k % 4 != 1]):
                    slots = list(slots)
                    session.engine_add_products(slots, [0] * len(slots), np.asfortranarray(B[:, slots]))
                    done, _ = session.engine_step(1)
                    assert all(done[s] for s in slots)
                    y = session.engine_take_batch(slots)
                    if len(slots) == 64:
                        out = y
                    else:
                        assert np.array_equal(y.view(np.uint32), out[:, slots].view(np.uint32)), (nwv, pd, len(slots))
    finally:
        session.set_gemm_mode("fp32")
        session.set_gemm_config(1, 1, 4)
