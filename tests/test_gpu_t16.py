"""The walk of the lower triangle (k_gemm_t16) at the sizes where few rows take
k_gemm_flat instead: every test here turns k_gemm_flat off.  The walk on the
three-byte triangle against the FP32 one bit by bit for both workgroups, both
depths and every width, before and after a leave-out range was subtracted in
place and added back; and the lower-triangle tests of the other files again."""
import numpy as np
import pytest

from fixtures import random_bed
from test_gpu_grm_24bit import test_launch_widths as launch_widths
from test_gpu_grm_pcg import (grm1000, grm1000_ref,  # noqa: F401
                              test_gemm_bf16x3_tri_mode as tri_mode, test_gemm_tri_mode_many_items as many_items,
                              test_scattered_slots_run_narrow_launches as scattered_slots,
                              test_split_grm_two_piece_gemm as two_piece)

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def no_flat(monkeypatch):
    monkeypatch.setenv("SAIGE_TRI_FLAT_MAX", "0")


@pytest.mark.parametrize("N,tile", [(200, "64"), (257, "128"), (513, "64"), (513, "256"), (2305, "128"), (7200, "256")])
def test_walk_of_the_three_byte_triangle(session, monkeypatch, N, tile):
    M = 320
    monkeypatch.setenv("SAIGE_SYRK_TILE", tile)
    print(f"case: walk of the three-byte triangle N={N} tile={tile}", flush=True)
    body, _, _ = random_bed(N, M, 0.01, seed=N, maf_lo=0.05, maf_hi=0.5)
    session.setminMAFforGRM(0.01)
    session.setmaxMissingRateforGRM(0.15)
    session.setgeno_bytes(body, N, M)
    session.build_grm("bf16_split")
    B = np.random.default_rng(N).standard_normal((N, 64)).astype(np.float32)

    def check():
        for rt in (1, 2):
            first = {}
            for pd in (1, 3):
                session.set_gemm_config(rt, pd, 8)
                for k in (64, 40, 20, 9):
                    monkeypatch.delenv("SAIGE_GEMM_S_PIECES", raising=False)
                    assert session.grm_triangle_bytes() == 3
                    a = session.grm_matvec(B[:, :k])
                    monkeypatch.setenv("SAIGE_GEMM_S_PIECES", "3")         # the FP32 triangle
                    b = session.grm_matvec(B[:, :k])
                    assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (rt, pd, k)
                    a0 = first.setdefault(k, a)
                    assert np.array_equal(a.view(np.uint32), a0.view(np.uint32)), (rt, pd, k)
        monkeypatch.delenv("SAIGE_GEMM_S_PIECES")

    try:
        session.set_gemm_mode("bf16x3_tri")
        check()
        monkeypatch.setenv("SAIGE_LOCO_INPLACE", "1")
        session.setStartEndIndex(40, 139, 0)
        session.getCrossprodMatAndKin_LOCO(B[:, 0])
        assert session.grm_triangle_bytes() == 4
        session.getCrossprodMatAndKin(B[:, 0])                             # the range goes back
        check()
    finally:
        session.set_gemm_mode("fp32")
        session.set_gemm_config(1, 1, 4)


@pytest.mark.parametrize("prec", ["bf16_split", "fp32"])
@pytest.mark.parametrize("N", [200, 700, 4700])
def test_walk_launch_widths(session, N, prec):
    launch_widths(session, N, prec)


def test_walk_tri_mode(session, grm1000):  # noqa: F811
    tri_mode(session, grm1000)


def test_walk_scattered_slots(session, grm1000):  # noqa: F811
    scattered_slots(session, grm1000)


def test_walk_many_items(session):
    many_items(session)


def test_walk_two_piece(session, monkeypatch):
    two_piece(session, monkeypatch)
