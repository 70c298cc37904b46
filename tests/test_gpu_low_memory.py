"""Calls that have to succeed with little device memory left: the rest of the
device is held by untouched allocations while they run."""
import contextlib
import ctypes
import time

import numpy as np
import pytest

from fixtures import random_bed

pytestmark = pytest.mark.gpu


def hip_runtime():
    return ctypes.CDLL("libamdhip64.so")


def free_memory():
    """Free device memory once it has stopped changing: the driver returns freed
    blocks some time after the call."""
    f, t = ctypes.c_size_t(), ctypes.c_size_t()
    last, same = -1, 0
    while same < 8:
        assert hip_runtime().hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        same = same + 1 if f.value == last else 0
        last = f.value
        time.sleep(0.02)
    return last


@contextlib.contextmanager
def only_free(left):
    """Holds device memory so that about `left` bytes stay free."""
    hip = hip_runtime()
    hip.hipMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
    hip.hipFree.argtypes = [ctypes.c_void_p]

    def take(n):
        p = ctypes.c_void_p()
        return p if hip.hipMalloc(ctypes.byref(p), n) == 0 else None

    # what hipMemGetInfo calls free is less than what can be allocated: hold
    # `left`, take all there is, let `left` go
    free_memory()
    room, held, piece = take(left), [], 1 << 38
    try:
        assert room
        while piece >= 1 << 22:
            p = take(piece)
            if p:
                held.append(p)
            else:
                piece //= 2
        hip.hipFree(room)
        hip.hipGetLastError()
        yield
    finally:
        for p in held:
            hip.hipFree(p)


def load(session, N, M, seed=3):
    body, _, _ = random_bed(N, M, 0.01, seed=seed, maf_lo=0.05, maf_hi=0.5)
    session.setminMAFforGRM(0.01)
    session.setmaxMissingRateforGRM(0.15)
    session.setgeno_bytes(body, N, M)


def test_fp32_grm_passes_add_up(session, monkeypatch):
    """The FP32 GRM in passes of 128 markers is the FP32 sum of the passes' GRMs
    (powers of two of markers, so that K names S exactly)."""
    N = 700
    print("case: FP32 GRM in passes", flush=True)
    body, _, _ = random_bed(N, 256, 0.0, seed=2, maf_lo=0.1, maf_hi=0.5)
    body = body.reshape(256, -1)
    session.setminMAFforGRM(0.01)
    session.setmaxMissingRateforGRM(0.15)
    part = []
    for j in (0, 128):
        session.setgeno_bytes(body[j:j + 128].ravel(), N, 128)
        assert session.getMsub_MAFge_minMAFtoConstructGRM() == 128
        session.build_grm("fp32")
        part.append(session.grm_block(0, 0, N, N) * np.float32(128))
    session.setgeno_bytes(body.ravel(), N, 256)
    monkeypatch.setenv("SAIGE_GRM_PANEL_MARKERS", "128")
    session.build_grm("fp32")
    S = session.grm_block(0, 0, N, N) * np.float32(256)
    assert np.array_equal(S, part[0] + part[1])
    # a range of two passes, taken off
    session.setStartEndIndex(30, 230, 0)
    monkeypatch.delenv("SAIGE_GRM_PANEL_MARKERS")
    e = np.zeros(N, np.float32)
    e[5] = 1.0
    y = session.getCrossprodMatAndKin_LOCO(e)
    session.setStartEndIndex(30, 230, 0)
    z = session.getCrossprodMatAndKin_LOCO(e)
    # FP32 sums of at most 256 products of |z| < 7 in two groupings
    assert np.max(np.abs(y - z)) <= 256 * 49 * 256 / 55 * 2.0 ** -24


def test_fp32_grm_without_room_for_all_markers(session):
    """Memory for a part of the markers' operands only: the build goes in passes."""
    N, M = 1000, 1 << 19
    print("case: FP32 GRM with little memory", flush=True)
    rng = np.random.default_rng(4)
    body = rng.integers(0, 256, (4096, (N + 3) // 4), dtype=np.uint8)
    session.setminMAFforGRM(0.0)
    session.setmaxMissingRateforGRM(1.0)
    try:
        session.setgeno_bytes(np.tile(body, (M // 4096, 1)).ravel(), N, M)
        session.build_grm("fp32")
        K = session.grm_block(0, 0, N, N)
        # all operands: 1024 / 4 bytes of genotypes and 56 of tables a marker
        with only_free(96 << 20):
            assert free_memory() < M * (256 + 56)
            session.build_grm("fp32")
        L = session.grm_block(0, 0, N, N)
        # FP32 sums over M markers in two groupings, random signs off the diagonal
        assert np.max(np.abs(K - L)) <= 4 * np.sqrt(M) * 2.0 ** -24 * np.max(np.abs(K))
        assert np.any(K != L)
    finally:
        load(session, 200, 64)


def many_markers(N, M):
    """A .bed body of M markers that repeats 1000 random ones."""
    body = np.random.default_rng(N).integers(0, 256, (1000, (N + 3) // 4), dtype=np.uint8)
    return np.tile(body, (M // 1000, 1)).ravel()


def test_kept_blocks_are_bounded(session):
    """A cohort of half the last one's size does not keep the last one's memory:
    at most 64 MB too much in each of an ingest's eight blocks."""
    print("case: kept blocks' bound", flush=True)
    N, large, small = 4000, 1250000, 650000
    session.setminMAFforGRM(0.0)
    session.setmaxMissingRateforGRM(1.0)
    try:
        load(session, 200, 64)
        session.setminMAFforGRM(0.0)
        session.setmaxMissingRateforGRM(1.0)
        before = free_memory()
        session.setgeno_bytes(many_markers(N, small), N, small)
        fresh = before - free_memory()
        session.setgeno_bytes(many_markers(N, large), N, large)
        session.setgeno_bytes(many_markers(N, small), N, small)
        assert before - free_memory() <= fresh + 8 * (64 << 20)
    finally:
        load(session, 200, 64)


def test_ingest_gives_up_kept_blocks(session):
    """A cohort that fits only without the last one's blocks."""
    print("case: ingest beside kept blocks", flush=True)
    session.setminMAFforGRM(0.0)
    session.setmaxMissingRateforGRM(1.0)
    try:
        session.setgeno_bytes(many_markers(4000, 1250000), 4000, 1250000)      # 1.3 GB of genotypes
        M = 7000000
        with only_free(200 << 20):
            # 0.26 GB of lists and stats first, then 1.0 GB of genotypes and tables
            session.setgeno_bytes(many_markers(8, M), 8, M)
        assert session.getMsub_MAFge_minMAFtoConstructGRM() == M
    finally:
        load(session, 200, 64)


COPY = 632 * 631 // 2 * 3072                         # bytes: 32 x 32 blocks left of the diagonal


@pytest.fixture
def split_grm(session):
    """A split GRM of 20,224 samples: 1.6 GB, its three-byte triangle 0.6."""
    session.setminMAFforGRM(0.0)
    session.setmaxMissingRateforGRM(1.0)
    session.setgeno_bytes(many_markers(20224, 1000), 20224, 1000)
    session.set_gemm_mode("bf16x3_tri")
    session.build_grm("bf16_split")
    assert session.grm_triangle_bytes() == 3
    yield np.random.default_rng(1).standard_normal((20224, 20)).astype(np.float32)
    session.set_gemm_mode("fp32")
    load(session, 200, 64)


def test_three_byte_copy_is_given_back(session, split_grm):
    """Allocations of the context take the copy's memory when there is no other,
    and the products' bits stay."""
    print("case: the three-byte triangle's memory", flush=True)
    B = split_grm
    free = free_memory()
    assert session.device_memory()[0] - free == COPY
    y = session.getCrossprodMatAndKin(B[:, 0])
    with only_free(64 << 20):
        Y = session.grm_matvec(B)                    # 0.15 GB of scratch on its first call
        assert session.grm_triangle_bytes() == 4
        assert np.array_equal(session.getCrossprodMatAndKin(B[:, 0]), y)
    session.build_grm("bf16_split")
    assert session.grm_triangle_bytes() == 3
    assert np.array_equal(session.grm_matvec(B), Y)
    with only_free(64 << 20):
        p = session.alloc_device(400 << 20)
        session.free_device(p)
        assert session.grm_triangle_bytes() == 4
        with pytest.raises(Exception):               # nothing left to give
            session.alloc_device(2 << 30)
        assert np.array_equal(session.getCrossprodMatAndKin(B[:, 0]), y)


def test_second_grm_takes_the_copys_memory(session, split_grm):
    """A leave-out range gets its own GRM (1.6 GB, with 4 GB to spare) where it
    fits without the copy."""
    print("case: a leave-out GRM beside the three-byte triangle", flush=True)
    with only_free((4 << 30) + 1300000000):
        before = free_memory()
        session.setStartEndIndex(10, 40, 0)
        assert session.grm_triangle_bytes() == 4
        assert before + COPY - free_memory() > 1500 << 20
