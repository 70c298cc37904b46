"""Rows and columns of S past the samples are zero whatever the operand form, the
tile and the pass (store, add, subtract): the products rely on it.  S is not
visible past the samples through the C ABI, so the SYRK is called directly."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BUILD = "_ZN5saige12SyrkOperands5buildEP12ihipStream_tiPKhPK15HIP_vector_typeIfLj4EEllllll"
RELEASE = "_ZN5saige12SyrkOperands7releaseEv"
SYRK = "_ZN5saige14launch_syrk_pkEP12ihipStream_tRKNS_12SyrkOperandsEPK15HIP_vector_typeIiLj2EEPfPKfiiPh"


@pytest.mark.parametrize("form", [0, 1, 2], ids=["hi", "split", "fp32"])
@pytest.mark.parametrize("tile", [64, 128, 256])
@pytest.mark.parametrize("N", [1, 300, 511])
def test_padding_is_zero(session, N, tile, form):
    print(f"case: padding of S N={N} tile={tile} form={form}", flush=True)
    from saige_gpu import _lib
    lib = _lib.load()
    build, release, syrk = (getattr(lib, n) for n in (BUILD, RELEASE, SYRK))
    p, i64 = ctypes.c_void_p, ctypes.c_int64
    build.argtypes = [p, p, ctypes.c_int, p, p] + [i64] * 6
    release.argtypes, release.restype = [p], None
    syrk.argtypes = [p, p, p, p, p, ctypes.c_int, ctypes.c_int, p]
    M, Np, ldp = 100, (N + 255) // 256 * 256, (N + 511) // 512 * 128
    rng = np.random.default_rng(N)
    code = np.zeros((M + 128, 4 * ldp), np.uint8)
    g = rng.integers(0, 3, (M, N))
    code[:M, :N] = np.array([3, 2, 0], np.uint8)[g]
    packed = code[:, 0::4] | code[:, 1::4] << 2 | code[:, 2::4] << 4 | code[:, 3::4] << 6
    f = rng.uniform(0.05, 0.5, M)
    lut = np.zeros((M + 128, 4), np.float32)
    lut[:M, :3] = (np.arange(3)[None] - 2 * f[:, None]) / np.sqrt(2 * f * (1 - f))[:, None]
    tiles = np.array([(i, j) for i in range(Np // tile) for j in range(i + 1)], np.int32)
    bufs = [session.alloc_device(b) for b in (packed.nbytes, lut.nbytes, tiles.nbytes, 4 * Np * Np)]
    op = ctypes.create_string_buffer(512)            # a SyrkOperands of zeros, its initial state
    try:
        for d, h in zip(bufs, (packed, lut, tiles)):
            session.copy_bytes_to_device(d, np.ascontiguousarray(h))
        d_packed, d_lut, d_tiles, d_S = bufs
        assert build(op, None, form, d_packed, d_lut, M, N, Np, ldp, 0, M) == 0
        for accumulate in (0, 1, -1):
            assert syrk(None, op, d_tiles, d_S, d_S, accumulate, tile, None) == 0
            S = session.copy_device_to_host(d_S, 4 * Np * Np).view(np.float32).reshape(Np, Np)
            assert np.any(S[:N, :N]) or accumulate
            assert not np.any(S[N:]) and not np.any(S[:, N:]), accumulate
    finally:
        release(op)
        for d in bufs:
            session.free_device(d)
