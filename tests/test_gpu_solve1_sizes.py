"""The single-right-hand-side solver at the sizes where its kernels change:
samples around a workgroup's 256 rows, the few-samples path's rows per wave
(2048, 4096 and 7168 rows) and the lower-triangle GEMV beyond it; the stop
rules; the full-GRM GEMV mode."""
import numpy as np
import pytest

from fixtures import random_bed

pytestmark = pytest.mark.gpu

TAU = np.array([1.0, 0.5], np.float32)


def _load(session, N, M=96):
    body, _, _ = random_bed(N, M, 0.01, seed=N, maf_lo=0.05)
    session.setminMAFforGRM(0.01)
    session.setmaxMissingRateforGRM(0.15)
    session.setminMAC_VarianceRatio(20, -1, False)
    session.setgeno_bytes(body, N, M)
    session.build_grm("fp32")
    rng = np.random.default_rng(N + 1)
    return rng.uniform(0.05, 0.25, N).astype(np.float32), rng.standard_normal(N).astype(np.float32)


def _pcg64(K, diag, w, tau, b, maxiter, tol):
    """The recurrence of FG.cpp:2696-2792 in FP64 on K."""
    w, b = w.astype(np.float64), b.astype(np.float64)
    minv = 1.0 / np.maximum(tau[1] * diag + tau[0] / w, 1e-4)
    x, r = np.zeros(len(b)), b.copy()
    z = minv * r
    p, rz, it = z.copy(), z @ r, 0
    while r @ r > np.float32(tol) and it < maxiter:
        ap = tau[0] * p / w + tau[1] * (K @ p)
        a = rz / (p @ ap)
        x, r = x + a * p, r - a * ap
        z = minv * r
        p, rz, it = z + (z @ r) / rz * p, z @ r, it + 1
    return x, it


@pytest.mark.parametrize("mode", ["tri", "full"])
@pytest.mark.parametrize("N", [5, 256, 257, 2048, 2049, 4096, 4097, 7168, 7169])
def test_solver_sizes(session, N, mode):
    """x and the iteration count of the FP64 recurrence on the GPU's own GRM,
    stopped by the tolerance, by maxiter and before the first iteration; the
    same bits on a second call."""
    if mode == "full" and N not in (257, 7169):
        pytest.skip("the full mode has one path: two sizes")
    print(f"case: single solve N={N} {mode}", flush=True)
    w, b = _load(session, N)
    K = session.grm_block(0, 0, N, N).astype(np.float64)
    d = session.get_DiagofKin().astype(np.float64)
    try:
        session.set_gemv_mode(mode)
        for maxiter, tol in [(500, 1e-5), (3, 1e-12), (0, 1e-5), (500, 1e9)]:
            x, it = session.getPCG1ofSigmaAndVector(w, TAU, b, maxiter, tol, return_iters=True)
            x64, it64 = _pcg64(K, d, w, TAU.astype(np.float64), b, maxiter, tol)
            assert it == it64
            # the same iterate in FP32: a few roundings of N-term FP32 sums per step
            assert np.max(np.abs(x - x64)) <= 1e-4 * max(np.max(np.abs(x64)), 1e-30), (maxiter, tol)
            assert np.array_equal(x, session.getPCG1ofSigmaAndVector(w, TAU, b, maxiter, tol))
        n0 = session.engine_stats("gemv")[1]
        _, it = session.getPCG1ofSigmaAndVector(w, TAU, b, return_iters=True)
        secs, n1 = session.engine_stats("gemv")
        assert n1 - n0 == it and secs > 0.0
    finally:
        session.set_gemv_mode("tri")
