"""Single-column products and solves on the split GRM have the same bits with its
three-byte triangle and without it (from the FP32 GRM), so they do not depend on
the device memory that was free when it was built: one row set (no strip of the
copy in use), a few rows of a second, several, and items of twelve chunks."""
import numpy as np
import pytest

from fixtures import random_bed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [200, 257, 2305, 7200, 18000])
def test_same_bits_without_the_copy(session, monkeypatch, N):
    print(f"case: single-column bits without the three-byte triangle N={N}", flush=True)
    body, _, _ = random_bed(N, 256, 0.01, seed=N, maf_lo=0.05, maf_hi=0.5)
    session.setminMAFforGRM(0.01)
    session.setmaxMissingRateforGRM(0.15)
    session.setgeno_bytes(body, N, 256)
    rng = np.random.default_rng(N)
    B = rng.standard_normal((N, 3)).astype(np.float32)
    w = rng.uniform(0.05, 0.25, N).astype(np.float32)
    tau = np.array([1.0, 0.3], np.float32)
    out = {}
    for env, width in (("1", 3), ("0", 4)):
        monkeypatch.setenv("SAIGE_GRM_24BIT", env)
        session.build_grm("bf16_split")
        assert session.grm_triangle_bytes() == width
        out[width] = [session.getCrossprodMatAndKin(B[:, j]) for j in range(3)]
        out[width].append(session.getPCG1ofSigmaAndVector(w, tau, B[:, 0]))
    for a, b in zip(out[3], out[4]):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
