"""The error of a single-column product on the split GRM against FP64: no larger
than that of the order in which the FP32 triangle's product (k_gemv_tri) adds,
modelled here: per 24 chunks of 256 columns a lane's sums of four products, then
the 64 lanes by halves, items one after another.  Rows of the last row set, which
are sums along their own rows of S alone."""
import numpy as np
import pytest

from fixtures import random_bed, round16

pytestmark = pytest.mark.gpu


def lanes(a):
    for o in (32, 16, 8, 4, 2, 1):
        a = a + a[..., np.arange(64) ^ o]
    return a[..., 0]


def model(S, x, R):
    """Rows of row set R of S x in k_gemv_tri's order."""
    k = (R + 23) // 24
    y = np.zeros(S.shape[0], np.float32)
    for a, b in [(R * i // k, R * (i + 1) // k) for i in range(k)] + [(R, R + 1)]:
        acc = np.zeros((S.shape[0], 64), np.float32)
        for c in range(a, b):
            v = S[:, 256 * c:256 * (c + 1)].reshape(-1, 64, 4)
            xj = x[256 * c:256 * (c + 1)].reshape(64, 4)
            t = v[:, :, 0] * xj[:, 0]
            for e in (1, 2, 3):
                t = t + v[:, :, e] * xj[:, e]
            acc = acc + t
        y = y + lanes(acc)
    return y


@pytest.mark.parametrize("signs", ["random", "equal"])
def test_split_gemv_error(session, signs):
    N, M = 20224, 320
    print(f"case: split GEMV error N={N} {signs}", flush=True)
    body, _, _ = random_bed(N, M, 0.01, seed=5, maf_lo=0.05, maf_hi=0.5)
    session.setminMAFforGRM(0.01)
    session.setmaxMissingRateforGRM(0.15)
    session.setgeno_bytes(body, N, M)
    session.build_grm("bf16_split")
    R = N // 256 - 1
    m = np.float32(session.getMsub_MAFge_minMAFtoConstructGRM())
    # S has 16 significant bits, so K = S / m, rounded to 24, names it
    S = round16((session.grm_block(256 * R, 0, 256, N).astype(np.float64) * m).astype(np.float32))
    rng = np.random.default_rng(7)
    err, ref = [], []
    for t in range(8 if signs == "random" else 64):
        b = rng.standard_normal(N).astype(np.float32)
        rows = slice(None)
        if signs == "equal":             # one row of the set meets terms of one sign
            b, rows = np.copysign(b, S[t]), slice(t, t + 1)
        exact = S[rows].astype(np.float64) @ b.astype(np.float64) / np.float64(m)
        err.append(session.getCrossprodMatAndKin(b)[256 * R:][rows] - exact)
        ref.append(model(S[rows], b, R) / m - exact)
    rms = lambda e: float(np.sqrt(np.mean(np.square(np.concatenate(e)))))
    # the spread of an RMS of n errors is 1 / sqrt(2 n) of it: five of them
    n = sum(len(e) for e in err)
    assert rms(err) <= (1 + 5 / np.sqrt(2 * n)) * rms(ref), (rms(err), rms(ref))
