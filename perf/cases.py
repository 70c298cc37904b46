"""The work that a user of saige_gpu has it do, as cases that can be timed:
genotype ingest, GRM builds, single and block solves, leave-one-chromosome-out
solves and whole null fits, each through saige_gpu.api.Session.

listed() are fixed cases, draw(rng) makes further ones of the same ranges,
prepare(case, seed) makes what a program holds before the call, run(state)
is one pass, work(case) the bytes and operations of a pass and
exact(case, seed) its outputs in 64 bits from plain torch.

Cohorts follow the repository's own: the 1000 x 10,000 marker fixture, C1
(10,000 samples, FP32 GRM) and C2 (100,000 samples, 150,000 markers).  The
GRMs of the large solves use 4096 to 5000 markers: a solve's cost does not
depend on the marker count once the GRM is resident.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "saige-gpu_amd"))

DEV = "cuda"
MIN_MAF, MAX_MISSING = 0.01, 0.15        # step 1's marker filter
TAU = (1.0, 0.3)
MAXITER, TOL = 500, 1e-5                 # getPCG1ofSigmaAndVector's defaults


def listed():
    return [
        # reading the fixture cohort: the smallest ingest
        {"name": "ingest_fixture", "kind": "ingest", "n": 1000, "m": 10000, "keep": 1.0},
        # a phenotype file that names 80% of the .fam's samples in an order of its own
        {"name": "ingest_subset", "kind": "ingest", "n": 30011, "m": 20003, "keep": 0.8},
        # C2's whole .bed
        {"name": "ingest_cohort", "kind": "ingest", "n": 100000, "m": 150000, "keep": 1.0},
        # the fixture's GRM, read back whole
        {"name": "grm_fixture", "kind": "grm", "n": 1000, "m": 10000, "precision": "bf16_split"},
        # build_grm's default precision, on C1's scale
        {"name": "grm_fp32", "kind": "grm", "n": 5003, "m": 20011, "precision": "fp32"},
        # a cohort's GRM as the fits use it, and the first block product with it
        {"name": "grm_cohort", "kind": "grm", "n": 40000, "m": 60000, "precision": "bf16_split"},
        # one chromosome left out of the GRM and a solve without it
        {"name": "loco_chromosome", "kind": "loco", "n": 20011, "m": 20000, "precision": "bf16_split"},
        # one right-hand side: the reference's own call, on the fixture ...
        {"name": "solve_fixture", "kind": "solve", "n": 1000, "m": 10000, "precision": "fp32"},
        # ... and on C2's samples
        {"name": "solve_cohort", "kind": "solve", "n": 100000, "m": 4096, "precision": "bf16_split"},
        # Sigma^-1 [Y, X] of one fit (three covariates) in the default GEMM arithmetic
        {"name": "block_coef", "kind": "block", "n": 10007, "m": 8000, "precision": "fp32", "k": 4, "mode": "fp32"},
        # a full block of trace probes on C2's samples, over the lower triangle
        {"name": "block_trace", "kind": "block", "n": 100000, "m": 4096, "precision": "bf16_split", "k": 64,
         "mode": "bf16x3_tri"},
        # whole null fits, batched: two binary and two quantitative phenotypes
        {"name": "null_fits", "kind": "fit", "n": 50000, "m": 5000, "precision": "bf16_split", "fits": 4,
         "nrun": 15, "mode": "bf16x3_tri"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["ingest", "ingest", "grm", "grm", "loco", "solve", "solve", "block", "block", "fit"])
    if kind == "ingest":
        n = _log(rng, 500, 100000)
        m = _log(rng, 2000, min(150000, int(4e9 / n)) if n > 20000 else 150000)
        return {"kind": kind, "n": n, "m": m, "keep": rng.choice([1.0, 1.0, 0.9, round(rng.uniform(0.3, 0.95), 3)])}
    if kind == "grm":
        precision = rng.choice(["bf16_split", "bf16_split", "fp32", "bf16"])
        n = _log(rng, 500, 10000 if precision == "fp32" else 40000)
        return {"kind": kind, "n": n, "m": _log(rng, 2000, 20000 if precision == "fp32" else 60000),
                "precision": precision}
    if kind == "loco":
        return {"kind": kind, "n": _log(rng, 1000, 30000), "m": _log(rng, 2000, 20000),
                "precision": rng.choice(["bf16_split", "bf16_split", "fp32"])}
    if kind == "solve":
        n = _log(rng, 500, 100000)
        return {"kind": kind, "n": n, "m": _log(rng, 1000, 4096 if n > 30000 else 10000),
                "precision": "bf16_split" if n > 10000 else rng.choice(["bf16_split", "fp32"])}
    if kind == "block":
        n = _log(rng, 1000, 100000)
        mode = "bf16x3_tri" if n > 30000 else rng.choice(["bf16x3_tri", "bf16x3_tri", "fp32"])
        return {"kind": kind, "n": n, "m": _log(rng, 1000, 4096 if n > 30000 else 10000),
                "precision": "bf16_split" if n > 10000 else rng.choice(["bf16_split", "fp32"]),
                "k": rng.choice([2, 4, rng.randint(5, 16), rng.randint(17, 32), rng.randint(33, 64), 64]),
                "mode": mode}
    return {"kind": kind, "n": _log(rng, 2000, 50000), "m": _log(rng, 2000, 5000), "precision": "bf16_split",
            "fits": rng.randint(1, 4), "nrun": 15, "mode": "bf16x3_tri"}


# ------------------------------------------------------------------ inputs

def _gen(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 16 + stream)
    return g


def _bed(n, m, seed):
    """A PLINK-1 .bed body (m x ceil(n/4) bytes): Binomial(2, p_j) calls,
    p_j ~ U(0.01, 0.5), 1% of them missing."""
    g = _gen(seed, 0)
    bpm = (n + 3) // 4
    p = 0.01 + 0.49 * torch.rand(m, 1, generator=g, device=DEV)
    out = torch.empty(m, bpm, dtype=torch.uint8, device=DEV)
    step = max(1, 100_000_000 // (4 * bpm))
    for j in range(0, m, step):
        q = p[j:j + step]
        u = torch.rand(q.shape[0], 4 * bpm, generator=g, device=DEV)
        code = 3 - (u < q * (2 - q)).byte() - 2 * (u < q * q).byte()     # 0, 1, 2 copies: 3, 2, 0
        code[torch.rand(u.shape, generator=g, device=DEV, out=u) < 0.01] = 1
        code[:, n:] = 0
        c = code.view(q.shape[0], bpm, 4)
        out[j:j + step] = c[:, :, 0] | (c[:, :, 1] << 2) | (c[:, :, 2] << 4) | (c[:, :, 3] << 6)
    return out


def _samples(case, seed):
    """1-based .fam rows of the phenotyped samples: all of them in order, or
    a share of them in an order of its own."""
    n = case["n"]
    if case.get("keep", 1.0) >= 1.0:
        return np.arange(1, n + 1, dtype=np.int32)
    rng = np.random.default_rng(int(seed))
    return (rng.permutation(n)[:max(1, int(n * case["keep"]))] + 1).astype(np.int32)


def _vectors(n, k, seed):
    """Working weights of a binary trait and k right-hand sides (column-major)."""
    rng = np.random.default_rng(int(seed) + 1)
    w = rng.uniform(0.05, 0.25, n).astype(np.float32)
    B = rng.standard_normal((k, n), np.float32).T
    return w, np.array(TAU, np.float32), B


def _loco_range(m):
    return m // 3, m // 3 + m // 20          # a chromosome of a twentieth of the markers


def _session(bed, n, sub):
    from saige_gpu import Session
    s = Session(0)
    s.setminMAFforGRM(MIN_MAF)
    s.setmaxMissingRateforGRM(MAX_MISSING)
    torch.cuda.synchronize()                 # the session works on a stream of its own
    if bed is not None:
        s.setgeno_device(bed.data_ptr(), n, bed.shape[0], sub)
    return s


def _phenotypes(case, bed, seed):
    """Jobs of fit_null_batch: covariates (intercept, age, sex), the genetic
    part from 200 causal markers, every second phenotype quantitative."""
    from saige_gpu import plink, synth
    n = case["n"]
    Xraw = synth.covariates(n, int(seed))
    X, _, _ = plink.covariate_transform(Xraw)
    rng = np.random.default_rng(int(seed) + 2)
    Z = _standardised(bed[torch.from_numpy(np.sort(rng.choice(case["m"], 200, replace=False))).to(DEV)],
                      np.arange(1, n + 1), qc=False)[0].cpu().numpy()
    jobs = []
    for k in range(case["fits"]):
        if k % 2 == 0:
            g = synth.polygenic(Z, 0.3, int(seed) + 10 * k)
            y, trait = synth.binary_phenotype(Xraw, g, (0.1, 0.1, 0.3, 0.3)[k], int(seed) + 10 * k), "binary"
        else:
            g = synth.polygenic(Z, 0.4, int(seed) + 10 * k)
            y, trait = synth.quantitative_phenotype(Xraw, g, 0.4, int(seed) + 10 * k), "quantitative"
        jobs.append({"trait": trait, "y": y, "X": X})
    return jobs


def prepare(case, seed):
    n, kind = case["n"], case["kind"]
    bed = _bed(n, case["m"], seed)
    sub = _samples(case, seed)
    if kind == "ingest":
        torch.cuda.synchronize()
        return {"kind": kind, "s": _session(None, n, sub), "bed": bed, "n": n, "sub": sub}
    s = _session(bed, n, sub)
    st = {"kind": kind, "s": s, "n": n}
    if kind == "grm":
        st["precision"] = case["precision"]
        st["B"] = _vectors(n, 8, seed)[2]
        return st
    s.build_grm(case["precision"])
    if "mode" in case:
        s.set_gemm_mode(case["mode"])
    if kind == "fit":
        from saige_gpu import driver
        st["jobs"] = _phenotypes(case, bed, seed)
        st["opt"] = driver.Options(nrun=case["nrun"])
        return st
    st["w"], st["tau"], B = _vectors(n, case.get("k", 1), seed)
    st["B"] = B if kind == "block" else np.ascontiguousarray(B[:, 0])
    if kind == "loco":
        st["range"] = _loco_range(s.getMsub_MAFge_minMAFtoConstructGRM())
    return st


# -------------------------------------------------------------------- runs

def run(st):
    s, kind = st["s"], st["kind"]
    if kind == "ingest":
        s.setgeno_device(st["bed"].data_ptr(), st["n"], st["bed"].shape[0], st["sub"])
        out = s.marker_stats()
        out["diag"] = s.Get_Diagof_StdGeno()
        return out
    if kind == "grm":
        s.build_grm(st["precision"])
        return s.grm_block(0, 0, st["n"], st["n"]) if st["n"] <= 2500 else s.grm_matvec(st["B"])
    if kind == "loco":
        s.setStartEndIndex(st["range"][0], st["range"][1], 0)
        return s.getPCG1ofSigmaAndVector_LOCO(st["w"], st["tau"], st["B"], MAXITER, TOL)
    if kind == "solve":
        return s.getPCG1ofSigmaAndVector(st["w"], st["tau"], st["B"], MAXITER, TOL)
    if kind == "block":
        X, iters = s.pcg_block(st["w"], st["tau"], st["B"], MAXITER, TOL)
        return {"X": X, "iters": iters}
    keys = ("theta", "coefficients", "linear_predictors", "fitted_values", "Y", "cov", "converged", "iterations")
    return [{k: r[k] for k in keys} for r in s.fit_null_batch(st["jobs"], st["opt"])]


def work(case):
    n, m, kind = case["n"], case["m"], case["kind"]
    bed = m * ((n + 3) // 4)
    tri = 2 * n * (n + 1)                    # the lower triangle of the FP32 GRM
    its = 3 + math.sqrt(n / m)               # GRM products of a solve: grows with samples per marker
    if kind == "ingest":
        return {"bytes": bed + m * ((int(n * case["keep"]) + 3) // 4) + 29 * m + 4 * n, "flops": 2 * n * m}
    if kind == "grm":
        return {"bytes": bed + 2 * tri, "flops": float(n) * (n + 1) * m}
    if kind == "loco":
        return {"bytes": bed / 20 + 2 * tri + its * tri, "flops": float(n) * (n + 1) * m / 20 + its * 2.0 * n * n}
    if kind == "solve":
        return {"bytes": its * tri, "flops": its * 2.0 * n * n}
    if kind == "block":
        return {"bytes": its * (tri + 20 * n * case["k"]), "flops": its * 2.0 * n * n * case["k"]}
    its *= 2.5 * 4                           # about three AI steps: coefficients, trace and score solves
    return {"bytes": its * tri, "flops": its * 2.0 * n * n * 10 * case["fits"]}


# ----------------------------------------------------------- 64-bit values

def _standardised(bed, sub, qc=True):
    """Z (samples x markers that pass) in FP64 and the per-marker values, by
    step 1's rules: missing calls become the rounded mean dosage, the
    frequency is taken after that, and markers are filtered on MAF and
    missing rate (compared in FP32, as they are stored)."""
    rows = torch.as_tensor(np.asarray(sub, np.int64) - 1, device=bed.device)
    codes = (bed[:, rows >> 2] >> ((rows & 3) * 2).to(torch.uint8)) & 3
    g = torch.tensor([2.0, 0.0, 1.0, 0.0], dtype=torch.float32, device=bed.device)[codes.long()]
    miss = codes == 1
    del codes
    ns = len(rows)
    ac, nm = g.sum(1, dtype=torch.float64), miss.sum(1, dtype=torch.float64)
    fill = torch.floor(ac / (ns - nm) + 0.5)
    g[miss] = fill.float()[:, None].expand_as(g)[miss]
    ac = ac + fill * nm
    f, rate = ac / (2.0 * ns), nm / ns
    std = torch.sqrt(2.0 * f * (1.0 - f))
    inv = torch.where(std > 0, 1.0 / std, torch.zeros_like(std))
    ok = (torch.minimum(f, 1.0 - f).float() >= MIN_MAF) & (rate.float() <= MAX_MISSING)
    if not qc:
        ok = torch.ones_like(ok)
    Z = ((g[ok].double() - 2.0 * f[ok, None]) * inv[ok, None]).t()
    return Z, {"freq": f, "missing_rate": rate, "inv_std": inv}


def _solve64(Z, w, tau, B, maxiter, tol):
    """The solver's recurrence in FP64, column by column: Jacobi
    preconditioner, stop when ||r||^2 <= tol."""
    m = Z.shape[1]
    w, B = torch.from_numpy(w).to(DEV).double(), torch.from_numpy(np.ascontiguousarray(B)).to(DEV).double()
    t0, t1 = (float(t) for t in tau)
    minv = 1.0 / torch.clamp(t1 * Z.square().sum(1) / m + t0 / w, min=1e-4)[:, None]
    X, R = torch.zeros_like(B), B.clone()
    Y = minv * R
    P, rz = Y.clone(), (Y * R).sum(0)
    live = R.square().sum(0) > float(np.float32(tol))
    for _ in range(maxiter):
        if not bool(live.any()):
            break
        AP = t0 * P / w[:, None] + t1 * (Z @ (Z.t() @ P)) / m
        a = torch.where(live, rz / (P * AP).sum(0), torch.zeros_like(rz))
        X += a * P
        R -= a * AP
        Y = minv * R
        new = (Y * R).sum(0)
        P = torch.where(live, Y + (new / rz) * P, P)
        rz = torch.where(live, new, rz)
        live = live & (R.square().sum(0) > float(np.float32(tol)))
    return X.cpu().numpy()


def exact(case, seed):
    n, m, kind = case["n"], case["m"], case["kind"]
    if kind == "fit":
        return None                          # a whole AI-REML fit: no plain 64-bit counterpart here
    sub = _samples(case, seed)
    bed = _bed(n, m, seed)
    if kind == "ingest":
        out = {"freq": [], "missing_rate": [], "inv_std": []}
        diag = torch.zeros(len(sub), dtype=torch.float64, device=DEV)
        step = max(1, int(2e8) // n)
        for j in range(0, m, step):
            Z, v = _standardised(bed[j:j + step], sub)
            diag += Z.square().sum(1)
            for k in out:
                out[k].append(v[k])
        out = {k: torch.cat(v).cpu().numpy() for k, v in out.items()}
        out.update({"diag": diag.cpu().numpy(), "allele_count": None, "num_missing": None, "mac": None,
                    "fill": None, "flags": None})
        return out
    if kind == "grm":
        step, K, B = max(1, int(2e8) // n), 0.0, None
        if n > 2500:
            B = torch.from_numpy(np.ascontiguousarray(_vectors(n, 8, seed)[2])).to(DEV).double()
        used = 0
        for j in range(0, m, step):
            Z = _standardised(bed[j:j + step], sub)[0]
            used += Z.shape[1]
            K = K + (Z @ Z.t() if B is None else Z @ (Z.t() @ B))
        return (K / used).cpu().numpy()
    Z = _standardised(bed, sub)[0]
    if kind == "loco":
        a, b = _loco_range(Z.shape[1])
        Z = torch.cat([Z[:, :a], Z[:, b + 1:]], 1)
    w, tau, B = _vectors(n, case.get("k", 1), seed)
    X = _solve64(Z, w, tau, B, MAXITER, TOL)
    return {"X": X, "iters": None} if kind == "block" else X[:, 0]
