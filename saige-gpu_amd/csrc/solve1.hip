// The single-right-hand-side solver (getPCG1ofSigmaAndVector, FG.cpp:2593-2809)
// and the vectors of every single-column product.
//
// One solve is a chain of launches without a host round trip in it.  Iteration
// j starts by deciding, from the FP64 partial sums the launch before left,
// whether the solve is over and beta; every workgroup forms those scalars for
// itself (the same partials in the same order), one also publishes them to the
// host.  The host stays P1_AHEAD iterations ahead of the last one published,
// and launches that find the solve over return at once.  Per iteration:
// * few samples (p1_small): k_p1_row (decide, p = z + beta p in LDS, its rows'
//   Sigma p from all of S, p'Ap) and k_p1_update (alpha, x, r, z, partial sums):
//   two launches, where the whole of S comes from the caches;
// * else: k_p1_dir (decide, p), the GEMV and its epilogue (Sigma p, p'Ap),
//   k_p1_update.
// 1000 samples: 76 us per solve of three iterations; six launches and a host
// round trip per iteration took 277 us.
#include "saige_internal.hpp"

#include <algorithm>

#pragma clang fp contract(off)

namespace saige {

namespace {

constexpr int P1_ROWS = 256;      // rows per workgroup of the vector kernels

// the workgroup's sum of v in a fixed tree order, to every thread
__device__ __forceinline__ double wg_sum(double v, double* sm) {
    const int tid = threadIdx.x;
    sm[tid] = v;
    for (int s = 128; s >= 1; s >>= 1) {
        __syncthreads();
        if (tid < s) sm[tid] += sm[tid + s];
    }
    __syncthreads();
    const double r = sm[0];
    __syncthreads();
    return r;
}

// the sums of partial[np][2] (r'z, r'r), every thread gets both
__device__ __forceinline__ void wg_sum2(const double* partial, int np, double2* sm, double& a, double& b) {
    const int tid = threadIdx.x;
    double2 v = make_double2(0.0, 0.0);
    for (int p = tid; p < np; p += 256) {
        v.x += partial[2 * p];
        v.y += partial[2 * p + 1];
    }
    sm[tid] = v;
    for (int s = 128; s >= 1; s >>= 1) {
        __syncthreads();
        if (tid < s) {
            sm[tid].x += sm[tid + s].x;
            sm[tid].y += sm[tid + s].y;
        }
    }
    __syncthreads();
    a = sm[0].x;
    b = sm[0].y;
}

// Iteration j's decision: true when the solve is over (the loop of
// FG.cpp:2696, after beta of FG.cpp:2770).  rz of iteration j is kept at
// st->rz[j & 1], so workgroups that still read the one before see it; over
// keeps the iteration number, so that a launch is ended by the decision of an
// earlier one only, never halfway by its own.
__device__ __forceinline__ bool p1_decide(int j, const double* partial, int np, P1State* st, P1Host* h, int maxiter,
                                          double tol, double2* sm, float& beta) {
    if (st->over < j) return true;
    double rz, rr;
    wg_sum2(partial, np, sm, rz, rr);
    beta = j == 0 ? 0.0f : (float)(rz / st->rz[(j + 1) & 1]);
    const bool done = !(rr > tol && j < maxiter);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        st->rz[j & 1] = rz;
        if (done) st->over = j;
        h->it = j;
        if (done) h->done = 1;
        __threadfence_system();
        h->decided = j;
    }
    return done;
}

// Sigma's diagonal as k_sigma_setup forms it, and the start x = 0, r = b,
// z = minv r (FG.cpp:2615-2690); the first direction is z.
__global__ __launch_bounds__(256) void k_p1_init(const float* __restrict__ w, const float* __restrict__ b,
                                                 const float* __restrict__ diag, int64_t Nnm, float tau0, float tau1,
                                                 float mqc, int diag_one, float* __restrict__ winv,
                                                 float* __restrict__ minv, float* __restrict__ x,
                                                 float* __restrict__ r, float* __restrict__ z,
                                                 double* __restrict__ partial, P1State* st) {
    __shared__ double2 sm[256];
    const int tid = threadIdx.x;
    const int64_t i = (int64_t)blockIdx.x * P1_ROWS + tid;
    float wi = 0.f, mi = 0.f, ri = 0.f;
    if (i < Nnm) {
        wi = div_rn(1.0f, w[i]);
        mi = div_rn(1.0f, sigma_diag(w[i], diag, i, tau0, tau1, mqc, diag_one));
        ri = b[i];
    }
    const float zi = __fmul_rn(mi, ri);
    winv[i] = wi;
    minv[i] = mi;
    x[i] = 0.0f;
    r[i] = ri;
    z[i] = zi;
    sm[tid] = make_double2((double)zi * (double)ri, (double)ri * (double)ri);
    for (int s = 128; s >= 1; s >>= 1) {
        __syncthreads();
        if (tid < s) {
            sm[tid].x += sm[tid + s].x;
            sm[tid].y += sm[tid + s].y;
        }
    }
    if (tid == 0) {
        partial[2 * blockIdx.x] = sm[0].x;
        partial[2 * blockIdx.x + 1] = sm[0].y;
        if (blockIdx.x == 0) st->over = INT32_MAX;
    }
}

// p = z + beta p (FG.cpp:2772)
__global__ __launch_bounds__(256) void k_p1_dir(int j, const double* __restrict__ partial, int np, P1State* st,
                                                P1Host* h, int maxiter, double tol, const float* __restrict__ z,
                                                float* __restrict__ p) {
    __shared__ double2 sm[256];
    float beta;
    if (p1_decide(j, partial, np, st, h, maxiter, tol, sm, beta)) return;
    const int64_t i = (int64_t)blockIdx.x * P1_ROWS + threadIdx.x;
    p[i] = j == 0 ? z[i] : __fadd_rn(z[i], __fmul_rn(beta, p[i]));
}

// alpha = r'z / p'Ap (FG.cpp:2710); x += alpha p; r -= alpha Ap; z = minv r
// (FG.cpp:2734-2767) and the partial sums r'z, r'r
__global__ __launch_bounds__(256) void k_p1_update(int j, const double* __restrict__ pap, int npap,
                                                   const P1State* __restrict__ st, const float* __restrict__ minv,
                                                   const float* __restrict__ p, const float* __restrict__ ap,
                                                   float* __restrict__ x, float* __restrict__ r,
                                                   float* __restrict__ z, double* __restrict__ partial) {
    __shared__ double2 sm[256];
    if (st->over <= j) return;
    const int tid = threadIdx.x;
    const int64_t i = (int64_t)blockIdx.x * P1_ROWS + tid;
    const float pi = p[i], api = ap[i], xi = x[i], ri = r[i], mi = minv[i];
    double v = 0.0;
    for (int k = tid; k < npap; k += 256) v += pap[k];
    const float a = (float)(st->rz[j & 1] / wg_sum(v, reinterpret_cast<double*>(sm)));
    const float r1 = __fsub_rn(ri, __fmul_rn(a, api));
    const float z1 = __fmul_rn(mi, r1);
    x[i] = __fadd_rn(xi, __fmul_rn(a, pi));
    r[i] = r1;
    z[i] = z1;
    sm[tid] = make_double2((double)z1 * (double)r1, (double)r1 * (double)r1);
    for (int s = 128; s >= 1; s >>= 1) {
        __syncthreads();
        if (tid < s) {
            sm[tid].x += sm[tid + s].x;
            sm[tid].y += sm[tid + s].y;
        }
    }
    if (tid == 0) {
        partial[2 * blockIdx.x] = sm[0].x;
        partial[2 * blockIdx.x + 1] = sm[0].y;
    }
}

// The few-samples iteration's first launch: a workgroup of four waves owns 4*RW
// rows.  It reads the first of its rows of S before the decision, forms the
// whole direction p in LDS (p_prev is the other buffer: workgroups that are
// still reading it must not see this one's), and its rows' Sigma p.  The launch
// that ends the solve stores x to the host.
template <int RW>
__global__ __launch_bounds__(256) void k_p1_row(int j, const float* __restrict__ S, int64_t ld, int64_t Nnm,
                                                const double* __restrict__ partial, int np, P1State* st, P1Host* h,
                                                int maxiter, double tol, const float* __restrict__ z,
                                                const float* __restrict__ p_prev, float* __restrict__ p_next,
                                                VecArgs a, float* __restrict__ ap, double* __restrict__ pap,
                                                const float* __restrict__ x, float* __restrict__ x_out) {
    extern __shared__ float4 sp4[];                       // p, ld floats
    __shared__ double2 sm[256];
    constexpr int PF = 4;                                 // float4 of each row requested ahead
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int64_t row0 = (int64_t)blockIdx.x * 4 * RW, rw = row0 + wv * RW;
    const int n4 = (int)(ld / 4);
    const float4* Sr = reinterpret_cast<const float4*>(S + rw * ld);
    float4 pre[RW][PF];
#pragma unroll
    for (int q = 0; q < RW; q++)
#pragma unroll
        for (int c = 0; c < PF; c++) pre[q][c] = Sr[(int64_t)q * n4 + min(lane + 64 * c, n4 - 1)];
    float beta;
    const bool late = st->over < j;                       // ended by an earlier launch, which stored x
    if (p1_decide(j, partial, np, st, h, maxiter, tol, sm, beta)) {
        if (!late && tid < 4 * RW) x_out[row0 + tid] = x[row0 + tid];
        return;
    }
    const float4* z4 = reinterpret_cast<const float4*>(z);
    const float4* q4 = reinterpret_cast<const float4*>(p_prev);
    for (int i = tid; i < n4; i += 256) {
        float4 v = z4[i];
        if (j > 0) {
            const float4 o = q4[i];
            v.x = __fadd_rn(v.x, __fmul_rn(beta, o.x));
            v.y = __fadd_rn(v.y, __fmul_rn(beta, o.y));
            v.z = __fadd_rn(v.z, __fmul_rn(beta, o.z));
            v.w = __fadd_rn(v.w, __fmul_rn(beta, o.w));
        }
        sp4[i] = v;
    }
    __syncthreads();
    const float* sp = reinterpret_cast<const float*>(sp4);
    if (tid < 4 * RW) p_next[row0 + tid] = sp[row0 + tid];
    float acc[RW];
#pragma unroll
    for (int q = 0; q < RW; q++) acc[q] = 0.0f;
    auto add = [&](int q, const float4& s, const float4& p) {
        acc[q] = __fmaf_rn(s.x, p.x, acc[q]);
        acc[q] = __fmaf_rn(s.y, p.y, acc[q]);
        acc[q] = __fmaf_rn(s.z, p.z, acc[q]);
        acc[q] = __fmaf_rn(s.w, p.w, acc[q]);
    };
#pragma unroll
    for (int c = 0; c < PF; c++)
        if (lane + 64 * c < n4) {
            const float4 p = sp4[lane + 64 * c];
#pragma unroll
            for (int q = 0; q < RW; q++) add(q, pre[q][c], p);
        }
#pragma unroll 4
    for (int c = lane + 64 * PF; c < n4; c += 64) {
        const float4 p = sp4[c];
#pragma unroll
        for (int q = 0; q < RW; q++) add(q, Sr[(int64_t)q * n4 + c], p);
    }
    double d = 0.0;
#pragma unroll
    for (int q = 0; q < RW; q++) {
        float y = acc[q];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) y += __shfl_xor(y, o, 64);
        if (lane == q) {
            const float p = sp[rw + q];
            const float o = rw + q < Nnm ? sigma_elem(p, y, a.winv[rw + q], a.tau0, a.tau1, a.mqc) : 0.0f;
            ap[rw + q] = o;
            d = (double)p * (double)o;
        }
    }
    const double s = wg_sum(lane < RW ? d : 0.0, reinterpret_cast<double*>(sm));
    if (tid == 0) pap[blockIdx.x] = s;
}

// Rows up to which a solve reads all of S (the caches hold it), two launches
// per iteration.  us per iteration at N = 1000, 3000, 5000, 7000, 8000: 15, 20,
// 33, 44, 62 against 60, 65, 62, 74, 75 with the lower-triangle GEMV's four
// launches, which reads half the bytes.
constexpr int64_t P1_SMALL_MAX = 7168;
int small_rows(int64_t Npad) { return Npad <= 2048 ? 1 : (Npad <= 4096 ? 2 : 4); }

constexpr int P1_AHEAD = 2;       // iterations enqueued past the last decided one

}  // namespace

hipError_t Solve1::reserve(int64_t Npad_) {
    if (block && Npad == Npad_) return hipSuccess;
    release();
    const int64_t np = std::max<int64_t>(gemv_max_parts(Npad_), Npad_ / P1_ROWS);
    // vectors, then the FP64 partial sums and the state
    const int64_t bytes = 4 * 10 * Npad_ + 8 * (np + 2 * (Npad_ / P1_ROWS)) + 256;
    hipError_t e = hipMalloc(&block, (size_t)bytes);
    if (e == hipSuccess) e = hipHostMalloc((void**)&host, sizeof(P1Host), hipHostMallocDefault);
    if (e == hipSuccess && Npad_ <= P1_SMALL_MAX)
        e = hipHostMalloc((void**)&hvec, sizeof(float) * (size_t)(3 * Npad_), hipHostMallocDefault);
    for (int k = 0; k < EVENTS && e == hipSuccess; k++) e = hipEventCreate(&ev[k]);
    if (e != hipSuccess) {
        release();
        return e;
    }
    Npad = Npad_;
    float* f = static_cast<float*>(block);
    for (float** v : {&w, &b, &winv, &minv, &x, &r, &z, &p, &p2, &ap}) {
        *v = f;
        f += Npad;
    }
    pap = reinterpret_cast<double*>(f);
    partial = pap + np;
    st = reinterpret_cast<P1State*>(partial + 2 * (Npad / P1_ROWS));
    return hipSuccess;
}

void Solve1::release() {
    if (block) (void)hipFree(block);
    if (host) (void)hipHostFree(host);
    if (hvec) (void)hipHostFree(hvec);
    for (hipEvent_t& e : ev) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
    const double s = seconds;
    const int64_t n = launches;
    *this = Solve1{};
    seconds = s;
    launches = n;
}

hipError_t solve1(hipStream_t s, Solve1& v, const float* w_host, const float* b_host, float* x_host, GrmMat S,
                  const float* diag, int64_t Nnm, float tau0, float tau1, float m, int diag_one, int maxiter,
                  double tol, const GemvPlan* tri, int* iters) {
    const int64_t Np = v.Npad;
    const int nb = (int)(Np / P1_ROWS);
    const bool small = tri && Np <= P1_SMALL_MAX;
    const int rw = small_rows(Np);
    VecArgs a;
    a.winv = v.winv;
    a.tau0 = tau0;
    a.tau1 = tau1;
    a.mqc = m;
    a.mode = 1;
    a.over = &v.st->over;
    P1Host* h = v.host;
    h->decided = -1;
    h->it = 0;
    h->done = 0;
    // a small solve's vectors are read and written in page-locked memory, which
    // spares the copies' round trips; longer ones are copied
    const float *w = v.w, *b = v.b;
    if (small) {
        std::copy(w_host, w_host + Nnm, v.hvec);
        std::copy(b_host, b_host + Nnm, v.hvec + Np);
        w = v.hvec;
        b = v.hvec + Np;
    } else {
        hipError_t c = hipMemcpyAsync(v.w, w_host, 4 * Nnm, hipMemcpyHostToDevice, s);
        if (c == hipSuccess) c = hipMemcpyAsync(v.b, b_host, 4 * Nnm, hipMemcpyHostToDevice, s);
        if (c != hipSuccess) return c;
    }
    hipLaunchKernelGGL(k_p1_init, dim3(nb), dim3(256), 0, s, w, b, diag, Nnm, tau0, tau1, m, diag_one, v.winv,
                       v.minv, v.x, v.r, v.z, v.partial, v.st);
    hipError_t e = hipGetLastError();
    // the products' device time: an event pair around each GEMV (read when its
    // pair comes round again or at the end), or around a small solve's whole
    // chain, whose products are not launches of their own
    constexpr int PAIRS = Solve1::EVENTS / 2;
    auto add_time = [&](int k) -> hipError_t {
        float ms = 0.f;
        const hipError_t t = hipEventElapsedTime(&ms, v.ev[2 * (k % PAIRS)], v.ev[2 * (k % PAIRS) + 1]);
        if (t == hipSuccess) v.seconds += ms * 1e-3;
        return t;
    };
    if (e == hipSuccess && small) e = hipEventRecord(v.ev[0], s);
    int j = 0;
    for (; e == hipSuccess; j++) {
        a.iter = j;
        int npap = nb;
        const float* p = v.p;
        if (small) {
            float* nx = (j & 1) ? v.p2 : v.p;
            const float* pv = (j & 1) ? v.p : v.p2;
            npap = (int)(Np / (4 * rw));
            const size_t lds = sizeof(float) * (size_t)Np;
            auto go = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, dim3((unsigned)npap), dim3(256), lds, s, j, S.S, Np, Nnm, v.partial, nb, v.st,
                                   h, maxiter, tol, v.z, pv, nx, a, v.ap, v.pap, v.x, v.hvec + 2 * Np);
            };
            if (rw == 1) go(k_p1_row<1>);
            else if (rw == 2) go(k_p1_row<2>);
            else go(k_p1_row<4>);
            p = nx;
        } else {
            // iteration j - PAIRS has been decided over: its pair's time is there
            if (j >= PAIRS && (e = add_time(j)) != hipSuccess) break;
            hipLaunchKernelGGL(k_p1_dir, dim3(nb), dim3(256), 0, s, j, v.partial, nb, v.st, h, maxiter, tol, v.z, v.p);
            int64_t n = 0;
            if ((e = hipEventRecord(v.ev[2 * (j % PAIRS)], s)) != hipSuccess) break;
            if ((e = launch_grm_gemv(s, S, Np, Nnm, v.p, v.ap, a, v.pap, &n, tri)) != hipSuccess) break;
            if ((e = hipEventRecord(v.ev[2 * (j % PAIRS) + 1], s)) != hipSuccess) break;
            npap = (int)n;
        }
        hipLaunchKernelGGL(k_p1_update, dim3(nb), dim3(256), 0, s, j, v.pap, npap, v.st, v.minv, p, v.ap, v.x, v.r,
                           v.z, v.partial);
        if ((e = hipGetLastError()) != hipSuccess) break;
        // wait until the device has decided iteration j - P1_AHEAD; an idle or
        // failed stream ends the wait whatever the host sees
        for (int spin = 0; !h->done && h->decided < j - P1_AHEAD; spin++) {
            if ((spin & 1023) == 1023) {
                const hipError_t q = hipStreamQuery(s);
                if (q == hipSuccess) break;
                if (q != hipErrorNotReady) {
                    e = q;
                    break;
                }
            }
        }
        if (h->done) break;
    }
    if (e == hipSuccess && small) e = hipEventRecord(v.ev[1], s);
    if (e == hipSuccess && !small) e = hipMemcpyAsync(x_host, v.x, 4 * Nnm, hipMemcpyDeviceToHost, s);
    const hipError_t end = hipStreamSynchronize(s);
    if (e == hipSuccess) e = end;
    if (e != hipSuccess) return e;
    if (small) std::copy(v.hvec + 2 * Np, v.hvec + 2 * Np + Nnm, x_host);
    *iters = h->it;
    if (small) {
        e = add_time(0);
    } else {
        // iterations j, j - 1, ... still unread; those past the end launched nothing
        for (int k = std::max(0, j + 1 - PAIRS); k < h->it && e == hipSuccess; k++) e = add_time(k);
    }
    v.launches += h->it;
    return e;
}

}  // namespace saige
