// Genotype kernels: PLINK-1 2-bit decode with allele / missing counts and
// QC, imputation + repacking, the standardisation lookup table, the FP32
// diagonal sum_j z_ij^2, standardised marker panels for the SYRK, and a
// counter-based synthetic genotype generator.
//
// Integer work is bit-exact with the reference by construction.  The FP32
// scalar formulas use explicitly rounded intrinsics (__fadd_rn ...) so no
// contraction into FMA changes a rounding step.
#include "saige_internal.hpp"

#include <algorithm>
#include <type_traits>

#pragma clang fp contract(off)

namespace saige {

namespace {

__device__ __forceinline__ int wave_sum_i(int v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// PLINK-1 codes (FG.cpp:343-357: b = bit0, a = bit1): (0,0) two A1 alleles,
// (1,0) missing, (0,1) one, (1,1) none.

// Counts of one 32-bit word of PLINK codes (16 samples) under a code mask
// (bit 2s set: sample s of the word is counted): with l, h the low and high
// bit of a code, missing = l & ~h (01), and a counted non-missing code adds
// 2 - l - h A1 alleles, where l = 1 only together with h = 1 (code 11).
// miss += missing codes, nonm += counted non-missing codes, t += sum of
// l + h over them; alleleCount = 2 nonm - t.
__device__ __forceinline__ void count_word(uint32_t w, uint32_t msk, uint32_t& miss, uint32_t& nonm,
                                           uint32_t& t) {
    const uint32_t L = w & msk, H = (w >> 1) & msk;
    const uint32_t Mi = L & ~H;
    const uint32_t nmiss = (uint32_t)__popc(Mi);
    miss += nmiss;
    nonm += (uint32_t)__popc(msk) - nmiss;
    t += (uint32_t)__popc(L & H) + (uint32_t)__popc(H);
}

// The reference's FP32 per-marker formulas in order (FG.cpp:424-547,
// 914-921) from the integer counts over the phenotyped samples.
__device__ __forceinline__ MarkerStat marker_stat(int alleleCount, int numMissing, const DecodeParams& p,
                                                  int inr) {
    const uint64_t nnm = (uint64_t)p.Nnm;
    // FG.cpp:424 and 442
    float altFreq = div_rn((float)alleleCount, (float)((nnm - (uint64_t)numMissing) * 2u));
    float missingRate = div_rn((float)numMissing, (float)nnm);
    // FG.cpp:447; NaN (all calls missing) maps to 0
    float twice = __fmul_rn(2.0f, altFreq);
    int fill = (twice != twice) ? 0 : (int)roundf(twice);
    if (numMissing > 0) alleleCount = alleleCount + fill * numMissing;   // FG.cpp:454
    altFreq = div_rn((float)alleleCount, (float)(nnm * 2u));          // FG.cpp:484
    float one_m = __fsub_rn(1.0f, altFreq);
    float maf = (one_m < altFreq) ? one_m : altFreq;                     // std::min
    int twoN = (int)p.Nnm * 2;
    int mac = (alleleCount < twoN - alleleCount) ? alleleCount : twoN - alleleCount;
    int passQC = (maf >= p.min_maf && missingRate <= p.max_missing) ? 1 : 0;
    int passVR = 0;
    if (p.vr_mode == 1) {
        if ((float)mac >= p.min_mac_vr && (float)mac < p.max_mac_vr) passVR = 1;
        else if ((float)mac >= p.max_mac_vr) passVR = inr;
    } else if (p.vr_mode == 2) {
        if ((float)mac >= p.min_mac_vr) passVR = inr;
    }
    if (passVR) passQC = 0;
    // FG.cpp:914-921
    float Std = sqrt_rn(__fmul_rn(__fmul_rn(2.0f, altFreq), one_m));
    float invStd = (Std == 0.0f) ? 0.0f : div_rn(1.0f, Std);
    MarkerStat st;
    st.allele_count = alleleCount;
    st.num_missing = numMissing;
    st.mac = mac;
    st.fill = fill;
    st.freq = altFreq;
    st.missing_rate = missingRate;
    st.inv_std = invStd;
    st.pass_qc = (uint8_t)passQC;
    st.pass_vr = (uint8_t)passVR;
    st.pad[0] = st.pad[1] = 0;
    return st;
}

// One wave per marker, four markers per workgroup, no workgroup barrier.
// A row of bpm bytes is read as the 16-byte chunks of the aligned span that
// covers it (a chunk always holds at least one byte of the row, so it never
// leaves the row's page), two chunks per lane in flight.  Bytes outside the
// row and the pad samples of its last byte are masked out: without a sample
// indicator (every .fam sample phenotyped) from the byte positions; with
// one (MASKED) from imask, 16 copies of the row's code mask (2 bits per
// sample, 0b11 when indicatorGenoSamplesWithPheno is set), copy r shifted by
// r bytes with stride ld, so that copy (row address mod 16) lines up with
// the aligned chunks.  Lane 0 evaluates the per-marker formulas.
template <bool MASKED>
__global__ __launch_bounds__(256) void k_decode_stats(const uint8_t* __restrict__ bed,
                                                      const uint8_t* __restrict__ imask, int64_t ld,
                                                      const uint8_t* __restrict__ randset, DecodeParams p,
                                                      MarkerStat* __restrict__ stats) {
    const int lane = threadIdx.x & 63;
    const int64_t m = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (m >= p.M) return;
    const uint8_t* row = bed + m * p.bpm;
    const int64_t r = (int64_t)((uintptr_t)row & 15u);
    const uint8_t* A = row - r;
    const int64_t span = r + p.bpm;                   // bytes from A to the row's end
    const int64_t nchunk = (span + 15) / 16;
    const uint8_t* mk = MASKED ? imask + r * ld : nullptr;
    // codes of the last byte that are samples (the rest is padding)
    const int last_codes = (int)(p.N - 4 * (p.bpm - 1));
    const uint32_t last_mask = last_codes >= 4 ? 0xFFu : ((1u << (2 * last_codes)) - 1u);
    uint32_t miss = 0, nonm = 0, t = 0;
    auto chunk = [&](int64_t q, const uint4& v) {
        const int64_t x0 = 16 * q;
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
        uint32_t mw[4];
        if (MASKED) {
            const uint4 mv = *reinterpret_cast<const uint4*>(mk + x0);
            mw[0] = mv.x; mw[1] = mv.y; mw[2] = mv.z; mw[3] = mv.w;
        } else if (x0 - r >= 0 && x0 - r + 16 <= p.bpm - 1) {
            mw[0] = mw[1] = mw[2] = mw[3] = 0xFFFFFFFFu;    // interior: every byte a full row byte
        } else {
#pragma unroll
            for (int d = 0; d < 4; d++) {
                uint32_t mm = 0;
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    const int64_t pos = x0 + 4 * d + b - r;
                    const uint32_t bm = (pos < 0 || pos >= p.bpm) ? 0u : (pos == p.bpm - 1 ? last_mask : 0xFFu);
                    mm |= bm << (8 * b);
                }
                mw[d] = mm;
            }
        }
#pragma unroll
        for (int d = 0; d < 4; d++) count_word(w[d], mw[d] & 0x55555555u, miss, nonm, t);
    };
    int64_t q = lane;
    for (; q + 64 < nchunk; q += 128) {
        const uint4 v0 = *reinterpret_cast<const uint4*>(A + 16 * q);
        const uint4 v1 = *reinterpret_cast<const uint4*>(A + 16 * (q + 64));
        chunk(q, v0);
        chunk(q + 64, v1);
    }
    if (q < nchunk) chunk(q, *reinterpret_cast<const uint4*>(A + 16 * q));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        miss += __shfl_xor(miss, o, 64);
        nonm += __shfl_xor(nonm, o, 64);
        t += __shfl_xor(t, o, 64);
    }
    if (lane == 0) {
        const int alleleCount = (int)(2u * nonm - t);
        stats[m] = marker_stat(alleleCount, (int)miss, p, randset ? (int)randset[m] : 0);
    }
}

// Repacking into subSampleInGeno order with imputation (FG.cpp:551-576).  The
// internal code of a PLINK code is its own bits (00 two copies, 10 one, 11
// none, FG.cpp:41-44), except that a missing call (01) takes the code of the
// marker's fill genotype: so a word of codes is repacked by finding its
// missing calls and replacing their two bits.  f0 / f1: the low / high bit of
// the fill's code, spread over the codes it applies to (all ones or zero per
// marker).
__device__ __forceinline__ uint32_t impute_word(uint32_t w, uint32_t f0, uint32_t f1) {
    const uint32_t m = w & ~(w >> 1) & 0x55555555u;      // low bit of every missing call
    return (w & ~m) | (m & f0) | ((m << 1) & f1);
}
// fill (0, 1 or 2 copies) -> internal code bits 11, 10, 00
__device__ __forceinline__ uint32_t fill_lo(int fill) { return fill == 0 ? 0xFFFFFFFFu : 0u; }
__device__ __forceinline__ uint32_t fill_hi(int fill) { return fill <= 1 ? 0xFFFFFFFFu : 0u; }

// four bytes at any address (one unaligned dword load)
__device__ __forceinline__ uint32_t load4(const uint8_t* p) {
    uint32_t v;
    __builtin_memcpy(&v, p, 4);
    return v;
}
// the bytes [o, o + 4) of a row of n bytes, zero past its end
__device__ __forceinline__ uint32_t row4(const uint8_t* row, int64_t o, int64_t n) {
    if (o + 4 <= n) return load4(row + o);
    uint32_t v = 0;
    for (int e = 0; e < 4; e++)
        if (o + e < n) v |= (uint32_t)row[o + e] << (8 * e);
    return v;
}

// k_repack_id: every .fam sample phenotyped, in .fam order.  One wave per
// marker, 16 output bytes per lane and step (rows start at any address, so
// the loads are unaligned, the stores aligned), four steps' loads in flight.
// Bound by its two streams: 1.43 ms for 7.5 GB at N = 100,000, M = 150,000,
// 5.2 TB/s (4.36 ms with a 256-entry byte table and one workgroup per
// marker).
__global__ __launch_bounds__(256) void k_repack_id(const uint8_t* __restrict__ bed, int64_t bpm,
                                                   const int32_t* __restrict__ markers, int64_t nmark,
                                                   const MarkerStat* __restrict__ stats, int64_t Nnm, int64_t ldp,
                                                   uint8_t* __restrict__ out) {
    const int lane = threadIdx.x & 63;
    const int64_t mi = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (mi >= nmark) return;
    const int64_t m = markers[mi];
    const uint8_t* row = bed + m * bpm;
    const int fill = stats[m].fill;
    const uint32_t f0 = fill_lo(fill), f1 = fill_hi(fill);
    uint4* orow = reinterpret_cast<uint4*>(out + mi * ldp);
    const int64_t whole = Nnm / 64;                      // 16-byte words full of samples
    const int64_t nw = ldp / 16;
    auto put = [&](int64_t q, uint4 v) {
        v.x = impute_word(v.x, f0, f1);
        v.y = impute_word(v.y, f0, f1);
        v.z = impute_word(v.z, f0, f1);
        v.w = impute_word(v.w, f0, f1);
        orow[q] = v;
    };
    int64_t q = lane;
    for (; q + 192 < whole; q += 256) {
        uint4 v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) __builtin_memcpy(&v[k], row + 16 * (q + 64 * k), 16);
#pragma unroll
        for (int k = 0; k < 4; k++) put(q + 64 * k, v[k]);
    }
    for (; q < whole; q += 64) {
        uint4 v;
        __builtin_memcpy(&v, row + 16 * q, 16);
        put(q, v);
    }
    // the last samples and the row's padding: code 00 past the samples, which
    // is no missing call
    for (; q < nw; q += 64) {
        uint32_t t[4];
#pragma unroll
        for (int d = 0; d < 4; d++) {
            const int64_t o = 16 * q + 4 * d, left = Nnm - 4 * o;
            const uint32_t keep = left >= 16 ? 0xFFFFFFFFu : (left <= 0 ? 0u : (1u << (2 * left)) - 1u);
            t[d] = keep ? row4(row, o, bpm) & keep : 0u;
        }
        put(q, make_uint4(t[0], t[1], t[2], t[3]));
    }
}

// k_repack_sub: the listed samples (1-based .fam rows) in the list's order,
// four markers per workgroup.  Their rows stand in LDS interleaved, a dword
// per .fam byte holding the four markers' bytes, so one read, shift and mask
// fetch a sample's codes of all four, and the sample list is read once for
// the four.  A thread makes four output bytes (16 samples) of each marker and
// transposes them into one dword per row.  LDS: 4 bytes per .fam byte, so
// rows of at most REPACK_LDS_BYTES / 4 bytes (163,840 samples); longer ones
// take k_repack_far.  24,008 of 30,011 samples, 20,003 markers: 89 us (957 us
// gathering bytes from global memory, one marker at a time).
constexpr int64_t REPACK_LDS_BYTES = 160 * 1024;
__global__ __launch_bounds__(512) void k_repack_sub(const uint8_t* __restrict__ bed, int64_t bpm,
                                                    const int32_t* __restrict__ markers, int64_t nmark,
                                                    const MarkerStat* __restrict__ stats,
                                                    const int32_t* __restrict__ subidx, int64_t Nnm, int64_t ldp,
                                                    uint8_t* __restrict__ out) {
    extern __shared__ uint32_t rows4[];                  // [4 * ceil(bpm / 4)]
    const int64_t mi0 = (int64_t)blockIdx.x * 4;
    const uint8_t* row[4];
    uint32_t f0 = 0, f1 = 0;                             // byte k: marker k's fill bits
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int64_t m = markers[min(mi0 + k, nmark - 1)];
        row[k] = bed + m * bpm;
        const int fill = stats[m].fill;
        f0 |= fill_lo(fill) & (0xFFu << (8 * k));
        f1 |= fill_hi(fill) & (0xFFu << (8 * k));
    }
    for (int64_t d = threadIdx.x; 4 * d < bpm; d += blockDim.x) {
        uint32_t t[4];
        transpose4x4(row4(row[0], 4 * d, bpm), row4(row[1], 4 * d, bpm), row4(row[2], 4 * d, bpm),
                     row4(row[3], 4 * d, bpm), t);
        *reinterpret_cast<uint4*>(rows4 + 4 * d) = make_uint4(t[0], t[1], t[2], t[3]);
    }
    __syncthreads();
    for (int64_t o = threadIdx.x; o < ldp / 4; o += blockDim.x) {
        const int64_t s0 = 16 * o;
        uint32_t acc[4] = {0u, 0u, 0u, 0u};              // output byte j of the four markers
        if (s0 < Nnm) {
            int32_t src[16];
            if (s0 + 16 <= Nnm) {
#pragma unroll
                for (int j = 0; j < 4; j++)
                    *reinterpret_cast<int4*>(src + 4 * j) = *reinterpret_cast<const int4*>(subidx + s0 + 4 * j);
            } else {
#pragma unroll
                for (int j = 0; j < 16; j++) src[j] = s0 + j < Nnm ? subidx[s0 + j] : 0;   // 0: no sample
            }
#pragma unroll
            for (int j = 0; j < 16; j++) {
                const uint32_t i = (uint32_t)max(src[j] - 1, 0);
                const uint32_t c = (rows4[i >> 2] >> (2 * (i & 3))) & 0x03030303u;
                acc[j >> 2] |= (src[j] > 0 ? c : 0u) << (2 * (j & 3));
            }
#pragma unroll
            for (int j = 0; j < 4; j++) acc[j] = impute_word(acc[j], f0, f1);
        }
        uint32_t t[4];
        transpose4x4(acc[0], acc[1], acc[2], acc[3], t);
#pragma unroll
        for (int k = 0; k < 4; k++)
            if (mi0 + k < nmark) reinterpret_cast<uint32_t*>(out + (mi0 + k) * ldp)[o] = t[k];
    }
}

// k_repack_far: as k_repack_sub for rows too long for LDS, gathered from
// global memory, one workgroup per marker.
__global__ __launch_bounds__(256) void k_repack_far(const uint8_t* __restrict__ bed, int64_t bpm,
                                                    const int32_t* __restrict__ markers, int64_t nmark,
                                                    const MarkerStat* __restrict__ stats,
                                                    const int32_t* __restrict__ subidx, int64_t Nnm, int64_t ldp,
                                                    uint8_t* __restrict__ out) {
    for (int64_t mi = blockIdx.x; mi < nmark; mi += gridDim.x) {
        const int64_t m = markers[mi];
        const uint8_t* row = bed + m * bpm;
        const int fill = stats[m].fill;
        const uint32_t f0 = fill_lo(fill), f1 = fill_hi(fill);
        uint8_t* orow = out + mi * ldp;
        for (int64_t o = threadIdx.x; o < ldp; o += blockDim.x) {
            uint32_t byte = 0;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int64_t indx = o * 4 + j;
                if (indx >= Nnm) break;
                const int64_t src = (int64_t)subidx[indx] - 1;
                byte |= ((row[src >> 2] >> ((src & 3) * 2)) & 3u) << (2 * j);
            }
            orow[o] = (uint8_t)impute_word(byte, f0, f1);
        }
    }
}

// setStdGenoLookUpArr (FG.cpp:152-159)
__global__ void k_lut(const int32_t* __restrict__ markers, int64_t nmark,
                      const MarkerStat* __restrict__ stats, float4* __restrict__ lut) {
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= nmark) return;
    const MarkerStat st = stats[markers[i]];
    float m2 = __fmul_rn(2.0f, st.freq);
    float4 L;
    L.x = __fmul_rn(__fsub_rn(0.0f, m2), st.inv_std);
    L.y = __fmul_rn(__fsub_rn(1.0f, m2), st.inv_std);
    L.z = __fmul_rn(__fsub_rn(2.0f, m2), st.inv_std);
    L.w = 0.0f;
    lut[i] = L;
}

// internal code -> 2-(a+b) (FG.cpp:596-600)
__device__ __forceinline__ int internal_geno(unsigned c) { return 2 - (int)((c & 1u) + (c >> 1)); }

__device__ __forceinline__ float lut_pick(const float4 L, int g) {
    return g == 0 ? L.x : (g == 1 ? L.y : L.z);
}

// Get_Diagof_StdGeno (FG.cpp:665-704): per sample the FP32 sum of z*z with
// the markers strictly in order (z*z rounded, then added).  The order makes
// it a chain of Mqc dependent additions per sample, so what bounds it is the
// number of instructions a wave issues between two of them.  A workgroup owns
// 256 samples (64 bytes of each marker's row) and walks tiles of DG_MK markers.
// Four waves make a tile:
// * its codes go to LDS per sample, a byte for every two markers: their two
//   codes, times 8;
// * its squares go to LDS as a 16-entry table (z^2 of the first marker, z^2 of
//   the second) for every two markers, so that byte is a table offset and one
//   8-byte read gives two addends;
// and four add up the one before it, a sample per thread: per two markers a
// bit-field extract, the read and two additions, the reads eight pairs ahead so
// that there is one wait for sixteen additions.  Both are double-buffered and the
// next tile's loads are in flight while a tile is made.  Markers past the end
// have zero tables.  1000 x 10,000: 61 us (115 with the same four waves making
// and adding, 863 with a byte load and two selects per marker and sample);
// 24,008 x 20,003: 126 us; 100,000 x 150,000: 1.66 ms (1.99, 15.3), where 391
// workgroups load 256 CUs unevenly.
constexpr int DG_MK = 128;                       // markers per tile
constexpr int DG_PITCH = DG_MK / 8 + 4;          // dwords per sample
constexpr int DG_PLANE = 16 * DG_PITCH + 4;      // samples s, s + 16, ... stand together
// sample s's codes in LDS: the transposed stores (samples 16 apart) and the
// 16-byte reads (consecutive samples) both spread over all banks
__device__ __forceinline__ int dg_sample(int s) { return (s & 15) * DG_PLANE + (s >> 4) * DG_PITCH; }

__global__ __launch_bounds__(512) void k_diag_std(const uint8_t* __restrict__ packed,
                                                  const float4* __restrict__ lut, int64_t Mqc,
                                                  int64_t Nnm, int64_t ldp,
                                                  float* __restrict__ diag) {
    __shared__ __attribute__((aligned(16))) float2 tab[2][DG_MK / 2 * 16];
    __shared__ __attribute__((aligned(16))) uint32_t cod[2][16 * DG_PLANE];
    const int tid = threadIdx.x & 255;
    const bool adds = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) == 0;
    const int64_t ntile = (Mqc + DG_MK - 1) / DG_MK;
    // loads: dword column c4 (samples 16*c4 + [0, 16)) of markers 8*mo + [0, 8)
    const int c4 = tid & 15, mo = tid >> 4;
    const uint8_t* src = packed + (int64_t)(8 * mo) * ldp + (int64_t)blockIdx.x * 64 + 4 * c4;
    // tables: entry nib (the first marker's code, 4 x the second's) of the
    // marker pairs tm + 16k
    const int nib = tid & 15, tm = tid >> 4;
    const int g0 = internal_geno(nib & 3), g1 = internal_geno(nib >> 2);
    uint32_t w[8];
    float4 L[8];
    // the next tile's codes and table values (rows past the end are in the
    // buffers' padding; their tables are zero), then on to the one after it
    const float4* lp = lut + 2 * tm;
    int64_t left = Mqc - 2 * tm;                             // markers from this thread's first pair to the end
    auto fetch = [&]() {
#pragma unroll
        for (int e = 0; e < 8; e++) w[e] = *reinterpret_cast<const uint32_t*>(src + e * ldp);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            L[2 * k] = lp[32 * k];
            L[2 * k + 1] = lp[32 * k + 1];
        }
        src += DG_MK * ldp;
        lp += DG_MK;
    };
    auto put = [&](auto buf) {
        // per marker pair and s < 4: the codes of sample 4e + s in byte e
        uint32_t p[4][4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t a = w[2 * j], b = w[2 * j + 1], m = 0x33333333u;
            const uint32_t ev = (a & m) | ((b << 2) & ~m), od = ((a >> 2) & m) | (b & ~m);
            p[0][j] = (ev & 0x0F0F0F0Fu) << 3;
            p[1][j] = (od & 0x0F0F0F0Fu) << 3;
            p[2][j] = (ev >> 1) & 0x78787878u;
            p[3][j] = (od >> 1) & 0x78787878u;
        }
#pragma unroll
        for (int s = 0; s < 4; s++) {
            uint32_t t[4];
            transpose4x4(p[s][0], p[s][1], p[s][2], p[s][3], t);
#pragma unroll
            for (int e = 0; e < 4; e++) cod[buf][dg_sample(16 * c4 + 4 * e + s) + mo] = t[e];
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const float z0 = lut_pick(L[2 * k], g0), z1 = lut_pick(L[2 * k + 1], g1);
            tab[buf][(tm + 16 * k) * 16 + nib] = make_float2(32 * k < left ? __fmul_rn(z0, z0) : 0.0f,
                                                             32 * k + 1 < left ? __fmul_rn(z1, z1) : 0.0f);
        }
        left -= DG_MK;
    };
    if (!adds) {
        // tile t + 1 is made while tile t is summed; its buffer's last reader
        // was tile t - 1, before the barrier
        fetch();
        put(std::integral_constant<int, 0>());
        if (ntile > 1) fetch();
        lds_barrier();
        auto step = [&](auto nxt, int64_t t) {
            if (t + 1 < ntile) {
                put(nxt);
                if (t + 2 < ntile) fetch();
            }
            lds_barrier();
        };
        for (int64_t t = 0; t < ntile; t += 2) {
            step(std::integral_constant<int, 1>(), t);
            if (t + 1 < ntile) step(std::integral_constant<int, 0>(), t + 1);
        }
        return;
    }
    float d = 0.0f;
    auto sum = [&](auto buf) {
        constexpr int NG = DG_MK / 16;               // groups of eight pairs
        const uint32_t* cp = cod[buf] + dg_sample(tid);
        const char* tp = reinterpret_cast<const char*>(tab[buf]);
        uint4 q[2];
        float2 s[2][8];
        auto codes = [&](int h) { q[h & 1] = *reinterpret_cast<const uint4*>(cp + 4 * h); };
        auto read = [&](int g) {
            const uint4 c = q[(g >> 1) & 1];
            const uint32_t v[2] = {g & 1 ? c.z : c.x, g & 1 ? c.w : c.y};
#pragma unroll
            for (int u = 0; u < 8; u++)
                s[g & 1][u] =
                    *reinterpret_cast<const float2*>(tp + 128 * (8 * g + u) + ((v[u >> 2] >> (8 * (u & 3))) & 255u));
        };
        codes(0);
        codes(1);
        read(0);
#pragma unroll
        for (int g = 0; g < NG; g++) {
            // the next group's addends are asked for before this one's are added:
            // one wait a group
            if (g + 1 < NG) read(g + 1);
            if ((g & 1) && g / 2 + 2 < NG / 2) codes(g / 2 + 2);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < 8; u++) d = __fadd_rn(__fadd_rn(d, s[g & 1][u].x), s[g & 1][u].y);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    lds_barrier();
    for (int64_t t = 0; t < ntile; t += 2) {
        sum(std::integral_constant<int, 0>());
        lds_barrier();
        if (t + 1 < ntile) {
            sum(std::integral_constant<int, 1>());
            lds_barrier();
        }
    }
    const int64_t i = (int64_t)blockIdx.x * 256 + tid;
    if (i < Nnm) diag[i] = d;
}

__global__ void k_get_geno(const uint8_t* __restrict__ row, int64_t Nnm, int32_t* __restrict__ out) {
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= Nnm) return;
    out[i] = internal_geno((row[i >> 2] >> ((i & 3) * 2)) & 3u);
}

__global__ void k_std_geno(const uint8_t* __restrict__ row, const float4* __restrict__ lut,
                           int64_t Nnm, float* __restrict__ out) {
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= Nnm) return;
    out[i] = lut_pick(lut[0], internal_geno((row[i >> 2] >> ((i & 3) * 2)) & 3u));
}

// Standardised panel: Zp[r][c] = z of panel marker c (global j0 + c) at
// sample r, for a 128-sample x 64-marker tile per workgroup, transposed
// through LDS so both the packed reads and the row writes are contiguous.
template <typename T>
__device__ __forceinline__ T to_elem(float v);
template <>
__device__ __forceinline__ __hip_bfloat16 to_elem<__hip_bfloat16>(float v) { return __float2bfloat16(v); }

template <typename T>
__global__ __launch_bounds__(256) void k_std_panel(const uint8_t* __restrict__ packed,
                                                   const float4* __restrict__ lut, int64_t j0,
                                                   int64_t np, int64_t Nnm, int64_t ldp,
                                                   int64_t ldz, T* __restrict__ Zp) {
    __shared__ float tile[128][65];
    const int tid = threadIdx.x;
    const int64_t s0 = (int64_t)blockIdx.x * 128;   // first sample of the tile
    const int64_t c0 = (int64_t)blockIdx.y * 64;    // first panel column of the tile
    {
        const int mk = tid >> 2;        // marker within tile 0..63
        const int part = tid & 3;       // 32 samples each
        const int64_t c = c0 + mk;
        const bool valid_m = c < np;
        float4 L = valid_m ? lut[j0 + c] : make_float4(0.f, 0.f, 0.f, 0.f);
        const uint8_t* row = packed + (j0 + c) * ldp;
#pragma unroll
        for (int bq = 0; bq < 8; bq++) {
            const int64_t sb = s0 + part * 32 + bq * 4;   // first sample of this byte
            unsigned byte = 0;
            if (valid_m && sb < Nnm) byte = row[sb >> 2];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int64_t s = sb + j;
                float z = 0.0f;
                if (valid_m && s < Nnm) z = lut_pick(L, internal_geno((byte >> (2 * j)) & 3u));
                tile[part * 32 + bq * 4 + j][mk] = z;
            }
        }
    }
    __syncthreads();
    const int lane = tid & 63, wv = tid >> 6;
    const int64_t c = c0 + lane;
    if (c < ldz) {
        for (int r = wv; r < 128; r += 4) {
            Zp[(s0 + r) * ldz + c] = to_elem<T>(tile[r][lane]);
        }
    }
}

// Counter-based uniform in [0, 1) from a 64-bit mix (splitmix64 finaliser).
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
__device__ __forceinline__ float unif(uint64_t seed, uint64_t a, uint64_t b, uint64_t k) {
    uint64_t h = mix64(seed ^ mix64(a * 0x9E3779B97F4A7C15ull + mix64(b * 0xC2B2AE3D27D4EB4Full + k)));
    return (float)(h >> 40) * (1.0f / 16777216.0f);
}

__device__ __forceinline__ int synth_geno(uint64_t seed, int64_t m, int64_t s, float pj) {
    return (unif(seed, m, s, 1) < pj ? 1 : 0) + (unif(seed, m, s, 2) < pj ? 1 : 0);
}

__device__ __forceinline__ void synth_byte(uint8_t* __restrict__ bed, int64_t t, int64_t N, int64_t bpm,
                                           float maf_lo, float maf_hi, float miss, int64_t npairs,
                                           uint64_t seed) {
    const int64_t m = t / bpm, b = t - m * bpm;
    const float pj = maf_lo + (maf_hi - maf_lo) * unif(seed, m, 0x7FFFFFFF, 0);
    unsigned byte = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int64_t s = b * 4 + j;
        if (s >= N) break;   // padding bits stay 00, as PLINK writes them
        int g = synth_geno(seed, m, s, pj);
        if (s < 2 * npairs && (s & 1) && unif(seed, m, s, 4) < 0.5f) g = synth_geno(seed, m, s - 1, pj);
        unsigned code;
        if (unif(seed, m, s, 3) < miss) code = 1u;
        else code = (g == 2) ? 0u : (g == 1 ? 2u : 3u);
        byte |= code << (2 * j);
    }
    bed[t] = (uint8_t)byte;
}

// Grid-stride over the M * bpm bytes: at N = 200k, M = 500k that is 2.5e10
// bytes, more work-items than one launch can address (2^32).
__global__ void k_synth_bed(uint8_t* __restrict__ bed, int64_t N, int64_t M, int64_t bpm,
                            float maf_lo, float maf_hi, float miss, int64_t npairs, uint64_t seed) {
    const int64_t total = M * bpm;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total; t += stride)
        synth_byte(bed, t, N, bpm, maf_lo, maf_hi, miss, npairs, seed);
}


// out = a - b, FP32 (diag(K) minus one chromosome's part, FG.cpp:4951)
__global__ void k_sub(const float* __restrict__ a, const float* __restrict__ b, int64_t n, float* __restrict__ out) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i < n) out[i] = __fsub_rn(a[i], b[i]);
}

inline unsigned grid_for(int64_t n, int64_t cap) { return (unsigned)(n < cap ? (n > 0 ? n : 1) : cap); }

}  // namespace

hipError_t launch_decode_stats(hipStream_t s, const uint8_t* bed, const uint8_t* imask, int64_t ld,
                               const uint8_t* randset, DecodeParams p, MarkerStat* stats) {
    const dim3 grid((unsigned)((p.M + 3) / 4));
    if (imask)
        hipLaunchKernelGGL(k_decode_stats<true>, grid, dim3(256), 0, s, bed, imask, ld, randset, p, stats);
    else
        hipLaunchKernelGGL(k_decode_stats<false>, grid, dim3(256), 0, s, bed, imask, ld, randset, p, stats);
    return hipGetLastError();
}

hipError_t launch_repack(hipStream_t s, const uint8_t* bed, int64_t bpm, const int32_t* markers,
                         int64_t nmark, const MarkerStat* stats, const int32_t* subidx, int64_t Nnm,
                         int64_t ldp, uint8_t* out) {
    if (nmark == 0) return hipSuccess;
    const int64_t lds = 16 * ((bpm + 3) / 4);
    if (subidx && lds > REPACK_LDS_BYTES) {
        hipLaunchKernelGGL(k_repack_far, dim3(grid_for(nmark, 16384)), dim3(256), 0, s, bed, bpm, markers, nmark,
                           stats, subidx, Nnm, ldp, out);
        return hipGetLastError();
    }
    if (subidx) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k_repack_sub),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)REPACK_LDS_BYTES);
        if (e != hipSuccess) return e;
    }
    // four markers per workgroup; a launch has fewer than 2^32 threads, so the
    // markers go in passes
    constexpr int64_t PASS = (int64_t)1 << 24;
    for (int64_t m0 = 0; m0 < nmark; m0 += PASS) {
        const int64_t n = std::min(PASS, nmark - m0);
        const dim3 grid((unsigned)((n + 3) / 4));
        if (!subidx)
            hipLaunchKernelGGL(k_repack_id, grid, dim3(256), 0, s, bed, bpm, markers + m0, n, stats, Nnm, ldp,
                               out + m0 * ldp);
        else
            hipLaunchKernelGGL(k_repack_sub, grid, dim3(512), (size_t)lds, s, bed, bpm, markers + m0, n, stats, subidx,
                               Nnm, ldp, out + m0 * ldp);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipGetLastError();
}

hipError_t launch_lut(hipStream_t s, const int32_t* markers, int64_t nmark, const MarkerStat* stats,
                      float4* lut) {
    if (nmark == 0) return hipSuccess;
    hipLaunchKernelGGL(k_lut, dim3((unsigned)((nmark + 255) / 256)), dim3(256), 0, s, markers, nmark,
                       stats, lut);
    return hipGetLastError();
}

hipError_t launch_diag_std(hipStream_t s, const uint8_t* packed, const float4* lut, int64_t Mqc,
                           int64_t Nnm, int64_t ldp, float* diag) {
    if (Mqc <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_diag_std, dim3((unsigned)((Nnm + 255) / 256)), dim3(512), 0, s, packed, lut,
                       Mqc, Nnm, ldp, diag);
    return hipGetLastError();
}

hipError_t launch_sub(hipStream_t s, const float* a, const float* b, int64_t n, float* out) {
    hipLaunchKernelGGL(k_sub, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a, b, n, out);
    return hipGetLastError();
}

hipError_t launch_get_geno(hipStream_t s, const uint8_t* row, int64_t Nnm, int32_t* out) {
    hipLaunchKernelGGL(k_get_geno, dim3((unsigned)((Nnm + 255) / 256)), dim3(256), 0, s, row, Nnm, out);
    return hipGetLastError();
}

hipError_t launch_std_geno(hipStream_t s, const uint8_t* row, const float4* lut_row, int64_t Nnm,
                           float* out) {
    hipLaunchKernelGGL(k_std_geno, dim3((unsigned)((Nnm + 255) / 256)), dim3(256), 0, s, row, lut_row,
                       Nnm, out);
    return hipGetLastError();
}

hipError_t launch_synth_bed(hipStream_t s, uint8_t* bed, int64_t N, int64_t M, float maf_lo,
                            float maf_hi, float miss, int64_t npairs, uint64_t seed) {
    const int64_t bpm = (N + 3) / 4;
    const int64_t n = M * bpm;
    hipLaunchKernelGGL(k_synth_bed, dim3(grid_for((n + 255) / 256, 1 << 16)), dim3(256), 0, s, bed, N, M, bpm,
                       maf_lo, maf_hi, miss, npairs, seed);
    return hipGetLastError();
}

hipError_t launch_std_panel_bf16(hipStream_t s, const uint8_t* packed, const float4* lut, int64_t j0,
                                 int64_t np, int64_t Nnm, int64_t Npad, int64_t ldp, int64_t ldz,
                                 __hip_bfloat16* Zp) {
    dim3 grid((unsigned)(Npad / 128), (unsigned)((ldz + 63) / 64));
    hipLaunchKernelGGL(k_std_panel<__hip_bfloat16>, grid, dim3(256), 0, s, packed, lut, j0, np, Nnm,
                       ldp, ldz, Zp);
    return hipGetLastError();
}

}  // namespace saige
