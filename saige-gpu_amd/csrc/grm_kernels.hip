// GRM SYRK on CDNA4 matrix cores: S = Z Z^T from the 2-bit genotypes
// (k_syrk_pk256, k_syrk_pk), or S (+)= Zp Zp^T for one marker panel
// (k_syrk_bf16).
//
// Both MFMA operands are marker-contiguous rows of the same matrix of
// standardised genotypes.
// Each workgroup computes one tile of the lower triangle (tile row >= tile
// column) and writes it and its mirror into the full row-major S.
// Tile order: the host lists the triangle's tiles grouped into 8x8-tile
// super-blocks, and the launch index is remapped so that each XCD (launch
// order round-robins over the 8 XCDs) walks a contiguous run of that list.
// The ~100 tiles an XCD holds at once then span one or two super-blocks,
// i.e. 16-24 distinct 128-row panels of Zp, whose current K chunk fits in
// that XCD's 4 MB L2.
//
// Operand staging: global -> registers (the next K chunk while the current one
// is multiplied; decoded there from 2 bits) -> LDS -> MFMA fragments.
#include <algorithm>
#include <cmath>
#include <cstdlib>

#include "saige_internal.hpp"

namespace saige {

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;   // native vector: stays in VGPRs
typedef __attribute__((ext_vector_type(16))) float f32x16;

constexpr int BT = 128;  // tile edge


// Launch index -> triangle tile index, grouping consecutive tiles per XCD.
__device__ __forceinline__ int64_t xcd_remap(int64_t bid, int64_t nblk) {
    const int64_t nx = 8;
    const int64_t x = bid % nx, loc = bid / nx;
    const int64_t q = nblk / nx, rem = nblk % nx;
    return (x < rem) ? x * (q + 1) + loc : rem * (q + 1) + (x - rem) * q + loc;
}

// x rounded to nearest (ties to even) at 16 significant bits: the FP32
// value with the low 8 of its 23 fraction bits cleared.  Such a value is
// exactly the sum of its two BF16 pieces by truncation (the upper half of
// its bits, then the upper half of the remainder's), which the block GEMM
// over the lower triangle relies on.  Finite x only.
__device__ __forceinline__ float round16(float x) {
    const uint32_t b = __float_as_uint(x);
    return __uint_as_float((b + 0x7Fu + ((b >> 8) & 1u)) & 0xFFFFFF00u);
}

// Store a wave's block of 32*MI rows from row0 and 32*NI columns from col0,
// mirrored for off-diagonal tiles; accumulate: +1 S = S0 + block, -1 S = S0 -
// block (LOCO: one chromosome's markers left out), 0 store.  S0 may be S.
// center: the column's value taken off each sum first (nullptr: none).  R16:
// the stored values (after the add or subtract) rounded by round16.
// Accumulator layout of a 32x32 MFMA block: lane l, register r holds row
// 8*(r/4) + 4*(l/32) + (r%4), column l%32.  A block's S0 values are requested
// before the block ahead of it is stored (no entry that is read is stored by
// another lane).  With few markers the store is a third of the launch and bound
// by its bytes (S0's triangle read, S written): 1000 of 20,000 markers left out
// at N = 20,000 take 1.54 ms; a copy of S first and requests at their use took
// 2.7.
// R16 and s24: each 32 x 32 block of the lower triangle is also stored in three
// bytes a value (s24_block), turned in the wave's scratch (S24_SCRATCH floats of
// LDS): about 1 ms of a 214 ms build at N = 40,000, a fifth more bytes in the
// stores between two tiles; a pass of its own over S takes as long there and 6.7
// ms at 100,000.
constexpr int S24_PITCH = 36;
constexpr int S24_SCRATCH = 32 * S24_PITCH;

template <int MI, int NI, bool R16>
__device__ __forceinline__ void store_block(float* S, const float* S0, int64_t ldS, int64_t row0, int64_t col0,
                                            bool mirror, int lane, const f32x16 (&acc)[MI][NI], int accumulate,
                                            const float* center = nullptr, uint8_t* s24 = nullptr,
                                            float* scratch = nullptr) {
    float s0[2][16];
    auto request = [&](int k) {
        const float* p = S0 + (row0 + k / NI * 32 + 4 * (lane >> 5)) * ldS + col0 + k % NI * 32 + (lane & 31);
#pragma unroll
        for (int r = 0; r < 16; r++) s0[k & 1][r] = p[(8 * (r >> 2) + (r & 3)) * ldS];
    };
    if (accumulate) request(0);
#pragma unroll
    for (int k = 0; k < MI * NI; k++) {
        const int mi = k / NI, ni = k % NI;
        const int64_t col = col0 + ni * 32 + (lane & 31);
        const float cc = center ? center[col] : 0.0f;
        if (accumulate && k + 1 < MI * NI) request(k + 1);
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int64_t row = row0 + mi * 32 + 8 * g + 4 * (lane >> 5);
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                v[e] = center ? acc[mi][ni][4 * g + e] - cc : acc[mi][ni][4 * g + e];
                if (accumulate > 0) v[e] = s0[k & 1][4 * g + e] + v[e];
                else if (accumulate < 0) v[e] = s0[k & 1][4 * g + e] - v[e];
                if (R16) v[e] = round16(v[e]);
            }
#pragma unroll
            for (int e = 0; e < 4; e++) S[(row + e) * ldS + col] = v[e];
            if (mirror) {
                float4* dst = reinterpret_cast<float4*>(S + col * ldS + row);
                *dst = make_float4(v[0], v[1], v[2], v[3]);
            }
            if constexpr (R16) {
                if (s24) {
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        scratch[(8 * g + 4 * (lane >> 5) + e) * S24_PITCH + (lane & 31)] = v[e];
                }
            }
        }
        if constexpr (R16) {
            const int64_t I = row0 / 32 + mi, J = col0 / 32 + ni;
            if (s24 && J < I) {
                const int ln = lane & 15, o = lane >> 4;
                u32x4* dst = reinterpret_cast<u32x4*>(s24 + s24_block(I, J) * S24_BLOCK) + lane;
                u32x4 lo;
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    const u32x4* p = reinterpret_cast<const u32x4*>(scratch + (16 * r + ln) * S24_PITCH + 8 * o);
                    const u32x4 a = p[0], b = p[1];
                    // upper halves; then byte 1 of two words each
                    dst[64 * r] = u32x4{__builtin_amdgcn_perm(a[1], a[0], 0x07060302u),
                                        __builtin_amdgcn_perm(a[3], a[2], 0x07060302u),
                                        __builtin_amdgcn_perm(b[1], b[0], 0x07060302u),
                                        __builtin_amdgcn_perm(b[3], b[2], 0x07060302u)};
                    lo[2 * r] = __builtin_amdgcn_perm(a[1], a[0], 0x0C0C0501u) |
                                (__builtin_amdgcn_perm(a[3], a[2], 0x0C0C0501u) << 16);
                    lo[2 * r + 1] = __builtin_amdgcn_perm(b[1], b[0], 0x0C0C0501u) |
                                    (__builtin_amdgcn_perm(b[3], b[2], 0x0C0C0501u) << 16);
                }
                dst[128] = lo;
                __builtin_amdgcn_wave_barrier();
            }
        }
    }
}

// ------------------------------------------------------------------ BF16
constexpr int BK16 = 64;            // markers per K chunk
constexpr int P16 = BK16 + 8;       // LDS row pitch (bf16 elements): 144 B, conflict-free b128 reads

__global__ __launch_bounds__(256) void k_syrk_bf16(const __hip_bfloat16* __restrict__ Zp, int64_t ldz,
                                                   int64_t kdim, const int2* __restrict__ tiles, int64_t nblk,
                                                   float* S, int64_t ldS, int accumulate) {
    __shared__ __attribute__((aligned(16))) __hip_bfloat16 sA[BT * P16];
    __shared__ __attribute__((aligned(16))) __hip_bfloat16 sB[BT * P16];
    const int2 t = tiles[xcd_remap(blockIdx.x, nblk)];
    const int64_t bi = t.x, bj = t.y;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int wr = wv >> 1, wc = wv & 1;

    // global chunk mapping: 16-byte chunk c = tid + 256 q : row c/8, k (c%8)*8
    const int lrow = tid >> 3, lk = (tid & 7) * 8;
    const __hip_bfloat16* gA = Zp + (bi * BT + lrow) * ldz + lk;
    const __hip_bfloat16* gB = Zp + (bj * BT + lrow) * ldz + lk;
    u32x4 ra[4], rb[4];
    const int64_t nk = kdim / BK16;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        ra[q] = *reinterpret_cast<const u32x4*>(gA + (int64_t)(32 * q) * ldz);
        rb[q] = *reinterpret_cast<const u32x4*>(gB + (int64_t)(32 * q) * ldz);
    }
    f32x16 acc[2][2];
#pragma unroll
    for (int mi = 0; mi < 2; mi++)
#pragma unroll
        for (int ni = 0; ni < 2; ni++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[mi][ni][r] = 0.0f;

    for (int64_t kc = 0; kc < nk; kc++) {
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 4; q++) {
            *reinterpret_cast<u32x4*>(sA + (lrow + 32 * q) * P16 + lk) = ra[q];
            *reinterpret_cast<u32x4*>(sB + (lrow + 32 * q) * P16 + lk) = rb[q];
        }
        __syncthreads();
        {
            // prefetch the next chunk (the last iteration re-reads its own chunk:
            // unconditional loads keep ra/rb in registers)
            const int64_t off = ((kc + 1 < nk) ? kc + 1 : kc) * BK16;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                ra[q] = *reinterpret_cast<const u32x4*>(gA + (int64_t)(32 * q) * ldz + off);
                rb[q] = *reinterpret_cast<const u32x4*>(gB + (int64_t)(32 * q) * ldz + off);
            }
        }
#pragma unroll
        for (int ks = 0; ks < BK16 / 16; ks++) {
            const int kk = ks * 16 + (lane >> 5) * 8;
            bf16x8 fa[2], fb[2];
#pragma unroll
            for (int mi = 0; mi < 2; mi++)
                fa[mi] = *reinterpret_cast<const bf16x8*>(sA + (wr * 64 + mi * 32 + (lane & 31)) * P16 + kk);
#pragma unroll
            for (int ni = 0; ni < 2; ni++)
                fb[ni] = *reinterpret_cast<const bf16x8*>(sB + (wc * 64 + ni * 32 + (lane & 31)) * P16 + kk);
#pragma unroll
            for (int mi = 0; mi < 2; mi++)
#pragma unroll
                for (int ni = 0; ni < 2; ni++)
                    acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[mi], fb[ni], acc[mi][ni], 0, 0, 0);
        }
    }
    store_block<2, 2, false>(S, S, ldS, bi * BT + wr * 64, bj * BT + wc * 64, bi != bj, lane, acc, accumulate);
}

// ------------------------------------------------------- BF16, 2-bit in
// Same tile and MFMA loop as k_syrk_bf16, but the operands arrive as 2-bit
// genotypes and are standardised in registers: 8x fewer bytes per element
// than a BF16 panel, so the K loop is no longer bound by L2-miss traffic.
//
// Input layout (built by k_pack_tiles): for each 128-sample panel p and
// 64-marker chunk c, a 2 KB block [b][m]: byte b (samples 4b..4b+3 of the
// panel, 2 bits each, low bits first) of marker m.  Code 0b01 marks padding
// (samples >= Nnm, markers >= Mqc); the internal codes are 00/10/11.
// lut64[j]: four BF16 values of marker j indexed by the internal code:
// 00 -> L[2], 01 -> 0, 10 -> L[1], 11 -> L[0].
//
// Eight consecutive markers' values of one sample (samples 4b + j of byte b;
// bytes: the eight markers' bytes), i.e. one 16-byte LDS row of an operand, by
// byte permutes: lo[e] / hi[e] hold the low / high bytes of marker e's four
// BF16 table entries (entry c in byte c), so the 8-byte pair table {lo[2k+1], lo[2k]} is indexed by c_even and
// 4 + c_odd.  (byte >> 2j) & 3 of all eight markers at once gives the
// selectors; four permutes pick the low and high bytes of two marker pairs
// and two more interleave them into packed BF16 pairs.
__device__ __forceinline__ u32x4 decode_row_perm(const uint32_t (&lo)[8], const uint32_t (&hi)[8], uint64_t bytes,
                                                 int j) {
    const uint64_t d = (bytes >> (2 * j)) & 0x0303030303030303ull;
    u32x4 r;
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const uint32_t sel = (uint32_t)(d >> (32 * q)) + 0x04000400u;   // [c0, c1+4, c2, c3+4]
        const uint32_t a01 = __builtin_amdgcn_perm(lo[4 * q + 1], lo[4 * q], sel);
        const uint32_t b01 = __builtin_amdgcn_perm(hi[4 * q + 1], hi[4 * q], sel);
        const uint32_t a23 = __builtin_amdgcn_perm(lo[4 * q + 3], lo[4 * q + 2], sel);
        const uint32_t b23 = __builtin_amdgcn_perm(hi[4 * q + 3], hi[4 * q + 2], sel);
        r[2 * q] = __builtin_amdgcn_perm(b01, a01, 0x05010400u);        // markers 4q, 4q+1
        r[2 * q + 1] = __builtin_amdgcn_perm(b23, a23, 0x07030602u);    // markers 4q+2, 4q+3
    }
    return r;
}

// The single-pass BF16 GRM on 256x256 tiles: 512 threads (8 waves as 4 x 2),
// each wave a 64 x 128 block of the tile (2 x 4 MFMA 32x32 blocks, 128
// accumulator registers).  The per-element accumulation order (chunk by
// chunk, 16 markers per MFMA) is that of every tile size, so all give
// bitwise equal S.
constexpr int BT2 = 256;

// Double-buffered: while the MFMAs run on chunk k from one LDS buffer, the
// same waves decode chunk k+1 into the other, so the matrix pipe and the
// VALU decode overlap (one workgroup per CU); one LDS-only barrier per chunk.
// The two buffers are separate arrays and the loop is unrolled by two, so
// the compiler sees that the decode's stores and the MFMA operand loads
// never alias and can interleave them; the loop body is one basic block (the
// last step decodes a clamped copy of the last chunk that nothing reads, and
// diagonal tiles, both panels the same, decode their B copy too).
// eight tables' low and high bytes of their BF16 entries
__device__ __forceinline__ void split_bytes(const uint64_t (&t)[8], uint32_t (&lo)[8], uint32_t (&hi)[8]) {
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const uint32_t l = (uint32_t)t[e], h = (uint32_t)(t[e] >> 32);
        lo[e] = __builtin_amdgcn_perm(h, l, 0x06040200u);
        hi[e] = __builtin_amdgcn_perm(h, l, 0x07050301u);
    }
}

__global__ __launch_bounds__(512) void k_syrk_pk256(const uint8_t* __restrict__ tp, int64_t nchunk, int64_t c0,
                                                    int64_t c1, const uint64_t* __restrict__ lut64,
                                                    const int2* __restrict__ tiles, int64_t nblk,
                                                    float* S, const float* S0, int64_t ldS, int accumulate) {
    __shared__ __attribute__((aligned(16))) __hip_bfloat16 sA0[BT2 * P16];
    __shared__ __attribute__((aligned(16))) __hip_bfloat16 sB0[BT2 * P16];
    __shared__ __attribute__((aligned(16))) __hip_bfloat16 sA1[BT2 * P16];
    __shared__ __attribute__((aligned(16))) __hip_bfloat16 sB1[BT2 * P16];
    const int2 t = tiles[xcd_remap(blockIdx.x, nblk)];
    const int64_t bi = t.x, bj = t.y;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int wr = wv >> 1, wc = wv & 1;
    // thread -> marker octet o, byte row b of the 256-sample panel (two
    // 128-sample blocks of the tiled layout)
    const int o = tid & 7, b = tid >> 3;
    const int64_t pa = 2 * bi + (b >> 5), pb = 2 * bj + (b >> 5);
    const uint64_t* gA = reinterpret_cast<const uint64_t*>(tp + (pa * nchunk * 32 + (b & 31)) * 64 + 8 * o);
    const uint64_t* gB = reinterpret_cast<const uint64_t*>(tp + (pb * nchunk * 32 + (b & 31)) * 64 + 8 * o);
    const uint64_t* gl = lut64 + 8 * o;

    f32x16 acc[2][4];
#pragma unroll
    for (int mi = 0; mi < 2; mi++)
#pragma unroll
        for (int ni = 0; ni < 4; ni++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[mi][ni][r] = 0.0f;

    uint64_t ra, rb, la[8];
    auto fetch = [&](int64_t kc) {
        ra = gA[kc * 256];
        rb = gB[kc * 256];
#pragma unroll
        for (int e = 0; e < 8; e++) la[e] = gl[kc * 64 + e];
    };
    // decode the chunk held in ra/rb/la into (dA, dB), fetching chunk kn
    auto decode_next = [&](__hip_bfloat16* dA, __hip_bfloat16* dB, int64_t kn) {
        const uint64_t ca = ra, cb = rb;
        uint32_t lo[8], hi[8];
        split_bytes(la, lo, hi);
        fetch(kn);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            *reinterpret_cast<u32x4*>(dA + (4 * b + j) * P16 + 8 * o) = decode_row_perm(lo, hi, ca, j);
            *reinterpret_cast<u32x4*>(dB + (4 * b + j) * P16 + 8 * o) = decode_row_perm(lo, hi, cb, j);
        }
    };
    auto multiply = [&](const __hip_bfloat16* pA, const __hip_bfloat16* pB) {
#pragma unroll
        for (int ks = 0; ks < BK16 / 16; ks++) {
            const int kk = ks * 16 + (lane >> 5) * 8;
            bf16x8 fa[2], fb[4];
#pragma unroll
            for (int mi = 0; mi < 2; mi++)
                fa[mi] = *reinterpret_cast<const bf16x8*>(pA + (wr * 64 + mi * 32 + (lane & 31)) * P16 + kk);
#pragma unroll
            for (int ni = 0; ni < 4; ni++)
                fb[ni] = *reinterpret_cast<const bf16x8*>(pB + (wc * 128 + ni * 32 + (lane & 31)) * P16 + kk);
#pragma unroll
            for (int mi = 0; mi < 2; mi++)
#pragma unroll
                for (int ni = 0; ni < 4; ni++)
                    acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[mi], fb[ni], acc[mi][ni], 0, 0, 0);
        }
    };
    // step: multiply chunk kc from (cA, cB) while decoding chunk kc+1 into (nA, nB)
    auto step = [&](const __hip_bfloat16* cA, const __hip_bfloat16* cB, __hip_bfloat16* nA, __hip_bfloat16* nB,
                    int64_t kc) {
        decode_next(nA, nB, kc + 2 < c1 ? kc + 2 : c1 - 1);
        multiply(cA, cB);
        // one MFMA, then about five decode instructions, 32 times
#pragma unroll
        for (int i = 0; i < 32; i++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
        }
        lds_barrier();
    };
    fetch(c0);
    decode_next(sA0, sB0, c0 + 1 < c1 ? c0 + 1 : c0);
    lds_barrier();
    int64_t kc = c0;
    for (; kc + 2 <= c1; kc += 2) {
        step(sA0, sB0, sA1, sB1, kc);
        step(sA1, sB1, sA0, sB0, kc + 1);
    }
    if (kc < c1) multiply(sA0, sB0);
    store_block<2, 4, false>(S, S0, ldS, bi * BT2 + wr * 64, bj * BT2 + wc * 128, bi != bj, lane, acc, accumulate);
}

// k_syrk_pk<T, F>: the GRM from 2-bit genotypes on T x T tiles, by operand
// form F:
// * SYRK_HI: one BF16 piece of z, hi.hi (the single-pass GRM; T < 256, the
//   256 tile is k_syrk_pk256);
// * SYRK_SPLIT: z in two BF16 pieces, hi.hi + hi.lo + lo.hi (the split GRM),
//   stored rounded to 16 significant bits (round16, after the add or subtract
//   of an accumulating pass), which moves each value by at most 2^-16 of
//   itself; the block GEMM then needs two BF16 pieces of S instead of three;
// * SYRK_FP32: z_i z_j = (g_i - c) beta z_j + (alpha + beta c) z_j with the
//   marker's z = alpha + beta g and c the whole number nearest its mean.  g - c
//   is a whole number, exact in one BF16 piece, so the row operand needs one
//   piece and only the column operand beta z needs three (24 bits and more):
//   three products instead of the six of two three-piece operands, on the
//   BF16 pipe instead of the FP32 one (1/16 of its rate).  The second term
//   depends on the column alone: its sum over the markers is formed in FP64
//   beforehand and taken off at the store (center).
// Per chunk of BK markers each decoding thread makes two operand rows' worth of
// its byte row through two tables (one for SYRK_HI), and every multiplying wave
// adds the products of its block in a fixed order.  LDS: two buffers of the operands
// (four for the multi-piece forms), so the next chunk's decode runs beside
// this chunk's MFMAs.  SYRK_SPLIT: threads of the lower half decode the row
// panel (hi, lo), of the upper half the column panel; SYRK_FP32: the lower
// half the row operand and the column's lo, the upper half its hi and mid.
//
// T: the 256 tile (8 waves of 64 x 128, each decoding too) does the most MFMA
// work per decoded value (split GRM at N = 40,000, M = 60,000: 1350 TFLOP/s of BF16
// products, the matrix pipe busy 63% of the cycles at 2.08 GHz); a small
// GRM has too few of its tiles for 256 CUs, each walking all markers, and takes
// 128 (4 waves of 64 x 64) or 64 (4 waves of 32 x 32) tiles, see syrk_pk_tile.
// There a wave has a SIMD to itself and issues one instruction in about seven
// cycles, so the 230 instructions of a chunk's decode took longer than its
// products: four waves multiply and two groups of four decode, each every other
// chunk.  us over 8192 markers with every wave doing both and so: one round of 64
// tiles 130 and 82, of 128 tiles 277 and 195; 2080 of 128 tiles (N = 8000) 1708
// and 1688.  The per-element order is the same for every T: bitwise equal S.
constexpr int syrk_pk_threads(int T) { return T == 256 ? 512 : 768; }

template <int T, int F>
__global__ __launch_bounds__(syrk_pk_threads(T)) void k_syrk_pk(const uint8_t* __restrict__ tp, int64_t nchunk,
                                                                  int64_t k0, int64_t k1, SyrkTables tb,
                                                                  const int2* __restrict__ tiles, int64_t nblk,
                                                                  float* S, const float* S0, int64_t ldS,
                                                                  int accumulate, uint8_t* __restrict__ s24) {
    constexpr int BK = T == 64 ? 64 : 32;            // markers per chunk
    constexpr int P = BK + 8;                        // LDS row pitch (bf16 elements), conflict-free 16-byte reads
    constexpr int NOP = F == SYRK_HI ? 2 : 4;        // operands in LDS
    constexpr int HALF = T == 256 ? 256 : 128;       // threads per panel
    constexpr int OCT = BK / 8;                      // marker octets per chunk
    constexpr int WC = 2;                            // waves across the tile's columns
    constexpr int MI = T == 64 ? 1 : 2, NI = T == 256 ? 4 : MI;
    constexpr int NPROD = F == SYRK_HI ? 1 : 3;
    constexpr bool ROLES = T != 256;                 // waves 0 to 3 multiply, two groups of four decode
    __shared__ __attribute__((aligned(16))) __hip_bfloat16 s0[NOP * T * P];
    __shared__ __attribute__((aligned(16))) __hip_bfloat16 s1[NOP * T * P];
    const int2 t = tiles[xcd_remap(blockIdx.x, nblk)];
    const int64_t bi = t.x, bj = t.y;
    const int tid = ROLES ? threadIdx.x & 255 : threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int wr = wv / WC, wc = wv % WC;
    // half (0, 1), octet and byte row of this thread
    const int h = tid / HALF, o = tid % OCT, b = (tid % HALF) / OCT;
    // its byte row of tile row / column index x: uint64 units, a 64-marker
    // chunk is 256 words on from the one before, its second 32 markers 4 words
    // into a byte row
    auto byte_row = [&](int64_t x) {
        const int64_t s4 = x * (T / 4) + b;          // byte row of the matrix: 32 per 128-sample panel
        return reinterpret_cast<const uint64_t*>(tp + ((s4 >> 5) * nchunk * 32 + (s4 & 31)) * 64 + 8 * o);
    };
    const bool lower = h == 0;
    const uint64_t* g0 = byte_row(lower ? bi : bj);
    const uint64_t* g1 = byte_row(F == SYRK_FP32 || !lower ? bj : bi);
    const uint64_t* t0 = (F == SYRK_FP32 && !lower ? tb.t[1] : tb.t[0]) + 8 * o;
    const uint64_t* t1 = (F == SYRK_FP32 ? (lower ? tb.t[3] : tb.t[2]) : tb.t[1]) + 8 * o;
    constexpr int OPS = T * P;                       // one operand
    const int dst = (F == SYRK_HI ? h : 2 * h) * OPS + (4 * b) * P + 8 * o;

    f32x16 acc[MI][NI];
#pragma unroll
    for (int mi = 0; mi < MI; mi++)
#pragma unroll
        for (int ni = 0; ni < NI; ni++)
#pragma unroll
            for (int q = 0; q < 16; q++) acc[mi][ni][q] = 0.0f;

    uint64_t raw0, raw1, l0[8], l1[8];
    auto fetch = [&](int64_t kc) {
        kc = kc < k1 ? kc : k1 - 1;                  // past the end: the last chunk again, unused
        const int64_t off = BK == 64 ? kc * 256 : (kc >> 1) * 256 + (kc & 1) * 4;
        raw0 = g0[off];
        if (F == SYRK_FP32) raw1 = g1[off];
#pragma unroll
        for (int e = 0; e < 8; e++) l0[e] = t0[kc * BK + e];
        if (F != SYRK_HI) {
#pragma unroll
            for (int e = 0; e < 8; e++) l1[e] = t1[kc * BK + e];
        }
    };
    // decode the chunk held in the registers, row by row to f(row, its operands),
    // fetching chunk kn
    constexpr int NW = F == SYRK_HI ? 1 : 2;         // operands a thread decodes
    auto decode = [&](int64_t kn, auto f) {
        const uint64_t c0 = raw0, c1 = F == SYRK_FP32 ? raw1 : raw0;
        uint32_t lo0[8], hi0[8], lo1[8], hi1[8];
        split_bytes(l0, lo0, hi0);
        if (F != SYRK_HI) split_bytes(l1, lo1, hi1);
        fetch(kn);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const u32x4 v0 = decode_row_perm(lo0, hi0, c0, j);
            f(j, v0, F != SYRK_HI ? decode_row_perm(lo1, hi1, c1, j) : v0);
        }
    };
    auto put_row = [&](__hip_bfloat16* d, int j, u32x4 v0, u32x4 v1) {
        *reinterpret_cast<u32x4*>(d + dst + j * P) = v0;
        if (F != SYRK_HI) *reinterpret_cast<u32x4*>(d + dst + OPS + j * P) = v1;
    };
    auto decode_to = [&](__hip_bfloat16* d, int64_t kn) {
        decode(kn, [&](int j, u32x4 v0, u32x4 v1) { put_row(d, j, v0, v1); });
    };
    auto multiply = [&](const __hip_bfloat16* d) {
#pragma unroll
        for (int ks = 0; ks < BK / 16; ks++) {
            const int kk = ks * 16 + (lane >> 5) * 8;
            // operand q of row block r
            auto frag = [&](int q, int r) {
                return *reinterpret_cast<const bf16x8*>(d + q * OPS + (r + (lane & 31)) * P + kk);
            };
            bf16x8 fa[MI], fl[MI];
#pragma unroll
            for (int mi = 0; mi < MI; mi++) {
                fa[mi] = frag(0, wr * 32 * MI + mi * 32);
                if (F == SYRK_SPLIT) fl[mi] = frag(1, wr * 32 * MI + mi * 32);
            }
#pragma unroll
            for (int ni = 0; ni < NI; ni++) {
                const int c = wc * 32 * NI + ni * 32;
                if (F == SYRK_HI) {
                    const bf16x8 fb = frag(1, c);
#pragma unroll
                    for (int mi = 0; mi < MI; mi++)
                        acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[mi], fb, acc[mi][ni], 0, 0, 0);
                } else if (F == SYRK_SPLIT) {
                    const bf16x8 fbh = frag(2, c), fbl = frag(3, c);
#pragma unroll
                    for (int mi = 0; mi < MI; mi++) {
                        acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[mi], fbh, acc[mi][ni], 0, 0, 0);
                        acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[mi], fbl, acc[mi][ni], 0, 0, 0);
                        acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fl[mi], fbh, acc[mi][ni], 0, 0, 0);
                    }
                } else {
                    const bf16x8 fbl = frag(1, c), fbh = frag(2, c), fbm = frag(3, c);
#pragma unroll
                    for (int mi = 0; mi < MI; mi++) {
                        acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[mi], fbl, acc[mi][ni], 0, 0, 0);
                        acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[mi], fbm, acc[mi][ni], 0, 0, 0);
                        acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[mi], fbh, acc[mi][ni], 0, 0, 0);
                    }
                }
            }
        }
    };
    // multiply chunk kc from cur while decoding chunk kc+1 into nxt: one MFMA,
    // then its share of the decode's VALU instructions
    auto step = [&](const __hip_bfloat16* cur, __hip_bfloat16* nxt, int64_t kc) {
        constexpr int NM = MI * NI * (BK / 16) * NPROD;
        decode_to(nxt, kc + 2);
        multiply(cur);
#pragma unroll
        for (int i = 0; i < NM; i++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, (F == SYRK_HI ? 72 : 144) / NM, 0);
        }
        lds_barrier();
    };
    // s1 is the waves' scratch: after the last chunk but one (behind its barrier)
    // nothing reads or writes it
    static_assert(sizeof(s1) >= sizeof(float) * S24_SCRATCH * (T == 256 ? 8 : 4), "");
    auto store = [&]() {
        store_block<MI, NI, F == SYRK_SPLIT>(S, S0, ldS, bi * T + wr * 32 * MI, bj * T + wc * 32 * NI, bi != bj, lane,
                                             acc, accumulate, F == SYRK_FP32 ? tb.center : nullptr, s24,
                                             reinterpret_cast<float*>(s1) + wv * S24_SCRATCH);
    };
    int64_t kc = k0;
    if constexpr (ROLES) {
        // one barrier per chunk: chunk kc is multiplied while kc + 1 is put into the
        // other buffer by the group that decoded it a chunk ago, and the other
        // group decodes kc + 2
        u32x4 dec[NW][4];
        auto hold = [&](int j, u32x4 v0, u32x4 v1) {
            dec[0][j] = v0;
            if (F != SYRK_HI) dec[NW - 1][j] = v1;
        };
        auto put = [&](__hip_bfloat16* d) {
#pragma unroll
            for (int j = 0; j < 4; j++) put_row(d, j, dec[0][j], dec[NW - 1][j]);
        };
        const int role = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
        if (role == 1) {
            fetch(k0);
            decode_to(s0, k0 + 2);
            lds_barrier();
            for (; kc + 2 <= k1; kc += 2) {
                decode(kc + 4, hold);
                lds_barrier();
                put(s0);
                lds_barrier();
            }
            return;
        }
        if (role == 2) {
            fetch(k0 + 1);
            decode(k0 + 3, hold);
            lds_barrier();
            for (; kc + 2 <= k1; kc += 2) {
                put(s1);
                lds_barrier();
                decode(kc + 5, hold);
                lds_barrier();
            }
            return;
        }
        lds_barrier();
        for (; kc + 2 <= k1; kc += 2) {
            multiply(s0);
            lds_barrier();
            multiply(s1);
            lds_barrier();
        }
        if (kc < k1) multiply(s0);
        store();
        return;
    }
    fetch(k0);
    decode_to(s0, k0 + 1);
    lds_barrier();
    for (; kc + 2 <= k1; kc += 2) {
        step(s0, s1, kc);
        step(s1, s0, kc + 1);
    }
    if (kc < k1) multiply(s0);
    store();
}

// Re-tile the packed genotypes for the SYRK: block (p, c) byte (b, m) = byte
// 32p + b of GRM marker 64(c0 + c) + m, with padding codes 0b01 (samples >= Nnm,
// markers >= Mqc).  A workgroup takes four panels (a cache line of each row)
// of one chunk: dwords of four markers' rows are transposed in registers,
// collected in LDS and stored 16 bytes per thread.  Bound by its two streams:
// 215 us for 1.2 GB at N = 40,000, M = 60,000, 5.6 TB/s (1431 us with a byte per
// thread and 32 bytes of a row at a time, which fetched the genotypes several
// times over).
__global__ __launch_bounds__(256) void k_pack_tiles(const uint8_t* __restrict__ packed, int64_t Mqc, int64_t Nnm,
                                                    int64_t ldp, int64_t npanel, int64_t c0, int64_t nchunk,
                                                    uint8_t* __restrict__ tp) {
    __shared__ uint32_t tile[128 * 17];              // [byte row of four panels][16 marker quads + 1]
    const int64_t p0 = 4 * (int64_t)blockIdx.x, c = blockIdx.y;
    const int tid = threadIdx.x, c4 = tid & 31, mq = tid >> 5;
    const int64_t left = Nnm - (p0 * 128 + 16 * c4); // samples from this dword on
    const uint32_t keep = left >= 16 ? 0xFFFFFFFFu : (left <= 0 ? 0u : (1u << (2 * left)) - 1u);
    const uint8_t* src = packed + p0 * 32 + 4 * c4;  // p0 * 32 + 128 <= ldp
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const int quad = mq + 8 * q;
        uint32_t w[4], t[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int64_t j = (c0 + c) * 64 + 4 * quad + e;
            // rows past the markers are the buffer's padding
            const uint32_t k = j < Mqc ? keep : 0u;
            w[e] = (*reinterpret_cast<const uint32_t*>(src + j * ldp) & k) | (0x55555555u & ~k);
        }
        transpose4x4(w[0], w[1], w[2], w[3], t);
#pragma unroll
        for (int e = 0; e < 4; e++) tile[(4 * c4 + e) * 17 + quad] = t[e];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const int i = tid + 256 * q;                 // 16 bytes: four marker quads of byte row i / 4
        const int64_t p = p0 + (i >> 7);
        const uint32_t* v = tile + (i >> 2) * 17 + 4 * (i & 3);
        if (p < npanel)
            *reinterpret_cast<uint4*>(tp + (p * nchunk + c) * 2048 + 16 * (i & 127)) =
                make_uint4(v[0], v[1], v[2], v[3]);
    }
}

// The SYRK's tables: entry j of a table is GRM marker base + j, four BF16
// values indexed by the internal code (00 -> two copies, 01 -> 0, 10 -> one,
// 11 -> none); zero outside markers [j0, j1).
// SYRK_HI / SYRK_SPLIT: t[0] z rounded to BF16 (hi), t[1] the remainder z - hi,
// exact in FP32, rounded to BF16 (lo), so that z - hi - lo is within 2^-16 |z|.
// SYRK_FP32: t[0] g - c, t[1..3] beta z in three BF16 pieces (each the rounded
// remainder of the ones before), and corr[j] = -(alpha + beta c) z in FP64 per
// genotype, from z(0), z(1), z(2) as alpha = z(0), beta = (z(2) - z(0)) / 2.
__device__ __forceinline__ uint64_t bf16_code(double x) { return __bfloat16_as_ushort(__float2bfloat16((float)x)); }
__device__ __forceinline__ uint64_t four_codes(uint64_t v0, uint64_t v1, uint64_t v2) {
    return v2 | (v1 << 32) | (v0 << 48);
}

__global__ void k_syrk_tables(const float4* __restrict__ lut, int64_t base, int64_t n, int64_t j0, int64_t j1,
                              int form, SyrkTables tb) {
    const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int64_t j = base + k;
    uint64_t out[4] = {0, 0, 0, 0};
    double cor[3] = {0.0, 0.0, 0.0};
    if (j >= j0 && j < j1) {
        const float4 L = lut[j];
        const float z[3] = {L.x, L.y, L.z};
        if (form != SYRK_FP32) {
            uint64_t hi[3], lo[3];
#pragma unroll
            for (int g = 0; g < 3; g++) {
                const __hip_bfloat16 h = __float2bfloat16(z[g]);
                hi[g] = __bfloat16_as_ushort(h);
                lo[g] = __bfloat16_as_ushort(__float2bfloat16(__fsub_rn(z[g], __bfloat162float(h))));
            }
            out[0] = four_codes(hi[0], hi[1], hi[2]);
            out[1] = four_codes(lo[0], lo[1], lo[2]);
        } else {
            const double alpha = z[0], beta = 0.5 * ((double)z[2] - (double)z[0]);
            // the mean genotype is -alpha / beta
            const double c = beta > 0.0 ? fmin(fmax(rint(-alpha / beta), 0.0), 2.0) : 0.0;
            out[0] = four_codes(bf16_code(0.0 - c), bf16_code(1.0 - c), bf16_code(2.0 - c));
            uint64_t pc[3][3];
#pragma unroll
            for (int g = 0; g < 3; g++) {
                double x = beta * (double)z[g];
                cor[g] = -(alpha + beta * c) * (double)z[g];
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    const __hip_bfloat16 h = __float2bfloat16((float)x);
                    pc[q][g] = __bfloat16_as_ushort(h);
                    x -= (double)__bfloat162float(h);
                }
            }
#pragma unroll
            for (int q = 0; q < 3; q++) out[1 + q] = four_codes(pc[q][0], pc[q][1], pc[q][2]);
        }
    }
    for (int q = 0; q < 4; q++)
        if (tb.t[q]) tb.t[q][k] = out[q];
    if (tb.corr)
        for (int g = 0; g < 3; g++) tb.corr[3 * k + g] = cor[g];
}

// SYRK_FP32's column terms: per sample the FP64 sum of corr over the markers'
// genotypes.  k_center_part: 16 samples (a dword of codes) per lane, one wave
// per 1024 samples and slice of the markers, four rows' loads in flight;
// k_center_sum adds the slices in order.
__global__ __launch_bounds__(64) void k_center_part(const uint8_t* __restrict__ packed, int64_t ldp,
                                                    const double* __restrict__ corr, int64_t base, int64_t n,
                                                    int64_t per, int64_t Npad, double* __restrict__ part) {
    const int64_t d = blockIdx.x * (int64_t)64 + threadIdx.x;    // dword of the row
    if (16 * d >= Npad) return;                                  // ldp >= Npad / 4
    const int64_t a = blockIdx.y * per, b = min(a + per, n);
    const uint8_t* src = packed + base * ldp + 4 * d;
    double s[16];
#pragma unroll
    for (int i = 0; i < 16; i++) s[i] = 0.0;
    for (int64_t j = a; j < b; j += 4) {
        uint32_t w[4];
        double c[4][3];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int64_t jj = min(j + u, b - 1);
            const double on = j + u < b ? 1.0 : 0.0;
            w[u] = *reinterpret_cast<const uint32_t*>(src + jj * ldp);
#pragma unroll
            for (int g = 0; g < 3; g++) c[u][g] = on * corr[3 * jj + g];
        }
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const uint32_t v = w[u] >> (2 * i);
                s[i] += (v & 2u) ? ((v & 1u) ? c[u][0] : c[u][1]) : c[u][2];
            }
    }
#pragma unroll
    for (int i = 0; i < 16; i++) part[blockIdx.y * Npad + 16 * d + i] = s[i];
}

__global__ __launch_bounds__(256) void k_center_sum(const double* __restrict__ part, int64_t nslice, int64_t Npad,
                                                    int64_t Nnm, float* __restrict__ center) {
    // 32 samples per workgroup, eight threads each: thread q adds slices q, q + 8, ...
    __shared__ double sm[8][32];
    const int l = threadIdx.x & 31, q = threadIdx.x >> 5;
    const int64_t i = blockIdx.x * (int64_t)32 + l;              // Npad is a multiple of 32
    double s = 0.0;
#pragma unroll 8
    for (int64_t k = q; k < nslice; k += 8) s += part[k * Npad + i];
    sm[q][l] = s;
    __syncthreads();
    if (q == 0) {
#pragma unroll
        for (int k = 1; k < 8; k++) s += sm[k][l];
        center[i] = i < Nnm ? (float)s : 0.0f;
    }
}

// Copy each diagonal tile's lower half onto its upper half: S[c][r] =
// S[r][c] for r > c inside tile t (rows and columns t*T + [0, T)).  The split
// GRM's cross terms add hi.lo and lo.hi to the two mirror entries of a
// diagonal tile in opposite orders; this keeps S exactly symmetric, with the
// lower triangle's values, as off-diagonal tiles are mirrored.  Block (t, r):
// row r of tile t; its threads write column r of the upper part.  Rows and
// columns from `rows` on (ld: none) are set to zero: the FP32 form's store takes
// the columns' centers off the padded rows' zeros too (leaving them out there
// took the SYRK of 5003 samples 8 us of 1350, here it takes 1.3).
__global__ __launch_bounds__(256) void k_mirror_diag(float* __restrict__ S, int64_t ld, int T, int64_t rows) {
    const int64_t t = blockIdx.x, r = blockIdx.y;
    const int64_t base = t * T, i = base + r;
    for (int64_t c = threadIdx.x; c < r; c += blockDim.x)
        S[(base + c) * ld + i] = i < rows ? S[i * ld + base + c] : 0.0f;
    for (int64_t c = (i < rows ? rows : 0) + threadIdx.x; c < ld; c += blockDim.x) S[i * ld + c] = 0.0f;
}

// out[nr][nc] = S[r0 + i][c0 + j] / m, rounded once (div_rn): the read-back of a
// block of K.  One row per blockIdx.y step, four columns per thread.
__global__ __launch_bounds__(256) void k_grm_block(const float* __restrict__ S, int64_t ld, int64_t nr, int64_t nc,
                                                   float m, float* __restrict__ out) {
    const int64_t j0 = 4 * (blockIdx.x * (int64_t)256 + threadIdx.x);
    for (int64_t i = blockIdx.y; i < nr; i += gridDim.y)
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (j0 + e < nc) out[i * nc + j0 + e] = div_rn(S[i * ld + j0 + e], m);
}

}  // namespace

int syrk_kchunk_bf16() { return BK16; }

// slices of the markers in k_center_part: enough waves to fill the chip,
// at least 32 markers each
static int64_t center_slices(int64_t n, int64_t Npad) {
    const int64_t blocks = (Npad + 1023) / 1024;
    return std::max<int64_t>(1, std::min<int64_t>({(n + 31) / 32, (2048 + blocks - 1) / blocks, (int64_t)512}));
}

namespace {
// the parts of SyrkOperands' block: tiled genotypes, tables, then (SYRK_FP32)
// corr, center, slices
struct OperandParts {
    int64_t c0, nchunk, n, npanel, ntab, nsl, tp, tab, cor, cen, total;
    OperandParts(int form, int64_t Npad, int64_t j0, int64_t j1) {
        c0 = j0 / 64;
        nchunk = (j1 + 63) / 64 - c0;
        npanel = Npad / BT;
        n = nchunk * 64;
        ntab = form == SYRK_HI ? 1 : (form == SYRK_SPLIT ? 2 : 4);
        nsl = form == SYRK_FP32 ? center_slices(n, Npad) : 0;
        tp = npanel * nchunk * 2048;
        tab = 8 * n;
        cor = nsl ? round_up(24 * n, 256) : 0;
        cen = nsl ? round_up(4 * Npad, 256) : 0;
        total = tp + ntab * tab + cor + cen + 8 * nsl * Npad;
    }
};
}  // namespace

int64_t SyrkOperands::bytes(int form, int64_t Npad, int64_t j0, int64_t j1) {
    return OperandParts(form, Npad, j0, j1).total;
}

hipError_t SyrkOperands::build(hipStream_t s, int form_, const uint8_t* packed, const float4* lut, int64_t Mqc,
                               int64_t Nnm, int64_t Npad_, int64_t ldp, int64_t j0, int64_t j1) {
    release();
    if (j0 < 0 || j1 > Mqc || j0 >= j1 || Npad_ % 256 != 0 || 4 * ldp < Npad_) return hipErrorInvalidValue;
    form = form_;
    Npad = Npad_;
    const OperandParts q(form, Npad, j0, j1);
    const int64_t c0 = q.c0, npanel = q.npanel, n = q.n, nsl = q.nsl;
    nchunk = q.nchunk;
    rows = Nnm;
    hipError_t e = hipMalloc(&block, (size_t)q.total);
    if (e != hipSuccess) {
        block = nullptr;
        return e;
    }
    uint8_t* p = static_cast<uint8_t*>(block);
    tp = p;
    p += q.tp;
    for (int k = 0; k < q.ntab; k++, p += q.tab) tb.t[k] = reinterpret_cast<uint64_t*>(p);
    double* part = nullptr;
    if (nsl) {
        tb.corr = reinterpret_cast<double*>(p);
        tb.center = reinterpret_cast<float*>(p + q.cor);
        part = reinterpret_cast<double*>(p + q.cor + q.cen);
    }
    hipLaunchKernelGGL(k_pack_tiles, dim3((unsigned)((npanel + 3) / 4), (unsigned)nchunk), dim3(256), 0, s, packed,
                       Mqc, Nnm, ldp, npanel, c0, nchunk, tp);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_syrk_tables, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, lut, c0 * 64, n, j0, j1,
                       form, tb);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (nsl) {
        const int64_t per = round_up((n + nsl - 1) / nsl, 4);
        hipLaunchKernelGGL(k_center_part, dim3((unsigned)((Npad + 1023) / 1024), (unsigned)nsl), dim3(64), 0, s, packed,
                           ldp, tb.corr, c0 * 64, n, per, Npad, part);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        hipLaunchKernelGGL(k_center_sum, dim3((unsigned)(Npad / 32)), dim3(256), 0, s, part, nsl, Npad, Nnm,
                           tb.center);
    }
    return hipGetLastError();
}

void SyrkOperands::release() {
    if (block) (void)hipFree(block);
    *this = SyrkOperands{};
}

template <int T, int F>
static void launch_pk(hipStream_t s, const SyrkOperands& op, const int2* tiles, float* S, const float* S0,
                      int accumulate, uint8_t* s24 = nullptr) {
    constexpr int BK = T == 64 ? 64 : 32;
    const int64_t nt = op.Npad / T, nblk = nt * (nt + 1) / 2;
    hipLaunchKernelGGL((k_syrk_pk<T, F>), dim3((unsigned)nblk), dim3(syrk_pk_threads(T)), 0, s, op.tp, op.nchunk,
                       (int64_t)0, op.nchunk * (64 / BK), op.tb, tiles, nblk, S, S0, op.Npad, accumulate,
                       s24);
}

hipError_t launch_syrk_pk(hipStream_t s, const SyrkOperands& op, const int2* tiles, float* S, const float* S0,
                          int accumulate, int tile, uint8_t* s24) {
    if ((tile != 64 && tile != BT && tile != BT2) || op.Npad % tile != 0 || !op.block) return hipErrorInvalidValue;
    if (op.form == SYRK_HI && tile == BT2) {
        const int64_t nt = op.Npad / BT2, nblk = nt * (nt + 1) / 2;
        hipLaunchKernelGGL(k_syrk_pk256, dim3((unsigned)nblk), dim3(512), 0, s, op.tp, op.nchunk, (int64_t)0, op.nchunk,
                           op.tb.t[0], tiles, nblk, S, S0, op.Npad, accumulate);
    } else if (op.form == SYRK_HI) {
        if (tile == BT) launch_pk<128, SYRK_HI>(s, op, tiles, S, S0, accumulate);
        else launch_pk<64, SYRK_HI>(s, op, tiles, S, S0, accumulate);
    } else if (op.form == SYRK_SPLIT) {
        if (tile == BT2) launch_pk<256, SYRK_SPLIT>(s, op, tiles, S, S0, accumulate, s24);
        else if (tile == BT) launch_pk<128, SYRK_SPLIT>(s, op, tiles, S, S0, accumulate, s24);
        else launch_pk<64, SYRK_SPLIT>(s, op, tiles, S, S0, accumulate, s24);
    } else {
        if (tile == BT2) launch_pk<256, SYRK_FP32>(s, op, tiles, S, S0, accumulate);
        else if (tile == BT) launch_pk<128, SYRK_FP32>(s, op, tiles, S, S0, accumulate);
        else launch_pk<64, SYRK_FP32>(s, op, tiles, S, S0, accumulate);
    }
    hipError_t e = hipGetLastError();
    // the multi-piece forms reach a diagonal tile's two mirror entries by
    // different sums: keep S exactly symmetric
    if (e == hipSuccess && op.form != SYRK_HI)
        e = launch_mirror_diag(s, S, op.Npad, tile, op.form == SYRK_FP32 ? op.rows : op.Npad);
    return e;
}

hipError_t launch_mirror_diag(hipStream_t s, float* S, int64_t Npad, int tile, int64_t rows) {
    if (tile <= 0 || Npad % tile != 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_mirror_diag, dim3((unsigned)(Npad / tile), (unsigned)tile), dim3(256), 0, s, S, Npad, tile,
                       rows);
    return hipGetLastError();
}

hipError_t launch_grm_block(hipStream_t s, const float* S, int64_t ld, int64_t nr, int64_t nc, float m, float* out) {
    if (nr <= 0 || nc <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_grm_block, dim3((unsigned)((nc + 1023) / 1024), (unsigned)std::min<int64_t>(nr, 32768)),
                       dim3(256), 0, s, S, ld, nr, nc, m, out);
    return hipGetLastError();
}

// Tile edge of the 2-bit-input SYRK at Npad rows (every size gives the same
// bits): the one of least time by a model of rounds of one tile per CU, in us
// over 8192 markers.  Measured us with 64, 128 and 256 tiles, split form: N = 1000
// 82, 171, 522; 1500 163, 185, 523; 2500 335, 195, 524; 3000 418, 367, 525; 4000
// 746, 574, 558; 5000 1031, 735, 574; 8000 2554, 1688, 1749; 12,000 5726, 3367,
// 3026; SYRK_FP32 within 5% of it; SYRK_HI: 1000 47, 87, 167; 2500 152, 94, 173;
// 3000 196, 182, 177; 4000 352, 276, 180; 8000 1117, 804, 616.
// SAIGE_SYRK_TILE=64, 128 or 256 sets it (the tests compare them).
int syrk_pk_tile(int64_t Npad, int form) {
    if (const char* env = std::getenv("SAIGE_SYRK_TILE")) {
        const int t = std::atoi(env);
        if (t == 64 || t == BT || t == BT2) return t;
    }
    auto rounds = [&](int64_t T) { return std::ceil((double)(Npad / T) * (double)(Npad / T + 1) / 512.0); };
    const bool hi = form == SYRK_HI;
    const double t64 = (hi ? 47.0 : 82.0) * rounds(64), t128 = (hi ? 92.0 : 190.0) * rounds(BT);
    const double r256 = rounds(BT2), t256 = hi ? (r256 > 1 ? 200.0 : 178.0) * r256 : (r256 > 1 ? 580.0 : 545.0) * r256;
    if (t256 <= t128 && t256 <= t64) return BT2;
    return t128 <= t64 ? BT : 64;
}

int syrk_tile() { return BT; }

// Lower-triangle tiles (bi >= bj) of an nt x nt tile grid, grouped into
// g x g super-blocks (super-block row >= column, each walked row by row).
std::vector<int2> syrk_tile_order(int64_t nt, int64_t g) {
    std::vector<int2> out;
    out.reserve((size_t)(nt * (nt + 1) / 2));
    const int64_t ns = (nt + g - 1) / g;
    for (int64_t SI = 0; SI < ns; SI++)
        for (int64_t SJ = 0; SJ <= SI; SJ++)
            for (int64_t bi = SI * g; bi < std::min(nt, (SI + 1) * g); bi++)
                for (int64_t bj = SJ * g; bj < std::min(bi + 1, (SJ + 1) * g); bj++)
                    out.push_back(make_int2((int)bi, (int)bj));
    return out;
}

hipError_t launch_syrk_bf16(hipStream_t s, const __hip_bfloat16* Zp, int64_t Npad, int64_t ldz,
                            int64_t kdim, const int2* tiles, float* S, int accumulate) {
    const int64_t nt = Npad / BT;
    const int64_t nblk = nt * (nt + 1) / 2;
    hipLaunchKernelGGL(k_syrk_bf16, dim3((unsigned)nblk), dim3(256), 0, s, Zp, ldz, kdim, tiles, nblk, S, Npad,
                       accumulate);
    return hipGetLastError();
}

}  // namespace saige
