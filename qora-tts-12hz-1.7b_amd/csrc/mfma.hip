// mfma.hip — the Q4 GEMM on the matrix cores (v_mfma_f32_32x32x16_f16) for
// row counts where the VALU GEMV's per-row cost dominates: gemm_q4
// (src/gemv.rs:311-375) at M >= 8, and the talker prefill's projections
// (src/talker.rs:364-462).
//
// Exactness.  The reference forms every term as f32(f32(s)*x)*(nib-8) and
// sums in f32.  Here each term is (xh + xl) * (sa*q + sb*q) with
//   q = nib - 8 in [-8, 7], exact in binary16;
//   s = sa + sb, sa the binary16 scale rounded to 7 significand bits and sb
//     the rest (at most 4 bits), so sa*q and sb*q are exact binary16 products
//     (formed with v_pk_mul_f16);
//   x = xh + xl, xh = f16(x), xl = f16(x - xh): |x - xh - xl| <= 2^-22 |x|.
// Products of binary16 values are exact in the f32 accumulator, and the
// xl*sb*q term (relative size 2^-19) is dropped, so every term carries a
// relative error of ~2^-19 or less before the f32 sums -- the f32 level the
// parity tolerance is set for.  With GemmMfmaParams::full that term is a
// fourth MFMA, and a term's error that of x's split, 2^-22 (the text
// projection, whose other path is the GEMV's f32 products).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "device_common.h"
#include "internal.h"

namespace qtts {

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4v __attribute__((ext_vector_type(4)));

// Repack of one panel-major Q4 weight into the MFMA B-operand order
// (DevQ4Mfma in internal.h): thread (p, s, l) gathers its 8 nibbles.
// A scale of magnitude above 8188 would overflow binary16 in sa * q; such a
// weight sets *too_large and stays on the VALU path.
__global__ void k_repack_mfma(DevQ4 w, uint32_t *wm, uint16_t *sa, uint16_t *sb, int *too_large) {
    const int Ks = w.K / 16, panels = w.N / 32;
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t total = (size_t)panels * Ks * 64;
    if (idx < total) {
        const int l = (int)(idx & 63);
        const size_t ps = idx >> 6;
        const int p = (int)(ps / Ks), s = (int)(ps - (size_t)p * Ks);
        const int col = l & 31, k0 = 16 * s + 8 * (l >> 5);
        const uint8_t *rows = reinterpret_cast<const uint8_t *>(w.wq + (size_t)p * w.K);
        uint32_t word = 0;
        for (int i = 0; i < 8; i++) {
            const uint8_t b = rows[(size_t)(k0 + i) * 16 + (col >> 1)];
            const uint32_t nib = (col & 1) ? (b >> 4) : (b & 15u);
            word |= nib << (4 * (i >> 1) + 16 * (i & 1));
        }
        wm[idx] = word;
    }
    // scales: one thread per (panel, row)
    const size_t nrows = (size_t)panels * w.K;
    if (idx < nrows) {
        const uint16_t s = w.ws[idx];
        if (fabsf((float)__builtin_bit_cast(_Float16, s)) > 8188.0f) atomicOr(too_large, 1);
        // top 7 significand bits, rounded to nearest unless that could
        // overflow sa * q (then truncated)
        uint16_t hi = (uint16_t)(s + 8u) & 0xFFF0u;
        if (fabsf((float)__builtin_bit_cast(_Float16, hi)) > 8128.0f) hi = s & 0xFFF0u;
        sa[idx] = hi;
        const float d = (float)__builtin_bit_cast(_Float16, s) - (float)__builtin_bit_cast(_Float16, hi);
        sb[idx] = __builtin_bit_cast(uint16_t, (_Float16)d);  // exact
    }
}

// One block per row m < Mpad: v = the row after the prologue (plain,
// rms_norm_f16 of src/gemv.rs:406-417, or silu(g)*u of
// src/talker.rs:342-345, with the same expression order as the GEMV path),
// then v * 2^e split into binary16 hi + lo, with e the per-row exponent that
// puts max|v| * 2^e in [2^14, 2^15) (no binary16 overflow; small entries keep
// their relative precision).  With RMSNorm, max|v| is taken as
// (1/rms) * max|x * gamma| from the same reduction as the sum of squares (one
// block barrier, and the gammas load with the row), which can miss max|v| by
// a few ulps: e is then one lower, putting max|v| * 2^e in [2^13, 2^15).
// rexp[m] = e; rows >= M are zero with e = 0.  xh and xl are stored in the
// MFMA A-operand order -- [M-tile][16-row step][lane][8], or
// [32-row step][lane][8] for k_gemm_mfma16 -- so that each wave's operand
// load of a step is one contiguous KiB.  One 8-value group per thread (K =
// 6144: 1024 threads a row).
template <int NT, bool M16>  // threads (K <= 8 * NT); the 16-row operand order
__global__ __launch_bounds__(NT) void k_mfma_rows(MfmaRowsParams P) {
    __shared__ float red[2][NT / 64];
    // Blocks of one XCD (every 8th) take neighbouring rows (Mpad is a multiple
    // of 16): 8 rows' 16-byte slots make up each 128-byte line of xh and xl,
    // which then leaves one L2 whole (1000 rows of 6144: 23.3 -> 15.0 us).
    const int m = (int)((blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3));
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int K = P.K, Ks = K / 16, ng = K / 8, g = tid;
    // 8-value group g = k / 8 of row m goes to the A-operand slot of lane
    // (m % 32) + 32 (g % 2) in step g / 2 of M-tile m / 32, or (16-row
    // operands) of lane m + 16 (g % 4) in 32-row step g / 4
    const size_t tile = M16 ? (size_t)m : (size_t)(m >> 5) * Ks * 64 + (m & 31);
    auto slot = [&](int g) {
        return (tile + (M16 ? (size_t)(g >> 2) * 64 + 16 * (g & 3) : (size_t)(g >> 1) * 64 + 32 * (g & 1))) * 8;
    };
    if (m >= P.M) {
        if (g < ng) {
            *reinterpret_cast<half8 *>(P.xh + slot(g)) = (half8){};
            *reinterpret_cast<half8 *>(P.xl + slot(g)) = (half8){};
        }
        if (tid == 0) P.rexp[m] = 0;
        return;
    }
    const float *src = P.x + (size_t)m * P.ldx;
    const bool norm = P.mode == MFMA_ROWS_RMSNORM;
    float v[8];
    uint32_t gw[4];
    // 1. the row's values and gammas (all loads first); the sum of squares
    //    and max|x * gamma| (RMSNorm) or max|v|
    if (g < ng) {
        const float4 a = *reinterpret_cast<const float4 *>(src + 8 * g);
        const float4 b = *reinterpret_cast<const float4 *>(src + 8 * g + 4);
        v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w;
        v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
        if (norm) {
            const uint4 q = *reinterpret_cast<const uint4 *>(P.gamma + 8 * g);
            gw[0] = q.x, gw[1] = q.y, gw[2] = q.z, gw[3] = q.w;
        }
        if (P.mode == MFMA_ROWS_SILU) {
#pragma unroll
            for (int i = 0; i < 8; i++) v[i] = v[i] / (1.0f + expf(-v[i]));
        }
        if (P.mode == MFMA_ROWS_SWIGLU) {
            const float4 c = *reinterpret_cast<const float4 *>(src + K + 8 * g);
            const float4 d = *reinterpret_cast<const float4 *>(src + K + 8 * g + 4);
            const float u[8] = {c.x, c.y, c.z, c.w, d.x, d.y, d.z, d.w};
#pragma unroll
            for (int i = 0; i < 8; i++) v[i] = (v[i] / (1.0f + expf(-v[i]))) * u[i];
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = 0.0f;
#pragma unroll
        for (int q = 0; q < 4; q++) gw[q] = 0u;
    }
    float ss = 0.0f, mx = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        ss += v[i] * v[i];
        // NaN entries drop out of the max here and stay NaN below
        mx = fmaxf(mx, fabsf(norm ? v[i] * f16_to_f32((uint16_t)(gw[i / 2] >> (16 * (i & 1)))) : v[i]));
    }
    ss = wave_sum(ss);
    mx = wave_max(mx);
    if (lane == 0) {
        red[0][wave] = ss;
        red[1][wave] = mx;
    }
    __syncthreads();
    mx = red[1][0];
#pragma unroll
    for (int w = 1; w < NT / 64; w++) mx = fmaxf(mx, red[1][w]);
    if (norm) {
        ss = 0.0f;
#pragma unroll
        for (int w = 0; w < NT / 64; w += 4) ss += (red[0][w] + red[0][w + 1]) + (red[0][w + 2] + red[0][w + 3]);
        const float inv = 1.0f / sqrtf(ss / (float)K + 1e-6f);
        mx *= inv;
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = v[i] * inv * f16_to_f32((uint16_t)(gw[i / 2] >> (16 * (i & 1))));
    }
    // 2. the row exponent
    int e = 0;
    if (mx > 0.0f && mx < INFINITY) {
        int E;
        (void)frexpf(mx, &E);  // mx = f * 2^E, f in [0.5, 1)
        e = min((norm ? 14 : 15) - E, 126);
    }
    if (tid == 0) P.rexp[m] = e;
    if (P.norm_out && g < ng) {
        float *dst = P.norm_out + (size_t)m * P.ldn + 8 * g;
#pragma unroll
        for (int i = 0; i < 8; i++) dst[i] = v[i];
    }
    // 3. the binary16 hi + lo split
    if (M16 && ng + tid < (ng + 3) / 4 * 4) {  // the last 32-row step's rows past K
        *reinterpret_cast<half8 *>(P.xh + slot(ng + tid)) = (half8){};
        *reinterpret_cast<half8 *>(P.xl + slot(ng + tid)) = (half8){};
    }
    if (g >= ng) return;
    half8 h, l;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const float s = ldexpf(v[i], e);
        h[i] = (_Float16)s;
        l[i] = (_Float16)(s - (float)h[i]);
    }
    *reinterpret_cast<half8 *>(P.xh + slot(g)) = h;
    *reinterpret_cast<half8 *>(P.xl + slot(g)) = l;
}

// One 32-column panel x one K chunk per block: 8 waves of `steps` 16-row
// steps, MT M-tiles of 32 rows sharing each step's B operand.  A wave's
// operands are loaded R steps ahead into a ring whose registers are loaded
// again as soon as their MFMAs are issued (a step past the end re-reads the
// last one and contributes zero: its nibbles are masked to q = 0); four waves
// a SIMD hide the rest.  The waves are summed through LDS in a fixed tree;
// with several chunks, each block stores its tile to `part` and the last
// block of a panel to arrive (a counter per panel) adds the chunks in chunk
// order -- deterministic -- and finishes: * 2^-rexp[m], + bias, store or
// accumulate.
// Row split and product, 64 rows, against blocks of 4 waves with all of a
// wave's 8 steps loaded at once (two waves a SIMD): 2048 -> 12288 27.4 ->
// 26.0 us, 6144 -> 2048 20.9 -> 18.3, 1024 -> 6144 12.8 -> 9.6 (no chunks to
// add).  Bound at 64 rows by the rows' operands from the L2, 512 KiB for
// every panel; two or four panels to a block measured slower (28.6-34.9).
template <int MT, bool FULL>
__global__ __launch_bounds__(64 * kMfmaWaves) void k_gemm_mfma(GemmMfmaParams P, int steps) {
    constexpr int NW = kMfmaWaves;
    __shared__ float red[NW][MT * 1024];
    __shared__ int s_last;
    const int p = blockIdx.x, ch = blockIdx.y, kc = gridDim.y;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: the operand addresses are scalar + lane
    const int K = P.w.K, N = P.w.N, Ks = K / 16, Mpad = 32 * MT;
    const int s0 = (ch * NW + wave) * steps, s1 = min(Ks, s0 + steps);
    const int half = lane >> 5, col = lane & 31;
    constexpr int R = MT == 1 ? 4 : 2;  // ring
    uint32_t wq[R];
    u32x4v sav[R], sbv[R];
    half8 xh[R][MT], xl[R][MT];
    auto load = [&](int i, int sw) {
        const int s = min(sw, Ks - 1);
        wq[i] = (P.w.wm + ((size_t)p * Ks + s) * 64)[lane];
        sav[i] = reinterpret_cast<const u32x4v *>(P.w.sa + (size_t)p * K + 16 * s)[half];
        sbv[i] = reinterpret_cast<const u32x4v *>(P.w.sb + (size_t)p * K + 16 * s)[half];
#pragma unroll
        for (int t = 0; t < MT; t++) {
            const size_t off = ((size_t)t * Ks + s) * 64 * 8;
            xh[i][t] = reinterpret_cast<const half8 *>(P.xh + off)[lane];
            xl[i][t] = reinterpret_cast<const half8 *>(P.xl + off)[lane];
        }
    };
#pragma unroll
    for (int i = 0; i < R; i++) load(i, s0 + i);
    __builtin_amdgcn_sched_barrier(0);
    f32x16 acc[MT];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[t][r] = 0.0f;
    for (int s = s0; s < s1; s += R) {
#pragma unroll
        for (int i = 0; i < R; i++) {
            const uint32_t w = s + i < s1 ? wq[i] : 0x88888888u;  // past the end: nibbles of 8, q = 0
            half8 ba, bb;
            const uint32_t sap[4] = {sav[i].x, sav[i].y, sav[i].z, sav[i].w};
            const uint32_t sbp[4] = {sbv[i].x, sbv[i].y, sbv[i].z, sbv[i].w};
#pragma unroll
            for (int j = 0; j < 4; j++) {
                typedef _Float16 half2v __attribute__((ext_vector_type(2)));
                const uint32_t bits = ((w >> (4 * j)) & 0x000F000Fu) | 0x64006400u;
                const half2v q = __builtin_bit_cast(half2v, bits) - (half2v){(_Float16)1032.0f, (_Float16)1032.0f};
                const half2v a = q * __builtin_bit_cast(half2v, sap[j]);
                const half2v b = q * __builtin_bit_cast(half2v, sbp[j]);
                ba[2 * j] = a.x;
                ba[2 * j + 1] = a.y;
                bb[2 * j] = b.x;
                bb[2 * j + 1] = b.y;
            }
#pragma unroll
            for (int t = 0; t < MT; t++) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xh[i][t], ba, acc[t], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < MT; t++) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xh[i][t], bb, acc[t], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < MT; t++) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xl[i][t], ba, acc[t], 0, 0, 0);
            if constexpr (FULL) {
#pragma unroll
                for (int t = 0; t < MT; t++)
                    acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xl[i][t], bb, acc[t], 0, 0, 0);
            }
            load(i, s + R + i);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // the waves through LDS.  D layout: lane l, register r -> row
    // (r/4)*8 + (l/32)*4 + r%4, column l%32
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++)
            red[wave][t * 1024 + ((r >> 2) * 8 + half * 4 + (r & 3)) * 32 + col] = acc[t][r];
    __syncthreads();
    constexpr int U = MT * 16 / NW;  // outputs i = tid + 64 NW u: row i / 32, column i % 32
    const int M = P.M, n = 32 * p + (tid & 31);
    float v[U];
    int mrow[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int i = tid + 64 * NW * u;
        mrow[u] = i >> 5;
        float t[NW];
#pragma unroll
        for (int w = 0; w < NW; w++) t[w] = red[w][i];
#pragma unroll
        for (int j = 1; j < NW; j *= 2)
#pragma unroll
            for (int w = 0; w < NW; w += 2 * j) t[w] += t[w + j];
        v[u] = t[0];
    }
    if (kc > 1) {
#pragma unroll
        for (int u = 0; u < U; u++)
            if (mrow[u] < M) st_dev(P.part + ((size_t)ch * Mpad + mrow[u]) * N + n, v[u]);
        wait_stores();
        __syncthreads();
        if (tid == 0) s_last = arrive_dev(&P.counters[p]) == (unsigned)(kc - 1);
        __syncthreads();
        if (!s_last) return;
        if (tid == 0) reset_dev(&P.counters[p]);
#pragma unroll
        for (int u = 0; u < U; u++) v[u] = 0.0f;
        for (int c0 = 0; c0 < kc; c0 += 4) {
            float t[4][U];
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int u = 0; u < U; u++)
                    t[j][u] = ld_dev(P.part + ((size_t)min(c0 + j, kc - 1) * Mpad + min(mrow[u], M - 1)) * N + n);
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int u = 0; u < U; u++)
                    if (c0 + j < kc) v[u] += t[j][u];
        }
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
        if (mrow[u] >= M) continue;
        float r = ldexpf(v[u], -P.rexp[mrow[u]]);
        if (P.bias) r += P.bias[n];
        float *dst = P.y + (size_t)mrow[u] * P.ldy + n;
        *dst = P.accumulate ? *dst + r : r;
    }
}

// The same for up to 16 rows: 16x16x32 MFMAs, so that no operand register or
// L2 read goes to rows that are not there.  A block of 4 waves owns one panel
// and 4 * SW 32-row steps; a wave holds twice the K of k_gemm_mfma's in as
// many registers, which halves the chunks (and their partials) and puts the
// whole weight in flight in one round of blocks.  Lane l: k rows 8 (l / 16)
// .. + 7 of a step, A row and B column l % 16; the panel's two 16-column
// tiles share the A operand and the scales.
// Row split and product, 16 rows, weights from memory: 2048 -> 12288 17.9 ->
// 13.2 us, 6144 -> 2048 15.9 -> 11.6, 1024 -> 6144 9.4 -> 6.8, 2048 -> 4096
// 9.7 -> 8.7.  Bound by launch, load and merge latency (the weights alone
// take 3 us of the first).
template <int SW, bool FULL>
__global__ __launch_bounds__(256) void k_gemm_mfma16(GemmMfmaParams P) {
    __shared__ float red[4][512];
    __shared__ int s_last;
    const int p = blockIdx.x, ch = blockIdx.y, kc = gridDim.y;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: the operand addresses are scalar + lane
    const int K = P.w.K, N = P.w.N, Ks = K / 16, K32 = (K + 31) / 32;
    const int s0 = (ch * 4 + wave) * SW;
    const int kg = lane >> 4, col = lane & 15;
    // K = 16 (mod 32): the last step's upper half re-reads its lower half, q = 0 (and x = 0)
    uint32_t wq[SW][2];
    u32x4v sav[SW], sbv[SW];
    half8 xh[SW], xl[SW];
#pragma unroll
    for (int i = 0; i < SW; i++) {
        const int s = min(s0 + i, K32 - 1);
        const int up = 2 * s + (kg >> 1) < Ks ? kg >> 1 : 0;  // 16-row step within the 32
        const uint32_t *wm = P.w.wm + ((size_t)p * Ks + 2 * s) * 64;
        wq[i][0] = wm[64 * up + 32 * (kg & 1) + col];
        wq[i][1] = wm[64 * up + 32 * (kg & 1) + col + 16];
        const size_t so = (size_t)p * K + 32 * s;
        sav[i] = reinterpret_cast<const u32x4v *>(P.w.sa + so)[2 * up + (kg & 1)];
        sbv[i] = reinterpret_cast<const u32x4v *>(P.w.sb + so)[2 * up + (kg & 1)];
        xh[i] = reinterpret_cast<const half8 *>(P.xh + (size_t)s * 512)[lane];
        xl[i] = reinterpret_cast<const half8 *>(P.xl + (size_t)s * 512)[lane];
    }
    __builtin_amdgcn_sched_barrier(0);  // keep every load ahead of the first wait
    f32x4 acc[2];
#pragma unroll
    for (int t = 0; t < 2; t++) acc[t] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < SW; i++) {
        const bool in = s0 + i < K32 && 2 * (s0 + i) + (kg >> 1) < Ks;
        const uint32_t sap[4] = {sav[i].x, sav[i].y, sav[i].z, sav[i].w};
        const uint32_t sbp[4] = {sbv[i].x, sbv[i].y, sbv[i].z, sbv[i].w};
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const uint32_t w = in ? wq[i][t] : 0x88888888u;
            half8 ba, bb;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                typedef _Float16 half2v __attribute__((ext_vector_type(2)));
                const uint32_t bits = ((w >> (4 * j)) & 0x000F000Fu) | 0x64006400u;
                const half2v q = __builtin_bit_cast(half2v, bits) - (half2v){(_Float16)1032.0f, (_Float16)1032.0f};
                const half2v a = q * __builtin_bit_cast(half2v, sap[j]);
                const half2v b = q * __builtin_bit_cast(half2v, sbp[j]);
                ba[2 * j] = a.x;
                ba[2 * j + 1] = a.y;
                bb[2 * j] = b.x;
                bb[2 * j + 1] = b.y;
            }
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[i], ba, acc[t], 0, 0, 0);
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[i], bb, acc[t], 0, 0, 0);
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl[i], ba, acc[t], 0, 0, 0);
            if constexpr (FULL) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl[i], bb, acc[t], 0, 0, 0);
        }
    }
    // D layout: lane l, register r -> row 4 (l / 16) + r, column l % 16
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) red[wave][(4 * kg + r) * 32 + 16 * t + col] = acc[t][r];
    __syncthreads();
    const int M = P.M;
    float v[2];
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int i = tid + 256 * u;
        v[u] = (red[0][i] + red[1][i]) + (red[2][i] + red[3][i]);
    }
    if (kc > 1) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int i = tid + 256 * u;
            if ((i >> 5) < M) st_dev(P.part + ((size_t)ch * 16 + (i >> 5)) * N + 32 * p + (i & 31), v[u]);
        }
        wait_stores();
        __syncthreads();
        if (tid == 0) s_last = arrive_dev(&P.counters[p]) == (unsigned)(kc - 1);
        __syncthreads();
        if (!s_last) return;
        if (tid == 0) reset_dev(&P.counters[p]);
        v[0] = v[1] = 0.0f;
        for (int c0 = 0; c0 < kc; c0 += 8) {
            float t[8][2];
#pragma unroll
            for (int j = 0; j < 8; j++)
#pragma unroll
                for (int u = 0; u < 2; u++)
                    t[j][u] = ld_dev(P.part + ((size_t)min(c0 + j, kc - 1) * 16 + min((tid + 256 * u) >> 5, M - 1)) * N +
                                     32 * p + (tid & 31));
#pragma unroll
            for (int j = 0; j < 8; j++)
#pragma unroll
                for (int u = 0; u < 2; u++)
                    if (c0 + j < kc) v[u] += t[j][u];
        }
    }
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int i = tid + 256 * u, m = i >> 5, n = 32 * p + (i & 31);
        if (m >= M) continue;
        float r = ldexpf(v[u], -P.rexp[m]);
        if (P.bias) r += P.bias[n];
        float *dst = P.y + (size_t)m * P.ldy + n;
        *dst = P.accumulate ? *dst + r : r;
    }
}

// The same product for many rows.  A block of NW waves owns 32 * MT rows x NW
// panels: wave w takes panel NW * n + w and all MT row tiles, so the nibbles
// become B operands once per wave and are used by 3 * MT MFMAs, and the
// block's A operands go through LDS once for its NW panels (two 16-row steps
// per stage, double buffered).  Loads run two stages ahead, and everything
// that is not an MFMA is issued between MFMAs.  Bound by the rows' operands
// from the L2: 1064 rows, 2048 -> 12288, take 159 us with the row split, 337
// TFLOP/s (1010 of binary16 MFMAs issued; a library binary16 product with as
// many MFMAs takes 149), where 17 passes of k_gemm_mfma took 410; 1000 rows,
// 6144 -> 2048, 342 -> 89 us (the library 189).
template <int MT, int NW, bool FULL>
__global__ __launch_bounds__(64 * NW, 2) void k_gemm_mfma_tile(GemmMfmaParams P, GemmTilePlan T) {
    constexpr int SS = 2;  // 16-row steps per stage
    constexpr int U = SS * MT * 2;  // 1 KiB operand units per stage
    constexpr int UW = U / NW;
    __shared__ __align__(16) half8 abuf[2][U][64];
    __shared__ int s_last;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5, col = lane & 31;
    // Blocks of one XCD (every 8th) take a contiguous run of (column block,
    // chunk, row block), row blocks innermost: the XCD's L2 then holds its
    // weights while the rows stream past them.
    const int total = T.mb * T.nb * T.kc, per = (int)(gridDim.x >> 3);
    const int L = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if (L >= total) return;
    const int nc = __builtin_amdgcn_readfirstlane(L / T.mb), m_blk = L - nc * T.mb;
    const int n_blk = __builtin_amdgcn_readfirstlane(nc / T.kc), ch = nc - n_blk * T.kc;
    const int K = P.w.K, N = P.w.N, Ks = K / 16, panels = N / 32;
    const int pw = NW * n_blk + wave, p = min(pw, panels - 1);
    const int sb = ch * T.cs, se = min(Ks, sb + T.cs);
    const int nst = (se - sb + SS - 1) / SS;

    const uint32_t *wm = P.w.wm + (size_t)p * Ks * 64 + lane;
    const uint16_t *sa = P.w.sa + (size_t)p * K + 8 * half, *sc = P.w.sb + (size_t)p * K + 8 * half;
    // this wave's units of a stage's A operands: u = wave * MT + j ->
    // (step u / (2 MT), tile, hi / lo)
    const half8 *asrc[UW];
    int astep[UW];
#pragma unroll
    for (int j = 0; j < UW; j++) {
        const int u = wave * UW + j, rem = u % (2 * MT);
        astep[j] = u / (2 * MT);
        asrc[j] = reinterpret_cast<const half8 *>((rem & 1) ? P.xl : P.xh) +
                  (size_t)(m_blk * MT + (rem >> 1)) * Ks * 64 + lane;
    }
    half8 ra[2][UW];
    uint32_t wq[2][SS];
    u32x4v va[2][SS], vb[2][SS];
    auto load = [&](int st, int b) {
#pragma unroll
        for (int i = 0; i < SS; i++) {
            const int s = min(sb + SS * st + i, Ks - 1);
            wq[b][i] = wm[(size_t)s * 64];
            va[b][i] = *reinterpret_cast<const u32x4v *>(sa + 16 * s);
            vb[b][i] = *reinterpret_cast<const u32x4v *>(sc + 16 * s);
        }
#pragma unroll
        for (int j = 0; j < UW; j++) ra[b][j] = asrc[j][(size_t)min(sb + SS * st + astep[j], Ks - 1) * 64];
    };
    auto put = [&](int b) {
#pragma unroll
        for (int j = 0; j < UW; j++) abuf[b][wave * UW + j][lane] = ra[b][j];
    };
    f32x16 acc[MT];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[t][r] = 0.0f;

    // The B operands of one step: q as binary16 1024 + nib (magic exponent)
    // minus 1032, times sa and sb.  A step past the end has nibbles of 8, q = 0.
    half8 ba[SS], bb[SS];
    auto form = [&](int st, int b, int i) {
        const uint32_t w = sb + SS * st + i < se ? wq[b][i] : 0x88888888u;  // uniform
        const uint32_t sap[4] = {va[b][i].x, va[b][i].y, va[b][i].z, va[b][i].w};
        const uint32_t sbp[4] = {vb[b][i].x, vb[b][i].y, vb[b][i].z, vb[b][i].w};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            typedef _Float16 half2v __attribute__((ext_vector_type(2)));
            const uint32_t bits = ((w >> (4 * j)) & 0x000F000Fu) | 0x64006400u;
            const half2v q = __builtin_bit_cast(half2v, bits) - (half2v){(_Float16)1032.0f, (_Float16)1032.0f};
            const half2v a = q * __builtin_bit_cast(half2v, sap[j]);
            const half2v c = q * __builtin_bit_cast(half2v, sbp[j]);
            ba[i][2 * j] = a.x;
            ba[i][2 * j + 1] = a.y;
            bb[i][2 * j] = c.x;
            bb[i][2 * j + 1] = c.y;
        }
    };
    // Tiles two at a time: the operands of the next two come from LDS under
    // the MFMAs of these two.
    constexpr int NG = (MT + 1) / 2;
    half8 xh[2][2], xl[2][2];
    auto get = [&](int b, int g) {  // group g = step g / NG, tiles 2 (g % NG) and the next
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int t = 2 * (g % NG) + u;
            if (t < MT) {
                xh[g & 1][u] = abuf[b][((g / NG) * MT + t) * 2][lane];
                xl[g & 1][u] = abuf[b][((g / NG) * MT + t) * 2 + 1][lane];
            }
        }
    };
    auto mma = [&](int g) {
        const int i = g / NG, t0 = 2 * (g % NG), n = t0 + 1 < MT ? 2 : 1;
#pragma unroll
        for (int u = 0; u < n; u++)
            acc[t0 + u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xh[g & 1][u], ba[i], acc[t0 + u], 0, 0, 0);
#pragma unroll
        for (int u = 0; u < n; u++)
            acc[t0 + u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xh[g & 1][u], bb[i], acc[t0 + u], 0, 0, 0);
#pragma unroll
        for (int u = 0; u < n; u++)
            acc[t0 + u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xl[g & 1][u], ba[i], acc[t0 + u], 0, 0, 0);
        if constexpr (FULL) {
#pragma unroll
            for (int u = 0; u < n; u++)
                acc[t0 + u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xl[g & 1][u], bb[i], acc[t0 + u], 0, 0, 0);
        }
    };
    // Stage st from buffer b = st % 2, its first step's B operands formed: the
    // second step's under the first step's MFMAs, the next stage's LDS writes
    // and first B operands and the loads of stage st + 2 under the second's.
    auto stage = [&](int st, int b) {
        get(b, 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int g = 0; g < SS * NG; g++) {
            if (g + 1 < SS * NG) get(b, g + 1);
            if (g == 0) form(st, b, 1);
            if (g == NG) {
                put(b ^ 1);  // stage st + 1
                form(min(st + 1, nst - 1), b ^ 1, 0);
            }
            if (g == SS * NG - 1) load(min(st + 2, nst - 1), b);
            mma(g);
#pragma unroll
            for (int u = 0; u < (FULL ? 8 : 6); u++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x020, 2, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
    };
    // Every 16 steps (8 with FULL) the accumulators move to a second level, so that a sum
    // over K = 2048 rounds as often as one over 16 steps and one over 8 such
    // sums: with one chain of 384 MFMAs its rounding (4.1e-7 of an
    // all-positive sum) was five times k_gemm_mfma's.
    f32x16 top[MT];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) top[t][r] = 0.0f;

    load(0, 0);
    put(0);
    load(min(1, nst - 1), 1);
    form(0, 0, 0);
    __syncthreads();
    for (int st = 0; st < nst; st += 2) {
        stage(st, 0);
        if (st + 1 < nst) stage(st + 1, 1);  // uniform
        if ((st & (FULL ? 2 : 6)) == (FULL ? 2 : 6) || st + 2 >= nst) {
#pragma unroll
            for (int t = 0; t < MT; t++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    top[t][r] += acc[t][r];
                    acc[t][r] = 0.0f;
                }
        }
    }
#pragma unroll
    for (int t = 0; t < MT; t++) acc[t] = top[t];

    const int m0 = m_blk * MT * 32, n = 32 * p + col;
    const int tile = n_blk * T.mb + m_blk;
    if (T.kc > 1) {
        // partials in accumulator order: [chunk][wave][tile][register][lane]
        float *mine = P.part + ((size_t)tile * T.kc + ch) * (size_t)(NW * MT * 1024) + wave * (MT * 1024) + lane;
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int r = 0; r < 16; r++) st_dev(mine + (t * 16 + r) * 64, acc[t][r]);
        wait_stores();
        __syncthreads();
        if (tid == 0) s_last = arrive_dev(&P.counters[tile]) == (unsigned)(T.kc - 1);
        __syncthreads();
        if (!s_last) return;
        if (tid == 0) reset_dev(&P.counters[tile]);
        // the last chunk to arrive adds all of them in chunk order
        const float *all = P.part + (size_t)tile * T.kc * (size_t)(NW * MT * 1024) + wave * (MT * 1024) + lane;
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[t][r] = 0.0f;
        for (int c = 0; c < T.kc; c++) {
            const float *pc = all + (size_t)c * (NW * MT * 1024);
            float v[MT][16];
#pragma unroll
            for (int t = 0; t < MT; t++)
#pragma unroll
                for (int r = 0; r < 16; r++) v[t][r] = ld_dev(pc + (t * 16 + r) * 64);
#pragma unroll
            for (int t = 0; t < MT; t++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[t][r] += v[t][r];
        }
    }
    if (pw >= panels) return;
    const float bias = P.bias ? P.bias[n] : 0.0f;
#pragma unroll
    for (int t = 0; t < MT; t++) {
        float old[16];
        int e[16];
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int m = m0 + 32 * t + (r >> 2) * 8 + half * 4 + (r & 3);
            e[r] = P.rexp[m];
            old[r] = P.accumulate ? P.y[(size_t)min(m, P.M - 1) * P.ldy + n] : 0.0f;
        }
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int m = m0 + 32 * t + (r >> 2) * 8 + half * 4 + (r & 3);
            if (m >= P.M) continue;
            float v = ldexpf(acc[t][r], -e[r]);
            if (P.bias) v += bias;
            P.y[(size_t)m * P.ldy + n] = P.accumulate ? old[r] + v : v;
        }
    }
}

// Causal attention of a whole prefill (src/talker.rs:404-441): row i of M
// sees cache rows 0..i.  A block takes one query head and 32 rows; its 4
// waves take every 4th run of 32 keys, and their softmax partials are merged
// in wave order.  The products are f32 MFMAs (32x32x2), so nothing is
// rounded below f32.
//   scores: S^T = K Q^T, lane l holding query l % 32 and the keys
//     key(r) = 8 (r / 4) + 4 (l / 32) + r % 4 in its 16 registers, so the
//     softmax of a query is a reduction over registers and one lane exchange;
//   values: O^T += V^T P^T with the registers of P as they are (MFMA r takes
//     key(r) of both lane halves), the MFMA row m of the t-th product being
//     dim 4 m + t, so a lane reads V and stores O four dims at a time.
// K and V are read from the cache straight into operand registers: an f32
// MFMA takes 64 cycles, 32 keys 8192, and their 32 KiB come from the L2
// meanwhile.  Longest rows first; the query heads of one kv head (and so its
// K and V) fall on one XCD where there are 8 kv heads.
// 1064 rows, 16 heads: 73 us per layer (the f32 MFMAs alone 37), where k_attn
// (one row per block) took 620; 300 rows 19.9, 96 rows 10.1.
__global__ __launch_bounds__(256, 2) void k_attn_prefill(AttnParams P, int M) {
    constexpr int HD = 128;
    __shared__ float part[4][16][4][64];  // [wave][register][t][lane]
    __shared__ float ml[4][2][32];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int half = lane >> 5, col = lane & 31;
    const int G = P.nq / P.nkv, tiles = (M + 31) / 32;
    const int hx = blockIdx.x % P.nq, qt = tiles - 1 - blockIdx.x / P.nq;
    const int kvh = hx % P.nkv, head = kvh * G + hx / P.nkv;
    const int q = 32 * qt + col;
    const float *K = P.kcache + (size_t)kvh * P.kv_cap * HD, *V = P.vcache + (size_t)kvh * P.kv_cap * HD;
    const float *qr = P.q + (size_t)min(q, M - 1) * P.ldq + (size_t)head * HD + 4 * half;

    f32x4 qv[16];  // dims 8 g + 4 half + j
#pragma unroll
    for (int g = 0; g < 16; g++) qv[g] = *reinterpret_cast<const f32x4 *>(qr + 8 * g);
    f32x16 acc[4];
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[t][r] = 0.0f;
    float mx = -INFINITY, sum = 0.0f;
    // K and V in batches of 4 registers' worth, one batch ahead of the MFMAs
    f32x4 kb[2][4], vb[2][4];
    auto load_k = [&](int kt, int c, int to) {
        const float *kr = K + (size_t)min(32 * kt + col, M - 1) * HD + 4 * half + 32 * c;
#pragma unroll
        for (int g = 0; g < 4; g++) kb[to][g] = *reinterpret_cast<const f32x4 *>(kr + 8 * g);
    };
    auto load_v = [&](int kt, int c, int to) {  // keys 32 kt + 8 c + 4 half + r
#pragma unroll
        for (int r = 0; r < 4; r++)
            vb[to][r] = *reinterpret_cast<const f32x4 *>(
                V + (size_t)min(32 * kt + 8 * c + 4 * half + r, M - 1) * HD + 4 * col);
    };
    // In the last run (the rows' own keys) an infinite or NaN V meets the
    // queries that do not see its key with weight 0, which makes them NaN too.
    // z, the largest |V| of that run or NaN, finds such a V.
    float z = 0.0f;
    load_k(min(wave, qt), 0, 0);
    for (int kt = wave; kt <= qt; kt += 4) {
        const bool diag = kt == qt;
        f32x16 s;
#pragma unroll
        for (int r = 0; r < 16; r++) s[r] = 0.0f;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            if (c < 3)
                load_k(kt, c + 1, (c + 1) & 1);
            else
                load_v(kt, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int g = 0; g < 4; g++)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    s = __builtin_amdgcn_mfma_f32_32x32x2f32(kb[c & 1][g][j], qv[4 * c + g][j], s, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        float m = mx;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int key = 32 * kt + 8 * (r >> 2) + 4 * half + (r & 3);
            s[r] = diag && key > q ? -INFINITY : s[r] * P.scale;
            m = fmaxf(m, s[r]);
        }
        m = halves_max(m);
        const float alpha = expf(mx - m);
        float l = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            s[r] = expf(s[r] - m);
            l += s[r];
        }
        sum = sum * alpha + halves_sum(l);
        mx = m;
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[t][r] *= alpha;
        z = diag ? 0.0f : z;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            if (c < 3)
                load_v(kt, c + 1, (c + 1) & 1);
            else
                load_k(min(kt + 4, qt), 0, 0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int t = 0; t < 4; t++)
                    acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(vb[c & 1][r][t], s[4 * c + r], acc[t], 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int t = 0; t < 4; t++) z = __builtin_elementwise_maximum(z, fabsf(vb[c & 1][r][t]));
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    if (wave == (qt & 3) && __any(!(z < INFINITY))) {  // uniform
        // the wave's keys again, one at a time for all 32 queries without the
        // matrix cores, a lane skipping those it does not see: for 1500 rows
        // 90 to 190 us more in a layer, however many rows are NaN (row by row
        // over all keys, for every tile after the bad row, it was 4 ms)
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[t][r] = 0.0f;
        for (int kt = wave; kt <= qt; kt += 4)
#pragma unroll 1
            for (int key = 32 * kt; key < min(32 * kt + 32, M); key++) {
                const float *kr = K + (size_t)key * HD + 4 * half, *vr = V + (size_t)key * HD + 16 * half;
                float d = 0.0f;
#pragma unroll
                for (int g = 0; g < 16; g++) {
                    const f32x4 k = *reinterpret_cast<const f32x4 *>(kr + 8 * g);
#pragma unroll
                    for (int j = 0; j < 4; j++) d = fmaf(k[j], qv[g][j], d);
                }
                d = halves_sum(d);
                if (key > q) continue;
                const float p = expf(d * P.scale - mx);
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const f32x4 v = *reinterpret_cast<const f32x4 *>(vr + 4 * (8 * (r >> 2) + (r & 3)));
#pragma unroll
                    for (int t = 0; t < 4; t++) acc[t][r] = fmaf(p, v[t], acc[t][r]);
                }
            }
    }
    // merge: weights exp(max of the wave - max of all), sums in wave order
    if (half == 0) {
        ml[wave][0][col] = mx;
        ml[wave][1][col] = sum;
    }
    __syncthreads();
    float m = ml[0][0][col];
#pragma unroll
    for (int w = 1; w < 4; w++) m = fmaxf(m, ml[w][0][col]);
    float l = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; w++)
        if (w <= qt) l += ml[w][1][col] * expf(ml[w][0][col] - m);
    const float f = wave <= qt ? expf(mx - m) : 0.0f;
#pragma unroll
    for (int r = 0; r < 16; r++)
#pragma unroll
        for (int t = 0; t < 4; t++) part[wave][r][t][lane] = acc[t][r] * f;
    __syncthreads();
    float *o = P.out + (size_t)q * P.ldo + (size_t)head * HD;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int r = 4 * wave + i;
        f32x4 v;
#pragma unroll
        for (int t = 0; t < 4; t++)
            v[t] = ((part[0][r][t][lane] + part[1][r][t][lane]) + (part[2][r][t][lane] + part[3][r][t][lane])) / l;
        if (q < M) *reinterpret_cast<f32x4 *>(o + 4 * (8 * (r >> 2) + 4 * half + (r & 3))) = v;
    }
}

}  // namespace

void launch_repack_mfma(hipStream_t st, const DevQ4 &w, uint32_t *wm, uint16_t *sa, uint16_t *sb, int *too_large) {
    const size_t total = (size_t)(w.N / 32) * (w.K / 16) * 64;
    const size_t nrows = (size_t)(w.N / 32) * w.K;
    const size_t n = total > nrows ? total : nrows;
    hipLaunchKernelGGL(k_repack_mfma, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, w, wm, sa, sb, too_large);
}

template <bool M16>
static void launch_mfma_rows_order(hipStream_t st, const MfmaRowsParams &p) {
    const dim3 grid((unsigned)p.Mpad);
    if (p.K <= 2048)
        hipLaunchKernelGGL((k_mfma_rows<256, M16>), grid, dim3(256), 0, st, p);
    else if (p.K <= 4096)
        hipLaunchKernelGGL((k_mfma_rows<512, M16>), grid, dim3(512), 0, st, p);
    else
        hipLaunchKernelGGL((k_mfma_rows<1024, M16>), grid, dim3(1024), 0, st, p);
}

void launch_mfma_rows(hipStream_t st, const MfmaRowsParams &p) {
    p.m16 ? launch_mfma_rows_order<true>(st, p) : launch_mfma_rows_order<false>(st, p);
}

template <bool FULL>
static void launch_gemm_mfma16_full(hipStream_t st, const GemmMfmaParams &p, int sw, int kc) {
    const dim3 grid((unsigned)(p.w.N / 32), (unsigned)kc);
    switch (sw) {
        case 8: hipLaunchKernelGGL((k_gemm_mfma16<8, FULL>), grid, dim3(256), 0, st, p); break;
        case 4: hipLaunchKernelGGL((k_gemm_mfma16<4, FULL>), grid, dim3(256), 0, st, p); break;
        case 2: hipLaunchKernelGGL((k_gemm_mfma16<2, FULL>), grid, dim3(256), 0, st, p); break;
        default: hipLaunchKernelGGL((k_gemm_mfma16<1, FULL>), grid, dim3(256), 0, st, p); break;
    }
}

void launch_gemm_mfma16(hipStream_t st, const GemmMfmaParams &p, int sw, int kc) {
    p.full ? launch_gemm_mfma16_full<true>(st, p, sw, kc) : launch_gemm_mfma16_full<false>(st, p, sw, kc);
}

void launch_gemm_mfma(hipStream_t st, const GemmMfmaParams &p, int mt, int steps, int kc) {
    const dim3 grid((unsigned)(p.w.N / 32), (unsigned)kc), block(64 * kMfmaWaves);
    if (mt == 1) {
        if (p.full)
            hipLaunchKernelGGL((k_gemm_mfma<1, true>), grid, block, 0, st, p, steps);
        else
            hipLaunchKernelGGL((k_gemm_mfma<1, false>), grid, block, 0, st, p, steps);
    } else {
        if (p.full)
            hipLaunchKernelGGL((k_gemm_mfma<2, true>), grid, block, 0, st, p, steps);
        else
            hipLaunchKernelGGL((k_gemm_mfma<2, false>), grid, block, 0, st, p, steps);
    }
}

template <bool FULL>
static void launch_gemm_mfma_tile_full(hipStream_t st, const GemmMfmaParams &p, const GemmTilePlan &t) {
    const int total = t.mb * t.nb * t.kc;
    const dim3 grid((unsigned)((total + 7) / 8 * 8)), block(64 * t.nw);
    if (t.nw == 8) {
        hipLaunchKernelGGL((k_gemm_mfma_tile<4, 8, FULL>), grid, block, 0, st, p, t);
        return;
    }
    switch (t.mt) {
        case 4: hipLaunchKernelGGL((k_gemm_mfma_tile<4, 4, FULL>), grid, block, 0, st, p, t); break;
        case 3: hipLaunchKernelGGL((k_gemm_mfma_tile<3, 4, FULL>), grid, block, 0, st, p, t); break;
        case 2: hipLaunchKernelGGL((k_gemm_mfma_tile<2, 4, FULL>), grid, block, 0, st, p, t); break;
        default: hipLaunchKernelGGL((k_gemm_mfma_tile<1, 4, FULL>), grid, block, 0, st, p, t); break;
    }
}

void launch_gemm_mfma_tile(hipStream_t st, const GemmMfmaParams &p, const GemmTilePlan &t) {
    p.full ? launch_gemm_mfma_tile_full<true>(st, p, t) : launch_gemm_mfma_tile_full<false>(st, p, t);
}

void launch_attn_prefill(hipStream_t st, const AttnParams &p, int M) {
    hipLaunchKernelGGL(k_attn_prefill, dim3((unsigned)(p.nq * ((M + 31) / 32))), dim3(256), 0, st, p, M);
}

}  // namespace qtts
