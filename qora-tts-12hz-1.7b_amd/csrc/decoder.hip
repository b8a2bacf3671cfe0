// decoder.hip — the speech decoder's kernels (decode_to_audio,
// src/decoder.rs:394-509), all f32 like the reference.
//
//  k_dec_gather   codebook rows of every frame: group 0's, and the sum of
//                 the other groups' in group order (src/decoder.rs:142-189)
//  k_dec_rmsnorm  rms_norm_f32 per frame (src/decoder.rs:515-525)
//  k_dec_rope     apply_rope_split_half of q and k (src/decoder.rs:556-578)
//  k_dec_attn     causal sliding-window attention, one wave per (frame, head)
//  k_dec_swiglu   silu(gate) * up
//  k_dec_dwconv   causal depthwise convolution (src/conv.rs:280-345)
//  k_dec_lnorm    channel-first LayerNorm per time step, channels summed in
//                 order (src/decoder.rs:580-602); k_dec_lnorm_tile over an
//                 LDS tile of 16 or 8 time steps, several threads a step
//  k_dec_snake    SnakeBeta (src/conv.rs:347-400), optionally recording
//                 max |out| for the convolution that reads it
//  k_dec_conv_mfma  every projection and convolution on the matrix cores
//                 (v_mfma_f32_32x32x16_f16 with binary16 hi + lo operands):
//                 causal convolutions as implicit GEMMs, a transposed
//                 convolution's phases as rows, linear layers as one tap;
//                 fused epilogues; k_dec_conv_win for convolutions of 3+
//                 taps (the input window split once into LDS; the variant
//                 k_dec_conv_win_tw, one channel tile per wave, at 3 and 4
//                 tiles, for 2+ taps),
//                 k_dec_conv_mfma_ks for launches too small to fill the GPU
//  k_dec_resunit  a residual unit of 96, 192 or 384 channels (both SnakeBetas,
//                 both convolutions, the residual) in one launch
//  k_dec_absmax   max |x| of a layer input (the operand scale)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <cstdint>

#include "device_common.h"
#include "internal.h"

namespace qtts {

namespace {

constexpr unsigned kSnakeBlocks = 8192;  // SnakeBeta grid size target (threads stride through their channel)
// Matrix-core launches of fewer blocks than this at one channel tile split
// K over a block's waves instead (measured: 1,024 ahead of 0 and 4,096).
constexpr size_t kDecFillBlocks = 1024;


__global__ void k_dec_gather(DecGatherParams P) {
    const int t = blockIdx.x, cd = P.cd;
    for (int d = threadIdx.x; d < cd; d += blockDim.x) {
        uint32_t c0 = P.codes[t];
        if (c0 >= (uint32_t)P.cb_size) {
            if (d == 0) atomicOr(P.status, 1);
            c0 = 0;
        }
        P.e0[(size_t)t * cd + d] = P.first[(size_t)c0 * cd + d];
        float s = 0.0f;
        for (int g = 0; g < P.num_rest; g++) {
            uint32_t c = P.codes[(size_t)(g + 1) * P.ld + t];
            if (c >= (uint32_t)P.cb_size) {
                if (d == 0) atomicOr(P.status, 1);
                c = 0;
            }
            s += P.rest[g][(size_t)c * cd + d];
        }
        P.es[(size_t)t * cd + d] = s;
    }
}

// GELU, the tanh form the reference uses.
__device__ __forceinline__ float dec_gelu(float x) { return x * 0.5f * (1.0f + tanhf(x * 0.7071067811865476f)); }

// max over a block of 256 threads into *slot: unsigned order is float order
// for non-negative values.  red: 4 words nothing reads any more.
__device__ __forceinline__ void block_amax(float m, float *red, unsigned *slot) {
    m = wave_max(m);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0)
        atomicMax(slot, __float_as_uint(fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]))));
}

// rms_norm_f32 of each of `rows` rows of n values: one block per row.
// max |out| (NaN excluded) goes into the slots of amax, as k_dec_snake's.
__global__ __launch_bounds__(256) void k_dec_rmsnorm(const float *x, const float *gamma, int n, float eps, float *out,
                                                     unsigned *amax) {
    __shared__ float red[4];
    const float *r = x + (size_t)blockIdx.x * n;
    float ss = 0.0f;
    for (int i = threadIdx.x; i < n; i += 256) ss += r[i] * r[i];
    ss = wave_sum(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    ss = (red[0] + red[1]) + (red[2] + red[3]);
    const float inv = 1.0f / sqrtf(ss / (float)n + eps);
    float m = 0.0f;
    for (int i = threadIdx.x; i < n; i += 256) {
        const float v = r[i] * inv * gamma[i];
        m = fmaxf(m, fabsf(v));
        out[(size_t)blockIdx.x * n + i] = v;
    }
    block_amax(m, red, &amax[blockIdx.x % kDecMaxSlots]);
}

// Split-half rotation of q and k at position = frame; no rotation past the
// table.  One thread per (frame, head, pair).
__global__ void k_dec_rope(float *q, float *k, int T, int heads, int hd, const float *cs, const float *sn, int rows,
                           int ld) {
    const int half = hd / 2;
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (size_t)T * heads * half) return;
    const int i = (int)(idx % half), h = (int)(idx / half % heads), t = (int)(idx / half / heads);
    if (t >= rows) return;
    const float c = cs[(size_t)t * half + i], s = sn[(size_t)t * half + i];
    float *qb = q + (size_t)t * ld + (size_t)h * hd, *kb = k + (size_t)t * ld + (size_t)h * hd;
    float x0 = qb[i], x1 = qb[half + i];
    qb[i] = x0 * c - x1 * s;
    qb[half + i] = x1 * c + x0 * s;
    x0 = kb[i], x1 = kb[half + i];
    kb[i] = x0 * c - x1 * s;
    kb[half + i] = x1 * c + x0 * s;
}

// Causal sliding-window attention (src/decoder.rs:248-275): one wave per
// (frame t, head h); scores over positions max(0, t+1-window) .. t, softmax,
// then out[d] = sum over positions in order of p * v[d] (lane = d).
__global__ __launch_bounds__(256) void k_dec_attn(DecAttnParams P) {
    __shared__ float ps[4][kDecMaxWindow];
    __shared__ float qs[4][kDecMaxHeadDim];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int pair = blockIdx.x * 4 + wave;
    const bool valid = pair < P.T * P.heads;  // wave-uniform; every wave reaches both barriers
    const int t = valid ? pair / P.heads : 0, h = valid ? pair - t * P.heads : 0;
    const int ad = P.heads * P.hd, ld = P.ld > 0 ? P.ld : ad;
    const int start = t + 1 > P.window ? t + 1 - P.window : 0, n = t + 1 - start;
    if (valid)
        for (int d = lane; d < P.hd; d += 64) qs[wave][d] = P.q[(size_t)t * ld + (size_t)h * P.hd + d];
    __syncthreads();
    float inv = 0.0f;
    if (valid) {
        float mx = -INFINITY;
        for (int s = lane; s < n; s += 64) {
            const float *k = P.k + (size_t)(start + s) * ld + (size_t)h * P.hd;
            float dot = 0.0f;
            for (int d = 0; d < P.hd; d++) dot += qs[wave][d] * k[d];
            dot *= P.scale;
            ps[wave][s] = dot;
            mx = fmaxf(mx, dot);
        }
        mx = wave_max(mx);
        float sum = 0.0f;
        for (int s = lane; s < n; s += 64) {
            const float e = expf(ps[wave][s] - mx);
            ps[wave][s] = e;
            sum += e;
        }
        inv = 1.0f / wave_sum(sum);
    }
    __syncthreads();
    float m = 0.0f;
    if (valid)
        for (int d = lane; d < P.hd; d += 64) {
            float o = 0.0f;
            for (int s = 0; s < n; s++) o += (ps[wave][s] * inv) * P.v[(size_t)(start + s) * ld + (size_t)h * P.hd + d];
            P.out[(size_t)t * ad + (size_t)h * P.hd + d] = o;
            m = fmaxf(m, fabsf(o));
        }
    block_amax(m, &qs[0][0], &P.amax[blockIdx.x % kDecMaxSlots]);  // qs was last read before the last barrier
}

// silu(g) * u, max |out| into the slots of amax.
__global__ __launch_bounds__(256) void k_dec_swiglu(const float *g, const float *u, int rows, int width, int ld,
                                                    float *out, unsigned *amax) {
    __shared__ float red[4];
    const size_t n = (size_t)rows * width, stride = (size_t)gridDim.x * blockDim.x;
    float m = 0.0f;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        const size_t t = i / width, j = i - t * width, a = t * ld + j;
        const float v = (g[a] / (1.0f + expf(-g[a]))) * u[a];
        m = fmaxf(m, fabsf(v));
        out[i] = v;
    }
    block_amax(m, red, &amax[blockIdx.x % kDecMaxSlots]);
}

// Causal depthwise convolution (padding kernel_size - 1), channel-first.
__global__ void k_dec_dwconv(const float *x, const float *w, const float *b, int ch, int len, int ks, float *out) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)ch * len) return;
    const int c = (int)(i / len), o = (int)(i - (size_t)c * len);
    float s = b[c];
    for (int k = 0; k < ks; k++) {
        const int p = o + k - (ks - 1);
        if (p >= 0) s += x[(size_t)c * len + p] * w[(size_t)c * ks + k];
    }
    out[i] = s;
}

// LayerNorm across channels at each time step (one thread per step; the
// channel sums run in channel order, 8 channels' loads issued together).
__global__ __launch_bounds__(64) void k_dec_lnorm(const float *x, const float *g, const float *b, int ch, int len,
                                                  float eps, float *out) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= len) return;
    const float *xt = x + t;
    float mean = 0.0f;
    int c = 0;
    for (; c + 8 <= ch; c += 8) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = xt[(size_t)(c + i) * len];
#pragma unroll
        for (int i = 0; i < 8; i++) mean += v[i];
    }
    for (; c < ch; c++) mean += xt[(size_t)c * len];
    mean /= (float)ch;
    float var = 0.0f;
    for (c = 0; c + 8 <= ch; c += 8) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = xt[(size_t)(c + i) * len];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float d = v[i] - mean;
            var += d * d;
        }
    }
    for (; c < ch; c++) {
        const float d = xt[(size_t)c * len] - mean;
        var += d * d;
    }
    const float inv = 1.0f / sqrtf(var / (float)ch + eps);
    for (c = 0; c < ch; c++) out[(size_t)c * len + t] = (xt[(size_t)c * len] - mean) * inv * g[c] + b[c];
}

// The same LayerNorm with TS time steps per block: the block's [ch][TS]
// input tile is loaded once into LDS (TS consecutive steps of a channel are
// consecutive addresses, 16 loads per thread in flight), 256 / TS threads
// share a step's channel sums (each a run of every (256 / TS)-th channel,
// then added in a fixed order), and every thread writes the normalised tile,
// with max |out| into the slots of amax.  With one thread per step the two
// sums over 1024 channels were 30 of 39 us at 26 steps.
template <int TS>
__global__ __launch_bounds__(256) void k_dec_lnorm_tile(const float *x, const float *g, const float *b, int ch, int len,
                                                        float eps, float *out, unsigned *amax) {
    extern __shared__ float tile[];  // [ch][TS]
    constexpr int U = 16, R = 256 / TS;
    __shared__ float part[R][TS];
    const int t0 = blockIdx.x * TS, tid = threadIdx.x;
    const int n = min(TS, len - t0);
    const int total = ch * TS;
    for (int base = 0; base < total; base += 256 * U) {
        float v[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i = base + u * 256 + tid, c = i / TS, j = i - c * TS;
            v[u] = i < total && j < n ? x[(size_t)c * len + t0 + j] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i = base + u * 256 + tid;
            if (i < total) tile[i] = v[u];
        }
    }
    __syncthreads();
    const int j = tid % TS, r = tid / TS;
    auto sum = [&](float v) {  // over the R threads of step j
        part[r][j] = v;
        __syncthreads();
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < R; i++) s += part[i][j];
        __syncthreads();
        return s;
    };
    float acc = 0.0f;
    for (int c = r; c < ch; c += R) acc += tile[c * TS + j];
    const float mean = sum(acc) / (float)ch;
    acc = 0.0f;
    for (int c = r; c < ch; c += R) {
        const float d = tile[c * TS + j] - mean;
        acc += d * d;
    }
    const float inv = 1.0f / sqrtf(sum(acc) / (float)ch + eps);
    float m = 0.0f;
    if (j < n)
        for (int c = r; c < ch; c += R) {
            const float v = (tile[c * TS + j] - mean) * inv * g[c] + b[c];
            m = fmaxf(m, fabsf(v));
            out[(size_t)c * len + t0 + j] = v;
        }
    block_amax(m, &part[0][0], &amax[blockIdx.x % kDecMaxSlots]);
}

// With add set, the input is x + add, stored to sum (which may be x: each
// element is read before it is written, by the same thread) before the
// activation: a residual sum made where it is next read.
// x + exp(-beta) * sin(exp(alpha) * x)^2 per channel, channel-first: block
// row y is channel y (its two exponentials computed once per thread, no
// division per element), and the blocks of a row stride through its
// samples.  With amax set, each block's largest |out| (NaN excluded) is
// folded into amax[block % kDecMaxSlots] by an unsigned atomicMax of the
// float bits, which orders non-negative floats as their values: the slots'
// maximum does not depend on the order of the blocks, and 64 slots keep the
// atomics from queueing on one address.
__global__ __launch_bounds__(256) void k_dec_snake(const float *x, const float *alpha, const float *beta, int ch,
                                                   int len, float *out, unsigned *amax, const float *add, float *sum) {
    const int c = blockIdx.y;
    const float a = expf(alpha[c]), inv_b = expf(-beta[c]);
    const size_t base = (size_t)c * len;
    float m = 0.0f;
    auto snake = [&](float v) {
        const float s = sinf(a * v);
        const float o = v + inv_b * s * s;
        m = fmaxf(m, fabsf(o));  // a NaN o leaves m as it was
        return o;
    };
    const int stride = gridDim.x * blockDim.x;
    if ((len & 3) == 0) {
        // rows of a multiple of 4 samples (every decoder stage): 16-byte
        // loads and stores, two in flight per thread
        const float4 *x4 = reinterpret_cast<const float4 *>(x + base);
        float4 *o4 = reinterpret_cast<float4 *>(out + base);
        const float4 *a4 = reinterpret_cast<const float4 *>(add + base);
        float4 *s4 = reinterpret_cast<float4 *>(sum + base);
        auto in = [&](int i) {  // x, or x + add stored to sum first
            float4 v = x4[i];
            if (add) {
                const float4 d = a4[i];
                v = make_float4(v.x + d.x, v.y + d.y, v.z + d.z, v.w + d.w);
                s4[i] = v;
            }
            return v;
        };
        const int n4 = len >> 2;
        int t = blockIdx.x * blockDim.x + threadIdx.x;
        for (; t + stride < n4; t += 2 * stride) {
            const float4 v0 = in(t), v1 = in(t + stride);
            o4[t] = make_float4(snake(v0.x), snake(v0.y), snake(v0.z), snake(v0.w));
            o4[t + stride] = make_float4(snake(v1.x), snake(v1.y), snake(v1.z), snake(v1.w));
        }
        if (t < n4) {
            const float4 v0 = in(t);
            o4[t] = make_float4(snake(v0.x), snake(v0.y), snake(v0.z), snake(v0.w));
        }
    } else {
        for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < len; t += stride) {
            float v = x[base + t];
            if (add) {
                v += add[base + t];
                sum[base + t] = v;
            }
            out[base + t] = snake(v);
        }
    }
    if (!amax) return;  // uniform
    __shared__ float red[4];
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
        atomicMax(&amax[(blockIdx.y * gridDim.x + blockIdx.x) % kDecMaxSlots], __float_as_uint(m));
    }
}

__global__ void k_dec_fill_u32(unsigned *p, int n, unsigned v) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// max |x| of n values into the kDecMaxSlots slots of amax, as k_dec_snake
// records it (for inputs of the matrix-core layers that no SnakeBeta makes).
__global__ __launch_bounds__(256) void k_dec_absmax(const float *x, size_t n, unsigned *amax) {
    float m = 0.0f;
    const size_t stride = (size_t)gridDim.x * blockDim.x, t0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if ((n & 3) == 0 && ((uintptr_t)x & 15) == 0) {
        // 16-byte loads, four in flight per thread
        const float4 *x4 = reinterpret_cast<const float4 *>(x);
        const size_t n4 = n >> 2;
#pragma unroll 4
        for (size_t i = t0; i < n4; i += stride) {
            const float4 v = x4[i];
            m = fmaxf(m, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
        }
    } else {
        for (size_t i = t0; i < n; i += stride) m = fmaxf(m, fabsf(x[i]));
    }
    __shared__ float red[4];
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
        atomicMax(&amax[blockIdx.x % kDecMaxSlots], __float_as_uint(m));
    }
}

// A bound on |v + eb sin(ea v)^2| over |v| <= m that no sine is needed for,
// from sin(t)^2 <= min(1, t^2).
__device__ __forceinline__ float dec_snake_bound(float m, float ea, float eb) {
    const float t = ea * m;
    return fmaf(eb, fminf(1.0f, t * t), m);
}

// |v|, or for a v that is not finite, whose SnakeBeta is NaN, NaN: a maximum
// leaves it out.
__device__ __forceinline__ float finite_abs(float v) { return fmaf(v, 0.0f, fabsf(v)); }

// Its maximum over x [ch][len] into the slots of amax; block row y is channel y.
__global__ __launch_bounds__(256) void k_dec_snake_bound(const float *x, const float *ea, const float *eb, int len,
                                                         unsigned *amax) {
    __shared__ float red[4];
    const int c = blockIdx.y, stride = gridDim.x * blockDim.x;
    const float a = ea[c], b = eb[c], *row = x + (size_t)c * len;
    float m = 0.0f;
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < len; t += stride) m = fmaxf(m, finite_abs(row[t]));
    block_amax(fmaxf(0.0f, dec_snake_bound(m, a, b)), red, &amax[(blockIdx.y * gridDim.x + blockIdx.x) % kDecMaxSlots]);
}

typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// The exponent e that puts a positive finite maximum m at m * 2^e in
// [2^14, 2^15) (0 for zero, infinite or NaN).
__device__ __forceinline__ int split_exponent(float m) {
    if (!(m > 0.0f && m < INFINITY)) return 0;
    int E;
    (void)frexpf(m, &E);  // m = f * 2^E, f in [0.5, 1)
    return min(15 - E, 126);
}

// A convolution's weights as binary16 hi + lo MFMA A operands, scaled by
// 2^ew: thread (tile, step, lane) writes the 8 values of row
// m = 32 * tile + lane % 32 for step = (16-channel block cb, tap) with the
// taps inner (cb = step / taps, tap = step % taps), channels
// ci = 16 cb + 8 (lane / 32) + i (zero past M or cin): the element
// w[m * sm + ci * sci + k0 + tap * kd] -- for a causal convolution
// W[m][ci][tap] (src/conv.rs:114-184: sm = cin * ksize, sci = ksize, k0 = 0,
// kd = 1).  up > 1: row m is output phase m % up of channel m / up of a
// transposed one, W[ci][m / up][m % up + (J-1-tap) up] (src/conv.rs:198-268:
// sm = ksize, sci = channels * ksize, k0 = (J - 1) up, kd = -up), so that tap
// t reads the input J - 1 - t steps back.
// hi = f16(w'), lo = f16(w' - hi).
__global__ void k_dec_conv_repack(const float *w, long long sm, long long sci, int k0, int kd, int M, int cin,
                                  int taps, int cin16, int mtiles, int ksteps, int ew, int up, _Float16 *wh,
                                  _Float16 *wl) {
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (size_t)mtiles * ksteps * 64) return;
    const int lane = (int)(idx & 63);
    const size_t ts = idx >> 6;
    const int tile = (int)(ts / ksteps), step = (int)(ts - (size_t)tile * ksteps);
    const int m = 32 * tile + (lane & 31), kb = 16 * step + 8 * (lane >> 5);
    const int cb = step / taps, tap = step - cb * taps;  // step = (16-channel block, tap), taps inner
    half8 h, l;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int ci = 16 * cb + (kb & 15) + i;
        const float v = (m < M && ci < cin && tap < taps)
                            ? ldexpf(w[(long long)(m / up) * sm + m % up + (long long)ci * sci + k0 + (long long)tap * kd], ew)
                            : 0.0f;
        const _Float16 hv = (_Float16)v;
        h[i] = hv;
        l[i] = (_Float16)(v - (float)hv);
    }
    reinterpret_cast<half8 *>(wh)[idx] = h;
    reinterpret_cast<half8 *>(wl)[idx] = l;
}

// Row m's channel and output phase (m = channel * up + phase; up_inv as
// launch_dec_conv_mfma sets it), and the output of row m at position n.
__device__ __forceinline__ int dec_row_channel(const DecConvMfmaParams &P, int m) {
    return P.up_inv ? (int)__umulhi((unsigned)m, P.up_inv) : m;
}
__device__ __forceinline__ float dec_conv_out(const DecConvMfmaParams &P, int m, int n, float v) {
    const int ch = dec_row_channel(P, m);
    if (P.bias) v += P.bias[ch];
    if (P.act == DEC_ACT_GELU) v = dec_gelu(v);
    float *dst = P.c + (long long)ch * P.ldc + (long long)n * P.out_stride + (m - ch * P.up);
    switch (P.epi) {
        case DEC_EPI_STORE: *dst = v; break;
        case DEC_EPI_ACCUM: *dst += v; break;
        case DEC_EPI_SCALED_RESID: *dst += P.scale[m] * v; break;
        case DEC_EPI_RESID_IN: *dst = P.resid[dst - P.c] + (P.scale ? P.scale[m] * v : v); break;
        default: *dst = v < -1.0f ? -1.0f : (v > 1.0f ? 1.0f : v); break;  // DEC_EPI_CLAMP (NaN stays)
    }
    return v;
}

// A causal convolution c[m][n] = bias[m] + sum_{ci, tap} W[m][ci][tap] *
// x[ci][n + (tap - (ksize - 1)) * dilation] (zero before the signal) as an
// implicit GEMM on the matrix cores.  Each wave owns 32 output steps n and
// the block's MT tiles of 32 channels.  The A operands of a stage of
// kConvStage 16-row K steps are loaded once per block -- each wave loads a
// quarter of the (tile, step, hi/lo) units -- and staged in LDS (double
// buffered, one barrier per stage), so the four waves share them.  Per step
// each wave gathers its own B operand -- lane l: step n0 + l % 32, channels
// ci0 + 8 (l / 32) + i of one tap (a step is one tap of one block of 16
// channels, the taps of a block consecutive, so a tap re-reads the lines
// the previous step gathered, shifted by the dilation) -- scales
// it by 2^ex (ex from the producer's max |x|), splits it into binary16 hi +
// lo, and runs three MFMAs per tile: wh * xh + wh * xl + wl * xh.  Every
// product of binary16 values is exact in the f32 accumulator; the dropped
// wl * xl term and the two splits leave a relative error of about 2^-21 per
// term, the f32 level.  The next stage's operands are loaded before the
// current stage's MFMAs.
template <int MT, bool KF>  // KF: channels contiguous (sxc == 1, cin % 8 == 0)
__global__ __launch_bounds__(256) void k_dec_conv_mfma(DecConvMfmaParams P) {
    static_assert(kDecMaxSlots == 64, "one max slot per lane");
    constexpr int G = kConvStage;
    constexpr int UNITS = 2 * MT * G;  // 1-KiB operand units per stage: (step, tile, hi/lo)
    constexpr int UPW = UNITS / 4;     // per wave
    static_assert(UNITS % 4 == 0, "units split evenly over the 4 waves");
    __shared__ half8 As[2][UNITS][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int col = lane & 31, half = lane >> 5;
    const int n = (blockIdx.x * 4 + wave) * 32 + col;  // this lane's output step
    const int t0 = blockIdx.y * MT;
    const int len = P.len, ksteps = P.ksteps, nstage = ksteps / G;
    const _Float16 *wh = P.wh, *wl = P.wl;
    // max |x| over the producer's slots, one per lane
    const int ex = split_exponent(wave_max(__uint_as_float(P.xmax[lane])));
    const float xs = ldexpf(1.0f, ex);
    const int cpl = P.cin - 8 * half;  // channels this lane's half may read at ci0 = 0

    // this wave's A units of stage g: unit u = (gs * MT + t) * 2 + hl
    auto load_a = [&](int g, half8 (&ua)[UPW]) {
#pragma unroll
        for (int k = 0; k < UPW; k++) {
            const int u = wave + 4 * k, hl = u & 1, t = (u >> 1) % MT, gs = (u >> 1) / MT;
            const size_t o = ((size_t)(t0 + t) * ksteps + g * G + gs) * 64 + lane;
            ua[k] = reinterpret_cast<const half8 *>(hl ? wl : wh)[o];
        }
    };
    // the 8 raw x values of this lane at step s (zero past the taps of a
    // padded last stage)
    auto load_b = [&](int s, float (&xv)[8]) {
        const int cb = s / P.ksize, tap = s - cb * P.ksize, ci0 = 16 * cb;  // wave-uniform
        const int p = n + (tap - (P.ksize - 1)) * P.dilation;
        const bool ok = n < len && p >= 0 && tap < P.ksize && ci0 < cpl;
        const float *xp = P.x + (long long)(ci0 + 8 * half) * P.sxc + (long long)(ok ? p : 0) * P.sxn;
        if constexpr (KF) {
            // all 8 channels exist (cin % 8 == 0): two 16-byte loads
            const float4 a = ok ? *reinterpret_cast<const float4 *>(xp) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            const float4 b = ok ? *reinterpret_cast<const float4 *>(xp + 4) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            xv[0] = a.x, xv[1] = a.y, xv[2] = a.z, xv[3] = a.w;
            xv[4] = b.x, xv[5] = b.y, xv[6] = b.z, xv[7] = b.w;
        } else {
#pragma unroll
            for (int i = 0; i < 8; i++) xv[i] = ok && ci0 + i < cpl ? xp[(long long)i * P.sxc] : 0.0f;
        }
    };
    f32x16 acc[MT];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[t][r] = 0.0f;
    half8 ua[UPW];
    float xv[G][8];
    load_a(0, ua);
#pragma unroll
    for (int gs = 0; gs < G; gs++) load_b(gs, xv[gs]);
#pragma unroll
    for (int k = 0; k < UPW; k++) As[0][wave + 4 * k][lane] = ua[k];
    __syncthreads();
    for (int g = 0; g < nstage; g++) {
        const int buf = g & 1;
        const bool more = g + 1 < nstage;  // uniform
        half8 na[UPW];
        float nx[G][8];
        if (more) {
            load_a(g + 1, na);
#pragma unroll
            for (int gs = 0; gs < G; gs++) load_b((g + 1) * G + gs, nx[gs]);
        }
#pragma unroll
        for (int gs = 0; gs < G; gs++) {
            half8 bh, bl;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float v = xv[gs][i] * xs;
                const _Float16 hv = (_Float16)v;
                bh[i] = hv;
                bl[i] = (_Float16)(v - (float)hv);
            }
#pragma unroll
            for (int t = 0; t < MT; t++) {
                const half8 ah = As[buf][(gs * MT + t) * 2][lane], al = As[buf][(gs * MT + t) * 2 + 1][lane];
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bh, acc[t], 0, 0, 0);
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bl, acc[t], 0, 0, 0);
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, bh, acc[t], 0, 0, 0);
            }
        }
        if (more) {
            // buf ^ 1 was last read in stage g - 1, before the last barrier
#pragma unroll
            for (int k = 0; k < UPW; k++) As[buf ^ 1][wave + 4 * k][lane] = na[k];
#pragma unroll
            for (int gs = 0; gs < G; gs++)
#pragma unroll
                for (int i = 0; i < 8; i++) xv[gs][i] = nx[gs][i];
        }
        __syncthreads();
    }
    // D layout: lane l, register r -> row (r / 4) * 8 + (l / 32) * 4 + r % 4,
    // column l % 32
    if (n >= len) return;
    const int sc = -(ex + P.ew);
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int m = 32 * (t0 + t) + (r >> 2) * 8 + half * 4 + (r & 3);
            if (m >= P.M) continue;
            float v = ldexpf(acc[t][r], sc);
            dec_conv_out(P, m, n, v);
        }
}

// The same product for launches too small to fill the GPU (the transformer's
// linears, the first Vocos stages; every layer of a short decode): one block
// per (32 output steps, channel tile), its NW waves splitting the K steps.
// Such a launch is one chain of loads, MFMAs and the sum, so each wave has
// the operands of U steps in flight at once, and the waves' partials go
// through LDS to all threads, one output each, added in wave order.
// 13 frames: the transformer's linears 18 -> 6-10 us, 768 -> 768 channels of
// 7 taps 85 -> 70 (four waves, one step ahead, before).
template <bool KF, int NW>
__global__ __launch_bounds__(64 * NW) void k_dec_conv_mfma_ks(DecConvMfmaParams P) {
    static_assert(kDecMaxSlots == 64, "one max slot per lane");
    constexpr int U = 4;
    __shared__ float red[NW][16][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 31, half = lane >> 5;
    // Blocks of one XCD (every 8th) take a contiguous run of (tile,
    // positions), positions innermost: a tile's weights then come into one
    // XCD's L2 only.
    const int len = P.len, ksteps = P.ksteps;
    const int nx = (len + 31) / 32, total = nx * P.mtiles, per = (int)(gridDim.x >> 3);
    const int L = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if (L >= total) return;
    const int tile = __builtin_amdgcn_readfirstlane(L / nx), n = (L - tile * nx) * 32 + col;
    const _Float16 *wh = P.wh, *wl = P.wl;
    const int q = (ksteps + NW - 1) / NW, s0 = wave * q, s1 = min(ksteps, s0 + q);
    const unsigned xmax = P.xmax[lane];
    const half8 *ah0 = reinterpret_cast<const half8 *>(wh) + (size_t)tile * ksteps * 64;
    const half8 *al0 = reinterpret_cast<const half8 *>(wl) + (size_t)tile * ksteps * 64;
    half8 ah[U], al[U];
    float xv[U][8];
    int cb = s0 / P.ksize, tap = s0 - cb * P.ksize;  // of the next step to load (uniform)
    // Steps s .. s + U - 1; one past the wave's last loads valid operands and
    // has a zero B.  A channel's row is a uniform address, the lane's
    // position (and upper half of the channels) a 32-bit offset.
    auto load = [&](int s) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int ci0 = 16 * cb, p = n + (tap - (P.ksize - 1)) * P.dilation;
            const bool ok = s + u < s1 && n < len && p >= 0;
            const size_t o = (size_t)min(s + u, ksteps - 1) * 64;
            ah[u] = (ah0 + o)[lane];
            al[u] = (al0 + o)[lane];
            if constexpr (KF) {
                // all 8 channels exist (cin % 8 == 0): two 16-byte loads
                const bool in = ok && ci0 + 8 * half < P.cin;
                const float *xp = P.x + (in ? (long long)p * P.sxn + ci0 + 8 * half : 0);
                const float4 a = *reinterpret_cast<const float4 *>(xp), b = *reinterpret_cast<const float4 *>(xp + 4);
                xv[u][0] = a.x, xv[u][1] = a.y, xv[u][2] = a.z, xv[u][3] = a.w;
                xv[u][4] = b.x, xv[u][5] = b.y, xv[u][6] = b.z, xv[u][7] = b.w;
#pragma unroll
                for (int i = 0; i < 8; i++) xv[u][i] = in ? xv[u][i] : 0.0f;
            } else {
                const long long lo = ok ? (long long)p * P.sxn : 0, hi = lo + 8 * half * P.sxc;
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const float *row = P.x + (long long)min(ci0 + i, P.cin - 1) * P.sxc;  // uniform
                    const bool in = ci0 + 8 * half + i < P.cin;
                    xv[u][i] = row[in ? hi : lo];
                    xv[u][i] = in && ok ? xv[u][i] : 0.0f;
                }
            }
            if (++tap == P.ksize) tap = 0, cb++;
        }
    };
    load(s0);
    // max |x| over the producer's slots, one per lane
    const int ex = split_exponent(wave_max(__uint_as_float(xmax)));
    const float xs = ldexpf(1.0f, ex);
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.0f;
    for (int s = s0; s < s1; s += U) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            half8 bh, bl;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float v = xv[u][i] * xs;
                const _Float16 hv = (_Float16)v;
                bh[i] = hv;
                bl[i] = (_Float16)(v - (float)hv);
            }
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[u], bh, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[u], bl, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[u], bh, acc, 0, 0, 0);
        }
        if (s + U < s1) load(s + U);  // uniform
    }
#pragma unroll
    for (int r = 0; r < 16; r++) red[wave][r][lane] = acc[r];
    __syncthreads();
    if (n >= len) return;
    // D layout: lane l, register r -> row (r / 4) * 8 + (l / 32) * 4 + r % 4,
    // column l % 32
    const int sc = -(ex + P.ew);
#pragma unroll
    for (int r0 = 0; r0 < 16; r0 += NW) {
        const int r = r0 + wave;
        const int m = 32 * tile + (r >> 2) * 8 + half * 4 + (r & 3);
        float v = red[0][r][lane];
#pragma unroll
        for (int w = 1; w < NW; w++) v += red[w][r][lane];
        if (m >= P.M) continue;
        v = ldexpf(v, sc);
        dec_conv_out(P, m, n, v);
    }
}

// A causal convolution with 3 or more taps over a channel-first input
// (sxn == 1), its input window staged in LDS: per block of 16 input
// channels, the block's window -- positions n0 - (ksize - 1) * dilation ..
// n0 + 127 of those channels -- is loaded once (thread t: position t, the
// 16 channels' values, each load coalesced over the threads), scaled by 2^ex
// and split into binary16 hi + lo, and stored position-major per half of the
// channels ([8-channel half][position][8 channels], 16-byte rows, so the 16
// lanes of a 16-byte LDS read hit 16 consecutive rows: no bank conflicts),
// and every tap's B operand is two 16-byte LDS reads at position n - n0 +
// tap * dilation: each value is split once instead of once per tap.  The
// next channel block's window is loaded into registers during the current
// block's taps (double-buffered, one barrier per channel block); A operands
// come from global memory one step ahead.  Same operand order and products as k_dec_conv_mfma.
template <int MT>
__global__ __launch_bounds__(256) void k_dec_conv_win(DecConvMfmaParams P) {
    static_assert(kDecMaxSlots == 64, "one max slot per lane");
    constexpr int WMAX = 256;  // window positions: 128 + (ksize - 1) * dilation <= the block's threads
    __shared__ __align__(16) _Float16 wh_s[2][2][WMAX][8], wl_s[2][2][WMAX][8];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int col = lane & 31, half = lane >> 5;
    const int n0 = blockIdx.x * 128, n = n0 + wave * 32 + col;
    const int t0 = blockIdx.y * MT;
    const int len = P.len, ks = P.ksize, dil = P.dilation, ksteps = P.ksteps;
    const _Float16 *wh = P.wh, *wl = P.wl;
    const int W = 128 + (ks - 1) * dil, wpos = n0 - (ks - 1) * dil + tid;  // this thread's window position
    const bool wok = tid < W && wpos >= 0 && wpos < len;
    const int ncb = P.cin16 / 16;
    const int ex = split_exponent(wave_max(__uint_as_float(P.xmax[lane])));
    const float xs = ldexpf(1.0f, ex);
    auto load_win = [&](int cb, float (&v)[16]) {
        const float *xp = P.x + (size_t)(16 * cb) * len + (wok ? wpos : 0);
#pragma unroll
        for (int c = 0; c < 16; c++) v[c] = wok && 16 * cb + c < P.cin ? xp[(size_t)c * len] : 0.0f;
    };
    auto store_win = [&](int buf, const float (&v)[16]) {
        if (tid >= W) return;
        half8 h[2], l[2];
#pragma unroll
        for (int c = 0; c < 16; c++) {
            const float x = v[c] * xs;
            const _Float16 hv = (_Float16)x;
            h[c >> 3][c & 7] = hv;
            l[c >> 3][c & 7] = (_Float16)(x - (float)hv);
        }
        *reinterpret_cast<half8 *>(&wh_s[buf][0][tid][0]) = h[0];
        *reinterpret_cast<half8 *>(&wh_s[buf][1][tid][0]) = h[1];
        *reinterpret_cast<half8 *>(&wl_s[buf][0][tid][0]) = l[0];
        *reinterpret_cast<half8 *>(&wl_s[buf][1][tid][0]) = l[1];
    };
    auto load_a = [&](int s, half8 (&ah)[MT], half8 (&al)[MT]) {
#pragma unroll
        for (int t = 0; t < MT; t++) {
            const size_t o = ((size_t)(t0 + t) * ksteps + s) * 64 + lane;
            ah[t] = reinterpret_cast<const half8 *>(wh)[o];
            al[t] = reinterpret_cast<const half8 *>(wl)[o];
        }
    };
    f32x16 acc[MT];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[t][r] = 0.0f;
    float wv[16];
    load_win(0, wv);
    store_win(0, wv);
    half8 ah[MT], al[MT];
    load_a(0, ah, al);
    __syncthreads();
    const int nsteps = ncb * ks;  // the steps past these (stage padding) hold zero weights
    for (int cb = 0; cb < ncb; cb++) {
        const int buf = cb & 1;
        const bool more = cb + 1 < ncb;  // uniform
        if (more) load_win(cb + 1, wv);
        for (int tap = 0; tap < ks; tap++) {
            const int s = cb * ks + tap;
            half8 nh[MT], nl[MT];
            load_a(s + 1 < nsteps ? s + 1 : s, nh, nl);
            const int p = wave * 32 + col + tap * dil;
            const half8 bh = *reinterpret_cast<const half8 *>(&wh_s[buf][half][p][0]);
            const half8 bl = *reinterpret_cast<const half8 *>(&wl_s[buf][half][p][0]);
#pragma unroll
            for (int t = 0; t < MT; t++) {
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[t], bh, acc[t], 0, 0, 0);
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[t], bl, acc[t], 0, 0, 0);
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[t], bh, acc[t], 0, 0, 0);
            }
#pragma unroll
            for (int t = 0; t < MT; t++) {
                ah[t] = nh[t];
                al[t] = nl[t];
            }
        }
        // buf ^ 1 was last read in channel block cb - 1, before the last barrier
        if (more) store_win(buf ^ 1, wv);
        __syncthreads();
    }
    // D layout: lane l, register r -> row (r / 4) * 8 + (l / 32) * 4 + r % 4,
    // column l % 32
    if (n >= len) return;
    const int sc = -(ex + P.ew);
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int m = 32 * (t0 + t) + (r >> 2) * 8 + half * 4 + (r & 3);
            if (m >= P.M) continue;
            float v = ldexpf(acc[t][r], sc);
            dec_conv_out(P, m, n, v);
        }
}

// k_dec_conv_win with the waves' roles swapped, for NW (3 or 4) channel
// tiles per block of NW waves: wave w owns channel tile NW * blockIdx.y + w
// -- its A operands loaded by it alone, where every wave of
// k_dec_conv_win<MT> loads all MT tiles' -- and all four 32-position tiles
// of the block, whose B operands it reads from the staged window (LDS,
// twice L1's bandwidth).  Per step a block reads NW * 2 KiB of A operands
// through L1 instead of 4 * NW * 2 KiB.  The window (up to 256 positions)
// is staged by the block's 64 * NW threads, position t + 64 * NW * q by
// thread t in pass q.  Same window, operands and product order per output
// as k_dec_conv_win: the same bits.
// The transposed convolutions (2 taps) come here with their phases as rows:
// the input is read for all of them at once and each stretch of the output
// is written whole, 16 bytes at a time where 4 rows are 4 phases of one
// channel.  As one launch row per phase (k_dec_conv_mfma, each gathering the
// input and writing every stride-th float) 768 -> 384 channels by 5 to
// 80,000 positions took 437 us, 384 -> 192 by 4 to 320,000 563, 192 -> 96 by
// 3 to 960,000 601 and 67 more for max |out|; here 424, 375 and 486 to 516,
// and 548 with the next unit's bound taken per channel (604 per element, whose
// two factors were then loaded for each; 16 maxima kept over the position
// tiles cost a wave a SIMD, 820).
template <int NW>
__global__ __launch_bounds__(64 * NW) void k_dec_conv_win_tw(DecConvMfmaParams P) {
    static_assert(kDecMaxSlots == 64, "one max slot per lane");
    constexpr int WMAX = 256, PT = 4;  // window positions; 32-position tiles per block
    constexpr int NT = 64 * NW, NP = (WMAX + NT - 1) / NT;  // threads; staging passes
    __shared__ __align__(16) _Float16 wh_s[2][2][WMAX][8], wl_s[2][2][WMAX][8];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, half = lane >> 5;
    // Blocks of one XCD (every 8th) take a contiguous run of (positions, tile
    // group), the tile groups innermost where the input is the larger operand
    // (it then comes into one XCD's L2 once), else the positions.
    const int nx = (P.len + 127) / 128, ny = P.mtiles / NW, per = (int)(gridDim.x >> 3);
    const int L = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if (L >= nx * ny) return;
    const bool inner = (long long)P.mtiles * 32 * P.ksize < P.len;  // weights: 4 bytes per value, as the input
    const int bx = inner ? L / ny : L % nx, by = inner ? L % ny : L / nx;
    const int n0 = bx * 128, tile = by * NW + wave;
    const int len = P.len, ks = P.ksize, dil = P.dilation, ksteps = P.ksteps;
    const _Float16 *wh = P.wh, *wl = P.wl;
    const int W = 128 + (ks - 1) * dil;  // window positions n0 - (ks - 1) * dil .. n0 + 127
    const int ncb = P.cin16 / 16;
    const int ex = split_exponent(wave_max(__uint_as_float(P.xmax[lane])));
    const float xs = ldexpf(1.0f, ex);
    auto load_win = [&](int cb, float (&v)[NP][16]) {
#pragma unroll
        for (int q = 0; q < NP; q++) {
            const int wi = tid + q * NT, wpos = n0 - (ks - 1) * dil + wi;
            const bool wok = wi < W && wpos >= 0 && wpos < len;
            const float *xp = P.x + (size_t)(16 * cb) * len + (wok ? wpos : 0);
#pragma unroll
            for (int c = 0; c < 16; c++) v[q][c] = wok && 16 * cb + c < P.cin ? xp[(size_t)c * len] : 0.0f;
        }
    };
    auto store_win = [&](int buf, const float (&v)[NP][16]) {
#pragma unroll
        for (int q = 0; q < NP; q++) {
            const int wi = tid + q * NT;
            if (wi >= W) continue;
            half8 h[2], l[2];
#pragma unroll
            for (int c = 0; c < 16; c++) {
                const float x = v[q][c] * xs;
                const _Float16 hv = (_Float16)x;
                h[c >> 3][c & 7] = hv;
                l[c >> 3][c & 7] = (_Float16)(x - (float)hv);
            }
            *reinterpret_cast<half8 *>(&wh_s[buf][0][wi][0]) = h[0];
            *reinterpret_cast<half8 *>(&wh_s[buf][1][wi][0]) = h[1];
            *reinterpret_cast<half8 *>(&wl_s[buf][0][wi][0]) = l[0];
            *reinterpret_cast<half8 *>(&wl_s[buf][1][wi][0]) = l[1];
        }
    };
    auto load_a = [&](int s, half8 &ah, half8 &al) {
        const size_t o = ((size_t)tile * ksteps + s) * 64 + lane;
        ah = reinterpret_cast<const half8 *>(wh)[o];
        al = reinterpret_cast<const half8 *>(wl)[o];
    };
    f32x16 acc[PT];
#pragma unroll
    for (int t = 0; t < PT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[t][r] = 0.0f;
    float wv[NP][16];
    load_win(0, wv);
    store_win(0, wv);
    half8 ah, al;
    load_a(0, ah, al);
    __syncthreads();
    const int nsteps = ncb * ks;  // the steps past these (stage padding) hold zero weights
    for (int cb = 0; cb < ncb; cb++) {
        const int buf = cb & 1;
        const bool more = cb + 1 < ncb;  // uniform
        if (more) load_win(cb + 1, wv);
        for (int tap = 0; tap < ks; tap++) {
            const int s = cb * ks + tap;
            half8 nh, nl;
            load_a(s + 1 < nsteps ? s + 1 : s, nh, nl);
#pragma unroll
            for (int t = 0; t < PT; t++) {
                const int p = t * 32 + col + tap * dil;
                const half8 bh = *reinterpret_cast<const half8 *>(&wh_s[buf][half][p][0]);
                const half8 bl = *reinterpret_cast<const half8 *>(&wl_s[buf][half][p][0]);
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bh, acc[t], 0, 0, 0);
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bl, acc[t], 0, 0, 0);
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, bh, acc[t], 0, 0, 0);
            }
            ah = nh;
            al = nl;
        }
        // buf ^ 1 was last read in channel block cb - 1, before the last barrier
        if (more) store_win(buf ^ 1, wv);
        __syncthreads();
    }
    // D layout: lane l, register r -> row (r / 4) * 8 + (l / 32) * 4 + r % 4,
    // column l % 32
    const int sc = -(ex + P.ew);
    float mx = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; r += 4) {
        const int m = 32 * tile + (r >> 2) * 8 + half * 4;
        if (P.quad) {  // 4 phases of one channel: one 16-byte store
            if (m >= P.M) continue;
            const int ch = dec_row_channel(P, m);
            const float b = P.bias ? P.bias[ch] : 0.0f;
            const float ea = P.omax ? P.oea[ch] : 0.0f, eb = P.omax ? P.oeb[ch] : 0.0f;
            float cm = 0.0f;  // the channel's largest |out|
#pragma unroll
            for (int t = 0; t < PT; t++) {
                const int n = n0 + t * 32 + col;
                if (n >= len) continue;
                float4 v;
                v.x = ldexpf(acc[t][r], sc) + b;
                v.y = ldexpf(acc[t][r + 1], sc) + b;
                v.z = ldexpf(acc[t][r + 2], sc) + b;
                v.w = ldexpf(acc[t][r + 3], sc) + b;
                cm = fmaxf(cm, fmaxf(fmaxf(finite_abs(v.x), finite_abs(v.y)), fmaxf(finite_abs(v.z), finite_abs(v.w))));
                *reinterpret_cast<float4 *>(P.c + (long long)ch * P.ldc + (long long)n * P.out_stride +
                                            (m - ch * P.up)) = v;
            }
            mx = fmaxf(mx, dec_snake_bound(cm, ea, eb));
            continue;
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (m + j >= P.M) continue;
            const int ch = P.omax ? dec_row_channel(P, m + j) : 0;
            const float ea = P.omax ? P.oea[ch] : 0.0f, eb = P.omax ? P.oeb[ch] : 0.0f;
            float cm = 0.0f;
#pragma unroll
            for (int t = 0; t < PT; t++) {
                const int n = n0 + t * 32 + col;
                if (n < len) cm = fmaxf(cm, finite_abs(dec_conv_out(P, m + j, n, ldexpf(acc[t][r + j], sc))));
            }
            mx = fmaxf(mx, dec_snake_bound(cm, ea, eb));
        }
    }
    if (P.omax) {  // uniform
        mx = wave_max(mx);
        if (lane == 0) atomicMax(&P.omax[(blockIdx.x * NW + wave) % kDecMaxSlots], __float_as_uint(mx));
    }
}

// sin(t)^2 of SnakeBeta.  r + e is t less the nearest multiple k of pi/2 (in
// three parts: the first subtraction is exact, e what the second rounds off),
// sin(r + e) = r + (e + r^3 p(r^2)) on [-pi/4, pi/4], p the least maximum
// relative error (Lawson's reweighted least squares; 8.3e-9 as rounded), and
// an odd k takes 1 - sin^2.  Error over 2^24 arguments N(0, 6) rms 1.85e-8,
// largest 9.8e-8; the square of sinf 3.13e-8 and 1.29e-7.  A polynomial over
// [-pi/2, pi/2] without e (3.7e-8, 2.5e-7) was 1 % of a decode faster.  Past
// |t| = 8192 the library's.
__device__ __forceinline__ float dec_sin2(float t) {
    const float k = rintf(t * 0.636619747f);
    const float r1 = fmaf(-k, 1.57079637f, t);
    const float r = fmaf(-k, -4.37113883e-8f, r1);
    const float e = fmaf(-k, -1.71509942e-15f, fmaf(-k, -4.37113883e-8f, r1 - r));
    const float z = r * r;
    float p = fmaf(z, -1.95149580e-4f, 8.33215844e-3f);
    p = fmaf(z, p, -0.166666552f);
    float s = r + fmaf(r * z, p, e);
    s = (int)k & 1 ? fmaf(-s, s, 1.0f) : s * s;
    if (!(fabsf(t) <= 8192.0f)) s = sinf(t), s *= s;
    return s;
}

// A residual unit (src/decoder.rs:462-480) in one launch: out = x + conv2(
// snake2(conv1(snake1(x)) + b1)) + b2, conv1 of 7 taps, conv2 of one, for C =
// 32 CT channels.  As five launches it read and wrote the signal nine times;
// here each block owns all C channels of P = 64 * 12 / CT positions:
//   conv1: as k_dec_conv_win_tw, the window of 16 channels at a time staged
//     position-major in LDS as binary16 hi + lo -- but from x, SnakeBeta
//     applied as it is staged (once per block, since the block has every
//     channel tile), interleaved with the MFMAs of the block before;
//   snake2 of the accumulators, split into LDS as conv2's operand, scaled by
//     the block's own largest value;
//   conv2 from LDS, and the residual added from x.
// 12 waves, wave w on channel tile w % CT and positions 64 (w / CT) ..: three
// waves a SIMD, each A operand used for two 32-position tiles and shared
// through L1 by the 12 / CT waves of its tile; A operands are loaded three
// to four taps ahead.  conv1's operand scale is a bound on SnakeBeta (per
// element, dec_snake_bound) that x's producer recorded, as this unit records
// the next one's.
// C = 96, 960,000 positions: 1130 us as five launches, 622 here; C = 192,
// 320,000 positions: 1060, 709; C = 384, 80,000: 810, 570 (averages of a
// trace whose fastest launches take 592, 666 and 548).
// Matrix cores a third busy, vector ALU (the sines and splits) a third, the
// rest latency: one block a CU, and of the 168 registers that 12 waves leave
// 0, 4 and 6 spill (96, 192 and 384 channels).  Blocks of 6 waves and half the
// positions measured slower (C = 96, 805 us: twice the A operands through the
// L2).
template <int CT, int NWV>
__global__ __launch_bounds__(64 * NWV, 3) void k_dec_resunit(DecResUnitParams P) {
    static_assert(kDecMaxSlots == 64, "one max slot per lane");
    constexpr int C = 32 * CT, PG = NWV / CT, NP = 64 * PG, TAPS = 7;
    constexpr int WMAX = NP + 64;                     // window positions: NP + 6 * dilation at most
    constexpr int SEG = WMAX / 64, ITEMS = 4 * SEG;   // (4 channels, 64 positions) per wave and pass
    constexpr int PASSES = (ITEMS + NWV - 1) / NWV;
    constexpr int NCB = C / 16;
    union Lds {
        struct {
            _Float16 h[2][2][WMAX][8], l[2][2][WMAX][8];  // [buffer][8-channel half][position][channel]
        } win;
        struct {
            _Float16 h[NCB][2][NP][8], l[NCB][2][NP][8];  // conv2's operand
        } act;
    };
    __shared__ __align__(16) Lds sm;
    __shared__ float red[NWV];
    __shared__ __align__(16) float last[3][C];  // b2, oea, oeb: read in the epilogue, where nothing hides a load (1 % of a decode)
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 31, half = lane >> 5;
    if (threadIdx.x < C) {
        last[0][threadIdx.x] = P.b2[threadIdx.x];
        last[1][threadIdx.x] = P.omax ? P.oea[threadIdx.x] : 0.0f;
        last[2][threadIdx.x] = P.omax ? P.oeb[threadIdx.x] : 0.0f;
    }
    const int tile = wave % CT, p0 = 64 * (wave / CT);  // this wave's channels and positions of the block
    const int n0 = blockIdx.x * NP, len = P.len, dil = P.dilation;
    const int w0 = n0 - (TAPS - 1) * dil, W = NP + (TAPS - 1) * dil;
    const int ex = split_exponent(wave_max(__uint_as_float(P.xmax[lane])));
    const float xs = ldexpf(1.0f, ex);

    float v[PASSES][4];
    auto load_win = [&](int cb) {
#pragma unroll
        for (int q = 0; q < PASSES; q++) {
            const int it = wave + NWV * q;
            if (it >= ITEMS) continue;  // uniform
            const int g = it / SEG, pos = w0 + 64 * (it % SEG) + lane;
            const float *xp = P.x + (size_t)(16 * cb + 4 * g) * len + min(max(pos, 0), len - 1);
#pragma unroll
            for (int j = 0; j < 4; j++) v[q][j] = xp[(size_t)j * len];
        }
    };
    auto put_win = [&](int cb, int q, int buf) {
        const int it = wave + NWV * q;
        if (it >= ITEMS) return;  // uniform
        const int g = it / SEG, wp = 64 * (it % SEG) + lane, pos = w0 + wp;
        const bool in = wp < W && pos >= 0 && pos < len;
        half4 h, l;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float x = in ? v[q][j] : 0.0f;
            const int c = 16 * cb + 4 * g + j;  // uniform
            const float o = (x + P.eb1[c] * dec_sin2(P.ea1[c] * x)) * xs;
            h[j] = (_Float16)o;
            l[j] = (_Float16)(o - (float)h[j]);
        }
        *reinterpret_cast<half4 *>(&sm.win.h[buf][g >> 1][wp][4 * (g & 1)]) = h;
        *reinterpret_cast<half4 *>(&sm.win.l[buf][g >> 1][wp][4 * (g & 1)]) = l;
    };
    // A operands in two runs of taps, each loaded while the other is used
    half8 a0h[4], a0l[4], a1h[3], a1l[3];
    const half8 *w1h = reinterpret_cast<const half8 *>(P.w1h) + (size_t)tile * P.ksteps1 * 64 + lane;
    const half8 *w1l = reinterpret_cast<const half8 *>(P.w1l) + (size_t)tile * P.ksteps1 * 64 + lane;
    auto load_a0 = [&](int cb) {
#pragma unroll
        for (int t = 0; t < 4; t++) a0h[t] = w1h[(cb * TAPS + t) * 64], a0l[t] = w1l[(cb * TAPS + t) * 64];
    };
    auto load_a1 = [&](int cb) {
#pragma unroll
        for (int t = 0; t < 3; t++) a1h[t] = w1h[(cb * TAPS + 4 + t) * 64], a1l[t] = w1l[(cb * TAPS + 4 + t) * 64];
    };
    f32x16 acc[2];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[t][r] = 0.0f;
    auto mma = [&](int buf, int tap, const half8 &ah, const half8 &al) {
        half8 bh[2], bl[2];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int p = p0 + 32 * t + col + tap * dil;
            bh[t] = *reinterpret_cast<const half8 *>(&sm.win.h[buf][half][p][0]);
            bl[t] = *reinterpret_cast<const half8 *>(&sm.win.l[buf][half][p][0]);
        }
#pragma unroll
        for (int t = 0; t < 2; t++) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bh[t], acc[t], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < 2; t++) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bl[t], acc[t], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < 2; t++) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, bh[t], acc[t], 0, 0, 0);
    };
    load_win(0);
    load_a0(0);
#pragma unroll
    for (int q = 0; q < PASSES; q++) put_win(0, q, 0);
    __syncthreads();
    for (int cb = 0; cb < NCB; cb++) {
        const int buf = cb & 1;
        const bool more = cb + 1 < NCB;  // uniform
        if (more) load_win(cb + 1);
        load_a1(cb);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < 4; t++) mma(buf, t, a0h[t], a0l[t]);
        __builtin_amdgcn_sched_barrier(0);
        load_a0(more ? cb + 1 : cb);
        if (more) put_win(cb + 1, 0, buf ^ 1);  // last read in channel block cb - 1
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < 3; t++) mma(buf, 4 + t, a1h[t], a1l[t]);
        __builtin_amdgcn_sched_barrier(0);
        if (more)
#pragma unroll
            for (int q = 1; q < PASSES; q++) put_win(cb + 1, q, buf ^ 1);
        __syncthreads();
    }

    // snake2 of this wave's [32 channels][64 positions]; D layout: lane l,
    // register r -> row (r / 4) * 8 + (l / 32) * 4 + r % 4, column l % 32
    const int sc1 = -(ex + P.ew1);
    float m = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int c = 32 * tile + 8 * j + 4 * half;
        const float4 b = *reinterpret_cast<const float4 *>(P.b1 + c);
        const float4 a = *reinterpret_cast<const float4 *>(P.ea2 + c), e = *reinterpret_cast<const float4 *>(P.eb2 + c);
        const float bv[4] = {b.x, b.y, b.z, b.w}, av[4] = {a.x, a.y, a.z, a.w}, ev[4] = {e.x, e.y, e.z, e.w};
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const bool in = n0 + p0 + 32 * t + col < len;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float x = ldexpf(acc[t][4 * j + i], sc1) + bv[i];
                const float o = x + ev[i] * dec_sin2(av[i] * x);
                acc[t][4 * j + i] = in ? o : 0.0f;
                m = fmaxf(m, fabsf(acc[t][4 * j + i]));
            }
        }
    }
    m = wave_max(m);
    if (lane == 0) red[wave] = m;
    __syncthreads();  // also: the last window is read
    m = red[0];
#pragma unroll
    for (int w = 1; w < NWV; w++) m = fmaxf(m, red[w]);
    const int ex2 = split_exponent(m);
    const float xs2 = ldexpf(1.0f, ex2);
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
        for (int t = 0; t < 2; t++) {
            half4 h, l;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float o = acc[t][4 * j + i] * xs2;
                h[i] = (_Float16)o;
                l[i] = (_Float16)(o - (float)h[i]);
            }
            const int p = p0 + 32 * t + col;
            *reinterpret_cast<half4 *>(&sm.act.h[2 * tile + (j >> 1)][j & 1][p][4 * half]) = h;
            *reinterpret_cast<half4 *>(&sm.act.l[2 * tile + (j >> 1)][j & 1][p][4 * half]) = l;
        }
    // the residual, under conv2
    float x[2][16];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int c = 32 * tile + (r >> 2) * 8 + half * 4 + (r & 3);
            x[t][r] = P.x[(size_t)c * len + min(n0 + p0 + 32 * t + col, len - 1)];
        }
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[t][r] = 0.0f;
    const half8 *w2h = reinterpret_cast<const half8 *>(P.w2h) + (size_t)tile * P.ksteps2 * 64 + lane;
    const half8 *w2l = reinterpret_cast<const half8 *>(P.w2l) + (size_t)tile * P.ksteps2 * 64 + lane;
    half8 ch[2][3], cl[2][3];
    auto load_c = [&](int s, int to) {
#pragma unroll
        for (int i = 0; i < 3; i++) ch[to][i] = w2h[(s + i) * 64], cl[to][i] = w2l[(s + i) * 64];
    };
    load_c(0, 0);
    __syncthreads();
#pragma unroll
    for (int s = 0; s < NCB; s += 3) {
        const int b = (s / 3) & 1;
        if (s + 3 < NCB) load_c(s + 3, b ^ 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 3; i++) {
            half8 bh[2], bl[2];
#pragma unroll
            for (int t = 0; t < 2; t++) {
                bh[t] = *reinterpret_cast<const half8 *>(&sm.act.h[s + i][half][p0 + 32 * t + col][0]);
                bl[t] = *reinterpret_cast<const half8 *>(&sm.act.l[s + i][half][p0 + 32 * t + col][0]);
            }
#pragma unroll
            for (int t = 0; t < 2; t++) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ch[b][i], bh[t], acc[t], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < 2; t++) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ch[b][i], bl[t], acc[t], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < 2; t++) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(cl[b][i], bh[t], acc[t], 0, 0, 0);
        }
    }
    const int sc2 = -(ex2 + P.ew2);
    m = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int c = 32 * tile + 8 * j + 4 * half;
        const float4 b = *reinterpret_cast<const float4 *>(&last[0][c]);
        const float bv[4] = {b.x, b.y, b.z, b.w};
        const float4 a = *reinterpret_cast<const float4 *>(&last[1][c]), e = *reinterpret_cast<const float4 *>(&last[2][c]);
        const float av[4] = {a.x, a.y, a.z, a.w}, ev[4] = {e.x, e.y, e.z, e.w};
        float cm[4] = {0.0f, 0.0f, 0.0f, 0.0f};  // the channels' largest |out|
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int n = n0 + p0 + 32 * t + col;
            if (n >= len) continue;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float o = x[t][4 * j + i] + (ldexpf(acc[t][4 * j + i], sc2) + bv[i]);
                cm[i] = fmaxf(cm[i], finite_abs(o));
                P.out[(size_t)(c + i) * len + n] = o;
            }
        }
#pragma unroll
        for (int i = 0; i < 4; i++) m = fmaxf(m, dec_snake_bound(cm[i], av[i], ev[i]));
    }
    if (!P.omax) return;
    m = wave_max(m);
    if (lane == 0) red[wave] = m;  // last read before the barrier ahead of conv2
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < NWV; w++) m = fmaxf(m, red[w]);
        atomicMax(&P.omax[blockIdx.x % kDecMaxSlots], __float_as_uint(m));
    }
}

// out[i] = exp(sign * x[i])
__global__ void k_dec_exp(const float *x, float sign, int n, float *out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = expf(sign * x[i]);
}

unsigned blocks_for(size_t n, unsigned per) { return (unsigned)((n + per - 1) / per); }

}  // namespace

void launch_dec_gather(hipStream_t st, const DecGatherParams &p, int frames) {
    hipLaunchKernelGGL(k_dec_gather, dim3((unsigned)frames), dim3(256), 0, st, p);
}

void launch_dec_rmsnorm(hipStream_t st, const float *x, const float *gamma, int rows, int n, float eps, float *out,
                        unsigned *amax) {
    hipLaunchKernelGGL(k_dec_rmsnorm, dim3((unsigned)rows), dim3(256), 0, st, x, gamma, n, eps, out, amax);
}

void launch_dec_rope(hipStream_t st, float *q, float *k, int T, int heads, int hd, const float *cs, const float *sn,
                     int rows, int ld) {
    const size_t n = (size_t)T * heads * (hd / 2);
    hipLaunchKernelGGL(k_dec_rope, dim3(blocks_for(n, 256)), dim3(256), 0, st, q, k, T, heads, hd, cs, sn, rows, ld);
}

void launch_dec_attn(hipStream_t st, const DecAttnParams &p) {
    hipLaunchKernelGGL(k_dec_attn, dim3(blocks_for((size_t)p.T * p.heads, 4)), dim3(256), 0, st, p);
}

void launch_dec_swiglu(hipStream_t st, const float *g, const float *u, int rows, int width, int ld, float *out,
                       unsigned *amax) {
    // at most 512 blocks, as launch_dec_absmax
    const unsigned blocks = std::min<unsigned>(blocks_for((size_t)rows * width, 256), 512u);
    hipLaunchKernelGGL(k_dec_swiglu, dim3(blocks), dim3(256), 0, st, g, u, rows, width, ld, out, amax);
}

void launch_dec_dwconv(hipStream_t st, const float *x, const float *w, const float *b, int ch, int len, int ks,
                       float *out) {
    hipLaunchKernelGGL(k_dec_dwconv, dim3(blocks_for((size_t)ch * len, 256)), dim3(256), 0, st, x, w, b, ch, len, ks,
                       out);
}

void launch_dec_lnorm(hipStream_t st, const float *x, const float *g, const float *b, int ch, int len, float eps,
                      float *out, unsigned *amax) {
    // the tiled kernel while its [ch][TS] tile fits 64 KiB of LDS
    const size_t lds16 = (size_t)ch * 16 * sizeof(float), lds8 = (size_t)ch * 8 * sizeof(float);
    if (lds16 <= 65536)
        hipLaunchKernelGGL(k_dec_lnorm_tile<16>, dim3((unsigned)((len + 15) / 16)), dim3(256), lds16, st, x, g, b, ch,
                           len, eps, out, amax);
    else if (lds8 <= 65536)
        hipLaunchKernelGGL(k_dec_lnorm_tile<8>, dim3((unsigned)((len + 7) / 8)), dim3(256), lds8, st, x, g, b, ch, len,
                           eps, out, amax);
    else {
        hipLaunchKernelGGL(k_dec_lnorm, dim3(blocks_for((size_t)len, 64)), dim3(64), 0, st, x, g, b, ch, len, eps, out);
        launch_dec_absmax(st, out, (size_t)ch * len, amax);
    }
}

void launch_dec_snake(hipStream_t st, const float *x, const float *alpha, const float *beta, int ch, int len,
                      float *out, unsigned *amax, const float *add, float *sum) {
    // about kSnakeBlocks blocks in all, at least one per channel (rows of a
    // multiple of 4 samples take 4 per thread and iteration)
    const size_t items = (len & 3) == 0 ? (size_t)len / 4 : (size_t)len;
    const unsigned per_row = std::max(1u, std::min<unsigned>(blocks_for(items, 256), kSnakeBlocks / (unsigned)ch));
    hipLaunchKernelGGL(k_dec_snake, dim3(per_row, (unsigned)ch), dim3(256), 0, st, x, alpha, beta, ch, len, out, amax,
                       add, sum);
}

void launch_dec_snake_bound(hipStream_t st, const float *x, const float *ea, const float *eb, int ch, int len,
                            unsigned *amax) {
    // at most 512 blocks where that leaves one per channel, as launch_dec_absmax
    const unsigned per_row = std::max(1u, std::min<unsigned>(blocks_for((size_t)len, 1024), 512u / (unsigned)ch));
    hipLaunchKernelGGL(k_dec_snake_bound, dim3(per_row, (unsigned)ch), dim3(256), 0, st, x, ea, eb, len, amax);
}

void launch_dec_fill_u32(hipStream_t st, unsigned *p, int n, unsigned v) {
    hipLaunchKernelGGL(k_dec_fill_u32, dim3(blocks_for((size_t)n, 256)), dim3(256), 0, st, p, n, v);
}

void launch_dec_conv_repack(hipStream_t st, const float *w, long long sm, long long sci, int k0, int kd, int M, int cin,
                            int taps, int cin16, int mtiles, int ksteps, int ew, int up, _Float16 *wh, _Float16 *wl) {
    const size_t n = (size_t)mtiles * ksteps * 64;
    hipLaunchKernelGGL(k_dec_conv_repack, dim3(blocks_for(n, 256)), dim3(256), 0, st, w, sm, sci, k0, kd, M, cin,
                       taps, cin16, mtiles, ksteps, ew, up, wh, wl);
}

// At least 4 steps (one batch of loads) per wave, and no more waves than the
// chip holds: 500 frames' 1024 -> 1536 channels of 7 taps (3,024 blocks) take
// 378 us with 4 waves a block, 507 with 16; 13 frames' 768 -> 768 (312
// blocks) 70 with 16, 85 with 4.
template <bool KF>
static void launch_conv_mfma_ks(hipStream_t st, const DecConvMfmaParams &p, dim3 grid) {
    if (p.ksteps >= 64 && grid.x <= 512)
        hipLaunchKernelGGL((k_dec_conv_mfma_ks<KF, 16>), grid, dim3(1024), 0, st, p);
    else if (p.ksteps >= 32 && grid.x <= 1024)
        hipLaunchKernelGGL((k_dec_conv_mfma_ks<KF, 8>), grid, dim3(512), 0, st, p);
    else
        hipLaunchKernelGGL((k_dec_conv_mfma_ks<KF, 4>), grid, dim3(256), 0, st, p);
}

template <bool KF>
static void launch_conv_mfma_kf(hipStream_t st, const DecConvMfmaParams &p, int mt) {
    const dim3 grid(blocks_for((size_t)p.len, 128), (unsigned)(p.mtiles / mt));
    switch (mt) {
        case 4: hipLaunchKernelGGL((k_dec_conv_mfma<4, KF>), grid, dim3(256), 0, st, p); break;
        case 3: hipLaunchKernelGGL((k_dec_conv_mfma<3, KF>), grid, dim3(256), 0, st, p); break;
        case 2: hipLaunchKernelGGL((k_dec_conv_mfma<2, KF>), grid, dim3(256), 0, st, p); break;
        default: hipLaunchKernelGGL((k_dec_conv_mfma<1, KF>), grid, dim3(256), 0, st, p); break;
    }
}

// MT: the largest of 4, 3, 2, 1 that divides the tile count (a block's
// tiles share each gathered B operand); a launch that would leave CUs idle
// even at MT = 1 (fewer than kDecFillBlocks blocks) splits K over the
// block's waves instead (k_dec_conv_mfma_ks); channel-first convolutions of
// 3 or more taps take k_dec_conv_win, of 2 where k_dec_conv_win_tw takes
// them.  QTTS_DEC_CONV=tiles or =split forces
// the long-decode kernels (MT by divisibility alone) or the K split for
// every launch, so that short decodes can check both against a reference.
bool launch_dec_conv_mfma(hipStream_t st, DecConvMfmaParams p) {
    const char *plan = std::getenv("QTTS_DEC_CONV");
    const bool force_tiles = plan && std::strcmp(plan, "tiles") == 0, force_split = plan && std::strcmp(plan, "split") == 0;
    const bool kf = p.sxc == 1 && p.cin % 8 == 0 && p.sxn % 4 == 0 && ((uintptr_t)p.x & 15) == 0;
    // m / up = umulhi(m, up_inv) while m * up < 2^32
    p.up_inv = p.up > 1 ? (unsigned)((1ull << 32) / (unsigned)p.up + 1) : 0;
    if (force_split ||
        (!force_tiles && (size_t)blocks_for((size_t)p.len, 128) * (size_t)p.mtiles < kDecFillBlocks)) {
        const dim3 grid(blocks_for(blocks_for((size_t)p.len, 32) * (size_t)p.mtiles, 8) * 8);
        if (kf)
            launch_conv_mfma_ks<true>(st, p, grid);
        else
            launch_conv_mfma_ks<false>(st, p, grid);
        return false;
    }
    int mt = p.mtiles % 4 == 0 ? 4 : p.mtiles % 3 == 0 ? 3 : p.mtiles % 2 == 0 ? 2 : 1;
    if (!force_tiles && (size_t)blocks_for((size_t)p.len, 128) * (size_t)(p.mtiles / mt) < 256) mt = 1;
    if (p.ksize >= (mt >= 3 ? 2 : 3) && p.sxn == 1 && p.sxc == p.len && 128 + (p.ksize - 1) * p.dilation <= 256) {
        // a channel-first convolution whose window fits the block's threads
        const dim3 grid(blocks_for((size_t)p.len, 128), (unsigned)(p.mtiles / mt));
        const dim3 flat(blocks_for((size_t)grid.x * grid.y, 8) * 8);
        p.quad = p.up > 1 && p.up % 4 == 0 && p.out_stride == p.up && p.ldc % 4 == 0 && p.epi == DEC_EPI_STORE &&
                 p.act == DEC_ACT_NONE && ((uintptr_t)p.c & 15) == 0;
        switch (mt) {
            case 4: hipLaunchKernelGGL(k_dec_conv_win_tw<4>, flat, dim3(256), 0, st, p); return true;
            case 3: hipLaunchKernelGGL(k_dec_conv_win_tw<3>, flat, dim3(192), 0, st, p); return true;
            case 2: hipLaunchKernelGGL(k_dec_conv_win<2>, grid, dim3(256), 0, st, p); break;
            default: hipLaunchKernelGGL(k_dec_conv_win<1>, grid, dim3(256), 0, st, p); break;
        }
        return false;
    }
    if (kf)
        launch_conv_mfma_kf<true>(st, p, mt);
    else
        launch_conv_mfma_kf<false>(st, p, mt);
    return false;
}

void launch_dec_absmax(hipStream_t st, const float *x, size_t n, unsigned *amax) {
    // at most 512 blocks: each folds its maximum into one of the 64 slots
    // with one atomic, so fewer blocks queue fewer atomics per slot
    const unsigned blocks = std::min<unsigned>(blocks_for((n + 3) / 4, 256), 512u);
    hipLaunchKernelGGL(k_dec_absmax, dim3(blocks), dim3(256), 0, st, x, n, amax);
}

// 3, 6 or 12 channel tiles (12 waves a block, conv2's operand 96 KiB of LDS)
// and a window of at most 64 positions before the block's.  C = 384, 80,000
// positions: 810 -> 565 us a unit, its weights read from the L2 for every 64
// positions; 768 channels would not fit the LDS.
bool dec_resunit_fits(int channels, int ksize1, int dilation, int ksize2) {
    return (channels == 96 || channels == 192 || channels == 384) && ksize1 == 7 && dilation >= 1 && dilation <= 10 && ksize2 == 1;
}

void launch_dec_resunit(hipStream_t st, const DecResUnitParams &p, int channels) {
    if (channels == 96)
        hipLaunchKernelGGL((k_dec_resunit<3, 12>), dim3(blocks_for((size_t)p.len, 256)), dim3(768), 0, st, p);
    else if (channels == 384)
        hipLaunchKernelGGL((k_dec_resunit<12, 12>), dim3(blocks_for((size_t)p.len, 64)), dim3(768), 0, st, p);
    else
        hipLaunchKernelGGL((k_dec_resunit<6, 12>), dim3(blocks_for((size_t)p.len, 128)), dim3(768), 0, st, p);
}

void launch_dec_exp(hipStream_t st, const float *x, float sign, int n, float *out) {
    hipLaunchKernelGGL(k_dec_exp, dim3(blocks_for((size_t)n, 256)), dim3(256), 0, st, x, sign, n, out);
}

}  // namespace qtts
