// Batched prompt processing ("prefill"): the decoder's matrix products for up to 1024
// tokens at once (128 through the product's own entry point), as a GEMM on the matrix cores.
// The reference has no such path -- it pushes the prompt through its batch-1 step one token at a time
// (wgml-chat/src/chat_llama2.rs:155-228 with the forced-token rule of
// wgml-chat/src/sampler.rs:102-107) -- so this is new functionality whose results are
// held against exactly that: N sequential decode steps.
//
//   out[t][r] = sum_k W[r][k] * X[t][k]      W: as stored for the GEMV (the kernels are in gemm_kernel.h)
//
// Activations are scaled per token by a power of two so that they stay in f16 range, products
// accumulate in fp32 on v_mfma_f32_16x16x32_f16.  Two precisions:
//   split f16 (default)  an activation is a pair of f16 numbers, hi = f16(v) and lo = f16(v - hi), scaled to
//                        512 < max |x| <= 1024 so that the low parts stay clear of the bottom of the f16
//                        range (the matrix cores take subnormal f16 inputs as they are); the weights'
//                        integers are exact, so the product is W X_hi + W X_lo: two MFMAs per term group
//                        (three for Q6_K), results to fp32 rounding (0.9e-7 to 2.4e-7 of their RMS, K = 512 .. 11008);
//   plain f16            the activations rounded to f16 once, one MFMA: about 2e-4 of a row's RMS (in runs
//                        of more than 128 tokens the weights are rounded once too: 3e-4).
//
// One launch can cover up to three matrices that multiply the same activations (Q, K
// and V; gate and up): their row tiles are numbered side by side.  A matrix too short to
// give every compute unit a tile has its K range split between ks workgroups; they leave
// partial sums that gemm_reduce_kernel adds in a fixed order (or, for a plain `x += W h`,
// the prep_x_kernel that reads x next).
//
// Activations are stored in the order the MFMA operand wants them (written by prep_x_kernel): for chunk
// c of 64 columns, token block n of NT, half s2 of the chunk, lane (g, j) finds the 8 halves
// X[16 n + j][64 c + 32 s2 + 8 g .. + 7] as one 16-byte word at word index
// ((c * NT + n) * 2 + s2) * 64 + 16 g + j: a chunk is NT x 2 KiB contiguous.  Behind them the sums of 32
// columns, for the formats with an offset per 32 weights: for unit u of 256 columns and token block n, word
// (u * NT + n) * 32 + 16 p + j holds the eight sums of token j as f16, part p (0: rounded, 1: what that left).
#include <hip/hip_fp16.h>

#include <type_traits>

#include "common.h"
#include "device_utils.h"
#include "gemm_args.h"

using namespace wgml;

namespace {

// p[0] + p[stride] + ..., n of them in this order, eight loads at a time (one by one they are a chain of trips to memory)
__device__ __forceinline__ float sum_of_parts(const float *p, size_t stride, uint32_t n) {
    float v = 0.f;
    uint32_t y = 0;
    for (; y + 8 <= n; y += 8) {
        float q[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) q[k] = p[(y + k) * stride];
#pragma unroll
        for (int k = 0; k < 8; ++k) v += q[k];
    }
    for (; y < n; ++y) v += p[y * stride];
    return v;
}

// out[t][r] (= or +=) xscale[t] * (part[0][t][r] + part[1][t][r] + ...) + bias[r]
__global__ __launch_bounds__(256) void gemm_reduce_kernel(const GemmArgs a) {
    const uint32_t rg = blockIdx.x * 256 + threadIdx.x, t = blockIdx.y;  // row among all matrices
    if (rg >= a.total_rows) return;
    uint32_t mi = 0;
    if (a.nmat > 1 && rg >= a.m[1].roff) mi = 1;
    if (a.nmat > 2 && rg >= a.m[2].roff) mi = 2;
    const GemmMat &m = a.m[mi];
    const uint32_t r = rg - m.roff;
    float v = sum_of_parts(a.part + (size_t)t * a.total_rows + rg, (size_t)a.T * a.total_rows, a.ks);
    v *= a.xscale ? a.xscale[t] : 1.f;
    if (m.bias) v += m.bias[r];
    float *o = m.out + (size_t)t * m.out_stride + r;
    *o = a.accumulate ? *o + v : v;
}

// The same for pairs of rows, with the rotary position encoding of the matrices marked for it
// (ops/rope.wgsl:35-78, the arithmetic of rope_rows_kernel below): thread (i, t) adds up the two
// rows of pair i of token t -- rows 2 i and 2 i + 1, or i' and i' + head_size / 2 within a head
// in the Neox variant -- and rotates them by the angle of position pos0 + t.  Every matrix of
// the launch has an even number of rows; nothing is accumulated onto the output.
__global__ __launch_bounds__(256) void gemm_reduce_rope_kernel(const GemmArgs a) {
    const uint32_t pg = blockIdx.x * 256 + threadIdx.x, t = blockIdx.y;  // pair among all matrices
    if (2 * pg >= a.total_rows) return;
    uint32_t mi = 0;
    if (a.nmat > 1 && 2 * pg >= a.m[1].roff) mi = 1;
    if (a.nmat > 2 && 2 * pg >= a.m[2].roff) mi = 2;
    const GemmMat &m = a.m[mi];
    const uint32_t i = pg - m.roff / 2, hs = a.rope_head_size;
    uint32_t ra = 2 * i, rb = 2 * i + 1;
    if (m.rope && a.rope_neox) {
        ra = i + (2 * i / hs) * (hs / 2);
        rb = ra + hs / 2;
    }
    const float *pa = a.part + (size_t)t * a.total_rows + m.roff + ra;
    const float *pb = a.part + (size_t)t * a.total_rows + m.roff + rb;
    float x = pa[0], y = pb[0];
    for (uint32_t k = 1; k < a.ks; ++k) {
        x += pa[(size_t)k * a.T * a.total_rows];
        y += pb[(size_t)k * a.T * a.total_rows];
    }
    const float xs_t = a.xscale ? a.xscale[t] : 1.f;
    x *= xs_t;
    y *= xs_t;
    if (m.bias) {
        x += m.bias[ra];
        y += m.bias[rb];
    }
    float *o = m.out + (size_t)t * m.out_stride;
    if (m.rope) {
        const float head_dim = (float)((i * 2) % hs);
        const float theta = powf(a.rope_base, -head_dim / (float)hs);
        float sn, cs;
        sincosf((float)(a.rope_pos0 + t) * theta, &sn, &cs);
        o[ra] = cs * x - sn * y;
        o[rb] = sn * x + cs * y;
    } else {
        o[ra] = x;
        o[rb] = y;
    }
}

// acc[n][0..7] += part[y .. y + B - 1][off[n] .. off[n] + 7], part by part in the order of y; the
// loads of all B parts are requested before the first sum (a chain of memory round trips
// otherwise).  ystride: floats from one part to the next.
template <int B, int N>
__device__ __forceinline__ void add_part_batch(float (&acc)[N][8], const float *__restrict__ part, size_t ystride,
                                               const size_t (&off)[N], uint32_t y) {
    float4 q[B][N][2];
#pragma unroll
    for (int b = 0; b < B; ++b) {
#pragma unroll
        for (int n = 0; n < N; ++n) {
            const float4 *p = reinterpret_cast<const float4 *>(part + (size_t)(y + b) * ystride + off[n]);
            q[b][n][0] = p[0];
            q[b][n][1] = p[1];
        }
    }
#pragma unroll
    for (int b = 0; b < B; ++b) {
#pragma unroll
        for (int n = 0; n < N; ++n) {
            acc[n][0] += q[b][n][0].x;
            acc[n][1] += q[b][n][0].y;
            acc[n][2] += q[b][n][0].z;
            acc[n][3] += q[b][n][0].w;
            acc[n][4] += q[b][n][1].x;
            acc[n][5] += q[b][n][1].y;
            acc[n][6] += q[b][n][1].z;
            acc[n][7] += q[b][n][1].w;
        }
    }
}
// all ks parts, eight (of one row), four, two or one at a time
template <int N>
__device__ __forceinline__ void add_parts(float (&acc)[N][8], const float *__restrict__ part, size_t ystride,
                                          const size_t (&off)[N], uint32_t ks) {
    uint32_t y = 0;
    if (N == 1)
        for (; y + 8 <= ks; y += 8) add_part_batch<8, N>(acc, part, ystride, off, y);
    for (; y + 4 <= ks; y += 4) add_part_batch<4, N>(acc, part, ystride, off, y);
    for (; y + 2 <= ks; y += 2) add_part_batch<2, N>(acc, part, ystride, off, y);
    for (; y < ks; ++y) add_part_batch<1, N>(acc, part, ystride, off, y);
}

__device__ __forceinline__ void load8(float (&o)[8], const float *p) {  // 16-byte aligned
    const float4 a = reinterpret_cast<const float4 *>(p)[0], b = reinterpret_cast<const float4 *>(p)[1];
    o[0] = a.x;
    o[1] = a.y;
    o[2] = a.z;
    o[3] = a.w;
    o[4] = b.x;
    o[5] = b.y;
    o[6] = b.z;
    o[7] = b.w;
}

// Token of workgroup w.  Eight neighbouring tokens share every 128-byte line of the packed activations (16 bytes each), and
// workgroup w runs on XCD w % 8: in runs of more than 64 tokens 8 i .. 8 i + 7 go to one XCD, whose L2 then writes whole
// lines; in the order of the tokens eight L2s write a sixteen-byte piece of each.  us per launch, in order / so: 1000 rows
// of 4096 to 14336 columns 36 -> 23, 128 rows 8.3 -> 7.7; 45 rows 5.8 / 5.9 (three XCDs have all the work).  A kernel of its
// own for each: the order chosen and workgroups beyond T ended at run time cost short runs 0.1 to 0.3 us of 4 to 5.
constexpr uint32_t kPrepInOrder = 64;
template <bool IN_ORDER>
__device__ __forceinline__ uint32_t prep_token(uint32_t w) {
    return IN_ORDER ? w : w / 64 * 64 + (w & 7) * 8 + (w / 8 & 7);
}

constexpr int PREP_THREADS = 1024;
constexpr int PREP_GROUPS = 2;  // groups of 8 columns a thread keeps in registers
// A form of its own for LayerNorm and for GELU: tested per element at run time they cost the other
// rows 3 % of a short prompt (8 layers of the 7B shape, 45 tokens in plain f16: 1620 us against 1574).
enum PrepMode { PREP_RMS, PREP_LN, PREP_GELU };
// Bound by its chain of one memory trip (row, partial sums and norm weights together), a reduction and
// a store: 7.7 us for 128 rows of 4096 that add four partial sums, 5.8 us for 21 rows of 3072 (9.5 and 6.4 with
// the weights requested after the first of two reductions).
// One workgroup per token: X[t] (fp32, optionally RMS-normalised with weights w as
// the reference does: (x * rsqrt(mean(x^2) + eps)) * w, ops/rms_norm.rs:55-63) -> f16
// in the packed order described at the top, times the power of two that brings the row's
// largest |x| into (512, 1024]; the factor to undo it goes to xscale[t].  Columns from K on are zero (tokens
// from T on hold anything: a token's results are its own).  With `up` non-null the input is the gated activation
// up[k] * silu(x[k]) (ops/silu.wgsl:13-27) instead of x itself (no normalisation then).
template <int MODE, bool IN_ORDER>
__global__ __launch_bounds__(PREP_THREADS) void prep_x_kernel(float *__restrict__ x, uint32_t x_stride,
                                                     const float *__restrict__ part, uint32_t part_ks,
                                                     uint32_t part_pair,
                                                     const float *__restrict__ up_or_beta,
                                                     const float *__restrict__ norm_w, float eps,
                                                     uint4 *__restrict__ xh, uint4 *__restrict__ xl,
                                                     _Float16 *__restrict__ xsum,
                                                     float *__restrict__ xscale, uint32_t K,
                                                     uint32_t kpad, uint32_t T, uint32_t nt) {
    __shared__ float red[32];
    const uint32_t t = prep_token<IN_ORDER>(blockIdx.x), tid = threadIdx.x;
    if (!IN_ORDER && t >= T) return;
    // 16-byte word of (token t, columns 8 k8 .. 8 k8 + 7)
    auto word_index = [&](uint32_t k8) {
        const uint32_t c = k8 >> 3, s2 = (k8 >> 2) & 1, g = k8 & 3;
        return (((size_t)c * nt + (t >> 4)) * 2 + s2) * 64 + 16 * g + (t & 15);
    };
    const uint32_t ngroups = kpad / 8;
    float *xr = x + (size_t)t * x_stride;
    // a LayerNorm has no gated rows: its beta comes in their place (an argument of its own made the
    // other form 3 % slower with the same instructions: 100 tokens, 4096 columns 7.7 us against 7.45)
    const float *const up = MODE == PREP_LN ? nullptr : up_or_beta;
    const float *ur = up ? up + (size_t)t * x_stride : nullptr;
    // Rows of up to 8 * PREP_GROUPS * PREP_THREADS columns are read once, 8 consecutive
    // columns per thread and group, and kept in registers (v); longer rows are re-read from
    // memory by the later passes.  (K is a multiple of 32 for every quantized format.)
    const bool cached = ngroups <= PREP_GROUPS * PREP_THREADS && K % 8 == 0 && x_stride % 4 == 0 &&
                        ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(up_or_beta) |
                          reinterpret_cast<uintptr_t>(norm_w) | reinterpret_cast<uintptr_t>(part)) & 15u) == 0;
    // (16-byte loads below)
    // the product before this kernel may have left  x[t] += xscale[t] * (part[0][t] + part[1][t]
    // + ...)  to be done here (part: [part_ks][T][K], xscale[t] still that product's factor)
    // With part_pair the partial sums are 2 K wide and hold a gate product in [0, K) and an up
    // product in [K, 2 K): the gated activation is formed from their sums, x and up are not
    // read (only for rows that fit the registers: the launcher sees to that).
    const float old_scale = part_ks ? xscale[t] : 0.f;
    if (part_ks && !cached) {
        for (uint32_t k = tid; k < K; k += PREP_THREADS) {
            const float *p = part + (size_t)t * K + k;
            float sum = p[0];
            for (uint32_t y = 1; y < part_ks; ++y) sum += p[(size_t)y * T * K];
            xr[k] += sum * old_scale;
        }
        __syncthreads();  // every thread reads what others wrote (same workgroup only)
    }
    float v[PREP_GROUPS][8];
    // the norm's weights, requested together with the row: after the reductions they would be one more
    // trip to memory
    const bool normed = MODE != PREP_GELU && norm_w;
    float nw[PREP_GROUPS][8], nb[PREP_GROUPS][8];
    if (cached && normed) {
#pragma unroll
        for (int i = 0; i < PREP_GROUPS; ++i) {
            const uint32_t k0 = 8 * (tid + i * PREP_THREADS);
#pragma unroll
            for (int e = 0; e < 8; ++e) nw[i][e] = nb[i][e] = 0.f;
            if (k0 >= K) continue;
            load8(nw[i], norm_w + k0);
            if (MODE == PREP_LN) load8(nb[i], up_or_beta + k0);
        }
    }
    auto raw = [&](uint32_t k) -> float {  // the value before normalisation
        if (k >= K) return 0.f;
        const float xv = xr[k];
        if (MODE == PREP_GELU) return gelu_tanh(xv);
        return ur ? ur[k] * (xv / (1.0f + expf(-xv))) : xv;
    };
    if (cached) {
#pragma unroll
        for (int i = 0; i < PREP_GROUPS; ++i) {
            const uint32_t k0 = 8 * (tid + i * PREP_THREADS);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[i][e] = 0.f;
            if (k0 < K && part_ks && part_pair) {
                const size_t wide = 2 * (size_t)K;
                float gu[2][8] = {};  // sums of the gate parts and of the up parts
                const size_t off[2] = {(size_t)t * wide + k0, (size_t)t * wide + K + k0};
                add_parts<2>(gu, part, (size_t)T * wide, off, part_ks);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float xv = gu[0][e] * old_scale;
                    v[i][e] = (gu[1][e] * old_scale) * (xv / (1.0f + expf(-xv)));
                }
            } else if (k0 < K) {
                float4 *xp = reinterpret_cast<float4 *>(xr + k0);
                float4 a0 = xp[0], a1 = xp[1];
                if (part_ks) {
                    float sp[1][8] = {};
                    const size_t off[1] = {(size_t)t * K + k0};
                    add_parts<1>(sp, part, (size_t)T * K, off, part_ks);
                    a0 = make_float4(a0.x + sp[0][0] * old_scale, a0.y + sp[0][1] * old_scale,
                                     a0.z + sp[0][2] * old_scale, a0.w + sp[0][3] * old_scale);
                    a1 = make_float4(a1.x + sp[0][4] * old_scale, a1.y + sp[0][5] * old_scale,
                                     a1.z + sp[0][6] * old_scale, a1.w + sp[0][7] * old_scale);
                    xp[0] = a0;
                    xp[1] = a1;
                }
                const float xv[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
                if (ur) {
                    const float4 *up4 = reinterpret_cast<const float4 *>(ur + k0);
                    const float4 u0 = up4[0], u1 = up4[1];
                    const float uv[8] = {u0.x, u0.y, u0.z, u0.w, u1.x, u1.y, u1.z, u1.w};
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[i][e] = uv[e] * (xv[e] / (1.0f + expf(-xv[e])));
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[i][e] = MODE == PREP_GELU ? gelu_tanh(xv[e]) : xv[e];
                }
            }
        }
    }
    float rs = 1.f, mean = 0.f;
    auto value = [&](uint32_t k, float r) { return normed && k < K ? (r * rs) * norm_w[k] : r; };  // not cached
    if (MODE == PREP_LN) {  // in registers only (the launcher sees to that)
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < PREP_GROUPS; ++i) {
#pragma unroll
            for (int e = 0; e < 8; ++e) sum += v[i][e];
        }
        mean = block_sum(sum, red) / (float)K;
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < PREP_GROUPS; ++i) {
            if (8 * (tid + i * PREP_THREADS) < K) {
#pragma unroll
                for (int e = 0; e < 8; ++e) ss = fmaf(v[i][e] - mean, v[i][e] - mean, ss);
            }
        }
        rs = 1.0f / sqrtf(block_sum(ss, red) / (float)K + eps);
    }
    float amax = 0.f;
    if (MODE == PREP_RMS && normed && cached) {
        // The sum of squares and the largest |x w| in one reduction: the factor between them is
        // positive and the same for the whole row, and only a power of two is taken from the largest value.
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < PREP_GROUPS; ++i) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                ss = fmaf(v[i][e], v[i][e], ss);
                amax = fmaxf(amax, fabsf(v[i][e] * nw[i][e]));
            }
        }
        ss = wave_sum(ss);
        amax = wave_max(amax);
        if ((tid & 63) == 0) {
            red[tid >> 6] = ss;
            red[16 + (tid >> 6)] = amax;
        }
        __syncthreads();
        ss = 0.f;
#pragma unroll
        for (int w = 0; w < PREP_THREADS / 64; ++w) {
            ss += red[w];
            amax = fmaxf(amax, red[16 + w]);
        }
        rs = 1.0f / sqrtf(ss / (float)K + eps);
        amax *= rs;
#pragma unroll
        for (int i = 0; i < PREP_GROUPS; ++i) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[i][e] = (v[i][e] * rs) * nw[i][e];
        }
    } else if (cached) {
#pragma unroll
        for (int i = 0; i < PREP_GROUPS; ++i) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                if (MODE == PREP_LN) v[i][e] = ((v[i][e] - mean) * rs) * nw[i][e] + nb[i][e];
                amax = fmaxf(amax, fabsf(v[i][e]));
            }
        }
        amax = block_max(amax, red);
    } else {
        if (normed) {
            float ss = 0.f;
            for (uint32_t k = tid; k < K; k += PREP_THREADS) ss = fmaf(xr[k], xr[k], ss);
            rs = 1.0f / sqrtf(block_sum(ss, red) / (float)K + eps);
        }
        for (uint32_t k = tid; k < K; k += PREP_THREADS) amax = fmaxf(amax, fabsf(value(k, raw(k))));
        amax = block_max(amax, red);
    }
    // the power of two that brings the largest value into (512, 1024], as far as 2^-120 .. 2^100 go
    int shift = 0;
    if (amax > 0.f) {
        const float f = frexpf(amax, &shift);  // f in [0.5, 1), shift 0 for infinities
        shift = amax <= 3.4028235e38f ? max(-120, min(100, 10 - shift + (f == 0.5f ? 1 : 0))) : -120;
    }
    const float down = ldexpf(1.f, shift), undo = ldexpf(1.f, -shift);
    // high parts f16(v); low parts f16(v - high) when the split-precision product is on
    auto store = [&](uint32_t k8, const float(&f)[8]) {
        _Float16 h[8], lo[8];
        float sum = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float v = f[e] * down;
            h[e] = (_Float16)v;
            lo[e] = (_Float16)(v - (float)h[e]);
            sum += (float)h[e] + (xl ? (float)lo[e] : 0.f);
        }
        uint4 w;
        __builtin_memcpy(&w, h, 16);
        xh[word_index(k8)] = w;
        if (xl) {
            __builtin_memcpy(&w, lo, 16);
            xl[word_index(k8)] = w;
        }
        // the sum of 32 columns (four neighbouring threads), in two parts
        sum += dpp_f32<0xB1>(sum);
        sum += dpp_f32<0x4E>(sum);
        if ((k8 & 3) == 0) {
            _Float16 *o = xsum + ((((size_t)(k8 >> 5) * nt + (t >> 4)) * 32 + (t & 15)) * 8 + ((k8 >> 2) & 7));
            const _Float16 sh = (_Float16)sum;
            o[0] = sh;
            o[16 * 8] = (_Float16)(sum - (float)sh);
        }
    };
    if (cached) {
#pragma unroll
        for (int i = 0; i < PREP_GROUPS; ++i) {
            const uint32_t k8 = tid + i * PREP_THREADS;
            if (k8 < ngroups) store(k8, v[i]);
        }
    } else {
        for (uint32_t k8 = tid; k8 < ngroups; k8 += PREP_THREADS) {
            float f[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] = value(8 * k8 + e, raw(8 * k8 + e));
            store(k8, f);
        }
    }
    if (tid == 0) xscale[t] = undo;
}

// X[t] = table[tokens[t]]  (embedding rows of the prompt tokens)
// pos_table (GPT-2's learned positions): the row of position pos0 + t is added.
__global__ void embed_rows_kernel(float *__restrict__ x, const float *__restrict__ table,
                                  const uint32_t *__restrict__ tokens, uint32_t dim,
                                  const float *__restrict__ pos_table, uint32_t pos0) {
    const uint32_t t = blockIdx.y, i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= dim) return;
    float v = table[(size_t)tokens[t] * dim + i];
    if (pos_table) v += pos_table[(size_t)(pos0 + t) * dim + i];
    x[(size_t)t * dim + i] = v;
}

// Rows of q, k and v side by side (3 n wide, n a multiple of 4): k and v of token t to its cache rows.
__global__ void cache_rows_kernel(const float *__restrict__ qkv, float *__restrict__ k, float *__restrict__ v,
                                  uint32_t n) {
    const uint32_t t = blockIdx.y, i = (blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (i >= 2 * n) return;
    const float4 w = *reinterpret_cast<const float4 *>(qkv + (size_t)t * 3 * n + n + i);
    *reinterpret_cast<float4 *>((i < n ? k + i : v + (i - n)) + (size_t)t * n) = w;
}

// RoPE of q[t] and of the K-cache row of position pos0 + t, for every token t
// (the arithmetic of rope_kernel in ops.hip; ops/rope.wgsl:35-78 of the reference).
__global__ void rope_rows_kernel(float *__restrict__ q, uint32_t q_stride, float *__restrict__ k,
                                 uint32_t k_stride, uint32_t n_pairs, uint32_t head_size,
                                 uint32_t kv_dim, uint32_t pos0, float base_freq, int neox) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x, t = blockIdx.y;
    if (i >= n_pairs) return;
    const uint32_t p = pos0 + t;
    float *qt = q + (size_t)t * q_stride, *kt = k + (size_t)t * k_stride;
    const float head_dim = (float)((i * 2) % head_size);
    const float theta = powf(base_freq, -head_dim / (float)head_size);
    float sn, cs;
    sincosf((float)p * theta, &sn, &cs);
    uint32_t a, b;
    if (!neox) {
        a = i * 2;
        b = a + 1;
    } else {
        const uint32_t head_id = (i * 2) / head_size;
        a = i + head_id * head_size / 2;
        b = a + head_size / 2;
    }
    if (q) {
        const float x = qt[a], y = qt[b];
        qt[a] = cs * x - sn * y;
        qt[b] = sn * x + cs * y;
    }
    if (k && i * 2 < kv_dim) {
        const float x = kt[a], y = kt[b];
        kt[a] = cs * x - sn * y;
        kt[b] = sn * x + cs * y;
    }
}


// Causal attention for a run of tokens: workgroup (h, t) computes head h of token t,
// which sits at position pos0 + t and attends to cache rows 0 .. pos0 + t (the rows of
// this run were written by the K and V products before).  Same arithmetic as the decode
// kernels (ops/batched_multiquery_attention.wgsl:24-97: scores q.k / sqrt(head_size),
// softmax, weighted sum of values), as an online softmax: 16 lanes share a position,
// a wave covers four positions at a time, the four waves stride over the positions.
struct AttnRowsArgs {
    const float *q;  // [T][q_stride]
    const float *kc, *vc;  // caches: rows kv_dim apart
    float *xb;  // [T][xb_stride]
    uint32_t q_stride, xb_stride, kv_dim, kv_mul, head_size, pos0;
};

__device__ __forceinline__ float dot4f(const float4 a, const float4 b, float acc) {
    acc = fmaf(a.x, b.x, acc);
    acc = fmaf(a.y, b.y, acc);
    acc = fmaf(a.z, b.z, acc);
    return fmaf(a.w, b.w, acc);
}
__device__ __forceinline__ float4 axpby4f(const float4 a, float sa, const float4 b, float sb) {
    return make_float4(fmaf(a.x, sa, b.x * sb), fmaf(a.y, sa, b.y * sb), fmaf(a.z, sa, b.z * sb),
                       fmaf(a.w, sa, b.w * sb));
}

template <int NV4>
__global__ __launch_bounds__(256) void attn_rows_kernel(const AttnRowsArgs a) {
    constexpr int HSP = NV4 * 64;
    __shared__ float sm_m[4], sm_l[4];
    __shared__ float sm_acc[4][HSP];
    const uint32_t h = blockIdx.x, t = blockIdx.y, pos = a.pos0 + t;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t sub = lane & 15, quarter = lane >> 4, hs = a.head_size;
    const float *kb = a.kc + (size_t)(h / a.kv_mul) * hs;
    const float *vb = a.vc + (size_t)(h / a.kv_mul) * hs;
    const float inv_sqrt_hs = 1.0f / sqrtf((float)hs);
    // float4 number sub + 16 v of the head; lanes beyond the head re-read its last one
    // with a zero q and never store
    uint32_t cv[NV4];
    float4 q[NV4], acc[NV4];
#pragma unroll
    for (int v = 0; v < NV4; ++v) {
        const bool inside = (sub + 16 * v) * 4 < hs;
        cv[v] = min(sub + 16 * v, hs / 4 - 1);
        const float4 qv =
            reinterpret_cast<const float4 *>(a.q + (size_t)t * a.q_stride + (size_t)h * hs)[cv[v]];
        q[v] = inside ? qv : make_float4(0.f, 0.f, 0.f, 0.f);
        acc[v] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    float mx = -INFINITY, l = 0.f;
    for (uint32_t p0 = wave * 4; p0 <= pos; p0 += 16) {  // uniform over the wave
        const uint32_t tt = p0 + quarter;
        const uint32_t tc = min(tt, pos);
        const float4 *kp = reinterpret_cast<const float4 *>(kb + (size_t)tc * a.kv_dim);
        const float4 *vp = reinterpret_cast<const float4 *>(vb + (size_t)tc * a.kv_dim);
        float4 kk[NV4], vv[NV4];
#pragma unroll
        for (int v = 0; v < NV4; ++v) kk[v] = kp[cv[v]];
#pragma unroll
        for (int v = 0; v < NV4; ++v) vv[v] = vp[cv[v]];
        float part = 0.f;
#pragma unroll
        for (int v = 0; v < NV4; ++v) part = dot4f(q[v], kk[v], part);
        const float s = row16_sum(part) * inv_sqrt_hs;
        if (tt <= pos) {  // uniform within a 16-lane row
            const float mn = fmaxf(mx, s);
            const float sc = __expf(mx - mn), p = __expf(s - mn);
            l = fmaf(l, sc, p);
#pragma unroll
            for (int v = 0; v < NV4; ++v) acc[v] = axpby4f(acc[v], sc, vv[v], p);
            mx = mn;
        }
    }
    // the four quarters of the wave
#pragma unroll
    for (int step = 16; step <= 32; step <<= 1) {
        const float om = __shfl_xor(mx, step, 64), ol = __shfl_xor(l, step, 64);
        const float M = fmaxf(mx, om);
        const float sa = mx == -INFINITY ? 0.f : __expf(mx - M);
        const float sb = om == -INFINITY ? 0.f : __expf(om - M);
        l = fmaf(l, sa, ol * sb);
#pragma unroll
        for (int v = 0; v < NV4; ++v) {
            float4 o;
            o.x = __shfl_xor(acc[v].x, step, 64);
            o.y = __shfl_xor(acc[v].y, step, 64);
            o.z = __shfl_xor(acc[v].z, step, 64);
            o.w = __shfl_xor(acc[v].w, step, 64);
            acc[v] = axpby4f(acc[v], sa, o, sb);
        }
        mx = M;
    }
    // the four waves
    if (lane == 0) {
        sm_m[wave] = mx;
        sm_l[wave] = l;
    }
    if (quarter == 0) {
#pragma unroll
        for (int v = 0; v < NV4; ++v) reinterpret_cast<float4 *>(&sm_acc[wave][0])[sub + 16 * v] = acc[v];
    }
    __syncthreads();
    for (uint32_t d = threadIdx.x; d < hs; d += 256) {
        const float M = fmaxf(fmaxf(sm_m[0], sm_m[1]), fmaxf(sm_m[2], sm_m[3]));
        float L = 0.f, o = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float wgt = sm_m[w] == -INFINITY ? 0.f : __expf(sm_m[w] - M);
            L = fmaf(sm_l[w], wgt, L);
            o = fmaf(wgt > 0.f ? sm_acc[w][d] : 0.f, wgt, o);
        }
        a.xb[(size_t)t * a.xb_stride + (size_t)h * hs + d] = o / L;
    }
}

// The same attention for 16 tokens of a run at once, on the fp32 matrix cores
// (v_mfma_f32_16x16x4_f32: operands and sums are fp32, so the arithmetic stays that of the
// step).  Workgroup (h, tb) computes head h of tokens 16 tb .. 16 tb + 15; its four waves
// share out the blocks of 16 cache rows and merge at the end, so a K or V row is read once
// per 16 tokens instead of once per token.  Per block of rows, with lane = (g, n):
//   S^T[row][token] = K · Q^T : A = K rows (lane n = row, k-slot g = dimension 16 c + 4 g + e in
//                     step (c, e)), B = Q^T (lane n = token), 4 HS16 steps -> each lane holds
//                     the scores of rows 4 g + i (i < 4) for token n;
//   online softmax per token: maximum and sum over the lane's 4 rows and the 4 lane groups;
//   O^T[dim][token] += V^T · P^T : A = V^T (lane n = dimension 16 b + n, k-slot g = row 4 g + i
//                     in step i), B = the lane's own P values -- no transposition anywhere.
// Both operands are loaded as they lie in memory.  A row of K belongs to lanes n, n + 16, ..., and loads in that order are 64
// pieces of 16 bytes: a wave brings its block in whole rows and turns it in LDS, in a place of its own (no barriers; KS keeps
// the sixteen rows of a read on different banks).  The products of PV take their dimensions so that a lane's are neighbours: one
// load of V for four products.  V is requested before the scores, the next block of K behind them.  us per launch, both in
// operand order -> so: 1000 tokens, 32 heads of 128 140 -> 106; 200 behind 1900 130 -> 92; 401 behind 1500 (32 heads of 64)
// 93 -> 80; 700 behind 100 (20 of 96) 50 -> 41; 128 9.5 -> 8.7; in eight waves 45 behind 300 17.9 -> 13.5, 21 behind 600 (24
// heads) 25 -> 18.5.  Bound by the fp32 MFMAs, 57 of those 106 us, and by a wave's vector instructions beside them.
// Three waves per SIMD, or four where the registers of a smaller head let them: 106 us, with two 117.
// WAVES 4: several workgroups fit a compute unit and cover each other's waits.  WAVES 8, where there are fewer
// workgroups than compute units (a short run behind a long context): twice the waves share the cache rows.
template <int HS16, int WAVES>
__global__ __launch_bounds__(WAVES * 64) __attribute__((amdgpu_waves_per_eu(HS16 > 5 ? 3 : 4))) void attn_block_kernel(const AttnRowsArgs a, uint32_t T) {
    constexpr int HS = HS16 * 16, KS = HS + 4;                      // KS: floats of a staged row of K
    constexpr int VW = HS16 % 4 == 0 ? 4 : HS16 % 2 == 0 ? 2 : 1;  // floats of V per load
    constexpr int STAGE = 16 * KS, MERGE = HS * 17, PER_WAVE = STAGE > MERGE ? STAGE : MERGE;
    typedef float vrow_t __attribute__((ext_vector_type(VW)));
    __shared__ float sm_m[WAVES][16], sm_l[WAVES][16];
    __shared__ __attribute__((aligned(16))) float sm[WAVES][PER_WAVE];  // a wave's block of K, then its results
    // the heads in eight groups, one on each XCD, and the longest workgroups first
    const uint32_t h = gridDim.x % 8 ? blockIdx.x : (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
    const uint32_t t0 = (gridDim.y - 1 - blockIdx.y) * 16;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t n = lane & 15, g = lane >> 4;
    const size_t head_off = (size_t)(h / a.kv_mul) * HS;
    const float inv_sqrt_hs = 1.0f / sqrtf((float)HS);
    // this lane's token (the B operand of the score product); tokens past the run repeat the last
    const uint32_t tq = min(t0 + n, T - 1), pos_q = a.pos0 + tq;
    const uint32_t last_pos = a.pos0 + min(t0 + 15, T - 1);  // rows 0 .. last_pos exist
    const uint32_t nblk = last_pos / 16 + 1;
    const uint32_t kv_bytes = a.kv_dim * 4;
    // a block of K as it lies in memory: 16-byte word 64 c + lane of its 16 rows
    floatx4 k[HS16];
    auto load_k = [&](uint32_t blk) {  // rows past the end repeat the last one and do not count
        const char *base = reinterpret_cast<const char *>(a.kc + (size_t)blk * 16 * a.kv_dim + head_off);
        const uint32_t last = last_pos - blk * 16;
#pragma unroll
        for (int c = 0; c < HS16; ++c) {
            const uint32_t w = 64 * c + lane, row = w / (HS / 4), col = w % (HS / 4) * 16;
            k[c] = *reinterpret_cast<const floatx4 *>(base + (min(row, last) * kv_bytes + col));
        }
    };
    // V^T: lane n has VW neighbouring dimensions of row 4 g + i, one for each of VW products
    vrow_t v[HS16 / VW][4];
    auto load_v = [&](uint32_t blk) {
        const char *base = reinterpret_cast<const char *>(a.vc + (size_t)blk * 16 * a.kv_dim + head_off);
        const uint32_t last = last_pos - blk * 16;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t at = min(4 * g + i, last) * kv_bytes + 4 * VW * n;
#pragma unroll
            for (int j = 0; j < HS16 / VW; ++j) v[j][i] = *reinterpret_cast<const vrow_t *>(base + at + 64 * VW * j);
        }
    };
    load_k(min(wave, nblk - 1));
    float4 q[HS16];
#pragma unroll
    for (int c = 0; c < HS16; ++c)
        q[c] = *reinterpret_cast<const float4 *>(a.q + (size_t)tq * a.q_stride + (size_t)h * HS + 16 * c + 4 * g);
    floatx4 acc[HS16];
#pragma unroll
    for (int b = 0; b < HS16; ++b) acc[b] = floatx4{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    for (uint32_t blk = wave; blk < nblk; blk += WAVES) {  // uniform over the wave
        const uint32_t pbase = blk * 16;
#pragma unroll
        for (int c = 0; c < HS16; ++c) {
            const uint32_t w = 64 * c + lane, row = w / (HS / 4), col = w % (HS / 4) * 4;
            *reinterpret_cast<floatx4 *>(&sm[wave][row * KS + col]) = k[c];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // (the wave's own rows: no barrier)
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        load_v(blk);
        __builtin_amdgcn_sched_barrier(0);  // requested before the products, not between them
        floatx4 s = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < HS16; ++c) {
            const float4 kf = *reinterpret_cast<const float4 *>(&sm[wave][n * KS + 16 * c + 4 * g]);
            s = __builtin_amdgcn_mfma_f32_16x16x4f32(kf.x, q[c].x, s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_16x16x4f32(kf.y, q[c].y, s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_16x16x4f32(kf.z, q[c].z, s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_16x16x4f32(kf.w, q[c].w, s, 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        load_k(min(blk + WAVES, nblk - 1));
        __builtin_amdgcn_sched_barrier(0);
        // s[i] = score of row pbase + 4 g + i for token n; rows after the token's position do not count
        float sc[4], mloc = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            sc[i] = pbase + 4 * g + i <= pos_q ? s[i] * inv_sqrt_hs : -INFINITY;
            mloc = fmaxf(mloc, sc[i]);
        }
        mloc = fmaxf(mloc, __shfl_xor(mloc, 16, 64));
        mloc = fmaxf(mloc, __shfl_xor(mloc, 32, 64));
        const float mn = fmaxf(m, mloc);
        const float scale = mn == -INFINITY ? 1.f : __expf(m - mn);
        float p[4], lsum = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            p[i] = sc[i] == -INFINITY ? 0.f : __expf(sc[i] - mn);
            lsum += p[i];
        }
        lsum += __shfl_xor(lsum, 16, 64);
        lsum += __shfl_xor(lsum, 32, 64);
        l = fmaf(l, scale, lsum);
        m = mn;
#pragma unroll
        for (int b = 0; b < HS16; ++b) {
            acc[b] = floatx4{acc[b][0] * scale, acc[b][1] * scale, acc[b][2] * scale, acc[b][3] * scale};
#pragma unroll
            for (int i = 0; i < 4; ++i)
                acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[b / VW][i][b % VW], p[i], acc[b], 0, 0, 0);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    // acc[b][i] = O^T[dimension dim(b, i)][token n] of this wave's rows; merge the waves, eight of
    // them in two steps (wave w takes up wave w + 4 first)
    auto dim = [&](int b, int i) { return 16 * VW * (b / VW) + VW * (4 * g + i) + b % VW; };
    auto leave = [&]() {
        if (g == 0) {
            sm_m[wave][n] = m;
            sm_l[wave][n] = l;
        }
#pragma unroll
        for (int b = 0; b < HS16; ++b) {
#pragma unroll
            for (int i = 0; i < 4; ++i) sm[wave][dim(b, i) * 17 + n] = acc[b][i];
        }
    };
    if (WAVES == 8) {
        if (wave >= 4) leave();
        __syncthreads();
        if (wave < 4) {
            const float m2 = sm_m[wave + 4][n], l2 = sm_l[wave + 4][n], mn = fmaxf(m, m2);
            const float s1 = m == -INFINITY ? 0.f : __expf(m - mn), s2 = m2 == -INFINITY ? 0.f : __expf(m2 - mn);
#pragma unroll
            for (int b = 0; b < HS16; ++b) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    acc[b][i] = fmaf(acc[b][i], s1, sm[wave + 4][dim(b, i) * 17 + n] * s2);
            }
            l = fmaf(l, s1, l2 * s2);
            m = mn;
        }
    }
    if (wave < 4) leave();
    __syncthreads();
    for (uint32_t idx = threadIdx.x; idx < 16 * HS; idx += WAVES * 64) {
        const uint32_t tok = idx / HS, d = idx % HS;
        if (t0 + tok >= T) continue;
        const float M = fmaxf(fmaxf(sm_m[0][tok], sm_m[1][tok]), fmaxf(sm_m[2][tok], sm_m[3][tok]));
        float L = 0.f, o = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float wgt = sm_m[w][tok] == -INFINITY ? 0.f : __expf(sm_m[w][tok] - M);
            L = fmaf(sm_l[w][tok], wgt, L);
            o = fmaf(sm[w][d * 17 + tok], wgt, o);
        }
        a.xb[(size_t)(t0 + tok) * a.xb_stride + (size_t)h * HS + d] = o / L;
    }
}



// T tokens as `tiles` tiles of `nt` blocks of 16: one tile of 1, 2, 3, 4, 6 or 8 blocks for up to 128
// tokens, tiles of 256 beyond.
void token_blocks(uint32_t T, uint32_t *tiles, uint32_t *nt) {
    const uint32_t n = (T + 15) / 16;
    *tiles = T <= kPrefillMaxTokens ? 1 : (T + TILE_TOKENS - 1) / TILE_TOKENS;
    *nt = T > kPrefillMaxTokens ? TILE_TOKENS / 16 : n == 5 ? 6 : n == 7 ? 8 : n;
}

template <int HS16>
void launch_attn_block(wgml_ctx *ctx, const AttnRowsArgs &a, uint32_t n_heads, uint32_t T, bool few) {
    const dim3 grid(n_heads, (T + 15) / 16);
    if (few)
        attn_block_kernel<HS16, 8><<<grid, dim3(512), 0, ctx->stream>>>(a, T);
    else
        attn_block_kernel<HS16, 4><<<grid, dim3(256), 0, ctx->stream>>>(a, T);
}

// How many workgroups share the K range of a row tile.
//   up to 128 tokens: several workgroups fit a compute unit and what a short product waits for is the
//   first bytes of each, so K is split into about 448 workgroups of the same number of units (256, 320,
//   384, 512, 600 instead: 0-6 % slower over a pass of 4 .. 128 tokens through the 7B shape, 3072 x 8192 and
//   768 x 2048; workgroups of one unit each up to 40 %).
//   Where the partial sums take a launch of their own (nothing behind the product adds or rotates its rows), no more than
//   pays: with T = 16 nt tokens a unit takes about 0.2 + 0.5 nt us (Q4_0 .. Q5_1, whose blocks come in pieces, 1.4 + 0.5 nt), the
//   launch 3.1 - 0.25 nt, a part 0.09 and 1.5 (1 + nt) ns per tile, and workgroups that share a compute unit slow each other by a
//   third (fitted to 1, 16, 45 and 128 tokens, 16 .. 4096 rows, 512 .. 65536 columns, Q8_0 and Q4_K, ks from 1 to 256: 1.1 % above
//   the best ks on average, 20 % at most).  Against 448 workgroups here too, one vector: 256 x 512 in Q8_0 11.9 us -> 9.2,
//   256 x 16384 26.7 -> 17.4; 128 vectors 40.1 -> 28.8.
//   longer runs: one workgroup per compute unit; the ks with the least time in units of K, one unit per
//   round of the grid for its start, end and results.
constexpr size_t kTilePartBytes = size_t(128) << 20;
uint32_t gemm_k_split(const wgml_ctx *ctx, int type, uint32_t tiles, uint32_t units, uint32_t nt, bool tall,
                      bool own_launch, size_t part_bytes) {
    const int forced = ctx->tuning[WGML_TUNE_GEMM_K_SPLIT];
    if (forced) return min((uint32_t)forced, units);
    const uint32_t cu = ctx->n_cu > 0 ? (uint32_t)ctx->n_cu : 256u;
    uint32_t best = 1;
    float best_cost = 1e30f;
    if (!tall) {
        const uint32_t want = 448, per = max(1u, (units * tiles + want / 2) / want);
        const uint32_t most = per >= units ? 1 : (units + per - 1) / per;
        if (!own_launch) return most;
        const bool pieces = type == WGML_Q4_0 || type == WGML_Q4_1 || type == WGML_Q5_0 || type == WGML_Q5_1;
        const float unit = (pieces ? 1.4f : 0.2f) + 0.5f * (float)nt;
        const float part = 0.09f + 1.5e-3f * (float)(tiles * (1 + nt));
        for (uint32_t ks = 1; ks <= most; ++ks) {
            const float shared = tiles * ks > cu ? (float)(tiles * ks - cu) / (float)cu : 0.f;
            const float cost = (float)((units + ks - 1) / ks) * unit * (1.f + 0.35f * shared) +
                               (ks > 1 ? 3.1f - 0.25f * (float)nt + (float)ks * part : 0.f);
            if (cost < best_cost) {
                best_cost = cost;
                best = ks;
            }
        }
        return best;
    }
    for (uint32_t ks = 1; ks <= 8 && ks <= units && (ks == 1 || ks * part_bytes <= kTilePartBytes); ++ks) {
        const float cost = (float)((tiles * ks + cu - 1) / cu) * ((float)((units + ks - 1) / ks) + 1.f);
        if (cost < best_cost) {
            best_cost = cost;
            best = ks;
        }
    }
    return best;
}

}  // namespace

namespace wgml {

uint32_t prefill_tpad(uint32_t T) {
    uint32_t tiles, nt;
    token_blocks(T, &tiles, &nt);
    return tiles * nt * 16;
}
uint32_t prefill_kpad(uint32_t K) { return (K + KU - 1) / KU * KU; }

bool gemm_supported(const wgml_qmat *q) {
    return q->type != WGML_F32 && gemv_fused_supported(q) && q->max_abs <= kGemmMaxWeight;  // the nine quantized formats
}

// The kernels address the rows of a tile in a plane with 32-bit offsets: at most 1 byte per element, but 292 per 256 in Q8_K,
// which matters to tiles of 2^32 bytes only.
bool gemm_addressable(const wgml_qmat *q) {
    constexpr uint64_t limit = (uint64_t(1) << 32) - 4096;
    const uint64_t rows = q->nrows < TILE_ROWS ? q->nrows : TILE_ROWS;
    return (uint64_t)q->nrows * q->ncols < limit && (q->type != WGML_Q8_K || rows * (q->ncols / 256) * 292 < limit);
}

// hipMalloc for a workspace: callers with a path that needs none of it go on with that where the
// memory is missing (WGML_E_OOM), and only there.
static int workspace_alloc(void **p, size_t bytes) {
    const hipError_t e = hipMalloc(p, bytes);
    if (e == hipSuccess) return WGML_OK;
    (void)hipGetLastError();  // not the next launch's error
    *p = nullptr;
    return set_error(WGML_E_OOM, "prompt workspace: hipMalloc(%zu) failed: %s", bytes, hipGetErrorString(e));
}

int ensure_prefill_scratch(wgml_ctx *ctx, size_t xh_bytes) {
    if (!ctx->prefill_xscale)
        WGML_TRY(workspace_alloc((void **)&ctx->prefill_xscale, kPrefillMaxRun * sizeof(float)));
    if (xh_bytes <= ctx->prefill_xh_bytes) return WGML_OK;
    xh_bytes = (xh_bytes + 255) & ~(size_t)255;
    // three arrays: the f16 activations, their low parts (split precision) and the sums of 32 of them
    void *xh = nullptr;
    WGML_TRY(workspace_alloc(&xh, 2 * xh_bytes + xh_bytes / 16));  // without it the old buffer stays in use
    // work already enqueued may still read the old buffer: retire it, free with the context
    if (ctx->prefill_xh) ctx->retired.push_back(ctx->prefill_xh);
    ctx->prefill_xh = xh;
    ctx->prefill_xl = (char *)ctx->prefill_xh + xh_bytes;
    ctx->prefill_xsum = (char *)ctx->prefill_xl + xh_bytes;
    ctx->prefill_xh_bytes = xh_bytes;
    return WGML_OK;
}

int launch_prefill_prep(wgml_ctx *ctx, float *x, uint32_t x_stride, const float *up,
                        const float *norm_w, float eps, void *xh, float *xscale, uint32_t K,
                        uint32_t T, const float *ln_beta, int gelu) {
    if (ln_beta && !(norm_w && !up && K % 8 == 0 && x_stride % 4 == 0 &&
                     prefill_kpad(K) / 8 <= (uint32_t)(PREP_GROUPS * PREP_THREADS) &&
                     (reinterpret_cast<uintptr_t>(x) & 15u) == 0))
        return set_error(WGML_E_UNSUPPORTED, "prefill_prep: LayerNorm of rows of %u columns", K);
    // partial sums a product with defer_reduce left: for x (K wide; x is its output), or for a
    // gate / up pair (2 K wide; x and up are then not read)
    const uint32_t pending = ctx->gemm_pending_ks, pair = ctx->gemm_pending_pair;
    ctx->gemm_pending_ks = 0;
    ctx->gemm_pending_pair = 0;
    if (pending && pair &&
        !(up && K % 8 == 0 && x_stride % 4 == 0 && prefill_kpad(K) / 8 <= (uint32_t)(PREP_GROUPS * PREP_THREADS) &&
          ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(up)) & 15u) == 0))
        return set_error(WGML_E_INVALID, "prefill_prep: pending gate/up partial sums need a gated row of at "
                                         "most %d columns", 8 * PREP_GROUPS * PREP_THREADS);
    const bool in_order = T <= kPrepInOrder;
    const auto kernel = ln_beta ? (in_order ? prep_x_kernel<PREP_LN, true> : prep_x_kernel<PREP_LN, false>)
                        : gelu  ? (in_order ? prep_x_kernel<PREP_GELU, true> : prep_x_kernel<PREP_GELU, false>)
                                : (in_order ? prep_x_kernel<PREP_RMS, true> : prep_x_kernel<PREP_RMS, false>);
    // (whole rounds of the eight XCDs, see prep_token; workgroups beyond T end at once)
    kernel<<<dim3(in_order ? T : (T + 63) / 64 * 64), dim3(PREP_THREADS), 0, ctx->stream>>>(
        x, x_stride, pending ? ctx->gemm_part : nullptr, pending, pair, ln_beta ? ln_beta : up, norm_w, eps,
        reinterpret_cast<uint4 *>(xh), ctx->gemm_precise ? reinterpret_cast<uint4 *>(ctx->prefill_xl) : nullptr,
        reinterpret_cast<_Float16 *>(ctx->prefill_xsum), xscale, K, prefill_kpad(K), T, prefill_tpad(T) / 16);
    WGML_CHECK_LAUNCH();
    ctx->launches++;
    return WGML_OK;
}

// x[t] += the partial sums a product with defer_reduce left, for callers whose next
// kernel is not launch_prefill_prep.
__global__ void gemm_flush_kernel(float *x, uint32_t x_stride, const float *part, uint32_t ks,
                                  const float *xscale, uint32_t K, uint32_t T) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x, t = blockIdx.y;
    if (k >= K) return;
    const float *p = part + (size_t)t * K + k;
    float sum = p[0];
    for (uint32_t y = 1; y < ks; ++y) sum += p[(size_t)y * T * K];
    x[(size_t)t * x_stride + k] += sum * xscale[t];
}

int launch_gemm_flush(wgml_ctx *ctx, float *x, uint32_t x_stride, const float *xscale, uint32_t K,
                      uint32_t T) {
    const uint32_t pending = ctx->gemm_pending_ks;
    ctx->gemm_pending_ks = 0;
    if (!pending) return WGML_OK;
    gemm_flush_kernel<<<dim3((K + 255) / 256, T), dim3(256), 0, ctx->stream>>>(x, x_stride, ctx->gemm_part,
                                                                          pending, xscale, K, T);
    WGML_CHECK_LAUNCH();
    ctx->launches++;
    return WGML_OK;
}

int ensure_gemm_partials(wgml_ctx *ctx, size_t bytes) {
    if (bytes <= ctx->gemm_part_bytes) return WGML_OK;
    // Old buffers stay until the context goes (queued work, or a graph the caller recorded, may read
    // them), so each is at least twice the one before, up to what a long run takes at most: together
    // they are no larger than the last.
    constexpr size_t kStep = size_t(8) << 20, kUsual = kTilePartBytes + kStep;
    // (half a MiB for the products of small models: K is split there too)
    const size_t need = bytes <= kStep / 16 ? kStep / 16 : (bytes + kStep) & ~((size_t(1) << 20) - 1);
    size_t size = need > 2 * ctx->gemm_part_bytes ? need : 2 * ctx->gemm_part_bytes;
    if (size > kUsual) size = need > kUsual ? need : kUsual;
    float *part = nullptr;
    int rc = workspace_alloc((void **)&part, size);
    if (rc != WGML_OK && size > need) rc = workspace_alloc((void **)&part, size = need);
    WGML_TRY(rc);  // without it the old buffer stays in use
    if (ctx->gemm_part) ctx->retired.push_back(ctx->gemm_part);
    ctx->gemm_part = part;
    ctx->gemm_part_bytes = size;
    return WGML_OK;
}

int launch_gemm_quant_multi(wgml_ctx *ctx, const GemmTarget *targets, int n, const void *xh,
                            const float *xscale, uint32_t T, int accumulate, bool defer_reduce,
                            GemmRope *rope) {
    if (T == 0 || T > kPrefillMaxRun)
        return set_error(WGML_E_INVALID, "gemm_quant: %u tokens (1..%u)", T, kPrefillMaxRun);
    const bool tall = T > kPrefillMaxTokens;
    const uint32_t tile_rows = tall ? TILE_ROWS : 64;
    if (n < 1 || n > 3) return set_error(WGML_E_INVALID, "gemm_quant: %d matrices (1..3)", n);
    const wgml_qmat *first = targets[0].m;
    GemmArgs a{};
    uint32_t tiles = 0;
    for (int i = 0; i < n; ++i) {
        const wgml_qmat *q = targets[i].m;
        if (q->type != first->type || q->ncols != first->ncols)
            return set_error(WGML_E_INVALID, "gemm_quant: matrices of one launch differ in format or width");
        if (!(q->max_abs <= kGemmMaxWeight))
            return set_error(WGML_E_UNSUPPORTED,
                             "gemm_quant: a weight of magnitude up to %g does not fit the f16 operands of "
                             "the batched product (up to %g only); use the per-token product",
                             (double)q->max_abs, (double)kGemmMaxWeight);
        if (!gemm_addressable(q))
            return set_error(WGML_E_UNSUPPORTED, "gemm_quant: a matrix of %u x %u elements (below 2^32 only, 128 rows below "
                             "2^32 bytes)", q->nrows, q->ncols);
        GemmMat &g = a.m[i];
        g.p0 = q->p0;
        g.p1 = q->p1;
        g.p2 = q->p2;
        g.p3 = q->p3;
        g.out = targets[i].out;
        g.bias = targets[i].bias;
        g.nrows = q->nrows;
        g.rope = targets[i].rope ? 1u : 0u;
        // offsets (no larger than a weight can be) up to 2^15: their second parts stay clear of the bottom of the f16 range
        int e = 0;
        if (q->max_abs > 0.f) frexpf(q->max_abs, &e);
        e = 15 - e < 100 ? 15 - e : 100;
        g.offset_up = ldexpf(1.f, e);
        g.offset_down = ldexpf(1.f, -e);
        g.out_stride = targets[i].out_stride;
        g.tile0 = tiles;
        g.roff = a.total_rows;
        tiles += (q->nrows + tile_rows - 1) / tile_rows;
        a.total_rows += q->nrows;
    }
    a.nmat = (uint32_t)n;
    a.xh = reinterpret_cast<const u32x4 *>(xh);
    a.xl = ctx->gemm_precise ? reinterpret_cast<const u32x4 *>(ctx->prefill_xl) : nullptr;
    if (a.xl) {
        // the kernel addresses the low parts relative to the high parts with 32 bits
        const ptrdiff_t d = reinterpret_cast<const char *>(a.xl) - reinterpret_cast<const char *>(a.xh);
        if (d <= 0 || d >= (ptrdiff_t(1) << 31))
            return set_error(WGML_E_INVALID, "gemm_quant: the activations are not the context's packed buffer");
        a.xl_offset = (uint32_t)d;
    }
    a.xscale = xscale;
    a.ncols = first->ncols;
    a.kpad = prefill_kpad(first->ncols);
    a.T = T;
    token_blocks(T, &a.ttiles, &a.nt);
    a.tall = tall;
    a.xsum = reinterpret_cast<const u32x4 *>(ctx->prefill_xsum);
    a.accumulate = accumulate;
    if (ctx->gemm_pending_ks)
        return set_error(WGML_E_INVALID, "gemm_quant: the partial sums a previous product left for its "
                                         "output were not added yet (launch_prefill_prep / launch_gemm_flush)");
    // the caller's next kernel adds the partial sums up itself: one matrix, plain += only, ...
    const bool residual = n == 1 && accumulate && !targets[0].bias;
    // ... or a gate / up pair whose next kernel is the gated launch_prefill_prep on (gate out, up out)
    const bool pair = n == 2 && !accumulate && !targets[0].bias && !targets[1].bias &&
                      targets[0].m->nrows == targets[1].m->nrows && targets[0].m->nrows % 8 == 0 &&
                      targets[0].m->nrows <= 8u * 2 * 1024;
    const bool defer = defer_reduce && (residual || pair);
    // the kernel that adds them rotates the marked targets, if rows come in pairs
    bool rotate = rope && !defer && !accumulate && rope->head_size >= 2 && rope->head_size % 2 == 0;
    for (int i = 0; rotate && i < n; ++i)
        rotate = targets[i].m->nrows % 2 == 0 && (!targets[i].rope || targets[i].m->nrows % rope->head_size == 0);
    a.ks = gemm_k_split(ctx, first->type, tiles * a.ttiles, a.kpad / KU, a.nt, a.tall, !defer && !rotate,
                        (size_t)T * a.total_rows * sizeof(float));
    if (a.ks > 1) {
        WGML_TRY(ensure_gemm_partials(ctx, (size_t)a.ks * T * a.total_rows * sizeof(float)));
        a.part = ctx->gemm_part;
        a.defer = defer;
        if (defer) {
            ctx->gemm_pending_ks = a.ks;
            ctx->gemm_pending_pair = pair ? 1 : 0;
        }
    }
    if (rope) {
        rope->applied = rotate && a.ks > 1;
        if (rope->applied) {
            a.rope_head_size = rope->head_size;
            a.rope_pos0 = rope->pos0;
            a.rope_base = rope->base_freq;
            a.rope_neox = rope->variant == WGML_ROPE_NEOX;
        }
    }
    int (*launch)(wgml_ctx *, const GemmArgs &, uint32_t) = nullptr;
    switch (first->type) {
    case WGML_Q4_K: launch = launch_gemm_q4_k; break;
    case WGML_Q6_K: launch = launch_gemm_q6_k; break;
    case WGML_Q8_0: launch = launch_gemm_q8_0; break;
    case WGML_Q5_K: launch = launch_gemm_q5_k; break;
    case WGML_Q8_K: launch = launch_gemm_q8_k; break;
    case WGML_Q4_0: launch = launch_gemm_q4_0; break;
    case WGML_Q4_1: launch = launch_gemm_q4_1; break;
    case WGML_Q5_0: launch = launch_gemm_q5_0; break;
    case WGML_Q5_1: launch = launch_gemm_q5_1; break;
    default:
        return set_error(WGML_E_UNSUPPORTED, "gemm_quant: matrix type %d has no batched product "
                                             "(the nine quantized block formats only)", first->type);
    }
    WGML_TRY(launch(ctx, a, tiles));
    if (a.ks > 1 && !a.defer) {
        if (a.rope_head_size)
            gemm_reduce_rope_kernel<<<dim3((a.total_rows / 2 + 255) / 256, a.T), dim3(256), 0, ctx->stream>>>(a);
        else
            gemm_reduce_kernel<<<dim3((a.total_rows + 255) / 256, a.T), dim3(256), 0, ctx->stream>>>(a);
        WGML_CHECK_LAUNCH();
        ctx->launches++;
    }
    return WGML_OK;
}

int launch_gemm_quant(wgml_ctx *ctx, float *out, uint32_t out_stride, const wgml_qmat *m,
                      const void *xh, const float *xscale, uint32_t T, const float *bias,
                      int accumulate, bool defer_reduce) {
    const GemmTarget t{m, out, out_stride, bias};
    return launch_gemm_quant_multi(ctx, &t, 1, xh, xscale, T, accumulate, defer_reduce);
}

int launch_embed_rows(wgml_ctx *ctx, float *x, const float *table, const uint32_t *d_tokens,
                      uint32_t dim, uint32_t T, const float *pos_table, uint32_t pos0) {
    embed_rows_kernel<<<dim3((dim + 255) / 256, T), dim3(256), 0, ctx->stream>>>(x, table, d_tokens, dim,
                                                                                 pos_table, pos0);
    WGML_CHECK_LAUNCH();
    ctx->launches++;
    return WGML_OK;
}

int launch_cache_rows(wgml_ctx *ctx, const float *qkv, float *k, float *v, uint32_t n, uint32_t T) {
    cache_rows_kernel<<<dim3((n / 2 + 255) / 256, T), dim3(256), 0, ctx->stream>>>(qkv, k, v, n);
    WGML_CHECK_LAUNCH();
    ctx->launches++;
    return WGML_OK;
}

int launch_rope_rows(wgml_ctx *ctx, int variant, uint32_t head_size, uint32_t kv_dim, uint32_t pos0,
                     float base_freq, float *q, uint32_t q_len, uint32_t q_stride, float *k,
                     uint32_t k_stride, uint32_t T) {
    const uint32_t n_pairs = q_len / 2;
    rope_rows_kernel<<<dim3((n_pairs + 63) / 64, T), dim3(64), 0, ctx->stream>>>(
        q, q_stride, k, k_stride, n_pairs, head_size, kv_dim, pos0, base_freq,
        variant == WGML_ROPE_NEOX);
    WGML_CHECK_LAUNCH();
    ctx->launches++;
    return WGML_OK;
}

int launch_attention_rows(wgml_ctx *ctx, const wgml_attn_params &p, uint32_t pos0, uint32_t T,
                          const float *q, uint32_t q_stride, const float *kc, const float *vc,
                          float *xb, uint32_t xb_stride) {
    if (p.head_size % 4 != 0 || p.head_size > 256 || p.kv_dim % 4 != 0 || q_stride % 4 != 0)
        return set_error(WGML_E_UNSUPPORTED,
                         "attention over a run of tokens: head_size %u (multiple of 4, <= 256)",
                         p.head_size);
    AttnRowsArgs a{q, kc, vc, xb, q_stride, xb_stride, p.kv_dim, p.kv_mul, p.head_size, pos0};
    if (p.head_size % 16 == 0 && p.head_size <= 128 && !ctx->tuning[WGML_TUNE_PREFILL_ATTENTION_PER_TOKEN]) {
        // 16 tokens per workgroup on the fp32 matrix cores
        const bool few = (uint64_t)p.n_heads * ((T + 15) / 16) < (uint64_t)(ctx->n_cu > 0 ? ctx->n_cu : 256);
        switch (p.head_size / 16) {
        case 1: launch_attn_block<1>(ctx, a, p.n_heads, T, few); break;
        case 2: launch_attn_block<2>(ctx, a, p.n_heads, T, few); break;
        case 3: launch_attn_block<3>(ctx, a, p.n_heads, T, few); break;
        case 4: launch_attn_block<4>(ctx, a, p.n_heads, T, few); break;
        case 5: launch_attn_block<5>(ctx, a, p.n_heads, T, few); break;
        case 6: launch_attn_block<6>(ctx, a, p.n_heads, T, few); break;
        case 7: launch_attn_block<7>(ctx, a, p.n_heads, T, few); break;
        default: launch_attn_block<8>(ctx, a, p.n_heads, T, few); break;
        }
        WGML_CHECK_LAUNCH();
        ctx->launches++;
        return WGML_OK;
    }
    const dim3 grid(p.n_heads, T), block(256);
    switch ((p.head_size + 63) / 64) {
    case 1: attn_rows_kernel<1><<<grid, block, 0, ctx->stream>>>(a); break;
    case 2: attn_rows_kernel<2><<<grid, block, 0, ctx->stream>>>(a); break;
    case 3: attn_rows_kernel<3><<<grid, block, 0, ctx->stream>>>(a); break;
    default: attn_rows_kernel<4><<<grid, block, 0, ctx->stream>>>(a); break;
    }
    WGML_CHECK_LAUNCH();
    ctx->launches++;
    return WGML_OK;
}

}  // namespace wgml

extern "C" {

// 1 (default): products of the batched path take the activations as pairs of f16 numbers (error
// about 2^-22 per term, two MFMAs per 32 terms); 0: plain f16 activations (2^-11, one MFMA).
int wgml_ctx_set_gemm_precision(wgml_ctx *ctx, int level) {
    WGML_REQUIRE(ctx != nullptr, "wgml_ctx_set_gemm_precision: null context");
    WGML_REQUIRE(level == 0 || level == 1, "wgml_ctx_set_gemm_precision: level %d not in {0, 1}", level);
    ctx->gemm_precise = level;
    return WGML_OK;
}

// out[t] = M x[t] for T <= 128 vectors at once (x: T x ncols, out: T x nrows, both
// row-major f32) on the matrix cores; the batched counterpart of wgml_gemv_quant.
int wgml_gemm_quant(wgml_ctx *ctx, wgml_view out, const wgml_qmat *m, wgml_view x, uint32_t n_tokens) {
    WGML_REQUIRE(ctx && m, "wgml_gemm_quant: null argument");
    WGML_TRY(check_view(out, "wgml_gemm_quant: out"));
    WGML_TRY(check_view(x, "wgml_gemm_quant: x"));
    WGML_REQUIRE(n_tokens >= 1 && n_tokens <= kPrefillMaxTokens,
                 "wgml_gemm_quant: %u tokens (1..%u)", n_tokens, kPrefillMaxTokens);
    WGML_REQUIRE((uint64_t)x.len == (uint64_t)n_tokens * m->ncols,
                 "Gemm: dimension mismatch (x has %u elements, expected %u x %u)", x.len, n_tokens,
                 m->ncols);
    WGML_REQUIRE((uint64_t)out.len == (uint64_t)n_tokens * m->nrows,
                 "Gemm: dimension mismatch (out has %u elements, expected %u x %u)", out.len,
                 n_tokens, m->nrows);
    const size_t xh_bytes = (size_t)kPrefillMaxTokens * prefill_kpad(m->ncols) * 2;
    WGML_TRY(ensure_prefill_scratch(ctx, xh_bytes));
    // a prompt pass that failed half way may have left partial sums owed to its next packing
    // kernel: they are not this product's (the packing kernel would add them to x)
    ctx->gemm_pending_ks = 0;
    ctx->gemm_pending_pair = 0;
    WGML_TRY(launch_prefill_prep(ctx, view_ptr(x), m->ncols, nullptr, nullptr, 0.f, ctx->prefill_xh,
                                 ctx->prefill_xscale, m->ncols, n_tokens));
    return launch_gemm_quant(ctx, view_ptr(out), m->nrows, m, ctx->prefill_xh, ctx->prefill_xscale,
                             n_tokens, nullptr, 0, false);
}

}  // extern "C"
