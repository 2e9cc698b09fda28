// Dequantize-and-GEMV kernels for Q8_0 / Q4_K / Q6_K and the dense f32 GEMV.
// Replaces GemvQuant::dispatch and its WGSL kernels (ops/gemv_quant.rs:243-348,
// ops/gemv_quant_{q8_0x2,q4_k,q6_kx2}.wgsl of the reference) and wgebra's f32
// Gemv/GemvTr.
//
// Scheme (wavefront-64, HBM-bound, no MFMA):
//   * the activation vector x is staged once per workgroup into LDS in a
//     lane-transposed order, so that lane L of a wave reads its k-th float4 at
//     LDS slot [k][L]: consecutive lanes hit consecutive 16-byte slots (no bank
//     conflicts);
//   * a wave owns R consecutive rows.  Per 64-tile step every lane loads one
//     tile of x from LDS into registers and reuses it for the R rows, so LDS
//     traffic is 1/R of the naive rate;
//   * weights stream from HBM as aligned 128-bit loads; a wave touches one
//     contiguous run of bytes per row and plane;
//   * sub-block minima / offsets are folded in through per-tile sums of x that
//     are computed once per workgroup (not once per row);
//   * the 64 partial sums of a row are reduced with DPP + v_readlane in a fixed
//     order (deterministic results).
//
// A "tile" is the span one lane covers per step:
//   Q4_K: one 64-element group of a super-block (32 bytes of qs) + the 16-byte
//         header {d, dmin, scales[12]};
//   Q6_K: 64 elements {e, e+32, e+64, e+96 : e in 16-run} of one 128-half: 16
//         bytes of ql, 16 of ql+32, 16 of qh, 8 scale bytes, d;
//   Q8_0: one 32-element block: 32 bytes of qs + d.
#pragma once

#include <type_traits>

#include "common.h"
#include "device_utils.h"

using namespace wgml;

namespace {

struct GemvParams {
    const uint8_t *p0, *p1, *p2, *p3;  // matrix planes
    const float *x;
    float *out;
    const float *bias;
    uint32_t nrows, ncols;
    int accumulate;
    const uint32_t *dyn_pos;  // out += *dyn_pos * out_pos_stride
    uint32_t out_pos_stride;
    const float *norm_w;  // optional fused RMSNorm of x
    float norm_eps;
    const float *ln_g, *ln_b;  // optional fused LayerNorm of x (integer-dot kernels)
    int act;                   // 1: GELU on acc + bias before the store
    // integer-dot kernels: the first `active_waves` waves of every workgroup walk
    // the row-groups with stride gridDim.x * active_waves
    uint32_t active_waves;
    // part_n > 0: x is the merged output of a decode-attention launch that left part_n partial
    // results per head (AttnPartials in common.h); x itself is then not read
    const float *part_o, *part_ml;
    uint32_t part_n, part_hsp, part_hs, part_hs_inv;  // part_hs_inv = ceil(2^32 / part_hs)
    // kernels with EXTRA_MAXIMA: (largest result, its row) of the wave whose first row-group is g goes to maxima[g]
    RowMaximum *maxima;
};

// What a single-matrix kernel can do beside the product (bits).  Kernels of their own (gemv_full.hip, gemv_maxima.hip): the
// code that the others jump over costs every launch 0.05 to 0.1 us.
enum { EXTRA_FULL = 1,     // x may go through a LayerNorm, results through an activation
       EXTRA_MAXIMA = 2 };  // every wave leaves the largest of its results

// Merging attention partial results (see AttnPartials) for float4 number g4 of the merged
// output: the partial results of its head are taken in eight at a time, the way an online
// softmax takes in new scores.  PartialChunk holds one round of loads, so that a caller can
// request it early and merge it later.
struct PartialChunk {
    float2 s[8];  // (maximum, sum of weights)
    float4 v[8];  // weighted sums of V
};
__device__ __forceinline__ void load_partials(PartialChunk &c, const GemvParams &p, uint32_t g4,
                                              uint32_t y0) {
    // h = e / head_size by multiplication with ceil(2^32 / head_size): exact for the e < 2^20
    // and head sizes up to 256 that occur here
    const uint32_t e = g4 * 4, h = __umulhi(e, p.part_hs_inv), d = e - h * p.part_hs, P = p.part_n;
    const float *o = p.part_o + (size_t)h * P * p.part_hsp + d;
    const float2 *ml = reinterpret_cast<const float2 *>(p.part_ml) + (size_t)h * P;
    // The loads are unconditional (a partial result beyond the last one re-reads the last one
    // and is masked out when it is merged): with a load under a condition the compiler cannot
    // count the loads in flight, and the wait for these would also wait for the weight tiles
    // requested after them.
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const uint32_t y = min(y0 + (uint32_t)k, P - 1);
        c.s[k] = ml[y];
        c.v[k] = *reinterpret_cast<const float4 *>(o + (size_t)y * p.part_hsp);
    }
}
struct PartialState {
    float M = -INFINITY, L = 0.f;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
};
// `n`: how many of the chunk's eight partial results exist.
__device__ __forceinline__ void merge_partials(PartialState &st, const PartialChunk &c, uint32_t n) {
    float Mc = st.M;
#pragma unroll
    for (int k = 0; k < 8; ++k) Mc = fmaxf(Mc, (uint32_t)k < n ? c.s[k].x : -INFINITY);
    // the running state is rescaled to the new maximum (M = -inf only while nothing has been
    // taken in, and then L and acc are zero)
    const float r = st.M == -INFINITY ? 0.f : __expf(st.M - Mc);
    st.L *= r;
    st.acc.x *= r;
    st.acc.y *= r;
    st.acc.z *= r;
    st.acc.w *= r;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        // a neutral partial (maximum -inf) has undefined values: they must not be touched
        const bool live = (uint32_t)k < n && c.s[k].x != -INFINITY;
        const float wk = live ? __expf(c.s[k].x - Mc) : 0.f;
        st.L = fmaf(c.s[k].y, wk, st.L);
        st.acc.x = fmaf(live ? c.v[k].x : 0.f, wk, st.acc.x);
        st.acc.y = fmaf(live ? c.v[k].y : 0.f, wk, st.acc.y);
        st.acc.z = fmaf(live ? c.v[k].z : 0.f, wk, st.acc.z);
        st.acc.w = fmaf(live ? c.v[k].w : 0.f, wk, st.acc.w);
    }
    st.M = Mc;
}
// `first`: the partial results 0..7, already requested; the others are fetched here.
__device__ __forceinline__ float4 merged_partials(const GemvParams &p, uint32_t g4,
                                                  const PartialChunk &first) {
    PartialState st;
    merge_partials(st, first, p.part_n);
    for (uint32_t y0 = 8; y0 < p.part_n; y0 += 8) {
        PartialChunk c;
        load_partials(c, p, g4, y0);
        merge_partials(st, c, p.part_n - y0);
    }
    return make_float4(st.acc.x / st.L, st.acc.y / st.L, st.acc.z / st.L, st.acc.w / st.L);
}
__device__ __forceinline__ float4 merged_partials(const GemvParams &p, uint32_t g4) {
    PartialChunk c;
    load_partials(c, p, g4, 0);
    return merged_partials(p, g4, c);
}

// Hides a value from the optimizer (no instruction is emitted).  Used on masked
// 32-bit words so that the four bytes are converted with v_cvt_f32_ubyte0..3 of
// the *shared* masked word instead of one bit-field extract per element.
__device__ __forceinline__ uint32_t opaque(uint32_t v) {
    asm("" : "+v"(v));
    return v;
}

// ------------------------------------------------------------------ Q4_K ----
struct FmtQ4K {
    static constexpr int TILE = 64;    // elements per lane tile
    static constexpr int CHUNKS = 16;  // float4 of x per tile
    static constexpr int NSUM = 2;     // x sums per tile (low-nibble half, high-nibble half)
    struct Row {
        uint4 hdr, qa, qb;
    };
    struct RowBase {
        const uint8_t *blocks;
    };
    __device__ static RowBase row_base(const GemvParams &p, uint32_t row) {
        return {p.p0 + (size_t)row * (p.ncols / 256) * 144};
    }
    // float4 index g of x -> (tile, chunk)
    __device__ static void map(uint32_t g, uint32_t &tile, uint32_t &chunk) {
        tile = g >> 4;
        chunk = g & 15;
    }
    __device__ static void load(Row &w, const RowBase &rb, uint32_t tile) {
        const uint8_t *blk = rb.blocks + (size_t)(tile >> 2) * 144;
        w.hdr = *reinterpret_cast<const uint4 *>(blk);
        const uint4 *q = reinterpret_cast<const uint4 *>(blk + 16 + (tile & 3) * 32);
        w.qa = q[0];
        w.qb = q[1];
    }
    // acc[r] += dot(row r tile, x tile).  xl points at this lane's slot of chunk 0
    // (chunk c is xl[c * 64]); s = the two half-tile sums of x.
    template <int R>
    __device__ static void accumulate(const Row (&w)[R], const float4 *xl, const float *s,
                                      uint32_t tile, float (&acc)[R]) {
        const uint32_t j = tile & 3;
        const uint32_t sh = (j & 1u) * 16u;
        float dlo[R], dhi[R];
#pragma unroll
        for (int r = 0; r < R; ++r) dlo[r] = dhi[r] = 0.f;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float4 xa = xl[k * 64], xb = xl[(8 + k) * 64];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const uint32_t q = k < 4 ? (&w[r].qa.x)[k] : (&w[r].qb.x)[k - 4];
                const uint32_t lo = opaque(q & 0x0f0f0f0fu);
                const uint32_t hi = opaque(q & 0xf0f0f0f0u);  // 16 * nibble per byte
                dlo[r] = fmaf(ub0(lo), xa.x, dlo[r]);
                dlo[r] = fmaf(ub1(lo), xa.y, dlo[r]);
                dlo[r] = fmaf(ub2(lo), xa.z, dlo[r]);
                dlo[r] = fmaf(ub3(lo), xa.w, dlo[r]);
                dhi[r] = fmaf(ub0(hi), xb.x, dhi[r]);
                dhi[r] = fmaf(ub1(hi), xb.y, dhi[r]);
                dhi[r] = fmaf(ub2(hi), xb.z, dhi[r]);
                dhi[r] = fmaf(ub3(hi), xb.w, dhi[r]);
            }
        }
        const float s0 = s[0], s1 = s[1];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float d = f16_bits_to_f32((uint16_t)(w[r].hdr.x & 0xffffu));
            const float dmin = f16_bits_to_f32((uint16_t)(w[r].hdr.x >> 16));
            // 6-bit scale/min pairs of sub-blocks 2j and 2j+1 (get_scale_min_k4).
            const uint32_t a = (w[r].hdr.y >> sh) & 0xffffu, b = (w[r].hdr.z >> sh) & 0xffffu,
                           c = (w[r].hdr.w >> sh) & 0xffffu;
            uint32_t sc2, m2;
            if (j < 2) {
                sc2 = a & 0x3f3fu;
                m2 = b & 0x3f3fu;
            } else {
                sc2 = (c & 0x0f0fu) | ((a >> 2) & 0x3030u);
                m2 = ((c >> 4) & 0x0f0fu) | ((b >> 2) & 0x3030u);
            }
            const float sc_lo = ub0(sc2), sc_hi = ub1(sc2), m_lo = ub0(m2), m_hi = ub1(m2);
            float v = (d * sc_lo) * dlo[r];
            v = fmaf((d * sc_hi) * 0.0625f, dhi[r], v);
            v = fmaf(-dmin, fmaf(m_lo, s0, m_hi * s1), v);
            acc[r] += v;
        }
    }
};

// ------------------------------------------------------------------ Q6_K ----
struct FmtQ6K {
    static constexpr int TILE = 64;
    static constexpr int CHUNKS = 16;
    static constexpr int NSUM = 4;  // one per 16-element sub-block
    struct Row {
        uint4 l0, l1, h;
        uint2 sc;
        uint16_t d;
    };
    struct RowBase {
        const uint8_t *ql, *qh, *sc, *d;
    };
    __device__ static RowBase row_base(const GemvParams &p, uint32_t row) {
        const size_t nb = (size_t)row * (p.ncols / 256);
        return {p.p0 + nb * 128, p.p1 + nb * 64, p.p2 + nb * 16, p.p3 + nb * 2};
    }
    __device__ static void map(uint32_t g, uint32_t &tile, uint32_t &chunk) {
        const uint32_t e = g * 4;
        const uint32_t blk = e >> 8, i = (e >> 7) & 1, quarter = (e >> 5) & 3, s = (e >> 4) & 1,
                       k4 = (e & 15) >> 2;
        tile = blk * 4 + i * 2 + s;
        chunk = quarter * 4 + k4;
    }
    __device__ static void load(Row &w, const RowBase &rb, uint32_t tile) {
        const size_t blk = tile >> 2;
        const uint32_t i = (tile >> 1) & 1, s = tile & 1;
        const uint8_t *ql = rb.ql + blk * 128 + i * 64 + s * 16;
        w.l0 = *reinterpret_cast<const uint4 *>(ql);
        w.l1 = *reinterpret_cast<const uint4 *>(ql + 32);
        w.h = *reinterpret_cast<const uint4 *>(rb.qh + blk * 64 + i * 32 + s * 16);
        w.sc = *reinterpret_cast<const uint2 *>(rb.sc + blk * 16 + i * 8);
        w.d = *reinterpret_cast<const uint16_t *>(rb.d + blk * 2);
    }
    template <int R>
    __device__ static void accumulate(const Row (&w)[R], const float4 *xl, const float *s,
                                      uint32_t tile, float (&acc)[R]) {
        float d1[R], d2[R], d3[R], d4[R];
#pragma unroll
        for (int r = 0; r < R; ++r) d1[r] = d2[r] = d3[r] = d4[r] = 0.f;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float4 x1 = xl[k * 64], x2 = xl[(4 + k) * 64], x3 = xl[(8 + k) * 64],
                         x4 = xl[(12 + k) * 64];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const uint32_t L0 = (&w[r].l0.x)[k], L1 = (&w[r].l1.x)[k], H = (&w[r].h.x)[k];
                const uint32_t q1 = opaque((L0 & 0x0f0f0f0fu) | ((H << 4) & 0x30303030u));
                const uint32_t q2 = opaque((L1 & 0x0f0f0f0fu) | ((H << 2) & 0x30303030u));
                const uint32_t q3 = opaque(((L0 >> 4) & 0x0f0f0f0fu) | (H & 0x30303030u));
                const uint32_t q4 = opaque(((L1 >> 4) & 0x0f0f0f0fu) | ((H >> 2) & 0x30303030u));
                d1[r] = fmaf(ub0(q1), x1.x, d1[r]);
                d1[r] = fmaf(ub1(q1), x1.y, d1[r]);
                d1[r] = fmaf(ub2(q1), x1.z, d1[r]);
                d1[r] = fmaf(ub3(q1), x1.w, d1[r]);
                d2[r] = fmaf(ub0(q2), x2.x, d2[r]);
                d2[r] = fmaf(ub1(q2), x2.y, d2[r]);
                d2[r] = fmaf(ub2(q2), x2.z, d2[r]);
                d2[r] = fmaf(ub3(q2), x2.w, d2[r]);
                d3[r] = fmaf(ub0(q3), x3.x, d3[r]);
                d3[r] = fmaf(ub1(q3), x3.y, d3[r]);
                d3[r] = fmaf(ub2(q3), x3.z, d3[r]);
                d3[r] = fmaf(ub3(q3), x3.w, d3[r]);
                d4[r] = fmaf(ub0(q4), x4.x, d4[r]);
                d4[r] = fmaf(ub1(q4), x4.y, d4[r]);
                d4[r] = fmaf(ub2(q4), x4.z, d4[r]);
                d4[r] = fmaf(ub3(q4), x4.w, d4[r]);
            }
        }
        const uint32_t sb = (tile & 1u) * 8u;  // bit offset of scales[is], is = tile & 1
        const float s0 = s[0], s1 = s[1], s2 = s[2], s3 = s[3];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float sc1 = sb0(w[r].sc.x >> sb), sc2 = sb0(w[r].sc.x >> (sb + 16)),
                        sc3 = sb0(w[r].sc.y >> sb), sc4 = sb0(w[r].sc.y >> (sb + 16));
            // q - 32 folded in through the sub-block sums of x.
            float v = sc1 * fmaf(-32.f, s0, d1[r]);
            v = fmaf(sc2, fmaf(-32.f, s1, d2[r]), v);
            v = fmaf(sc3, fmaf(-32.f, s2, d3[r]), v);
            v = fmaf(sc4, fmaf(-32.f, s3, d4[r]), v);
            acc[r] = fmaf(f16_bits_to_f32(w[r].d), v, acc[r]);
        }
    }
};

// ------------------------------------------------------------------ Q8_0 ----
struct FmtQ8_0 {
    static constexpr int TILE = 32;
    static constexpr int CHUNKS = 8;
    static constexpr int NSUM = 1;  // sum of the tile's x: quants are used as q + 128
    struct Row {
        uint4 a, b;
        uint16_t d;
    };
    struct RowBase {
        const uint8_t *qs, *d;
    };
    __device__ static RowBase row_base(const GemvParams &p, uint32_t row) {
        return {p.p0 + (size_t)row * p.ncols, p.p1 + (size_t)row * (p.ncols / 32) * 2};
    }
    __device__ static void map(uint32_t g, uint32_t &tile, uint32_t &chunk) {
        tile = g >> 3;
        chunk = g & 7;
    }
    __device__ static void load(Row &w, const RowBase &rb, uint32_t tile) {
        const uint4 *q = reinterpret_cast<const uint4 *>(rb.qs + (size_t)tile * 32);
        w.a = q[0];
        w.b = q[1];
        w.d = *reinterpret_cast<const uint16_t *>(rb.d + (size_t)tile * 2);
    }
    template <int R>
    __device__ static void accumulate(const Row (&w)[R], const float4 *xl, const float *s,
                                      uint32_t, float (&acc)[R]) {
        float dt[R];
#pragma unroll
        for (int r = 0; r < R; ++r) dt[r] = 0.f;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float4 xv = xl[k * 64];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const uint32_t q = k < 4 ? (&w[r].a.x)[k] : (&w[r].b.x)[k - 4];
                const uint32_t u = opaque(q ^ 0x80808080u);  // q + 128 per byte, unsigned
                dt[r] = fmaf(ub0(u), xv.x, dt[r]);
                dt[r] = fmaf(ub1(u), xv.y, dt[r]);
                dt[r] = fmaf(ub2(u), xv.z, dt[r]);
                dt[r] = fmaf(ub3(u), xv.w, dt[r]);
            }
        }
        const float s0 = s[0];
#pragma unroll
        for (int r = 0; r < R; ++r)
            acc[r] = fmaf(f16_bits_to_f32(w[r].d), fmaf(-128.f, s0, dt[r]), acc[r]);
    }
};

// ----------------------------------------- the 32-element GGUF blocks ----
// Q4_0, Q4_1, Q5_0, Q5_1 (quantization.rs:47-162 of the reference) as planes of nibbles, scales (with
// minima) and fifth bits.  Element k of a block is the low nibble of qs[k] for k < 16, the high nibble
// of qs[k-16] otherwise, plus bit k of qh as its fifth bit.  A tile is B = 1 or 2 blocks (kLegacyWide).
// Bound by the bytes in flight: 16 or 32 aligned bytes of nibbles per lane and request (blocks of 18 to
// 24 bytes as in the file made them straddle; 24 tokens of eight layers of 3072 x 8192 in Q4_0, with
// 21 of a prompt, 9.55 ms -> 8.08).  Integer-dot kernels only.
template <bool HAS_M, bool HAS_QH, int B>
struct FmtLegacy {
    struct Row {
        uint4 q[B];
        uint32_t qh[HAS_QH ? B : 1], dm[HAS_M ? B : 1];  // dm without minima: the d of both blocks in one word
    };
    struct RowBase {
        const uint8_t *qs, *dm, *qh;
    };
    __device__ static RowBase row_base(const GemvParams &p, uint32_t row) {
        const size_t nb = (size_t)row * (p.ncols / 32);
        return {p.p0 + nb * 16, p.p1 + nb * (HAS_M ? 4 : 2), p.p2 + nb * 4};
    }
    __device__ static void load(Row &w, const RowBase &rb, uint32_t tile) {
        const size_t blk = (size_t)tile * B;
#pragma unroll
        for (int b = 0; b < B; ++b) w.q[b] = reinterpret_cast<const uint4 *>(rb.qs)[blk + b];
        if constexpr (HAS_QH) __builtin_memcpy(w.qh, __builtin_assume_aligned(rb.qh + blk * 4, 4 * B), 4 * B);
        if constexpr (HAS_M)
            __builtin_memcpy(w.dm, __builtin_assume_aligned(rb.dm + blk * 4, 4 * B), 4 * B);
        else if constexpr (B == 2)
            w.dm[0] = *reinterpret_cast<const uint32_t *>(rb.dm + blk * 2);
        else
            w.dm[0] = *reinterpret_cast<const uint16_t *>(rb.dm + blk * 2);
    }
    __device__ static float d(const Row &w, int b) {
        return f16_bits_to_f32((uint16_t)(HAS_M ? w.dm[HAS_M ? b : 0] & 0xffffu : (w.dm[0] >> (16 * b)) & 0xffffu));
    }
    __device__ static float m(const Row &w, int b) { return f16_bits_to_f32((uint16_t)(w.dm[HAS_M ? b : 0] >> 16)); }
};

// Q8_K (292 B: f32 d, 256 int8, 16 block sums that dequantization does not use;
// quantization.rs:170-199).  A tile is 32 of the 256 quants.
struct FmtQ8K {
    struct Row {
        uint4 a, b;
        float d;
    };
    struct RowBase {
        const uint8_t *blocks;
    };
    __device__ static RowBase row_base(const GemvParams &p, uint32_t row) {
        return {p.p0 + (size_t)row * (p.ncols / 256) * 292};
    }
    __device__ static void load(Row &w, const RowBase &rb, uint32_t tile) {
        const uint8_t *b = rb.blocks + (size_t)(tile >> 3) * 292;
        __builtin_memcpy(&w.d, b, 4);
        __builtin_memcpy(&w.a, b + 4 + (tile & 7) * 32, 16);
        __builtin_memcpy(&w.b, b + 4 + (tile & 7) * 32 + 16, 16);
    }
};

// Q5_K (176 B: d, dmin, scales[12] as Q4_K, 32 bytes of fifth bits, 128 bytes of nibbles;
// quantization.rs:249-317).  A tile is a 64-element group as for Q4_K: sub-blocks 2j (low
// nibbles) and 2j+1 (high nibbles), whose fifth bits are bits 2j and 2j+1 of qh[l].
struct FmtQ5K {
    struct Row {
        uint4 hdr, qa, qb, ha, hb;
    };
    struct RowBase {
        const uint8_t *blocks;
    };
    __device__ static RowBase row_base(const GemvParams &p, uint32_t row) {
        return {p.p0 + (size_t)row * (p.ncols / 256) * 176};
    }
    __device__ static void load(Row &w, const RowBase &rb, uint32_t tile) {
        const uint8_t *blk = rb.blocks + (size_t)(tile >> 2) * 176;
        w.hdr = *reinterpret_cast<const uint4 *>(blk);
        w.ha = *reinterpret_cast<const uint4 *>(blk + 16);
        w.hb = *reinterpret_cast<const uint4 *>(blk + 32);
        const uint4 *q = reinterpret_cast<const uint4 *>(blk + 48 + (tile & 3) * 32);
        w.qa = q[0];
        w.qb = q[1];
    }
};

// ------------------------------------------------------------- dense f32 ----
// Rows of a multiple of 16 floats (F32 tensors, and F16 ones that are expanded when the matrix
// is created, see gemv_keeps_f16).  A tile is 16 elements, 64 bytes: a wave's step covers 1024 columns and asks for
// 4 KB, as the quantized formats do.  No sums of x are needed.  HBM-bound where tall (GPT-2's
// 50257x768 output projection), launch-bound elsewhere: what it brings is the folded norms,
// epilogues and Q/K/V launch, and with them the recorded step -- GPT-2 124M with its matrices in f32
// 283 us per token, 625 with a launch per operation and gemv_f32_kernel.
struct FmtF32 {
    static constexpr int TILE = 16;
    static constexpr int CHUNKS = 4;
    static constexpr int NSUM = 0;
    struct Row {
        float4 a[4];
    };
    struct RowBase {
        const float4 *row;
    };
    __device__ static RowBase row_base(const GemvParams &p, uint32_t row) {
        return {reinterpret_cast<const float4 *>(p.p0) + (size_t)row * (p.ncols / 4)};
    }
    __device__ static void map(uint32_t g, uint32_t &tile, uint32_t &chunk) {
        tile = g >> 2;
        chunk = g & 3;
    }
    __device__ static void load(Row &w, const RowBase &rb, uint32_t tile) {
#pragma unroll
        for (int c = 0; c < 4; ++c) w.a[c] = rb.row[(size_t)tile * 4 + c];
    }
    template <int R>
    __device__ static void accumulate(const Row (&w)[R], const float4 *xl, const float *, uint32_t,
                                      float (&acc)[R]) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float4 xv = xl[c * 64];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                acc[r] = fmaf(w[r].a[c].x, xv.x, acc[r]);
                acc[r] = fmaf(w[r].a[c].y, xv.y, acc[r]);
                acc[r] = fmaf(w[r].a[c].z, xv.z, acc[r]);
                acc[r] = fmaf(w[r].a[c].w, xv.w, acc[r]);
            }
        }
    }
};

// An F16 tensor as the file has it: the same tiles and the same multiply-adds in the same order as FmtF32 with the values
// expanded, so the same results.  Half the bytes that the expanded values take: GPT-2 124M 283 -> 251 us per token (8 tokens in,
// 16 out: 6.80 -> 6.04 ms), four layers of 1024 x 4096 with its 50257 rows of output 140 -> 100.
struct FmtF16 {
    static constexpr int TILE = 16;
    static constexpr int CHUNKS = 4;
    static constexpr int NSUM = 0;
    struct Row {
        uint4 a[2];
    };
    struct RowBase {
        const uint4 *row;
    };
    __device__ static RowBase row_base(const GemvParams &p, uint32_t row) {
        return {reinterpret_cast<const uint4 *>(p.p0) + (size_t)row * (p.ncols / 8)};
    }
    __device__ static void map(uint32_t g, uint32_t &tile, uint32_t &chunk) { FmtF32::map(g, tile, chunk); }
    __device__ static void load(Row &w, const RowBase &rb, uint32_t tile) {
#pragma unroll
        for (int c = 0; c < 2; ++c) w.a[c] = rb.row[(size_t)tile * 2 + c];
    }
    template <int R>
    __device__ static void accumulate(const Row (&w)[R], const float4 *xl, const float *, uint32_t,
                                      float (&acc)[R]) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float4 xv = xl[c * 64];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const uint32_t bits[2] = {c & 1 ? w[r].a[c / 2].z : w[r].a[c / 2].x, c & 1 ? w[r].a[c / 2].w : w[r].a[c / 2].y};
                _Float16 v[4];
                __builtin_memcpy(v, bits, 8);
                acc[r] = fmaf((float)v[0], xv.x, acc[r]);
                acc[r] = fmaf((float)v[1], xv.y, acc[r]);
                acc[r] = fmaf((float)v[2], xv.z, acc[r]);
                acc[r] = fmaf((float)v[3], xv.w, acc[r]);
            }
        }
    }
};

// F16 and F32 tensors in one launch (a file may mix them in a layer): plane pointer p1 is null for F32.  The values and order of the
// other two, a matrix' rows as words of 16 bytes (F16: the second word again in place of the third and fourth).
struct FmtDenseMix {
    static constexpr int TILE = 16;
    static constexpr int CHUNKS = 4;
    static constexpr int NSUM = 0;
    struct Row {
        uint4 a[4];
        bool half;
    };
    struct RowBase {
        const uint4 *row;
        bool half;
    };
    __device__ static RowBase row_base(const GemvParams &p, uint32_t row) {
        const bool half = p.p1 != nullptr;
        return {reinterpret_cast<const uint4 *>(p.p0) + (size_t)row * (p.ncols / (half ? 8 : 4)), half};
    }
    __device__ static void map(uint32_t g, uint32_t &tile, uint32_t &chunk) { FmtF32::map(g, tile, chunk); }
    __device__ static void load(Row &w, const RowBase &rb, uint32_t tile) {
        const uint32_t n = rb.half ? 2 : 4;
        w.half = rb.half;
#pragma unroll
        for (uint32_t c = 0; c < 4; ++c) w.a[c] = rb.row[(size_t)tile * n + min(c, n - 1)];
    }
    template <int R>
    __device__ static void accumulate(const Row (&w)[R], const float4 *xl, const float *, uint32_t,
                                      float (&acc)[R]) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float4 xv = xl[c * 64];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const uint32_t bits[2] = {c & 1 ? w[r].a[c / 2].z : w[r].a[c / 2].x, c & 1 ? w[r].a[c / 2].w : w[r].a[c / 2].y};
                _Float16 h[4];
                __builtin_memcpy(h, bits, 8);
                float v[4];
                __builtin_memcpy(v, &w[r].a[c], 16);
                acc[r] = fmaf(w[r].half ? (float)h[0] : v[0], xv.x, acc[r]);
                acc[r] = fmaf(w[r].half ? (float)h[1] : v[1], xv.y, acc[r]);
                acc[r] = fmaf(w[r].half ? (float)h[2] : v[2], xv.z, acc[r]);
                acc[r] = fmaf(w[r].half ? (float)h[3] : v[3], xv.w, acc[r]);
            }
        }
    }
};

// LDS layout: x as float4 xs[step][chunk][lane]; then sums[sum][tile_padded].
template <class F>
__device__ __forceinline__ uint32_t lds_slot(uint32_t tile, uint32_t chunk) {
    return ((tile >> 6) * F::CHUNKS + chunk) * 64 + (tile & 63);
}

// rsqrt(mean(x^2) + eps) over the whole vector, computed by the workgroup
// (ops/rms_norm.wgsl:36-60 of the reference).  Contains barriers.
__device__ __forceinline__ float block_rms_scale(const GemvParams &p, float *red) {
    const float4 *x4 = reinterpret_cast<const float4 *>(p.x);
    const uint32_t n4 = p.ncols >> 2;
    float ss = 0.f;
    for (uint32_t g4 = threadIdx.x; g4 < n4; g4 += blockDim.x) {
        const float4 v = x4[g4];
        ss = fmaf(v.x, v.x, ss);
        ss = fmaf(v.y, v.y, ss);
        ss = fmaf(v.z, v.z, ss);
        ss = fmaf(v.w, v.w, ss);
    }
    const float total = block_sum(ss, red);
    return 1.0f / sqrtf(total / (float)p.ncols + p.norm_eps);
}

__device__ __forceinline__ float4 apply_norm(float4 v, float rms, const float4 w) {
    v.x = (v.x * rms) * w.x;
    v.y = (v.y * rms) * w.y;
    v.z = (v.z * rms) * w.z;
    v.w = (v.w * rms) * w.w;
    return v;
}

// Loads the tiles of the R rows of row-group `g` for tile index `tile`.
template <class F, int R>
__device__ __forceinline__ void load_group(typename F::Row (&w)[R], const GemvParams &p,
                                           uint32_t g, uint32_t tile) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t row = min(g * R + r, p.nrows - 1);
        F::load(w[r], F::row_base(p, row), tile);
    }
}

// =========================================================================
// Integer-dot path (default).  The fp32 path above spends ~3 VALU operations
// per weight element (convert, multiply-add, unpack), which makes the 4-bit
// formats issue-bound on the four SIMD16 units of a CU well below HBM speed.
// Here the activation vector is staged once per workgroup as 16-bit block
// fixed point: per block of XB elements a scale s = max|x| / 32512 and
// X = round(x / s), stored as two int8 planes X = 256*hi + lo (hi in
// [-127,127], lo in [-128,127]).  Weights are unpacked to bytes and multiplied
// with v_dot4c_i32_i8 (four exact integer MACs per lane-operation); the two
// int32 partial sums are recombined as 256*hi + lo and scaled once per
// sub-block in fp32.  The rounding of x is at most 2^-16 of the block maximum
// per element (about 3e-5 of a block's RMS), i.e. ~30x inside the 1e-3
// tolerance of the GEMV.  The result is the product of the exactly dequantized
// weights with the rounded activation vector: the block sums used for the
// minima / offsets are sums of the rounded values too.  Everything after the
// sub-block dot product is fp32.
// =========================================================================

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ int sdot4(uint32_t a, uint32_t b, int c) {
    return __builtin_amdgcn_sdot4((int)a, (int)b, c, false);
}

template <int CTRL>
__device__ __forceinline__ float dpp_max(float v) {
    return fmaxf(v, dpp_f32<CTRL>(v));
}

// --- formats: TILE elements per lane, XB elements per activation block ------
struct IFmtQ4K {
    using W = FmtQ4K;
    static constexpr bool F32X = false;
    static constexpr int TILE = 64, XB = 32, NXB = 2, NSUM = 2;
    // element index e of x -> tile, element within tile, block within tile
    __device__ static void locate(uint32_t e, uint32_t &tile, uint32_t &local, uint32_t &xb) {
        tile = e >> 6;
        local = e & 63;
        xb = local >> 5;
    }
    // A lane's tile of the staged activations.
    struct X {
        uint4 xh[4], xl[4];
        float4 mt;  // s0, s1, S0, S1
    };
    // xq: this lane's slot of chunk 0 of the hi plane; chunk c at xq[c*64], lo plane 4 chunks on
    __device__ static void load_x(X &x, const uint4 *xq, const float *meta) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            x.xh[c] = xq[c * 64];
            x.xl[c] = xq[(4 + c) * 64];
        }
        x.mt = *reinterpret_cast<const float4 *>(meta);
    }
    template <int R>
    __device__ static void accumulate(const W::Row (&w)[R], const X &x, uint32_t tile,
                                      float (&acc)[R]) {
        const uint4(&xh)[4] = x.xh;
        const uint4(&xl)[4] = x.xl;
        const float4 mt = x.mt;
        const uint32_t j = tile & 3;
        const uint32_t sh = (j & 1u) * 16u;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            int hlo = 0, llo = 0, hhi = 0, lhi = 0;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const uint32_t q = k < 4 ? (&w[r].qa.x)[k] : (&w[r].qb.x)[k - 4];
                const uint32_t lo = q & 0x0f0f0f0fu, hi = (q >> 4) & 0x0f0f0f0fu;
                hlo = sdot4(lo, (&xh[k >> 2].x)[k & 3], hlo);
                llo = sdot4(lo, (&xl[k >> 2].x)[k & 3], llo);
                hhi = sdot4(hi, (&xh[2 + (k >> 2)].x)[k & 3], hhi);
                lhi = sdot4(hi, (&xl[2 + (k >> 2)].x)[k & 3], lhi);
            }
            const float flo = (float)((hlo << 8) + llo) * mt.x;
            const float fhi = (float)((hhi << 8) + lhi) * mt.y;
            const float d = f16_bits_to_f32((uint16_t)(w[r].hdr.x & 0xffffu));
            const float dmin = f16_bits_to_f32((uint16_t)(w[r].hdr.x >> 16));
            const uint32_t a = (w[r].hdr.y >> sh) & 0xffffu, b = (w[r].hdr.z >> sh) & 0xffffu,
                           c = (w[r].hdr.w >> sh) & 0xffffu;
            uint32_t sc2, m2;
            if (j < 2) {
                sc2 = a & 0x3f3fu;
                m2 = b & 0x3f3fu;
            } else {
                sc2 = (c & 0x0f0fu) | ((a >> 2) & 0x3030u);
                m2 = ((c >> 4) & 0x0f0fu) | ((b >> 2) & 0x3030u);
            }
            float v = (d * ub0(sc2)) * flo;
            v = fmaf(d * ub1(sc2), fhi, v);
            v = fmaf(-dmin, fmaf(ub0(m2), mt.z, ub1(m2) * mt.w), v);
            acc[r] += v;
        }
    }
};

struct IFmtQ6K {
    using W = FmtQ6K;
    static constexpr bool F32X = false;
    static constexpr int TILE = 64, XB = 16, NXB = 4, NSUM = 4;
    __device__ static void locate(uint32_t e, uint32_t &tile, uint32_t &local, uint32_t &xb) {
        const uint32_t blk = e >> 8, i = (e >> 7) & 1, quarter = (e >> 5) & 3, s = (e >> 4) & 1;
        tile = blk * 4 + i * 2 + s;
        xb = quarter;
        local = quarter * 16 + (e & 15);
    }
    struct X {
        uint4 xh[4], xl[4];  // chunk = quarter
        float4 ms, mS;       // scales of the 4 quarters, sums of the rounded values
    };
    __device__ static void load_x(X &x, const uint4 *xq, const float *meta) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            x.xh[c] = xq[c * 64];
            x.xl[c] = xq[(4 + c) * 64];
        }
        x.ms = *reinterpret_cast<const float4 *>(meta);
        x.mS = *reinterpret_cast<const float4 *>(meta + 4);
    }
    template <int R>
    __device__ static void accumulate(const W::Row (&w)[R], const X &x, uint32_t tile,
                                      float (&acc)[R]) {
        const uint4(&xh)[4] = x.xh;
        const uint4(&xl)[4] = x.xl;
        const float4 ms = x.ms, mS = x.mS;
        const uint32_t sb = (tile & 1u) * 8u;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            int h1 = 0, l1 = 0, h2 = 0, l2 = 0, h3 = 0, l3 = 0, h4 = 0, l4 = 0;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const uint32_t L0 = (&w[r].l0.x)[k], L1 = (&w[r].l1.x)[k], H = (&w[r].h.x)[k];
                const uint32_t q1 = (L0 & 0x0f0f0f0fu) | ((H << 4) & 0x30303030u);
                const uint32_t q2 = (L1 & 0x0f0f0f0fu) | ((H << 2) & 0x30303030u);
                const uint32_t q3 = ((L0 >> 4) & 0x0f0f0f0fu) | (H & 0x30303030u);
                const uint32_t q4 = ((L1 >> 4) & 0x0f0f0f0fu) | ((H >> 2) & 0x30303030u);
                h1 = sdot4(q1, (&xh[0].x)[k], h1);
                l1 = sdot4(q1, (&xl[0].x)[k], l1);
                h2 = sdot4(q2, (&xh[1].x)[k], h2);
                l2 = sdot4(q2, (&xl[1].x)[k], l2);
                h3 = sdot4(q3, (&xh[2].x)[k], h3);
                l3 = sdot4(q3, (&xl[2].x)[k], l3);
                h4 = sdot4(q4, (&xh[3].x)[k], h4);
                l4 = sdot4(q4, (&xl[3].x)[k], l4);
            }
            const float f1 = fmaf((float)((h1 << 8) + l1), ms.x, -32.f * mS.x);
            const float f2 = fmaf((float)((h2 << 8) + l2), ms.y, -32.f * mS.y);
            const float f3 = fmaf((float)((h3 << 8) + l3), ms.z, -32.f * mS.z);
            const float f4 = fmaf((float)((h4 << 8) + l4), ms.w, -32.f * mS.w);
            const float sc1 = sb0(w[r].sc.x >> sb), sc2 = sb0(w[r].sc.x >> (sb + 16)),
                        sc3 = sb0(w[r].sc.y >> sb), sc4 = sb0(w[r].sc.y >> (sb + 16));
            float v = sc1 * f1;
            v = fmaf(sc2, f2, v);
            v = fmaf(sc3, f3, v);
            v = fmaf(sc4, f4, v);
            acc[r] = fmaf(f16_bits_to_f32(w[r].d), v, acc[r]);
        }
    }
};

struct IFmtQ8_0 {
    using W = FmtQ8_0;
    static constexpr bool F32X = false;
    static constexpr int TILE = 32, XB = 32, NXB = 1, NSUM = 0;
    __device__ static void locate(uint32_t e, uint32_t &tile, uint32_t &local, uint32_t &xb) {
        tile = e >> 5;
        local = e & 31;
        xb = 0;
    }
    struct X {
        uint4 xh[2], xl[2];
        float s0;
    };
    __device__ static void load_x(X &x, const uint4 *xq, const float *meta) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            x.xh[c] = xq[c * 64];
            x.xl[c] = xq[(2 + c) * 64];
        }
        x.s0 = meta[0];
    }
    template <int R>
    __device__ static void accumulate(const W::Row (&w)[R], const X &x, uint32_t,
                                      float (&acc)[R]) {
        const uint4(&xh)[2] = x.xh;
        const uint4(&xl)[2] = x.xl;
        const float s0 = x.s0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            int h = 0, l = 0;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const uint32_t q = k < 4 ? (&w[r].a.x)[k] : (&w[r].b.x)[k - 4];
                h = sdot4(q, (&xh[k >> 2].x)[k & 3], h);
                l = sdot4(q, (&xl[k >> 2].x)[k & 3], l);
            }
            acc[r] = fmaf(f16_bits_to_f32(w[r].d) * s0, (float)((h << 8) + l), acc[r]);
        }
    }
};

// Bits 0..3 of b moved to bit 4 of bytes 0..3 (the fifth bits of four 5-bit quants).
__device__ __forceinline__ uint32_t spread_bit4(uint32_t b) {
    return ((b * 0x00204081u) & 0x01010101u) << 4;
}

template <bool HAS_M, bool HAS_QH, int B = 1>
struct IFmtLegacy {
    using W = FmtLegacy<HAS_M, HAS_QH, B>;
    static constexpr bool F32X = false;
    static constexpr int TILE = 32 * B, XB = 32, NXB = B, NSUM = B;
    __device__ static void locate(uint32_t e, uint32_t &tile, uint32_t &local, uint32_t &xb) {
        tile = e / TILE;
        local = e % TILE;
        xb = local >> 5;
    }
    struct X {
        uint4 xh[2 * B], xl[2 * B];
        float s[B], S[B];  // scales of the blocks' fixed-point activations, sums of the rounded values
    };
    __device__ static void load_x(X &x, const uint4 *xq, const float *meta) {
#pragma unroll
        for (int c = 0; c < 2 * B; ++c) {
            x.xh[c] = xq[c * 64];
            x.xl[c] = xq[(2 * B + c) * 64];
        }
        __builtin_memcpy(x.s, __builtin_assume_aligned(meta, 8 * B), 4 * B);
        __builtin_memcpy(x.S, meta + B, 4 * B);
    }
    template <int R>
    __device__ static void accumulate(const typename W::Row (&w)[R], const X &x, uint32_t,
                                      float (&acc)[R]) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
#pragma unroll
            for (int b = 0; b < B; ++b) {
                int h = 0, l = 0;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const uint32_t q = (&w[r].q[b].x)[k];
                    uint32_t lo = q & 0x0f0f0f0fu, hi = (q >> 4) & 0x0f0f0f0fu;
                    if constexpr (HAS_QH) {
                        lo |= spread_bit4((w[r].qh[b] >> (4 * k)) & 15u);
                        hi |= spread_bit4((w[r].qh[b] >> (16 + 4 * k)) & 15u);
                    }
                    h = sdot4(lo, (&x.xh[2 * b].x)[k], h);
                    l = sdot4(lo, (&x.xl[2 * b].x)[k], l);
                    h = sdot4(hi, (&x.xh[2 * b + 1].x)[k], h);
                    l = sdot4(hi, (&x.xl[2 * b + 1].x)[k], l);
                }
                const float dot = (float)((h << 8) + l) * x.s[b];  // sum of quant * x over the block
                const float d = W::d(w[r], b);
                if (HAS_M)  // y = d q + m   (quantization.rs:93-96, 160-165)
                    acc[r] += fmaf(d, dot, W::m(w[r], b) * x.S[b]);
                else  // y = d (q - 8) or d (q - 16)   (quantization.rs:62-66, 123-129)
                    acc[r] = fmaf(d, fmaf(HAS_QH ? -16.f : -8.f, x.S[b], dot), acc[r]);
            }
        }
    }
};

struct IFmtQ8K {
    using W = FmtQ8K;
    static constexpr bool F32X = false;
    static constexpr int TILE = 32, XB = 32, NXB = 1, NSUM = 0;
    __device__ static void locate(uint32_t e, uint32_t &tile, uint32_t &local, uint32_t &xb) {
        tile = e >> 5;
        local = e & 31;
        xb = 0;
    }
    using X = IFmtQ8_0::X;
    __device__ static void load_x(X &x, const uint4 *xq, const float *meta) {
        IFmtQ8_0::load_x(x, xq, meta);
    }
    template <int R>
    __device__ static void accumulate(const W::Row (&w)[R], const X &x, uint32_t,
                                      float (&acc)[R]) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            int h = 0, l = 0;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const uint32_t q = k < 4 ? (&w[r].a.x)[k] : (&w[r].b.x)[k - 4];
                h = sdot4(q, (&x.xh[k >> 2].x)[k & 3], h);
                l = sdot4(q, (&x.xl[k >> 2].x)[k & 3], l);
            }
            acc[r] = fmaf(w[r].d * x.s0, (float)((h << 8) + l), acc[r]);
        }
    }
};

struct IFmtQ5K {
    using W = FmtQ5K;
    static constexpr bool F32X = false;
    static constexpr int TILE = 64, XB = 32, NXB = 2, NSUM = 2;
    __device__ static void locate(uint32_t e, uint32_t &tile, uint32_t &local, uint32_t &xb) {
        IFmtQ4K::locate(e, tile, local, xb);
    }
    using X = IFmtQ4K::X;
    __device__ static void load_x(X &x, const uint4 *xq, const float *meta) {
        IFmtQ4K::load_x(x, xq, meta);
    }
    template <int R>
    __device__ static void accumulate(const W::Row (&w)[R], const X &x, uint32_t tile,
                                      float (&acc)[R]) {
        const uint4(&xh)[4] = x.xh;
        const uint4(&xl)[4] = x.xl;
        const float4 mt = x.mt;
        const uint32_t j = tile & 3;
        const uint32_t sh = (j & 1u) * 16u;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            int hlo = 0, llo = 0, hhi = 0, lhi = 0;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const uint32_t q = k < 4 ? (&w[r].qa.x)[k] : (&w[r].qb.x)[k - 4];
                const uint32_t H = (k < 4 ? (&w[r].ha.x)[k] : (&w[r].hb.x)[k - 4]) >> (2 * j);
                const uint32_t lo = (q & 0x0f0f0f0fu) | ((H & 0x01010101u) << 4);
                const uint32_t hi = ((q >> 4) & 0x0f0f0f0fu) | (((H >> 1) & 0x01010101u) << 4);
                hlo = sdot4(lo, (&xh[k >> 2].x)[k & 3], hlo);
                llo = sdot4(lo, (&xl[k >> 2].x)[k & 3], llo);
                hhi = sdot4(hi, (&xh[2 + (k >> 2)].x)[k & 3], hhi);
                lhi = sdot4(hi, (&xl[2 + (k >> 2)].x)[k & 3], lhi);
            }
            const float flo = (float)((hlo << 8) + llo) * mt.x;
            const float fhi = (float)((hhi << 8) + lhi) * mt.y;
            const float d = f16_bits_to_f32((uint16_t)(w[r].hdr.x & 0xffffu));
            const float dmin = f16_bits_to_f32((uint16_t)(w[r].hdr.x >> 16));
            // 6-bit scale / min pairs of sub-blocks 2j and 2j+1 (get_scale_min_k4)
            const uint32_t a = (w[r].hdr.y >> sh) & 0xffffu, b = (w[r].hdr.z >> sh) & 0xffffu,
                           c = (w[r].hdr.w >> sh) & 0xffffu;
            uint32_t sc2, m2;
            if (j < 2) {
                sc2 = a & 0x3f3fu;
                m2 = b & 0x3f3fu;
            } else {
                sc2 = (c & 0x0f0fu) | ((a >> 2) & 0x3030u);
                m2 = ((c >> 4) & 0x0f0fu) | ((b >> 2) & 0x3030u);
            }
            float v = (d * ub0(sc2)) * flo;
            v = fmaf(d * ub1(sc2), fhi, v);
            v = fmaf(-dmin, fmaf(ub0(m2), mt.z, ub1(m2) * mt.w), v);
            acc[r] += v;
        }
    }
};

// The fp32-activation twin of a format: x is staged in LDS as it is (RMSNorm / LayerNorm applied),
// float4 xs[step][chunk][lane] followed by the NSUM sums of x per tile, and the weights are
// expanded with one conversion and one multiply-add per element (FmtQ4K / FmtQ6K / FmtQ8_0
// ::accumulate).  The arithmetic the reference's shaders use (ops/gemv_quant.rs:243-348 multiply
// f32 vectors); about 3 VALU operations per weight against 1 on the integer-dot path.
template <class WFmt>
struct FFmt {
    using W = WFmt;
    static constexpr bool F32X = true;
    static constexpr int TILE = WFmt::TILE, CHUNKS = WFmt::CHUNKS, NSUM = WFmt::NSUM;
    // elements per sum of x
    static constexpr int XB = WFmt::NSUM ? WFmt::TILE / (WFmt::NSUM ? WFmt::NSUM : 1) : WFmt::TILE, NXB = 0;
    struct X {};
};

// Row source / sink of a plain single-matrix GEMV: group g = rows g*R .. g*R+R-1.
template <int EXTRA>
struct PlainPolicy {
    static constexpr bool FULL = EXTRA & EXTRA_FULL;
    static constexpr int S = 1;  // passes per group
    const GemvParams &p;
    // `ok` false: the load still happens, from row-group 0 (a wave's loads are never
    // skipped, see gemv_i8_body)
    template <class WF, int R>
    __device__ void load(typename WF::Row (&w)[R], uint32_t g, uint32_t, uint32_t tile,
                         bool ok) const {
        load_group<WF, R>(w, p, ok ? g : 0u, tile);
    }
    // Lane n holds finished result n of the wave, whose first group is g0: result n
    // belongs to row (g0 + (n / R) * GW) * R + n % R.  The operands the epilogue needs
    // are fetched by prefetch() at kernel start: fetched at the end they would add a
    // memory round trip to every wave's tail.
    float *out;
    float pre_bias, pre_out;
    uint32_t pos;
    __device__ const uint32_t *pos_ptr() const { return p.dyn_pos; }
    __device__ void set_pos(uint32_t fetched) { pos = fetched; }
    // `late` false: at kernel start, whatever does not need the position; true: behind the
    // first weight tiles, once the position is there, the rest.
    template <int R>
    __device__ void prefetch(bool late, uint32_t g0, uint32_t GW, uint32_t my_groups, uint32_t lane) {
        const uint32_t row = (g0 + (lane / R) * GW) * R + lane % R;
        const bool mine = lane < my_groups * R && row < p.nrows;
        if (!late) {
            out = p.out;
            pre_bias = pre_out = 0.f;
            if (mine && p.bias) pre_bias = p.bias[row];
            if (mine && p.accumulate && !p.dyn_pos) pre_out = out[row];
        } else if (p.dyn_pos) {
            out += (size_t)pos * p.out_pos_stride;
            if (mine && p.accumulate) pre_out = out[row];
        }
    }
    template <int R>
    __device__ void finish(float mine, uint32_t n, uint32_t g0, uint32_t GW, uint32_t lane) {
        const uint32_t row = (g0 + (lane / R) * GW) * R + lane % R;
        if (lane < n && row < p.nrows) {
            float v = mine + pre_bias;
            if constexpr (FULL) {
                if (p.act == 1) v = gelu_tanh(v);
            }
            out[row] = v + pre_out;
            if constexpr ((EXTRA & EXTRA_MAXIMA) != 0) mine = v + pre_out;
        }
        if constexpr ((EXTRA & EXTRA_MAXIMA) != 0) {
            // The first of the largest results: rows ascend with the lane.  A sequential scan for v > best from row 0 on
            // passes over NaN, except in row 0, which then stays the best.
            if (!p.maxima) return;
            float v = lane < n && row < p.nrows && mine == mine ? mine : -INFINITY;
            if (row == 0 && mine != mine) v = INFINITY;
            const float best = wave_max(v);
            const uint64_t at = __ballot(lane < n && v == best);
            if (lane == (uint32_t)__builtin_ctzll(at)) p.maxima[g0] = RowMaximum{best, row};
        }
    }
};

// The body shared by the single-matrix and the fused multi-matrix kernels.  `p`
// supplies x, ncols and the optional norm folding; `pol` the rows.
// The workgroup is number `wg` of the `nwg` that share the matrix; its waves
// w < nw take the row-groups (wg * nw + w) + i * (nwg * nw) < ngroups, so that at
// any time the machine reads one contiguous window of the matrix.  A group is
// Policy::S passes over R rows each (a fused pair is two single-row passes of
// the same wave).  The (group, pass, step) triples
// of a wave form one sequence that is software-pipelined D deep.
// LDS: uint4 xq[step][plane(2)][chunk(PCH)][lane(64)], then float meta[tile][MF].
// XREG: rows fit one step (ncols <= 64 tiles), so a lane's tile of x is the same
// for every row and is read from LDS once instead of once per row.
// XPART: x is not read from p.x but merged from attention partial results (merged_partials).
// FULL: x may go through a LayerNorm (p.ln_g) on its way, and results through an activation.
template <class F, int R, int D, bool XREG, class Policy, bool XPART = false, bool FULL = false>
__device__ __forceinline__ void gemv_i8_body(const GemvParams &p, Policy &pol, uint32_t wg,
                                             uint32_t nwg, uint32_t nw, uint32_t ngroups) {
    using WF = typename F::W;
    constexpr int S = Policy::S;
    constexpr int PCH = F::TILE / 16;         // 16-byte chunks per plane per tile
    constexpr int MF = F::NXB + F::NSUM;      // floats of meta per tile
    constexpr int LPB = F::XB / 4;            // lanes (float4) per activation block (fp32: per sum)
    static_assert(!(F::F32X && XREG), "fp32 activations are read from LDS tile by tile");
    extern __shared__ float4 smem4[];
    uint4 *xq = reinterpret_cast<uint4 *>(smem4);
    // the wave index is read through readfirstlane: the compiler then knows that it,
    // and the loop control derived from it, are the same in every lane (scalar registers
    // and branches instead of vector compares and masks)
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t nwaves = blockDim.x >> 6;
    const uint32_t ntiles = p.ncols / F::TILE;
    const uint32_t nsteps = (ntiles + 63) >> 6;
    const uint32_t ntiles_pad = nsteps << 6;
    float *meta = reinterpret_cast<float *>(xq + (size_t)ntiles_pad * 2 * PCH);
    // fp32 activations: the tile sums follow the ntiles_pad * CHUNKS float4 of x
    float *fsums = reinterpret_cast<float *>(smem4 + (size_t)ntiles_pad * (F::TILE / 4));

    const uint32_t first = wg * nw + wave, GW = nwg * nw;
    const uint32_t my_groups = (wave < nw && first < ngroups) ? (ngroups - first + GW - 1) / GW : 0;
    const uint32_t n_it = my_groups * S * nsteps;

    // the epilogue's operands that do not depend on the position (bias, RoPE table entry,
    // the value to accumulate into) are requested before anything else
    pol.template prefetch<R>(false, first, GW, my_groups, lane);

    // The requests for x go out first, the first D weight requests after them: a
    // wave's loads return in order, so x, a cache hit, is not held up behind the
    // weights and is staged while they are in flight.
    // The position (when it lives in device memory) is requested by a vector load ahead of
    // x: it returns in order with x, so it is there once x has been staged, and no scalar
    // round trip for it stands between the kernel's start and its first weight request.
    const uint32_t *pos_src = pol.pos_ptr();
    uint32_t pos_fetched = 0;
    if (pos_src) pos_fetched = pos_src[opaque(0u)];
    constexpr int XP = 3;  // float4 of x per thread requested up front
    const float4 *x4 = reinterpret_cast<const float4 *>(p.x);
    const float4 *nw4 = reinterpret_cast<const float4 *>(p.norm_w);
    const uint32_t n4 = p.ncols >> 2;
    // (The x loads stay under their conditions: clamping the out-of-range ones to a
    // valid address instead makes every idle thread of the machine hit the same
    // cache line, which cost 1 us on a 4096x4096 launch.)
    // nv: the RMSNorm weights, or gamma of a folded LayerNorm; bv: its beta.  They are
    // requested here, ahead of the weights, so that waiting for them later does not
    // mean waiting for a weight tile.
    // Only the first `ns` waves stage x (as few as cover it with their XP float4 per lane,
    // in fours so that every SIMD takes part): the waves of a 1024-thread workgroup start
    // up to a microsecond apart, and the staging would otherwise end a whole prologue after
    // the last of them has arrived.  The other waves request their weights and wait at the
    // barrier.  (The folded LayerNorm has barriers of its own, so there every wave stages.)
    // (Merging partial results is several loads per float4: every wave takes a share.)
    uint32_t ns = ((n4 + 64 * XP - 1) / (64 * XP) + 3) & ~3u;
    const float *const ln_g = FULL ? p.ln_g : nullptr;
    if (ns > nwaves || ln_g || XPART) ns = nwaves;
    // LayerNorm of up to LN_ROW float4: as many waves as hold them at one per lane stage, and each of these reads the
    // whole vector and finds its mean and variance by itself.  Shared out over all waves that is two more barriers
    // (with kernels without arguments of a second mode: GPT-2 124M in Q8_0 205 us per token -> 190, from an F16 file 331 -> 290).
    constexpr int LN_REGS = 4;
    constexpr uint32_t LN_ROW = 64 * LN_REGS;
    const bool ln_row = ln_g && n4 <= LN_ROW;
    if (ln_row) ns = (n4 + 63) / 64;
    const bool stager = wave < ns;
    // a wave with neither rows nor a share of x is done: the barrier below counts only the
    // waves that are still running, and it would be the last to reach it
    if (n_it == 0 && !stager) return;
    const uint32_t sthreads = ns * 64;
    float4 xv[XP], nv[XP], bv[XP];
    const float4 *gsrc = ln_g ? reinterpret_cast<const float4 *>(ln_g) : nw4;
    const float4 *bsrc = FULL ? reinterpret_cast<const float4 *>(p.ln_b) : nullptr;
#pragma unroll
    for (int i = 0; i < XP; ++i) {
        xv[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        nv[i] = make_float4(1.f, 1.f, 1.f, 1.f);
        bv[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    // such a row takes the places of the second and third float4, which nobody has then (sixteen registers of its own: 128 and a
    // spill in the Q/K/V kernel of Q5_1)
    auto row_part = [&](int i) -> float4 & { return i < 2 ? xv[1 + i] : nv[i - 1]; };
    if constexpr (FULL) {
        if (ln_row && stager) {
#pragma unroll
            for (int i = 0; i < LN_REGS; ++i)
                row_part(i) = lane + 64 * i < n4 ? x4[lane + 64 * i] : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    }
#pragma unroll
    for (int i = 0; i < XP; ++i) {
        const uint32_t g4 = stager ? tid + i * sthreads : n4;
        if (g4 < n4) {
            if constexpr (!XPART) xv[i] = x4[g4];
            if (gsrc) nv[i] = gsrc[g4];
            if (ln_g && bsrc) bv[i] = bsrc[g4];
        }
    }
    // XPART: the first eight partial results of each thread's first float4 are requested here,
    // ahead of the weights, and merged in stage_x once they are there (merging them here would
    // put a memory round trip in front of the first weight request)
    PartialChunk early;
    if constexpr (XPART) {
        load_partials(early, p, min(tid, n4 - 1), 0);  // unconditional, see there
        // the compiler must not move the weight requests below ahead of these (a wave's loads
        // return in the order they were issued)
        asm volatile("" ::: "memory");
    }

    // Stage x as 16-bit block fixed point (two int8 planes) + per-block scale and sum.
    // A fused RMSNorm costs no extra pass and no extra barrier: the normalisation
    // factor rsqrt(mean(x^2) + eps) is one scalar for the whole vector, so x * w is
    // staged, the sum of squares is gathered on the way and the factor multiplies
    // the finished dot products instead.
    __shared__ float red[16], red_a[16], red_b[16];
    auto stage_x = [&]() -> float {
        float out_scale = 1.f;
        uint32_t *xq32 = reinterpret_cast<uint32_t *>(xq);
        float ss = 0.f;
        if constexpr (XPART) {  // every wave stages (sthreads == blockDim.x)
            if (tid < n4) xv[0] = merged_partials(p, tid, early);
#pragma unroll
            for (int i = 1; i < XP; ++i)
                if (tid + i * sthreads < n4) xv[i] = merged_partials(p, tid + i * sthreads);
        }
        if constexpr (FULL) if (ln_row) {
            float s1 = 0.f;
#pragma unroll
            for (int i = 0; i < LN_REGS; ++i) {
                const float4 v = row_part(i);
                s1 += (v.x + v.y) + (v.z + v.w);
            }
            const float mean = wave_sum(s1) / (float)p.ncols;
            float s2 = 0.f;
#pragma unroll
            for (int i = 0; i < LN_REGS; ++i) {
                const bool there = lane + 64 * i < n4;
                const float4 v = row_part(i);
                const float a = there ? v.x - mean : 0.f, b = there ? v.y - mean : 0.f, c = there ? v.z - mean : 0.f,
                            d = there ? v.w - mean : 0.f;
                s2 = fmaf(a, a, s2);
                s2 = fmaf(b, b, s2);
                s2 = fmaf(c, c, s2);
                s2 = fmaf(d, d, s2);
            }
            const float rstd = 1.0f / sqrtf(wave_sum(s2) / (float)p.ncols + 1.0e-5f);
            xv[0].x = ((xv[0].x - mean) * rstd) * nv[0].x + bv[0].x;
            xv[0].y = ((xv[0].y - mean) * rstd) * nv[0].y + bv[0].y;
            xv[0].z = ((xv[0].z - mean) * rstd) * nv[0].z + bv[0].z;
            xv[0].w = ((xv[0].w - mean) * rstd) * nv[0].w + bv[0].w;
        } else if (ln_g) {
            // LayerNorm folded in (host guarantees that the XP float4 per thread cover
            // x): mean, then variance about the mean (two exact passes over registers,
            // ops/layernorm.rs:46-53), then x <- (x - mean) * rstd * gamma + beta.
            auto block_total = [&](float v, float *buf) {
                v = wave_sum(v);
                if (lane == 0) buf[wave] = v;
                __syncthreads();
                const float part = lane < nwaves ? buf[lane] : 0.f;
                return readlane_f32(row16_sum(part), 0);
            };
            float s1 = 0.f;
#pragma unroll
            for (int i = 0; i < XP; ++i)
                if (tid + i * blockDim.x < n4) s1 += (xv[i].x + xv[i].y) + (xv[i].z + xv[i].w);
            const float mean = block_total(s1, red_a) / (float)p.ncols;
            float s2 = 0.f;
#pragma unroll
            for (int i = 0; i < XP; ++i) {
                if (tid + i * blockDim.x < n4) {
                    xv[i].x -= mean;
                    xv[i].y -= mean;
                    xv[i].z -= mean;
                    xv[i].w -= mean;
                    s2 = fmaf(xv[i].x, xv[i].x, s2);
                    s2 = fmaf(xv[i].y, xv[i].y, s2);
                    s2 = fmaf(xv[i].z, xv[i].z, s2);
                    s2 = fmaf(xv[i].w, xv[i].w, s2);
                }
            }
            const float rstd = 1.0f / sqrtf(block_total(s2, red_b) / (float)p.ncols + 1.0e-5f);
#pragma unroll
            for (int i = 0; i < XP; ++i) {
                const uint32_t g4 = tid + i * blockDim.x;
                if (g4 < n4) {
                    const float4 ga = nv[i], be = bv[i];
                    xv[i].x = (xv[i].x * rstd) * ga.x + be.x;
                    xv[i].y = (xv[i].y * rstd) * ga.y + be.y;
                    xv[i].z = (xv[i].z * rstd) * ga.z + be.z;
                    xv[i].w = (xv[i].w * rstd) * ga.w + be.w;
                }
            }
        }
        auto stage_one = [&](uint32_t g4, float4 v, const float4 nw) {
            if constexpr (F::F32X) {
                if (p.norm_w) {
                    ss = fmaf(v.x, v.x, ss);
                    ss = fmaf(v.y, v.y, ss);
                    ss = fmaf(v.z, v.z, ss);
                    ss = fmaf(v.w, v.w, ss);
                    v.x *= nw.x;
                    v.y *= nw.y;
                    v.z *= nw.z;
                    v.w *= nw.w;
                }
                uint32_t tile, chunk;
                WF::map(g4, tile, chunk);
                smem4[lds_slot<WF>(tile, chunk)] = v;
                if constexpr (F::NSUM > 0) {
                    // the sum of x over the LPB consecutive float4 that one sum covers
                    float sum = (v.x + v.y) + (v.z + v.w);
                    sum += dpp_f32<0xB1>(sum);
                    sum += dpp_f32<0x4E>(sum);
                    if (LPB == 8) sum += dpp_f32<0x141>(sum);
                    constexpr int CPS = F::CHUNKS / F::NSUM;  // chunks per sum
                    if ((g4 & (LPB - 1)) == 0) fsums[tile * F::NSUM + chunk / CPS] = sum;
                }
            } else {
            if (p.norm_w) {
                ss = fmaf(v.x, v.x, ss);
                ss = fmaf(v.y, v.y, ss);
                ss = fmaf(v.z, v.z, ss);
                ss = fmaf(v.w, v.w, ss);
                v.x *= nw.x;
                v.y *= nw.y;
                v.z *= nw.z;
                v.w *= nw.w;
            }
            float amax = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
            float sum;
            amax = dpp_max<0xB1>(amax);
            amax = dpp_max<0x4E>(amax);
            if (LPB == 8) amax = dpp_max<0x141>(amax);
            const float inv = amax > 0.f ? 32512.f / amax : 0.f;
            const int X0 = __float2int_rn(v.x * inv), X1 = __float2int_rn(v.y * inv),
                      X2 = __float2int_rn(v.z * inv), X3 = __float2int_rn(v.w * inv);
            // block sum of the *rounded* activations, so that the minima / offset terms
            // see exactly the same vector as the dot products (exact in fp32: |sum| < 2^21)
            sum = (float)((X0 + X1) + (X2 + X3));
            sum += dpp_f32<0xB1>(sum);
            sum += dpp_f32<0x4E>(sum);
            if (LPB == 8) sum += dpp_f32<0x141>(sum);
            sum *= amax * (1.0f / 32512.f);
            // X = 256 hi + lo with lo the sign-extended low byte: lo is byte 0 of X as it stands
            // and hi = (X + 128) >> 8 is byte 1 of X + 128 (|X| <= 32512, so 16 bits hold both).
            // Two values per register as 16-bit halves, one packed add, and two byte
            // permutes gather the four lo bytes and the four hi bytes.
            const uint32_t p01 = __builtin_amdgcn_perm((uint32_t)X1, (uint32_t)X0, 0x05040100u);
            const uint32_t p23 = __builtin_amdgcn_perm((uint32_t)X3, (uint32_t)X2, 0x05040100u);
            const u16x2 bias128 = {128, 128};
            u16x2 y01, y23;
            __builtin_memcpy(&y01, &p01, 4);
            __builtin_memcpy(&y23, &p23, 4);
            y01 += bias128;
            y23 += bias128;
            uint32_t q01, q23;
            __builtin_memcpy(&q01, &y01, 4);
            __builtin_memcpy(&q23, &y23, 4);
            const uint32_t lo = __builtin_amdgcn_perm(p23, p01, 0x06040200u);
            const uint32_t hi = __builtin_amdgcn_perm(q23, q01, 0x07050301u);
            uint32_t tile, local, xb;
            F::locate(g4 * 4, tile, local, xb);
            const uint32_t dl = local >> 2, chunk = dl >> 2, sub = dl & 3;
            const uint32_t slot = ((tile >> 6) * 2 * PCH + chunk) * 64 + (tile & 63);
            xq32[(size_t)slot * 4 + sub] = hi;
            xq32[(size_t)(slot + PCH * 64) * 4 + sub] = lo;
            if ((g4 & (LPB - 1)) == 0) {
                meta[tile * MF + xb] = amax * (1.0f / 32512.f);
                if (F::NSUM > 0) meta[tile * MF + F::NXB + xb] = sum;
            }
            }  // integer-dot staging
        };
        // ncols is a multiple of the tile size, so the LPB lanes of a block are
        // active together in every one of these branches
#pragma unroll
        for (int i = 0; i < XP; ++i) {
            const uint32_t g4 = stager ? tid + i * sthreads : n4;
            if (g4 < n4) stage_one(g4, xv[i], nv[i]);
        }
        for (uint32_t g4 = stager ? tid + XP * sthreads : n4; g4 < n4; g4 += sthreads)
            stage_one(g4, XPART ? merged_partials(p, g4) : x4[g4],
                      p.norm_w ? nw4[g4] : make_float4(1.f, 1.f, 1.f, 1.f));
        if (p.norm_w && stager) {
            ss = wave_sum(ss);
            if (lane == 0) red[wave] = ss;
        }
        __syncthreads();
        if (p.norm_w) {
            // one LDS read per lane and a 16-lane DPP sum instead of a chain of
            // dependent reads (a workgroup has at most 16 waves; only the staging ones
            // have written a partial sum)
            const float part = lane < ns ? red[lane] : 0.f;
            const float total = readlane_f32(row16_sum(part), 0);
            out_scale = 1.0f / sqrtf(total / (float)p.ncols + p.norm_eps);
        }
        return out_scale;
    };

    // The weight loads below and in the main loop are issued unconditionally (a lane
    // without a tile re-reads tile 0; a register set beyond the wave's last iteration
    // re-reads the wave's own first tile, a cache hit).  Only then can the compiler
    // count the loads in flight and wait for exactly the one it needs: with a load
    // under a condition it falls back to waiting for all of them, and the staging of
    // x, a cache hit, would wait for the first weight tile to arrive from HBM.
    // A wave without any row re-reads row-group 0: the host sizes the workgroups so that
    // only the last one can have such waves (thousands of idle waves asking for one and
    // the same tile would queue up on a single cache line).
    typename WF::Row w[D][R];
    uint32_t lg = first, lsub = 0, ls = 0;  // (group, pass, step) of the next load
    // A wave's finished row sums are parked one per lane (result n in lane n) until the
    // policy's epilogue at the end, so a wave takes at most 64 results: the host sizes
    // the grid accordingly (plan_groups).  The loads of the first D iterations go out
    // here; with fewer than D iterations the other register sets take a dummy load and
    // are never consumed.
    auto advance_load_cursor = [&]() {
        if (++ls == nsteps) {
            ls = 0;
            if (++lsub == S) {
                lsub = 0;
                lg += GW;
            }
        }
    };
#pragma unroll
    for (int d = 0; d < D; ++d) {
        const bool ok = (uint32_t)d < n_it;
        const uint32_t tile = ok ? ls * 64 + lane : lane;
        // no tile left: the wave's own first one again, or, for a wave without rows, the
        // first one of its workgroup (a hit in the CU's cache either way)
        const uint32_t spare = n_it ? first : (wg * nw < ngroups ? wg * nw : 0u);
        pol.template load<WF, R>(w[d], ok ? lg : spare, ok ? lsub : 0u, tile < ntiles ? tile : 0u, true);
        if (ok) advance_load_cursor();
    }

    const float out_scale = stage_x();
    if (n_it == 0) return;
    // The epilogue's operands whose addresses depend on the position are requested here,
    // behind the first weight tiles: the position is a second memory round trip away from
    // the kernel arguments, and nothing before this point waits for it.
    pol.set_pos((uint32_t)__builtin_amdgcn_readfirstlane((int)pos_fetched));
    pol.template prefetch<R>(true, first, GW, my_groups, lane);

    // XREG: a lane without a tile (rows shorter than 64 tiles) keeps an all-zero tile of
    // x, so that the row loop needs no condition on the lane
    typename F::X xr{};
    if constexpr (XREG) {
        if (lane < ntiles) F::load_x(xr, xq + lane, meta + (size_t)lane * MF);
    }
    uint32_t step = 0;  // step within the row being computed
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.f;
    uint32_t nres = 0;
    float mine = 0.f;
    // one iteration on a register set: the dot products of a tile, and the row
    // reduction when the row is complete (no memory operation, LDS aside)
    auto compute = [&](typename WF::Row(&wd)[R]) {
        const uint32_t tile = step * 64 + lane;
        if constexpr (F::F32X) {
            if (tile < ntiles)
                WF::template accumulate<R>(wd, smem4 + (size_t)step * F::CHUNKS * 64 + lane,
                                           fsums + (size_t)tile * F::NSUM, tile, acc);
        } else if constexpr (XREG) {
            F::template accumulate<R>(wd, xr, lane, acc);
        } else if (tile < ntiles) {
            typename F::X xt;
            F::load_x(xt, xq + (size_t)step * 2 * PCH * 64 + lane, meta + (size_t)tile * MF);
            F::template accumulate<R>(wd, xt, tile, acc);
        }
        if (XREG || ++step == nsteps) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const float t = wave_sum(acc[r]) * out_scale;
                mine = lane == nres ? t : mine;
                ++nres;
                acc[r] = 0.f;
            }
            step = 0;
        }
    };
    // refills a register set with the next triple of the load cursor
    auto refill = [&](typename WF::Row(&wd)[R]) {
        const uint32_t tile_n = ls * 64 + lane;
        pol.template load<WF, R>(wd, lg, lsub, tile_n < ntiles ? tile_n : 0u, true);
        advance_load_cursor();
    };
    // The last K < 2 D iterations as straight-line code: iteration i runs on
    // register set i mod D and refills it only if iteration i + D exists.  No load sits
    // under a run-time condition, so every wait is for exactly the tile that is needed.
    auto tail = [&](auto kc) {
        constexpr int K = decltype(kc)::value;
#pragma unroll
        for (int i = 0; i < K; ++i) {
            compute(w[i % D]);
            if (i + D < K) refill(w[i % D]);
        }
    };
    uint32_t left = n_it;
    // rounds of D iterations whose refills all exist
    for (; left >= 2u * D; left -= D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            compute(w[d]);
            refill(w[d]);
        }
    }
    switch (left) {  // 1 .. 2 D - 1
#define WGML_TAIL_CASE(K)                                                 \
    case K:                                                               \
        if constexpr (K < 2 * D) tail(std::integral_constant<int, K>{});  \
        break;
        WGML_TAIL_CASE(1)
        WGML_TAIL_CASE(2)
        WGML_TAIL_CASE(3)
        WGML_TAIL_CASE(4)
        WGML_TAIL_CASE(5)
        WGML_TAIL_CASE(6)
        WGML_TAIL_CASE(7)
#undef WGML_TAIL_CASE
    default: break;
    }
    // The policy's epilogue: its loads (bias, RoPE table, the value to accumulate into)
    // were requested at kernel start, its stores come after the last weight tile.
    pol.template finish<R>(mine, nres, first, GW, lane);
}

// MINW: waves per SIMD the register allocation must leave room for (MAXT / 256 = one
// workgroup per CU; twice that caps the kernel at 64 vector registers, so that two
// 1024-thread workgroups share a CU).
template <class F, int R, int D, int MAXT, int MINW = MAXT / 256, bool XPART = false, int EXTRA = 0>
__global__ __launch_bounds__(MAXT, MINW) void gemv_quant_i8_kernel(const GemvParams p) {
    using Policy = PlainPolicy<EXTRA>;
    constexpr bool FULL = Policy::FULL;
    Policy pol{p, nullptr, 0.f, 0.f, 0};
    const uint32_t ngroups = (p.nrows + R - 1) / R;
    if constexpr (!F::F32X) {
        if (p.ncols <= 64 * F::TILE) {
            gemv_i8_body<F, R, D, true, Policy, XPART, FULL>(p, pol, blockIdx.x, gridDim.x,
                                                             p.active_waves, ngroups);
            return;
        }
    }
    gemv_i8_body<F, R, D, false, Policy, XPART, FULL>(p, pol, blockIdx.x, gridDim.x, p.active_waves,
                                                      ngroups);
}

// ------------------------------------------------------------------------
// Fused multi-matrix launches.  Up to three matrices that consume the same input vector share one launch
// (Q, K and V): each workgroup works on one of them (so mixed quantization formats are fine: the format
// decides the workgroup's staging layout and inner loop), and the row pairs of a wave get an epilogue:
//   PLAIN  out[row] = dot (+ bias) (+ out)
//   ROPE   the pair (2g, 2g+1) is rotated by the RoPE angle of pair g before it
//          is stored (ops/rope.wgsl:35-58, adjacent-pair variant)
// Outputs may be displaced by pos * out_pos_stride (KV-cache column of the current position).
// A gate and an up matrix share one launch of another kernel (GatedPolicy):
//   SILU   the wave holds row g of the gate matrix and row g of the up matrix and
//          stores up * gate / (1 + exp(-gate))   (ops/silu.wgsl:13-27)
// One kernel for all three modes took longer: the arguments lie in memory that no cache holds when a launch starts (two
// unused job records of 112 bytes 0.24 us), and both matrices' planes were fetched and picked from (0.35 us).  us per launch in a
// recorded graph, Q8_0: gate and up 768x288 4.01 -> 3.12, plain rows 3.81 -> 3.38 (the single-matrix kernel 2.8); gate and
// up 11008x4096 in Q4_K 12.6 -> 11.8.
enum { JOB_PLAIN = 0, JOB_ROPE = 1, JOB_SILU = 2 };

struct GemvJob {
    const uint8_t *a0, *a1, *a2, *a3;  // matrix planes
    float *out;
    const float *bias;
    uint32_t nrows;
    uint32_t kind;  // format, mode and whether out is added to: GEMV_KIND
    uint32_t out_pos_stride;
    uint32_t wg_begin, wg_count;  // workgroups assigned to this matrix
    uint32_t active_waves;        // waves of a workgroup that walk its row pairs
    __host__ __device__ int type() const { return (int)(kind & 0xffu); }
    __host__ __device__ int mode() const { return (int)((kind >> 8) & 0xffu); }
    __device__ bool accumulate() const { return kind >> 16; }
};
constexpr uint32_t gemv_kind(int type, int mode, int accumulate) {
    return (uint32_t)type | (uint32_t)mode << 8 | (accumulate ? 1u << 16 : 0u);
}

struct FusedParams {
    GemvJob jobs[3];
    const float *ln_g, *ln_b;
    const float *x;
    uint32_t ncols;
    float norm_eps;
    const float *norm_w;
    DynPos pos;
    uint32_t head_size;
    float rope_base;
    const float2 *rope_cs;  // optional: (cos, sin) of the current position per pair of a head
    // The first field a workgroup needs sits in the last cache line of the arguments, so that
    // the first batch of scalar loads touches every line (a line first touched by a later
    // batch is another round trip to memory).
    int njobs;
};

// A group is the pair of rows 2g and 2g+1, whose tiles a wave loads together and multiplies with one
// read of its tile of x.
struct JobPolicy {
    static constexpr int S = 1;
    const GemvJob &j;
    const GemvParams &p;
    DynPos dpos;
    uint32_t head_size;
    float rope_base;
    const float2 *rope_cs;
    template <class WF, int R>
    __device__ void load(typename WF::Row (&w)[R], uint32_t g, uint32_t, uint32_t tile,
                         bool ok) const {
        static_assert(R == 2, "fused launches work on row pairs");
        if (!ok) g = 0;
        WF::load(w[0], WF::row_base(p, 2 * g), tile);
        WF::load(w[1], WF::row_base(p, min(2 * g + 1, j.nrows - 1)), tile);
    }
    // Lanes 2i and 2i+1 hold the two results of group g0 + i * GW.  prefetch()
    // fetches what the epilogue of the first segment needs at kernel start.
    float pre_bias, pre_out;
    float2 pre_cs;
    uint32_t pos;
    __device__ const uint32_t *pos_ptr() const { return dpos.ptr; }
    __device__ void set_pos(uint32_t fetched) { pos = dpos.ptr ? fetched : dpos.val; }
    __device__ float2 rope_entry(uint32_t row) const {
        if (rope_cs) return rope_cs[((row & ~1u) % head_size) >> 1];
        const float head_dim = (float)((row & ~1u) % head_size);
        const float theta = powf(rope_base, -head_dim / (float)head_size);
        float sn, cs;
        sincosf((float)pos * theta, &sn, &cs);
        return make_float2(cs, sn);
    }
    template <int R>
    __device__ void prefetch(bool late, uint32_t g0, uint32_t GW, uint32_t my_groups, uint32_t lane) {
        if (!late) {
            pre_bias = pre_out = 0.f;
            pre_cs = make_float2(1.f, 0.f);
        }
        const uint32_t row = 2 * (g0 + (lane >> 1) * GW) + (lane & 1);
        if (!(lane < 2 * my_groups && row < j.nrows)) return;
        // what depends on the position waits for the late call: the output column of a
        // position-strided destination, and RoPE angles when there is no table of them
        const bool out_needs_pos = dpos.ptr && j.out_pos_stride;
        const bool cs_needs_pos = dpos.ptr && !rope_cs;
        if (!late) {
            if (j.bias) pre_bias = j.bias[row];
            if (j.accumulate() && !out_needs_pos) pre_out = (j.out + (size_t)dpos.val * j.out_pos_stride)[row];
            if (j.mode() == JOB_ROPE && !cs_needs_pos) {
                pos = dpos.val;
                pre_cs = rope_entry(row);
            }
        } else {
            if (j.accumulate() && out_needs_pos) pre_out = (j.out + (size_t)pos * j.out_pos_stride)[row];
            if (j.mode() == JOB_ROPE && cs_needs_pos) pre_cs = rope_entry(row);
        }
    }
    template <int R>
    __device__ void finish(float mine, uint32_t n, uint32_t g0, uint32_t GW, uint32_t lane) {
        const uint32_t g = g0 + (lane >> 1) * GW, sub = lane & 1;
        const bool valid = lane < n;
        float *out = j.out + (size_t)pos * j.out_pos_stride;
        const uint32_t row = 2 * g + sub;
        float t = mine + pre_bias;
        if (j.mode() == JOB_ROPE) {  // ROPE matrices have an even number of rows
            const float other = dpp_f32<0xB1>(t);
            // (x, y) = (even row, odd row):  x' = cs x - sn y,  y' = sn x + cs y
            t = sub ? pre_cs.y * other + pre_cs.x * t : pre_cs.x * t - pre_cs.y * other;
        }
        if (valid && row < j.nrows) out[row] = j.accumulate() ? pre_out + t : t;
    }
};

// Row g of the gate matrix and row g of the up matrix.
struct GatedPolicy {
    static constexpr int S = 1;
    const GemvParams &gate, &up;
    template <class WF, int R>
    __device__ void load(typename WF::Row (&w)[R], uint32_t g, uint32_t, uint32_t tile, bool ok) const {
        static_assert(R == 2, "fused launches work on row pairs");
        if (!ok) g = 0;
        WF::load(w[0], WF::row_base(gate, g), tile);
        WF::load(w[1], WF::row_base(up, g), tile);
    }
    __device__ const uint32_t *pos_ptr() const { return nullptr; }
    __device__ void set_pos(uint32_t) {}
    template <int R>
    __device__ void prefetch(bool, uint32_t, uint32_t, uint32_t, uint32_t) {}
    template <int R>
    __device__ void finish(float mine, uint32_t n, uint32_t g0, uint32_t GW, uint32_t lane) {
        const float u = dpp_f32<0xB1>(mine);  // the neighbouring lane's value
        if (lane < n && (lane & 1) == 0) gate.out[g0 + (lane >> 1) * GW] = u * (mine / (1.0f + expf(-mine)));
    }
};

template <class F, int D, bool FULL>
__device__ __forceinline__ void fused_job_body(const FusedParams &P, const GemvJob &j) {
    GemvParams p{};
    p.x = P.x;
    p.ncols = P.ncols;
    p.norm_w = P.norm_w;
    p.norm_eps = P.norm_eps;
    if constexpr (FULL) {
        p.ln_g = P.ln_g;
        p.ln_b = P.ln_b;
    }
    p.nrows = j.nrows;
    p.p0 = j.a0;
    p.p1 = j.a1;
    p.p2 = j.a2;
    p.p3 = j.a3;
    JobPolicy pol{j, p, P.pos, P.head_size, P.rope_base, P.rope_cs, 0.f, 0.f, make_float2(1.f, 0.f), 0};
    const uint32_t ngroups = (j.nrows + 1) / 2, wg = blockIdx.x - j.wg_begin;
    if constexpr (!F::F32X) {
        if (P.ncols <= 64 * F::TILE) {
            gemv_i8_body<F, 2, D, true, JobPolicy, false, FULL>(p, pol, wg, j.wg_count, j.active_waves, ngroups);
            return;
        }
    }
    gemv_i8_body<F, 2, D, false, JobPolicy, false, FULL>(p, pol, wg, j.wg_count, j.active_waves, ngroups);
}

// The format struct of a GGUF type: integer-dot (F32 false) or fp32-activation.
template <int TYPE, bool F32> struct FusedFmt;
template <> struct FusedFmt<WGML_Q4_K, false> { using T = IFmtQ4K; };
template <> struct FusedFmt<WGML_Q6_K, false> { using T = IFmtQ6K; };
template <> struct FusedFmt<WGML_Q8_0, false> { using T = IFmtQ8_0; };
template <> struct FusedFmt<WGML_Q4_K, true> { using T = FFmt<FmtQ4K>; };
template <> struct FusedFmt<WGML_Q6_K, true> { using T = FFmt<FmtQ6K>; };
template <> struct FusedFmt<WGML_Q8_0, true> { using T = FFmt<FmtQ8_0>; };
// (WGML_F32 is 0, which as FMT stands for mixed formats)
constexpr int kFusedDenseF32 = 1000, kFusedDenseF16 = 1001, kFusedDenseMix = 1002;
template <> struct FusedFmt<kFusedDenseF32, true> { using T = FFmt<FmtF32>; };
template <> struct FusedFmt<kFusedDenseF16, true> { using T = FFmt<FmtF16>; };
template <> struct FusedFmt<kFusedDenseMix, true> { using T = FFmt<FmtDenseMix>; };
// A format number for kernels whose tiles are two blocks of a 32-element format.
constexpr int kLegacyWide = 2000;
template <> struct FusedFmt<WGML_Q5_K, false> { using T = IFmtQ5K; };
template <> struct FusedFmt<WGML_Q8_K, false> { using T = IFmtQ8K; };
template <> struct FusedFmt<WGML_Q4_0, false> { using T = IFmtLegacy<false, false>; };
template <> struct FusedFmt<WGML_Q4_1, false> { using T = IFmtLegacy<true, false>; };
template <> struct FusedFmt<WGML_Q5_0, false> { using T = IFmtLegacy<false, true>; };
template <> struct FusedFmt<WGML_Q5_1, false> { using T = IFmtLegacy<true, true>; };
// the same with tiles of two blocks (kLegacyWide)
template <> struct FusedFmt<kLegacyWide + WGML_Q4_0, false> { using T = IFmtLegacy<false, false, 2>; };
template <> struct FusedFmt<kLegacyWide + WGML_Q4_1, false> { using T = IFmtLegacy<true, false, 2>; };
template <> struct FusedFmt<kLegacyWide + WGML_Q5_0, false> { using T = IFmtLegacy<false, true, 2>; };
template <> struct FusedFmt<kLegacyWide + WGML_Q5_1, false> { using T = IFmtLegacy<true, true, 2>; };

// MINW: waves per SIMD the register budget must allow.  FMT: 0 = the matrices of
// a launch may differ in format (Q4_K / Q6_K / Q8_0, decided per workgroup), else the one
// format all of them have (smaller code, registers of that format only).  F32: fp32
// activations (the three main formats only).
template <int D, int MAXT, int MINW, int FMT, bool F32 = false, bool FULL = false>
__global__ __launch_bounds__(MAXT, MINW) void gemv_fused_kernel(const FusedParams P) {
    // All three job records are fetched at once and the workgroup's own is picked field by
    // field afterwards: indexing the kernel arguments with the job number would put a second
    // scalar-memory round trip (a microsecond when the arguments come from HBM) in front of
    // the first weight request.
    const bool is1 = P.njobs > 1 && blockIdx.x >= P.jobs[1].wg_begin;
    const bool is2 = P.njobs > 2 && blockIdx.x >= P.jobs[2].wg_begin;
    const GemvJob &j0 = P.jobs[0], &j1 = P.jobs[1], &j2 = P.jobs[2];
#define WGML_PICK(f) (is2 ? j2.f : (is1 ? j1.f : j0.f))
    const GemvJob j{WGML_PICK(a0), WGML_PICK(a1), WGML_PICK(a2), WGML_PICK(a3),
                    WGML_PICK(out), WGML_PICK(bias), WGML_PICK(nrows), WGML_PICK(kind),
                    WGML_PICK(out_pos_stride), WGML_PICK(wg_begin), WGML_PICK(wg_count),
                    WGML_PICK(active_waves)};
    if constexpr (FMT != 0) {
        fused_job_body<typename FusedFmt<FMT, F32>::T, D, FULL>(P, j);
    } else {
        switch (j.type()) {
        case WGML_Q4_K: fused_job_body<typename FusedFmt<WGML_Q4_K, F32>::T, D, FULL>(P, j); break;
        case WGML_Q6_K: fused_job_body<typename FusedFmt<WGML_Q6_K, F32>::T, D, FULL>(P, j); break;
        default: fused_job_body<typename FusedFmt<WGML_Q8_0, F32>::T, D, FULL>(P, j); break;
        }
    }
}

// The launch of a gate and an up matrix (of one format).
struct GatedParams {
    const uint8_t *a0, *a1, *a2, *a3;  // gate
    const uint8_t *b0, *b1, *b2, *b3;  // up
    const float *x, *norm_w;
    float *out;
    float norm_eps;
    uint32_t nrows, ncols, active_waves;
};
template <int MAXT, int FMT, bool F32 = false>
__global__ __launch_bounds__(MAXT, 1) void gemv_gated_kernel(const GatedParams P) {
    using F = typename FusedFmt<FMT, F32>::T;
    GemvParams a{};
    a.x = P.x;
    a.out = P.out;
    a.nrows = P.nrows;
    a.ncols = P.ncols;
    a.norm_w = P.norm_w;
    a.norm_eps = P.norm_eps;
    GemvParams b = a;
    a.p0 = P.a0;
    a.p1 = P.a1;
    a.p2 = P.a2;
    a.p3 = P.a3;
    b.p0 = P.b0;
    b.p1 = P.b1;
    b.p2 = P.b2;
    b.p3 = P.b3;
    GatedPolicy pol{a, b};
    if constexpr (!F::F32X) {
        if (P.ncols <= 64 * F::TILE) {
            gemv_i8_body<F, 2, 1, true>(a, pol, blockIdx.x, gridDim.x, P.active_waves, P.nrows);
            return;
        }
    }
    gemv_i8_body<F, 2, 1, false>(a, pol, blockIdx.x, gridDim.x, P.active_waves, P.nrows);
}

// A format's kernels (the fp32-activation ones with F32).  (gemv.hip has other single-matrix kernels for Q4_K and Q8_0; `plain` of these
// two stays in its code object because the others lie elsewhere without it, and a token of the 7B shape took 0.2 % longer.)
template <int TYPE, bool F32, bool FULL>
GemvKernels gemv_kernels_of() {
    using F = typename FusedFmt<TYPE, F32>::T;
    GemvKernels k{};
    k.plain = (const void *)gemv_quant_i8_kernel<F, 1, 1, 1024, 4, false, FULL ? EXTRA_FULL | EXTRA_MAXIMA : 0>;
    k.fused1024 = (const void *)gemv_fused_kernel<1, 1024, 1, TYPE, F32, FULL>;
    k.fused768 = (const void *)gemv_fused_kernel<1, 768, 1, TYPE, F32, FULL>;
    if constexpr (!FULL) {
        k.gated1024 = (const void *)gemv_gated_kernel<1024, TYPE, F32>;
        k.gated768 = (const void *)gemv_gated_kernel<768, TYPE, F32>;
    }
    return k;
}

// Pairs of the jobs in ROPE mode in the Neox variant: half a head, and 2^32 over it rounded up (g / half is
// the high word of their product for all g < 2^32 / half).
struct NeoxPairs {
    uint32_t half, magic;
};

}  // namespace
