// The batched product's kernel and its weight formats; one source file per format instantiates it.
#pragma once

#include <hip/hip_fp16.h>

#include <type_traits>

#include "device_utils.h"
#include "gemm_args.h"

namespace {

using namespace wgml;

// A load from uniform base + 32-bit lane offset.  The empty asm keeps the offset a 32-bit VGPR
// at the point of use, so that the load takes the base from scalar registers and the offset as
// it is: no 64-bit address arithmetic per lane and iteration.
template <class T>
__device__ __forceinline__ T load_at(const uint8_t *uniform_base, uint32_t lane_offset) {
    asm volatile("" : "+v"(lane_offset));
    return *reinterpret_cast<const T *>(uniform_base + lane_offset);
}

template <class T>
struct __attribute__((packed, aligned(2))) Half2Aligned {
    T v;
};

// ---- weight operands -------------------------------------------------------------
// A weight of every format is an exact small integer times the scale of its block (plus, in some,
// an offset shared by 32 elements).  The matrix cores multiply the integers, which f16 holds
// exactly, and the scale multiplies the fp32 sums of a block:
//   Q8_0, Q8_K    q in [-128, 127], d per 32 (Q8_K: 256) elements
//   Q4_0, Q5_0    q - 8, q - 16, d per 32
//   Q4_1, Q5_1    q - 7.5, q - 15.5, d per 32
//   Q4_K, Q5_K    (q - 7.5) * scale, (q - 15.5) * scale: up to 977, d per 256
//   Q6_K          (q - 32) * scale up to 4096: f16 holds 11 bits, so a pair hi + lo (exact), d per 256
// What these integers leave of a weight d q + m (Q4_1, Q5_1) or d scale q - dmin min (Q4_K, Q5_K) is an offset shared by
// 32 elements, 7.5 d + m and the like, which meets the sums of 32 activations in one more MFMA per 256 elements, as a pair
// of f16 numbers of which the second holds what rounding the first left.
// The integers are taken from the middle of q's range because d q and m alone are each about a hundred times the result
// where activations have one sign, and cancel only in the fp32 sums: error of Q4_K, |N(0,1)| activations, K = 4096, 3.6e-6 of
// the result's rms with q from 0, 3.9e-7 around 8, 2.8e-7 around 7.5 (zero-mean activations 4.1e-7, 1.8e-7, 1.9e-7;
// shorter chains of MFMAs take it further, CHAIN below).
// Nothing else is rounded on the weights' side, and an element takes about one vector instruction (a
// byte permutation makes f16 numbers 1024 + q out of two bytes of q at a time; one packed multiply-add
// takes the 1024 off again and applies the block's integer scale).
//
// Lane (g, j) of a wave holds, for half chunk Q of row j of its row block, the elements
// 256 u + 32 Q + 8 g .. + 7 (u: unit of 256 columns, Q in 0..7).  A format provides
//   Unit      the bytes of one unit, in four pieces (piece c: what half chunks 2 c and 2 c + 1 need
//             and the pieces before it have not fetched)
//   to_row    moves a matrix to the first row of a tile; its lanes' rows are 32-bit offsets from there
//   Dec       what is decoded once per unit
//   operand   the 8 halves of half chunk Q, and the low parts where the format has them
//   scale     of half chunk Q (blocks of 32) or of the unit
//   offsets   of sub-blocks 2 g and 2 g + 1 times `up`, as f16 pairs hi and lo
// Elements beyond the row's end (32-element blocks, last unit) are whatever follows in the matrix or
// in the zeroed bytes behind it: finite, and multiplied by activations that are zero.
__device__ __forceinline__ half2v as_half2(uint32_t v) {
    half2v h;
    __builtin_memcpy(&h, &v, 4);
    return h;
}
__device__ __forceinline__ uint32_t as_u32(half2v h) {
    uint32_t v;
    __builtin_memcpy(&v, &h, 4);
    return v;
}
// bytes 2 P and 2 P + 1 of `four` as f16 numbers 1024 + byte (0x6400 is 1024, its last place is 1)
template <int P>
__device__ __forceinline__ half2v bytes_1024(uint32_t four) {
    return as_half2(__builtin_amdgcn_perm(0x64646464u, four, P ? 0x04030402u : 0x04010400u));
}
__device__ __forceinline__ half2v splat(float v) {
    const _Float16 h = (_Float16)v;
    return half2v{h, h};
}
// byte B of a word as a pair of equal f16 numbers 1024 + byte
template <int B>
__device__ __forceinline__ half2v byte_1024(uint32_t w) {
    return as_half2(__builtin_amdgcn_perm(0x64646464u, w, 0x04000400u | (B * 0x00010001u)));
}
// eight bytes q (two words) to q + off
__device__ __forceinline__ void bytes_plus(uint32_t (&o)[4], uint32_t lo4, uint32_t hi4, float off) {
    const half2v k = splat(off - 1024.f);
    o[0] = as_u32(bytes_1024<0>(lo4) + k);
    o[1] = as_u32(bytes_1024<1>(lo4) + k);
    o[2] = as_u32(bytes_1024<0>(hi4) + k);
    o[3] = as_u32(bytes_1024<1>(hi4) + k);
}
// eight bytes b (two words) to b / 2 + off (0x6000 is 512, its last place is 1/2)
__device__ __forceinline__ void bytes_halved(uint32_t (&o)[4], uint32_t lo4, uint32_t hi4, float off) {
    const half2v k = splat(off - 512.f);
    o[0] = as_u32(as_half2(__builtin_amdgcn_perm(0x60606060u, lo4, 0x04010400u)) + k);
    o[1] = as_u32(as_half2(__builtin_amdgcn_perm(0x60606060u, lo4, 0x04030402u)) + k);
    o[2] = as_u32(as_half2(__builtin_amdgcn_perm(0x60606060u, hi4, 0x04010400u)) + k);
    o[3] = as_u32(as_half2(__builtin_amdgcn_perm(0x60606060u, hi4, 0x04030402u)) + k);
}
// eight bytes n q + n / 2 (two words) to (q - c) * n s, c = 128 / n - 1/2 (the middle of q's range), where n s is a scale of
// up to 63: s, 1152 s and the result (multiples of 1/2 up to 977) are numbers that f16 holds
__device__ __forceinline__ void bytes_times(uint32_t (&o)[4], uint32_t lo4, uint32_t hi4, half2v s) {
    const half2v k = s * splat(-(1024.f + 128.f));
    o[0] = as_u32(__builtin_elementwise_fma(bytes_1024<0>(lo4), s, k));
    o[1] = as_u32(__builtin_elementwise_fma(bytes_1024<1>(lo4), s, k));
    o[2] = as_u32(__builtin_elementwise_fma(bytes_1024<0>(hi4), s, k));
    o[3] = as_u32(__builtin_elementwise_fma(bytes_1024<1>(hi4), s, k));
}
// two offsets, and what rounding them to f16 left
__device__ __forceinline__ void offset_pair(uint32_t &hi, uint32_t &lo, float a, float b) {
    const half2v h{(_Float16)a, (_Float16)b};
    hi = as_u32(h);
    lo = as_u32(half2v{(_Float16)(a - (float)h[0]), (_Float16)(b - (float)h[1])});
}

// Plain f16 in runs of more than 128 tokens: the weight itself, rounded to f16 once, times 2^8 (undone at
// the end), so that nothing is left to scale per block: fp32 s q + off for eight bytes q.
constexpr float kDirectScale = 256.f;
__device__ __forceinline__ void bytes_direct(uint32_t (&o)[4], uint32_t lo4, uint32_t hi4, float s, float off) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t w = (k < 2 ? lo4 : hi4) >> (16 * (k & 1));
        o[k] = as_u32(half2v{(_Float16)fmaf(s, (float)(w & 0xffu), off), (_Float16)fmaf(s, (float)((w >> 8) & 0xffu), off)});
    }
}

// scales and minima of Q4_K and Q5_K: eight 6-bit numbers each, one per 32 elements
// (get_scale_min_k4, quantization.rs:381-389, on words of four)
struct ScalesK {
    uint32_t s[2], m[2];
    float d, dmin;
    __device__ void decode(const u32x4 &h) {
        d = f16_bits_to_f32((uint16_t)(h.x & 0xffffu));
        dmin = f16_bits_to_f32((uint16_t)(h.x >> 16));
        s[0] = h.y & 0x3f3f3f3fu;
        m[0] = h.z & 0x3f3f3f3fu;
        s[1] = (h.w & 0x0f0f0f0fu) | ((h.y >> 2) & 0x30303030u);
        m[1] = ((h.w >> 4) & 0x0f0f0f0fu) | ((h.z >> 2) & 0x30303030u);
    }
    // of sub-block Q over N (16 or 8)
    template <int Q, int N>
    __device__ half2v scale() const {
        return __builtin_elementwise_fma(byte_1024<Q & 3>(s[Q >> 2]), splat(1.f / N), splat(-1024.f / N));
    }
    template <int N>
    __device__ void offsets(uint32_t &hi, uint32_t &lo, uint32_t g, float up) const {
        const uint32_t sc = (g & 2 ? s[1] : s[0]) >> (16 * (g & 1)), mn = (g & 2 ? m[1] : m[0]) >> (16 * (g & 1));
        const float centre = d * up * (128.f / N - 0.5f), least = dmin * up;
        offset_pair(hi, lo, fmaf(centre, (float)(sc & 0xffu), -(least * (float)(mn & 0xffu))),
                    fmaf(centre, (float)((sc >> 8) & 0xffu), -(least * (float)((mn >> 8) & 0xffu))));
    }
    template <int Q, int N>
    __device__ void direct(uint32_t (&o)[4], uint32_t lo4, uint32_t hi4) const {
        bytes_direct(o, lo4, hi4, d * (kDirectScale / N) * (float)((s[Q >> 2] >> (8 * (Q & 3))) & 0xffu),
                     -(dmin * kDirectScale * (float)((m[Q >> 2] >> (8 * (Q & 3))) & 0xffu)));
    }
};

struct GemmQ4K {
    static constexpr int GROUP = 256;
    static constexpr bool OFFSET = true, PAIR = false;
    struct Unit {
        u32x4 hdr;    // d, dmin, 12 bytes of packed scales
        u32x2 qs[4];  // per chunk: bytes 8 g .. 8 g + 7 of its 32; low nibbles half 0, high half 1
    };
    using Dec = ScalesK;
    struct Lane {
        uint32_t hdr, qs;
    };
    __device__ static void to_row(GemmMat &m, uint32_t ncols, uint32_t row) { m.p0 += (size_t)row * (ncols / 256) * 144; }
    __device__ static void lane_init(Lane &l, uint32_t ncols, uint32_t row, uint32_t g) {
        l.hdr = row * (ncols / 256) * 144;
        l.qs = l.hdr + 16 + 8 * g;
    }
    template <int C>
    __device__ static void load(Unit &r, const GemmMat &m, const Lane &l, uint32_t u) {
        const uint8_t *blk = m.p0 + (size_t)u * 144;
        if (C == 0) r.hdr = load_at<u32x4>(blk, l.hdr);
        r.qs[C] = load_at<u32x2>(blk + C * 32, l.qs);
    }
    __device__ static void decode(Dec &d, const Unit &r, uint32_t) { d.decode(r.hdr); }
    template <int Q>
    __device__ static u32x2 bytes(const Unit &r) {  // 16 q
        return (Q & 1 ? r.qs[Q / 2] : r.qs[Q / 2] << 4) & 0xf0f0f0f0u;
    }
    template <int Q>
    __device__ static void operand(uint32_t (&hi)[4], uint32_t (&)[4], const Dec &d, const Unit &r, uint32_t) {
        const u32x2 q = bytes<Q>(r) | 0x08080808u;
        bytes_times(hi, q.x, q.y, d.scale<Q, 16>());
    }
    template <int Q>
    __device__ static void direct(uint32_t (&o)[4], const Dec &d, const Unit &r, uint32_t) {
        const u32x2 q = bytes<Q>(r);
        d.direct<Q, 16>(o, q.x, q.y);
    }
    __device__ static float unit_scale(const Dec &d) { return d.d; }
    __device__ static void offsets(uint32_t &hi, uint32_t &lo, const Dec &d, uint32_t g, float up) {
        d.offsets<16>(hi, lo, g, up);
    }
};

// Q5_K (176 B: d, dmin, scales[12] as Q4_K, 32 bytes of fifth bits, 128 bytes of nibbles;
// quantization.rs:249-317): bit Q of qh[8 g + i] belongs to half chunk Q.
struct GemmQ5K {
    static constexpr int GROUP = 256;
    static constexpr bool OFFSET = true, PAIR = false;
    struct Unit {
        u32x4 hdr;
        u32x2 qh, qs[4];
    };
    struct Dec {
        ScalesK k;
        u32x2 qh;
    };
    struct Lane {
        uint32_t hdr, qh, qs;
    };
    __device__ static void to_row(GemmMat &m, uint32_t ncols, uint32_t row) { m.p0 += (size_t)row * (ncols / 256) * 176; }
    __device__ static void lane_init(Lane &l, uint32_t ncols, uint32_t row, uint32_t g) {
        l.hdr = row * (ncols / 256) * 176;
        l.qh = l.hdr + 16 + 8 * g;
        l.qs = l.hdr + 48 + 8 * g;
    }
    template <int C>
    __device__ static void load(Unit &r, const GemmMat &m, const Lane &l, uint32_t u) {
        const uint8_t *blk = m.p0 + (size_t)u * 176;
        if (C == 0) {
            r.hdr = load_at<u32x4>(blk, l.hdr);
            r.qh = load_at<u32x2>(blk, l.qh);
        }
        r.qs[C] = load_at<u32x2>(blk + C * 32, l.qs);
    }
    __device__ static void decode(Dec &d, const Unit &r, uint32_t) {
        d.k.decode(r.hdr);
        d.qh = r.qh;
    }
    template <int Q>
    __device__ static u32x2 bytes(const Dec &d, const Unit &r) {  // 8 q
        return ((Q & 1 ? r.qs[Q / 2] >> 1 : r.qs[Q / 2] << 3) & 0x78787878u) | (((d.qh >> Q) & 0x01010101u) << 7);
    }
    template <int Q>
    __device__ static void operand(uint32_t (&hi)[4], uint32_t (&)[4], const Dec &d, const Unit &r, uint32_t) {
        const u32x2 q = bytes<Q>(d, r) | 0x04040404u;
        bytes_times(hi, q.x, q.y, d.k.scale<Q, 8>());
    }
    template <int Q>
    __device__ static void direct(uint32_t (&o)[4], const Dec &d, const Unit &r, uint32_t) {
        const u32x2 q = bytes<Q>(d, r);
        d.k.direct<Q, 8>(o, q.x, q.y);
    }
    __device__ static float unit_scale(const Dec &d) { return d.k.d; }
    __device__ static void offsets(uint32_t &hi, uint32_t &lo, const Dec &d, uint32_t g, float up) {
        d.k.offsets<8>(hi, lo, g, up);
    }
};

// Element 32 Q + 8 g + i of a super-block: nibble (Q >> 1) & 1 of ql[64 (Q >> 2) + 32 (Q & 1) + 8 g + i],
// bit pair Q & 3 of qh[32 (Q >> 2) + 8 g + i], scale 2 Q + g / 2.
struct GemmQ6K {
    static constexpr int GROUP = 256;
    static constexpr bool OFFSET = false, PAIR = true;
    struct Unit {
        u32x2 ql[2][2], qh[2];  // per 128 elements
        u32x4 sc;
        uint32_t d;
    };
    struct Dec {
        uint32_t sc[4];
        float d;
    };
    struct Lane {
        uint32_t ql, qh, sc, d;
    };
    __device__ static void to_row(GemmMat &m, uint32_t ncols, uint32_t row) {
        const size_t blk = (size_t)row * (ncols / 256);
        m.p0 += blk * 128;
        m.p1 += blk * 64;
        m.p2 += blk * 16;
        m.p3 += blk * 2;
    }
    __device__ static void lane_init(Lane &l, uint32_t ncols, uint32_t row, uint32_t g) {
        const uint32_t blk = row * (ncols / 256);
        l.ql = blk * 128 + 8 * g;
        l.qh = blk * 64 + 8 * g;
        l.sc = blk * 16;
        l.d = blk * 2;
    }
    template <int C>
    __device__ static void load(Unit &r, const GemmMat &m, const Lane &l, uint32_t u) {
        if (C == 0) {
            r.sc = load_at<u32x4>(m.p2 + (size_t)u * 16, l.sc);
            r.d = load_at<uint16_t>(m.p3 + (size_t)u * 2, l.d);
        }
        if (C & 1) {  // two chunks share their bytes: fetched again when the second is done with them
            constexpr int i = C / 2;
            const uint8_t *ql = m.p0 + (size_t)u * 128 + 64 * i;
            r.ql[i][0] = load_at<u32x2>(ql, l.ql);
            r.ql[i][1] = load_at<u32x2>(ql + 32, l.ql);
            r.qh[i] = load_at<u32x2>(m.p1 + (size_t)u * 64 + 32 * i, l.qh);
        }
    }
    __device__ static void decode(Dec &d, const Unit &r, uint32_t g) {
        // bytes 2 Q + g / 2 of the 16: lanes of the upper half shift them down
        const uint32_t sh = (g >> 1) * 8;
        d.sc[0] = r.sc.x >> sh;
        d.sc[1] = r.sc.y >> sh;
        d.sc[2] = r.sc.z >> sh;
        d.sc[3] = r.sc.w >> sh;
        d.d = f16_bits_to_f32((uint16_t)r.d);
    }
    template <int Q>
    __device__ static u32x2 bytes(const Unit &r) {
        return ((r.ql[Q / 4][Q & 1] >> (4 * ((Q >> 1) & 1))) & 0x0f0f0f0fu) |
               (((r.qh[Q / 4] >> (2 * (Q & 3))) & 0x03030303u) << 4);
    }
    template <int Q>
    __device__ static float block_scale(const Dec &d) {
        return (float)(int8_t)((d.sc[Q / 2] >> (16 * (Q & 1))) & 0xffu);
    }
    template <int Q>
    __device__ static void operand(uint32_t (&hi)[4], uint32_t (&lo)[4], const Dec &d, const Unit &r, uint32_t) {
        const half2v s = splat(block_scale<Q>(d));
        const u32x2 b = bytes<Q>(r);
        uint32_t q[4];
        bytes_plus(q, b.x, b.y, -32.f);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            // the product rounded to f16, and what the rounding left (0 or +-1), exactly
            const half2v p = as_half2(q[k]) * s;
            hi[k] = as_u32(p);
            lo[k] = as_u32(__builtin_elementwise_fma(as_half2(q[k]), s, -p));
        }
    }
    template <int Q>
    __device__ static void direct(uint32_t (&o)[4], const Dec &d, const Unit &r, uint32_t) {
        const u32x2 b = bytes<Q>(r);
        const float s = d.d * kDirectScale * block_scale<Q>(d);
        bytes_direct(o, b.x, b.y, s, -32.f * s);
    }
    __device__ static float unit_scale(const Dec &d) { return d.d; }
};

// signed bytes: with the top bit flipped they are q + 128
struct GemmQ8_0 {
    static constexpr int GROUP = 32;
    static constexpr bool OFFSET = false, PAIR = false;
    struct __attribute__((packed, aligned(2))) Half8 {
        u32x4 v;
    };
    struct Unit {
        u32x2 q[8];
        u32x4 d;  // the unit's eight scales
    };
    struct Dec {
        uint32_t d[4];
    };
    struct Lane {
        uint32_t q, d;
    };
    __device__ static void to_row(GemmMat &m, uint32_t ncols, uint32_t row) {
        m.p0 += (size_t)row * ncols;
        m.p1 += (size_t)row * (ncols / 32) * 2;
    }
    __device__ static void lane_init(Lane &l, uint32_t ncols, uint32_t row, uint32_t g) {
        l.q = row * ncols + 8 * g;
        l.d = row * (ncols / 32) * 2;
    }
    template <int C>
    __device__ static void load(Unit &r, const GemmMat &m, const Lane &l, uint32_t u) {
        const uint8_t *q = m.p0 + (size_t)u * 256 + 64 * C;
        if (C == 0) r.d = load_at<Half8>(m.p1 + (size_t)u * 16, l.d).v;
        r.q[2 * C] = load_at<u32x2>(q, l.q);
        r.q[2 * C + 1] = load_at<u32x2>(q + 32, l.q);
    }
    __device__ static void decode(Dec &d, const Unit &r, uint32_t) {
        d.d[0] = r.d.x;
        d.d[1] = r.d.y;
        d.d[2] = r.d.z;
        d.d[3] = r.d.w;
    }
    template <int Q>
    __device__ static void operand(uint32_t (&hi)[4], uint32_t (&)[4], const Dec &, const Unit &r, uint32_t) {
        bytes_plus(hi, r.q[Q].x ^ 0x80808080u, r.q[Q].y ^ 0x80808080u, -128.f);
    }
    template <int Q>
    __device__ static void direct(uint32_t (&o)[4], const Dec &d, const Unit &r, uint32_t) {
        const float s = scale<Q>(d) * kDirectScale;
        bytes_direct(o, r.q[Q].x ^ 0x80808080u, r.q[Q].y ^ 0x80808080u, s, -128.f * s);
    }
    template <int Q>
    __device__ static float scale(const Dec &d) {
        return f16_bits_to_f32((uint16_t)(d.d[Q / 2] >> (16 * (Q & 1))));
    }
};

// Q8_K (292 B: f32 d, 256 int8, 16 sums that dequantization does not use; quantization.rs:170-199).
struct GemmQ8K {
    static constexpr int GROUP = 256;
    static constexpr bool OFFSET = false, PAIR = false;
    struct Unit {
        u32x2 q[8];
        float d;
    };
    struct Dec {
        float d;
    };
    struct Lane {
        uint32_t d, q;
    };
    __device__ static void to_row(GemmMat &m, uint32_t ncols, uint32_t row) { m.p0 += (size_t)row * (ncols / 256) * 292; }
    __device__ static void lane_init(Lane &l, uint32_t ncols, uint32_t row, uint32_t g) {
        l.d = row * (ncols / 256) * 292;
        l.q = l.d + 4 + 8 * g;
    }
    template <int C>
    __device__ static void load(Unit &r, const GemmMat &m, const Lane &l, uint32_t u) {
        const uint8_t *blk = m.p0 + (size_t)u * 292;
        if (C == 0) r.d = load_at<float>(blk, l.d);
        r.q[2 * C] = load_at<Half2Aligned<u32x2>>(blk + 64 * C, l.q).v;
        r.q[2 * C + 1] = load_at<Half2Aligned<u32x2>>(blk + 64 * C + 32, l.q).v;
    }
    __device__ static void decode(Dec &d, const Unit &r, uint32_t) { d.d = r.d; }
    template <int Q>
    __device__ static void operand(uint32_t (&hi)[4], uint32_t (&)[4], const Dec &, const Unit &r, uint32_t) {
        bytes_plus(hi, r.q[Q].x ^ 0x80808080u, r.q[Q].y ^ 0x80808080u, -128.f);
    }
    template <int Q>
    __device__ static void direct(uint32_t (&o)[4], const Dec &d, const Unit &r, uint32_t) {
        const float s = d.d * kDirectScale;
        bytes_direct(o, r.q[Q].x ^ 0x80808080u, r.q[Q].y ^ 0x80808080u, s, -128.f * s);
    }
    __device__ static float unit_scale(const Dec &d) { return d.d; }
};

// The 32-element blocks Q4_0, Q4_1, Q5_0, Q5_1 (quantization.rs:47-162), as planes of nibbles (p0), d or {d, m} (p1) and
// fifth bits (p2).  Element t of a block is the low nibble of qs[t] for t < 16 and the high nibble of qs[t - 16]
// otherwise, with bit t of qh as its fifth bit.  Half chunk Q is block 8 u + Q; a lane's t = 8 g + i, so
// lanes g < 2 take low nibbles and g >= 2 high nibbles of the same eight bytes.
template <bool HAS_M, bool HAS_QH>
struct GemmLegacy {
    static constexpr int GROUP = 32;
    static constexpr bool OFFSET = HAS_M, PAIR = false;
    struct Unit {
        u32x2 q[8];
        u32x2 qh[4];
        u32x2 dm;   // d (low half) and m (high half) of blocks 2 g and 2 g + 1 where there is an m
        u32x4 d;    // the unit's eight scales where there is none
    };
    struct Dec {
        uint32_t dm[HAS_M ? 8 : 4], own[HAS_M ? 2 : 1];  // of all blocks (two to a word without m); of blocks 2 g and 2 g + 1
    };
    struct Lane {
        uint32_t q, dm, qh;
    };
    __device__ static void to_row(GemmMat &m, uint32_t ncols, uint32_t row) {
        const size_t blk = (size_t)row * (ncols / 32);
        m.p0 += blk * 16;
        m.p1 += blk * (HAS_M ? 4 : 2);
        m.p2 += blk * 4;
    }
    __device__ static void lane_init(Lane &l, uint32_t ncols, uint32_t row, uint32_t g) {
        const uint32_t blk = row * (ncols / 32);
        l.q = blk * 16 + 8 * (g & 1);
        l.dm = HAS_M ? blk * 4 + 8 * g : blk * 2;
        l.qh = blk * 4;
    }
    template <int C>
    __device__ static void load(Unit &r, const GemmMat &m, const Lane &l, uint32_t u) {
        if (C == 0) {
            if constexpr (HAS_M)
                r.dm = load_at<Half2Aligned<u32x2>>(m.p1 + (size_t)u * 32, l.dm).v;
            else
                r.d = load_at<Half2Aligned<u32x4>>(m.p1 + (size_t)u * 16, l.dm).v;
        }
        if constexpr (HAS_QH) r.qh[C] = load_at<Half2Aligned<u32x2>>(m.p2 + (size_t)u * 32 + 8 * C, l.qh).v;
        r.q[2 * C] = load_at<u32x2>(m.p0 + (size_t)u * 128 + 32 * C, l.q);
        r.q[2 * C + 1] = load_at<u32x2>(m.p0 + (size_t)u * 128 + 32 * C + 16, l.q);
    }
    // With minima the eight pairs of a row come from its four lanes (all eight of them in every lane take six registers more
    // through the whole unit).
    __device__ static void decode(Dec &d, const Unit &r, uint32_t) {
        if constexpr (HAS_M) {
            const int j4 = (int)(threadIdx.x & 15) * 4;
#pragma unroll
            for (int b = 0; b < 8; ++b) d.dm[b] = (uint32_t)__builtin_amdgcn_ds_bpermute((b / 2) * 64 + j4, (int)(b & 1 ? r.dm.y : r.dm.x));
            d.own[0] = r.dm.x;
            d.own[1] = r.dm.y;
        } else {
            d.dm[0] = r.d.x;
            d.dm[1] = r.d.y;
            d.dm[2] = r.d.z;
            d.dm[3] = r.d.w;
        }
    }
    // q << SHIFT in eight bytes
    template <int Q, int SHIFT>
    __device__ static u32x2 bytes(const Unit &r, uint32_t g) {
        const uint32_t right = (4 * (g >> 1) - SHIFT) & 31u, mask = 0x0f0f0f0fu << SHIFT;  // (a rotation)
        uint32_t a = __builtin_amdgcn_alignbit(r.q[Q].x, r.q[Q].x, right) & mask;
        uint32_t b = __builtin_amdgcn_alignbit(r.q[Q].y, r.q[Q].y, right) & mask;
        if (HAS_QH) {
            // bits 8 g .. 8 g + 7 of qh moved to bit 4 of the eight bytes
            const uint32_t bits = (Q & 1 ? r.qh[Q / 2].y : r.qh[Q / 2].x) >> (8 * g);
            a |= (((bits & 15u) * 0x00204081u) & 0x01010101u) << (4 + SHIFT);
            b |= ((((bits >> 4) & 15u) * 0x00204081u) & 0x01010101u) << (4 + SHIFT);
        }
        return u32x2{a, b};
    }
    static constexpr float CENTRE = HAS_QH ? 16.f : 8.f;
    template <int Q>
    __device__ static void operand(uint32_t (&hi)[4], uint32_t (&)[4], const Dec &, const Unit &r, uint32_t g) {
        const u32x2 q = HAS_M ? bytes<Q, 1>(r, g) | 0x01010101u : bytes<Q, 0>(r, g);
        if constexpr (HAS_M)
            bytes_halved(hi, q.x, q.y, -CENTRE);  // q - 7.5, q - 15.5 out of bytes 2 q + 1
        else
            bytes_plus(hi, q.x, q.y, -CENTRE);
    }
    template <int Q>
    __device__ static void direct(uint32_t (&o)[4], const Dec &d, const Unit &r, uint32_t g) {
        const u32x2 q = bytes<Q, 0>(r, g);
        const float s = scale<Q>(d) * kDirectScale;
        bytes_direct(o, q.x, q.y, s, HAS_M ? f16_bits_to_f32((uint16_t)(d.dm[HAS_M ? Q : 0] >> 16)) * kDirectScale : -CENTRE * s);
    }
    template <int Q>
    __device__ static float scale(const Dec &d) {
        return f16_bits_to_f32((uint16_t)(HAS_M ? d.dm[HAS_M ? Q : 0] & 0xffffu : d.dm[Q / 2] >> (16 * (Q & 1))));
    }
    __device__ static void offsets(uint32_t &hi, uint32_t &lo, const Dec &d, uint32_t, float up) {
        float c[2];
#pragma unroll
        for (int b = 0; b < 2; ++b)
            c[b] = fmaf(CENTRE - 0.5f, f16_bits_to_f32((uint16_t)(d.own[HAS_M ? b : 0] & 0xffffu)),
                        f16_bits_to_f32((uint16_t)(d.own[HAS_M ? b : 0] >> 16))) * up;
        offset_pair(hi, lo, c[0], c[1]);
    }
};
using GemmQ4_0 = GemmLegacy<false, false>;
using GemmQ4_1 = GemmLegacy<true, false>;
using GemmQ5_0 = GemmLegacy<false, true>;
using GemmQ5_1 = GemmLegacy<true, true>;

template <int I, int N, class Fn>
__device__ __forceinline__ void static_for(Fn &&fn) {
    if constexpr (I < N) {
        fn(std::integral_constant<int, I>{});
        static_for<I + 1, N>(fn);
    }
}

// Tokens tok0 + 16 n + k of one row: into the workgroup's partial sums, or scaled, with the bias, to (or
// onto) the output.  What the latter reads is requested before the first store (as one load, add and
// store per value the last rows of a short product cost more than its multiplications).
template <int N>
__device__ __forceinline__ void store_row(const GemmArgs &a, const GemmMat &m, const floatx4 (&acc)[N], float unit,
                                          uint32_t row, uint32_t tok0, uint32_t ky) {
    if (row >= m.nrows) return;
    if (a.ks > 1) {
        float *o = a.part + ((size_t)ky * a.T + tok0) * a.total_rows + m.roff + row;
#pragma unroll
        for (int n = 0; n < N; ++n) {
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (tok0 + 16 * n + k < a.T) o[(size_t)(16 * n + k) * a.total_rows] = acc[n][k] * unit;
        }
        return;
    }
    float *o = m.out + (size_t)tok0 * m.out_stride + row;
    const float bias = m.bias ? m.bias[row] : 0.f;
    float xs[N][4], old[N][4];
#pragma unroll
    for (int n = 0; n < N; ++n) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t t = 16 * n + k;
            const bool there = tok0 + t < a.T;
            xs[n][k] = there ? a.xscale[tok0 + t] : 0.f;
            old[n][k] = there && a.accumulate ? o[(size_t)t * m.out_stride] : 0.f;
        }
    }
#pragma unroll
    for (int n = 0; n < N; ++n) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t t = 16 * n + k;
            const float v = (acc[n][k] * unit) * xs[n][k] + bias;
            if (tok0 + t < a.T) o[(size_t)t * m.out_stride] = a.accumulate ? old[n][k] + v : v;
        }
    }
}

// The matrix of a row tile, copied out of the arguments: indexed, its pointers would be loaded again
// in every iteration.
__device__ __forceinline__ GemmMat matrix_of_tile(const GemmArgs &a, uint32_t tile) {
    GemmMat m = a.m[0];
    if (a.nmat > 1 && tile >= a.m[1].tile0) m = a.m[1];
    if (a.nmat > 2 && tile >= a.m[2].tile0) m = a.m[2];
    return m;
}

__device__ __forceinline__ half8 as_half8(const uint32_t (&v)[4]) {
    half8 h;
    __builtin_memcpy(&h, v, 16);
    return h;
}
__device__ __forceinline__ half8 as_half8(const u32x4 &v) {
    half8 h;
    __builtin_memcpy(&h, &v, 16);
    return h;
}
// Tokens come first: lane (g, j) of the result holds tokens 4 g .. 4 g + 3 of row j, the row whose
// weights (and scales) it supplies.
__device__ __forceinline__ floatx4 mfma(const half8 &x, const half8 &w, const floatx4 &c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(x, w, c, 0, 0, 0);
}
__device__ __forceinline__ void add_scaled(floatx4 &acc, const floatx4 &t, float s) {
#pragma unroll
    for (int k = 0; k < 4; ++k) acc[k] = fmaf(t[k], s, acc[k]);
}

// Offsets as an MFMA operand: lane (g, j) comes with hi and lo of its two sub-blocks and leaves with the eight hi of row j
// for g < 2, the eight lo otherwise.  The sums opposite are their first part for even g and their second for odd,
// so that the four products of parts are summed.
__device__ __forceinline__ void gather_offsets(uint32_t (&o)[4], uint32_t hi, uint32_t lo) {
    // rows of 16 lanes: [h0 h1 h2 h3] twice -> [h0 h0 h2 h2], [h1 h1 h3 h3]; then the upper halves of those against the
    // lower halves of lo's
    const u32x2 h = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(hi, hi, false, false));
    const u32x2 l = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(lo, lo, false, false));
    const u32x2 even = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(h.x, l.x, false, false));
    const u32x2 odd = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(h.y, l.y, false, false));
    o[0] = even.x;
    o[1] = odd.x;
    o[2] = even.y;
    o[3] = odd.y;
}

// What computes `v` stays in front of this: instruction selection would move sums that nothing in the
// loop reads to its end, and keep what they are made of in registers until there.
__device__ __forceinline__ void keep_here(floatx4 &v) { asm volatile("" : "+v"(v)); }

// ---- up to 128 tokens --------------------------------------------------------------
// A workgroup of 4 waves owns 64 rows of one matrix, a wave 16 of them, and a range of units.  The
// activations of all tokens pass through LDS (two buffers in turn, one barrier per stage); a wave makes
// its operands in registers, each weight once, while the matrix cores multiply the half chunk
// before, and refills the bytes of a unit piece by piece as they are used up.
// What bounds it: with few tokens the first bytes of each workgroup and about 2.6 vector instructions per
// weight, with many the activations, which every 64 rows read again (leave-one-out at 128 tokens, with one sum per result
// and unit: LDS reads 11 %, staging 12 %, weight loads 7 %, no single one dominates; now MFMAs for 29 % of the cycles, 2.8 other vector
// instructions each).  Four layers, one pass, us, with operands
// expanded to fp32 and three MFMAs per term -> now: 7B shape Q4_K_M 4 tokens 594 -> 471, 45: 801 -> 618, 128: 1199 ->
// 1015 (plain f16 886 -> 745); 768 x 2048 Q8_0 4: 297 -> 206, 128: 458 -> 299.
// Measured and dropped: two row blocks per wave (128 tokens 1048 -> 1272: fewer workgroups, and no shorter
// a time per unit); 8 waves that share rows and tokens out; activations requested two stages ahead
// (spills below 128 registers, no faster where it fits).
//
// Chunks of 64 columns staged per barrier: 16 KB of activations in split precision for up to 16, 32 and 64 tokens, 24 KB
// for 48 and 96, 32 KB for 128, half of that in plain f16; twice, with 512 bytes of sums per 16 tokens.
constexpr int gemm_stage_chunks(int nt) { return nt == 1 ? 4 : nt <= 3 ? 2 : 1; }
template <class F, bool SPLIT>
constexpr uint32_t gemm_lds_words(int nt) {  // 16-byte words
    return 2 * (gemm_stage_chunks(nt) * nt * 128 * (SPLIT ? 2 : 1) + (F::OFFSET ? nt * 32 : 0));
}
// Workgroups per compute unit that registers are kept for (128 each at four, 168 at three): no more than fit its 160 KB of LDS
// in split precision (three for 48 tokens, two or three for 96, two for 128), and three for 64 tokens, where four fit: at
// 128 registers the formats with most to decode spill (four layers, 2080 x 5600 in Q5_1, us: 45 tokens 507 with four ->
// 410, 64 tokens 482 -> 438; 4096 x 11008 in Q5_K 651 -> 604, 703 -> 663) and the others gain nothing (+-0.6 %).
template <class F, bool SPLIT>
constexpr int gemm_workgroups(int nt) {
    const int fit = (int)(160 * 1024 / (16 * gemm_lds_words<F, SPLIT>(nt)));
    const int most = nt >= 8 ? 2 : nt >= (SPLIT ? 3 : 6) ? 3 : 4;
    return fit < most ? fit : most;
}

template <class F, int NT, bool SPLIT>
__global__ __launch_bounds__(256, (gemm_workgroups<F, SPLIT>(NT))) void gemm_lds_kernel(const GemmArgs a) {
    extern __shared__ u32x4 xs[];  // [2][chunks][high: NT * 128 words (, low: the same)], [2][sums: NT * 32]
    constexpr int PARTS = SPLIT ? 2 : 1, CPS = gemm_stage_chunks(NT), NS = 4 / CPS;
    constexpr uint32_t CW = NT * 128, CWX = CW * PARTS, STAGE = CPS * CWX, SUMS = F::OFFSET ? NT * 32 : 0;
    constexpr int SW = STAGE / 256;  // staged words per thread
    constexpr bool WLO = F::PAIR && SPLIT, G32 = F::GROUP == 32;
    // Half chunks whose products pile up before the scale multiplies them.  An MFMA's own additions round more than a
    // multiply-add does: eight half chunks of high and low parts in one sum, as in the other formats with a scale per unit, give
    // 2.7e-7 of the result's rms (Q4_K, |N(0,1)| activations, K = 512 .. 4096); weights expanded to fp32 first gave 2.1e-7.
    // Where weights have an offset the low parts, a thousandth as large, have a sum of their own, and the high parts one of four
    // half chunks: 1.9e-7 (in one sum of two half chunks 2.0e-7, and 4 % slower at 128 tokens of the 7B widths).
    constexpr int CHAIN = F::OFFSET && SPLIT && !G32 ? 4 : 8;
    constexpr bool APART = F::OFFSET && SPLIT && !G32;
    const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t j = lane & 15, g = lane >> 4;
    const uint32_t ky = blockIdx.x % a.ks, tile = blockIdx.x / a.ks;
    GemmMat m = matrix_of_tile(a, tile);
    const uint32_t tile_row = (tile - m.tile0) * 64, row0 = tile_row + wave * 16;
    F::to_row(m, a.ncols, tile_row);
    typename F::Lane wl;
    F::lane_init(wl, a.ncols, min(wave * 16 + j, m.nrows - 1 - tile_row), g);
    const uint32_t nunits = a.kpad / KU, u0 = nunits * ky / a.ks, u1 = nunits * (ky + 1) / a.ks;

    floatx4 acc[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[n] = zero;
    uint32_t soff[SW];
#pragma unroll
    for (int q = 0; q < SW; ++q) {
        const uint32_t w = tid + 256 * q, ch = w / CWX, ww = w % CWX;
        soff[q] = ch * (NT * 2048) + (SPLIT && ww >= CW ? a.xl_offset + (ww - CW) * 16 : ww * 16);
    }
    // Loads are unconditional: past the end the last unit is fetched again and not used.
    auto unit_at = [&](uint32_t u) { return min(u, nunits - 1); };
    u32x4 st[SW], ss;
    auto stage_load = [&](uint32_t u, int s) {
        const uint8_t *base = reinterpret_cast<const uint8_t *>(a.xh) + (size_t)(u * 4 + s * CPS) * (NT * 2048);
#pragma unroll
        for (int q = 0; q < SW; ++q) st[q] = load_at<u32x4>(base, soff[q]);
        if (F::OFFSET && s == 0)
            ss = load_at<u32x4>(reinterpret_cast<const uint8_t *>(a.xsum) + (size_t)u * (NT * 512),
                                min(tid, SUMS - 1) * 16);
    };
    // weights of a half chunk as MFMA operands
    struct Op {
        uint32_t hi[4], lo[4];
        float scale;
    };
    auto make = [&](auto q_c, Op &o, const typename F::Dec &d, const typename F::Unit &r) {
        constexpr int Q = decltype(q_c)::value;
        F::template operand<Q>(o.hi, o.lo, d, r, g);
        if constexpr (G32) o.scale = F::template scale<Q>(d);
    };
    typename F::Unit un;
    typename F::Dec dec;
    Op op[2];
    floatx4 late = zero;  // blocks of 32: sums whose scaling is still to come
    float late_scale = 0.f;
    stage_load(u0, 0);
    static_for<0, 4>([&](auto c) { F::template load<decltype(c)::value>(un, m, wl, u0); });
    F::decode(dec, un, g);
    make(std::integral_constant<int, 0>{}, op[0], dec, un);
    for (uint32_t u = u0; u < u1; ++u) {
        const uint32_t next = unit_at(u + 1);
        typename F::Dec ndec;
        floatx4 tmp[G32 ? 1 : NT], low[APART ? NT : 1];
        uint32_t off_hi = 0, off_lo = 0;
        if constexpr (F::OFFSET) F::offsets(off_hi, off_lo, dec, g, m.offset_up);
        static_for<0, NS>([&](auto s_c) {
            constexpr int s = decltype(s_c)::value;
            u32x4 *buf = xs + (NS > 1 ? (uint32_t)(s & 1) : (u & 1)) * STAGE;
#pragma unroll
            for (int q = 0; q < SW; ++q) buf[tid + 256 * q] = st[q];
            if constexpr (F::OFFSET && s == 0) {
                if (SUMS % 256 == 0 || tid < SUMS) xs[2 * STAGE + (u & 1) * SUMS + tid] = ss;
            }
            __syncthreads();
            if (s + 1 < NS)
                stage_load(u, s + 1);
            else
                stage_load(next, 0);
            // Steps of one token block and half chunk each: the LDS words of a later step are
            // requested, the step's MFMAs issued and, once per half chunk, the operands of the next one
            // made (nothing is scheduled across a step's end).
            const u32x4 *bsrc = buf + lane;
            constexpr int NSTEP = CPS * 2 * NT, AHEAD = NT >= 6 ? 3 : 2;
            u32x4 bh[AHEAD + 1], bl[AHEAD + 1];
            auto fetch = [&](auto i_c) {
                constexpr int i = decltype(i_c)::value, slot = i % (AHEAD + 1);
                constexpr uint32_t at = (i / (2 * NT)) * CWX + ((i % NT) * 2 + (i / NT) % 2) * 64;
                bh[slot] = bsrc[at];
                if (SPLIT) bl[slot] = bsrc[at + CW];
            };
            static_for<0, AHEAD>(fetch);
            __builtin_amdgcn_sched_barrier(0);
            static_for<0, NSTEP>([&](auto i_c) {
                constexpr int i = decltype(i_c)::value, n = i % NT, q = s * CPS * 2 + i / NT, slot = i % (AHEAD + 1);
                Op &o = op[q & 1];
                if constexpr (i + AHEAD < NSTEP) fetch(std::integral_constant<int, i + AHEAD>{});
                const half8 x8 = as_half8(bh[slot]);
                floatx4 t = mfma(x8, as_half8(o.hi), G32 || q % CHAIN == 0 ? zero : tmp[G32 ? 0 : n]);
                if constexpr (APART)
                    low[n] = mfma(as_half8(bl[slot]), as_half8(o.hi), q == 0 ? zero : low[n]);
                else if constexpr (SPLIT)
                    t = mfma(as_half8(bl[slot]), as_half8(o.hi), t);
                if constexpr (WLO) t = mfma(x8, as_half8(o.lo), t);
                if constexpr (n == 0) {
                    if constexpr (q < 7) {
                        make(std::integral_constant<int, q + 1>{}, op[(q + 1) & 1], dec, un);
                    } else {
                        F::decode(ndec, un, g);
                        make(std::integral_constant<int, 0>{}, op[0], ndec, un);
                    }
                    // the bytes of the next unit where the old ones have served
                    if constexpr (q % 2 == 0) F::template load<q / 2>(un, m, wl, next);
                }
                if constexpr (G32) {
                    // the sums of the step before: its MFMAs have ended meanwhile
                    add_scaled(acc[(n + NT - 1) % NT], late, late_scale);
                    late = t;
                    late_scale = o.scale;
                } else {
                    if constexpr (q % CHAIN == CHAIN - 1 && n > 0) add_scaled(acc[n - 1], tmp[n - 1], F::unit_scale(dec));
                    if constexpr (q % CHAIN == 0 && q > 0 && n == 0)
                        add_scaled(acc[NT - 1], tmp[NT - 1], F::unit_scale(dec));
                    tmp[n] = t;
                }
                __builtin_amdgcn_sched_barrier(0);
            });
        });
        if constexpr (!G32 || F::OFFSET) {
            const u32x4 *sums = xs + 2 * STAGE + (u & 1) * SUMS + (lane & 31);
            uint32_t offs[4];
            if constexpr (F::OFFSET) gather_offsets(offs, off_hi, off_lo);
            if constexpr (!G32) add_scaled(acc[NT - 1], tmp[NT - 1], F::unit_scale(dec));
            if constexpr (F::OFFSET) {
#pragma unroll
                for (int n = 0; n < NT; ++n) {
                    if constexpr (APART) add_scaled(acc[n], low[n], F::unit_scale(dec));
                    add_scaled(acc[n], mfma(as_half8(sums[n * 32]), as_half8(offs), zero), m.offset_down);
                }
            }
        }
        dec = ndec;
    }
    if constexpr (G32) add_scaled(acc[NT - 1], late, late_scale);
    store_row(a, m, acc, 1.f, row0 + j, 4 * g, ky);
}

// ---- runs of more than 128 tokens ----------------------------------------------------
// A workgroup owns 128 rows x 256 tokens and a wave 64 x 64 of them: a word of weights or of activations
// read from LDS serves four products, and a weight is expanded once per 256 tokens.  The weights meet in
// LDS too: wave w makes the operands of row block w of the tile, every wave reads the four row
// blocks it multiplies.  K is walked in half chunks of 32 columns, two LDS slots in turn, one barrier
// each: during half chunk Q slot Q & 1 is multiplied, the other one takes the activations (requested
// during Q - 1) and weights (made during Q - 1) of Q + 1, and the operands of Q + 2 are made.
// What bounds it (Q8_0): a half chunk takes 2350 cycles for 1090 of MFMAs (17 each), 1100 of LDS and, per MFMA, 2.7
// vector instructions, which hide beside each other only in part (two waves per SIMD: 8 MFMAs, then 32
// multiply-adds take 452 cycles, apart 271 and 289).  So sums are scaled per unit where the format
// allows it (tmp), not per 32 columns, and not at all in plain f16, where the weight itself is rounded.
// Four layers, one pass of 1000 tokens, us, with three MFMAs per term -> now: 3072 x 8192 Q8_0 3508 -> 2830, plain
// f16 2441 -> 2144; 7B shape Q4_K_M 5503 -> 4733, 3306 -> 3164.  Measured and dropped: activations requested two
// half chunks ahead (5262 against 5042), tiles of 128 tokens in workgroups of 4 waves (5750), Q8_0 as pairs of
// f16 products with a third MFMA (3535 against 3137).
template <class F, bool SPLIT>
struct TileLds {  // 16-byte words
    static constexpr uint32_t WPARTS = F::PAIR && SPLIT ? 2 : 1, XPARTS = SPLIT ? 2 : 1;
    static constexpr uint32_t W = 8 * WPARTS * 64, X = XPARTS * 16 * 64, SLOT = W + X + 32;  // + 128 scales
    // per unit, twice: 128 scales, the offsets (per row block 16 words of their first parts, 16 of the second), the sums
    static constexpr uint32_t UNIT = !SPLIT ? 0 : F::OFFSET ? 32 + 8 * 32 + 16 * 32 : F::GROUP == 256 ? 32 : 0;
    static constexpr uint32_t WORDS = 2 * (SLOT + UNIT);
};

template <class F, bool SPLIT>
__global__ __launch_bounds__(512) void gemm_tile_kernel(const GemmArgs a) {
    extern __shared__ u32x4 xs[];
    using L = TileLds<F, SPLIT>;
    // plain f16: the sums need no scaling per block (direct), split f16: per 32 columns or per unit (tmp)
    constexpr bool DIRECT = !SPLIT, OFFSET = F::OFFSET && SPLIT, WLO = L::WPARTS == 2;
    constexpr bool G32 = F::GROUP == 32 && SPLIT, TMP = F::GROUP == 256 && SPLIT;
    constexpr int CHAIN = F::OFFSET ? 4 : 8;  // see gemm_lds_kernel: 2.2e-7 (expanded weights 2.7e-7 to 3.7e-7)
    constexpr int SW = 2 * L::XPARTS;  // staged words of activations per thread and half chunk
    const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t j = lane & 15, g = lane >> 4;
    const uint32_t wr = wave & 1, wc = wave >> 1;
    // Workgroup w runs on XCD w % 8: give each XCD a contiguous range of the tiles, token tiles
    // varying fastest, so that the workgroups an XCD runs at a time share weights and activations
    // in its L2.
    const uint32_t n_wg = gridDim.x, xcd = blockIdx.x & 7, q8 = n_wg >> 3, r8 = n_wg & 7;
    const uint32_t v = xcd * q8 + min(xcd, r8) + (blockIdx.x >> 3);
    const uint32_t tt = v % a.ttiles, rtiles = n_wg / (a.ttiles * a.ks);
    const uint32_t tile = (v / a.ttiles) % rtiles, ky = v / a.ttiles / rtiles;
    GemmMat m = matrix_of_tile(a, tile);
    const uint32_t row0 = (tile - m.tile0) * TILE_ROWS;
    F::to_row(m, a.ncols, row0);
    typename F::Lane wl;
    F::lane_init(wl, a.ncols, min(16 * wave + j, m.nrows - 1 - row0), g);
    const uint32_t nunits = a.kpad / KU, u0 = nunits * ky / a.ks, u1 = nunits * (ky + 1) / a.ks;

    floatx4 acc[4][4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
#pragma unroll
        for (int n = 0; n < 4; ++n) acc[b][n] = zero;
    }
    // Loads are unconditional: past the end the last unit is fetched again and not used.
    auto unit_at = [&](uint32_t u) { return min(u, nunits - 1); };
    const uint32_t nt = a.ttiles * 16;
    u32x4 st[SW], ss;
    auto stage_load = [&](uint32_t u, int q) {  // blocks wave and wave + 8 of the half chunk, 1 KiB each
        const uint8_t *base = reinterpret_cast<const uint8_t *>(a.xh) +
                              (((size_t)(u * 4 + q / 2) * nt + tt * 16) * 2 + (q & 1)) * 1024;
#pragma unroll
        for (int i = 0; i < SW; ++i)
            st[i] = load_at<u32x4>(base, (wave + 8 * (i & 1)) * 2048 + lane * 16 + (i >= 2 ? a.xl_offset : 0));
    };
    auto stage_store = [&](uint32_t slot) {
#pragma unroll
        for (int i = 0; i < SW; ++i) xs[slot * L::SLOT + L::W + (wave + 8 * i) * 64 + lane] = st[i];
    };
    auto sums_load = [&](uint32_t u) {  // 16 blocks x 32 words: one per thread
        ss = load_at<u32x4>(reinterpret_cast<const uint8_t *>(a.xsum) + ((size_t)u * nt + tt * 16) * 512, tid * 16);
    };
    struct Op {
        uint32_t hi[4], lo[4];
        float scale;
    } op;
    auto make = [&](auto q_c, const typename F::Dec &d, const typename F::Unit &r) {
        constexpr int Q = decltype(q_c)::value;
        if constexpr (DIRECT)
            F::template direct<Q>(op.hi, d, r, g);
        else
            F::template operand<Q>(op.hi, op.lo, d, r, g);
        if constexpr (G32) op.scale = F::template scale<Q>(d);
    };
    auto op_store = [&](uint32_t slot) {
        u32x4 *dst = xs + slot * L::SLOT + wave * L::WPARTS * 64 + lane;
        u32x4 w;
        __builtin_memcpy(&w, op.hi, 16);
        dst[0] = w;
        if constexpr (WLO) {
            __builtin_memcpy(&w, op.lo, 16);
            dst[64] = w;
        }
        if constexpr (G32) {
            if (g == 0) reinterpret_cast<float *>(xs + slot * L::SLOT + L::W + L::X)[wave * 16 + j] = op.scale;
        }
    };
    // what is shared per unit: scales, offsets, sums
    auto unit_words = [&](uint32_t parity) { return xs + 2 * L::SLOT + parity * L::UNIT; };
    auto unit_store = [&](uint32_t parity, const typename F::Dec &d) {
        u32x4 *w = unit_words(parity);
        if constexpr (TMP) {
            if (g == 0) reinterpret_cast<float *>(w)[wave * 16 + j] = F::unit_scale(d);
        }
        if constexpr (OFFSET) {
            uint32_t hi, lo;
            F::offsets(hi, lo, d, g, m.offset_up);
            uint32_t *o = reinterpret_cast<uint32_t *>(w + 32 + wave * 32 + j) + g;
            o[0] = hi;
            o[16 * 4] = lo;
            w[32 + 8 * 32 + tid] = ss;
        }
    };
    typename F::Unit un;
    typename F::Dec dec;
    stage_load(u0, 0);
    if constexpr (OFFSET) sums_load(u0);
    static_for<0, 4>([&](auto c) { F::template load<decltype(c)::value>(un, m, wl, u0); });
    F::decode(dec, un, g);
    make(std::integral_constant<int, 0>{}, dec, un);
    stage_store(0);
    op_store(0);
    unit_store(u0 & 1, dec);
    make(std::integral_constant<int, 1>{}, dec, un);
    F::template load<0>(un, m, wl, unit_at(u0 + 1));
    stage_load(u0, 1);
    __syncthreads();
    for (uint32_t u = u0; u < u1; ++u) {
        const uint32_t next = unit_at(u + 1);
        floatx4 tmp[TMP ? 4 : 1][TMP ? 4 : 1], late[4];
        float sc[4];
        static_for<0, 8>([&](auto q_c) {
            constexpr int q = decltype(q_c)::value, q2 = (q + 2) & 7;
            const u32x4 *aw = xs + (q & 1) * L::SLOT + wr * 4 * L::WPARTS * 64 + lane;
            const u32x4 *bw = xs + (q & 1) * L::SLOT + L::W + wc * 4 * 64 + lane;
            u32x4 ah[4], al[4], bh[2], bl[2];
            bh[0] = bw[0];
            if (SPLIT) bl[0] = bw[16 * 64];
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                ah[b] = aw[b * L::WPARTS * 64];
                if (WLO) al[b] = aw[b * L::WPARTS * 64 + 64];
                if (G32)
                    sc[b] = reinterpret_cast<const float *>(xs + (q & 1) * L::SLOT + L::W + L::X)[(wr * 4 + b) * 16 + j];
                if (TMP && q % CHAIN == CHAIN - 1)
                    sc[b] = reinterpret_cast<const float *>(unit_words(u & 1))[(wr * 4 + b) * 16 + j];
            }
            __builtin_amdgcn_sched_barrier(0);
            stage_store(1 - (q & 1));
            op_store(1 - (q & 1));
            stage_load(q < 6 ? u : next, q2);
            if constexpr (OFFSET && q == 0) sums_load(next);
            __builtin_amdgcn_sched_barrier(0);
            static_for<0, 4>([&](auto n_c) {
                constexpr int n = decltype(n_c)::value, cur = n & 1;
                if constexpr (n < 3) {
                    bh[1 - cur] = bw[(n + 1) * 64];
                    if (SPLIT) bl[1 - cur] = bw[(16 + n + 1) * 64];
                }
                const half8 x8 = as_half8(bh[cur]);
                floatx4 t[4];
#pragma unroll
                for (int b = 0; b < 4; ++b)
                    t[b] = mfma(x8, as_half8(ah[b]), DIRECT ? acc[b][n] : G32 || q % CHAIN == 0 ? zero : tmp[TMP ? b : 0][TMP ? n : 0]);
                if constexpr (SPLIT) {
                    const half8 l8 = as_half8(bl[cur]);
#pragma unroll
                    for (int b = 0; b < 4; ++b) t[b] = mfma(l8, as_half8(ah[b]), t[b]);
                }
                if constexpr (WLO) {
#pragma unroll
                    for (int b = 0; b < 4; ++b) t[b] = mfma(x8, as_half8(al[b]), t[b]);
                }
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    if constexpr (G32) {
                        // the sums of the token block before: its MFMAs have ended meanwhile
                        if constexpr (n > 0) {
                            add_scaled(acc[b][n - 1], late[b], sc[b]);
                            keep_here(acc[b][n - 1]);
                        }
                        late[b] = t[b];
                    } else if constexpr (DIRECT) {
                        acc[b][n] = t[b];
                    } else {
                        if constexpr (q % CHAIN == CHAIN - 1 && n > 0) {
                            add_scaled(acc[b][n - 1], tmp[b][n - 1], sc[b]);
                            keep_here(acc[b][n - 1]);
                        }
                        tmp[b][n] = t[b];
                    }
                }
                if constexpr (n == 0 && q == 6) F::decode(dec, un, g);
                if constexpr (n == 1) {
                    make(std::integral_constant<int, q2>{}, dec, un);
                    // the bytes of the next unit where the old ones have served
                    if constexpr (q2 & 1) F::template load<q2 / 2>(un, m, wl, q == 7 ? unit_at(u + 2) : next);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
            if constexpr (TMP && q % CHAIN == CHAIN - 1) {
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    add_scaled(acc[b][3], tmp[b][3], sc[b]);
                    keep_here(acc[b][3]);
                }
            }
            if constexpr (G32) {
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    add_scaled(acc[b][3], late[b], sc[b]);
                    keep_here(acc[b][3]);
                }
            }
            if constexpr (q == 7 && (TMP || OFFSET)) {
                const u32x4 *w = unit_words(u & 1);
                u32x4 o[4];
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    if (OFFSET) o[b] = w[32 + (wr * 4 + b) * 32 + 16 * (g >> 1) + j];
                }
                static_for<0, 4>([&](auto n_c) {
                    constexpr int n = decltype(n_c)::value;
                    u32x4 sums;
                    if (OFFSET) sums = w[32 + 8 * 32 + (wc * 4 + n) * 32 + (lane & 31)];
#pragma unroll
                    for (int b = 0; b < 4; ++b) {
                        if constexpr (OFFSET)
                            add_scaled(acc[b][n], mfma(as_half8(sums), as_half8(o[b]), zero), m.offset_down);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                });
                unit_store((u + 1) & 1, dec);
            }
            __syncthreads();
        });
    }
#pragma unroll
    for (int b = 0; b < 4; ++b)
        store_row(a, m, acc[b], DIRECT ? 1.f / kDirectScale : 1.f, row0 + (wr * 4 + b) * 16 + j,
                  tt * TILE_TOKENS + wc * 64 + 4 * g, ky);
}

template <class K>
int launch_with_lds(wgml_ctx *ctx, K kernel, const GemmArgs &a, uint32_t grid, uint32_t threads, size_t lds) {
    wgml_kernel_info &ki = ctx->kernel_info[(const void *)kernel];
    if (lds > 64 * 1024 && !ki.opted_in) {
        // gfx950 has 160 KB of LDS per CU; above 64 KB a kernel must opt in once
        WGML_CHECK_HIP(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        ki.opted_in = true;
    }
    kernel<<<dim3(grid), dim3(threads), lds, ctx->stream>>>(a);
    WGML_CHECK_LAUNCH();
    ctx->launches++;
    return WGML_OK;
}

template <class F, int NT, bool SPLIT>
int launch_rows(wgml_ctx *ctx, const GemmArgs &a, uint32_t tiles) {
    return launch_with_lds(ctx, gemm_lds_kernel<F, NT, SPLIT>, a, tiles * a.ks, 256,
                           gemm_lds_words<F, SPLIT>(NT) * sizeof(u32x4));
}

template <class F, bool SPLIT>
int launch_gemm_prec(wgml_ctx *ctx, const GemmArgs &a, uint32_t tiles) {
    if (a.tall)
        return launch_with_lds(ctx, gemm_tile_kernel<F, SPLIT>, a, tiles * a.ttiles * a.ks, 512,
                               TileLds<F, SPLIT>::WORDS * sizeof(u32x4));
    switch (a.nt) {  // token_blocks
    case 1: return launch_rows<F, 1, SPLIT>(ctx, a, tiles);
    case 2: return launch_rows<F, 2, SPLIT>(ctx, a, tiles);
    case 3: return launch_rows<F, 3, SPLIT>(ctx, a, tiles);
    case 4: return launch_rows<F, 4, SPLIT>(ctx, a, tiles);
    case 6: return launch_rows<F, 6, SPLIT>(ctx, a, tiles);
    default: return launch_rows<F, 8, SPLIT>(ctx, a, tiles);
    }
}

template <class F>
int launch_gemm_fmt(wgml_ctx *ctx, const GemmArgs &a, uint32_t tiles) {
    return a.xl ? launch_gemm_prec<F, true>(ctx, a, tiles) : launch_gemm_prec<F, false>(ctx, a, tiles);
}

}  // namespace
