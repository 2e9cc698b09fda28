// What the kernels of the batched products (gemm_kernel.h, prefill.hip) share.
#pragma once

#include "common.h"

namespace wgml {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));  // plain vector: arrays of it stay in registers

constexpr uint32_t KU = 256;  // elements of K per unit, the step in which K is walked and split
constexpr uint32_t TILE_ROWS = 128, TILE_TOKENS = 256;  // of a workgroup in runs of more than 128 tokens

struct GemmMat {
    const uint8_t *p0, *p1, *p2, *p3;  // matrix planes (as wgml_qmat)
    float *out;                        // [T][out_stride]
    const float *bias;                 // optional, per row
    uint32_t nrows, out_stride;
    uint32_t tile0;                    // first row tile of this matrix in the launch (64 or TILE_ROWS rows)
    uint32_t roff;                     // rows of the matrices before this one in the launch
    uint32_t rope;                     // the reduction rotates this matrix' rows (GemmArgs::rope_*)
    float offset_up, offset_down;      // power of two that brings offsets of weights into f16 range, and its inverse
};

struct GemmArgs {
    GemmMat m[3];
    uint32_t nmat;
    const u32x4 *xh;                   // packed f16 activations (order: top of prefill.hip)
    const u32x4 *xl;                   // their low parts in the same order (split precision only)
    uint32_t xl_offset;                // bytes from xh to xl
    const u32x4 *xsum;                 // sums of 32 activations (order: top of prefill.hip)
    uint32_t ttiles;                   // tiles of tokens
    uint32_t tall;                     // gemm_tile_kernel
    const float *xscale;               // [tpad] factor to multiply a token's results with
    uint32_t ncols, kpad, T, nt;       // nt: blocks of 16 tokens per tile
    int accumulate;                    // out += result
    float *part;                       // [ks][T][total_rows] partial sums (ks > 1)
    uint32_t ks;                       // ways K is split between workgroups (its part varies fastest in the grid up to 128 tokens, slowest beyond)
    uint32_t total_rows;               // rows of all matrices of the launch
    int defer;                         // ks > 1: leave the partial sums to the next kernel
    // rotary encoding applied by gemm_reduce_rope_kernel to the matrices marked `rope`
    uint32_t rope_head_size, rope_pos0;
    float rope_base;
    int rope_neox;
};

#define WGML_GEMM_FORMATS(X) X(q4_k) X(q5_k) X(q6_k) X(q8_0) X(q8_k) X(q4_0) X(q4_1) X(q5_0) X(q5_1)
#define WGML_GEMM_DECLARE(name) int launch_gemm_##name(wgml_ctx *ctx, const GemmArgs &a, uint32_t tiles);
WGML_GEMM_FORMATS(WGML_GEMM_DECLARE)

}  // namespace wgml
