// Dense f32 products, and the host side of every matrix-vector product (the kernels are in gemv_kernels.h).
#include "gemv_kernels.h"

namespace {

// The kernels a decode step launches by default come first and side by side: 16 tokens of the 7B shape take 22.59 ms, with
// the same kernels scattered over the code object 22.64 to 22.69.
template __global__ void gemv_fused_kernel<1, 1024, 5, 0, false>(const FusedParams);
template __global__ void gemv_fused_kernel<1, 1024, 1, WGML_Q4_K, false>(const FusedParams);
template __global__ void gemv_quant_i8_kernel<IFmtQ4K, 1, 1, 1024, 8, false>(const GemvParams);
template __global__ void gemv_gated_kernel<1024, WGML_Q4_K>(const GatedParams);
template __global__ void gemv_quant_i8_kernel<IFmtQ6K, 1, 1, 1024, 4, false>(const GemvParams);
template __global__ void gemv_fused_kernel<1, 1024, 1, WGML_Q6_K, false>(const FusedParams);
template __global__ void gemv_fused_kernel<1, 768, 1, WGML_Q6_K, false>(const FusedParams);
template __global__ void gemv_gated_kernel<1024, WGML_Q6_K>(const GatedParams);
template __global__ void gemv_fused_kernel<1, 1024, 1, WGML_Q8_0, false>(const FusedParams);
template __global__ void gemv_quant_i8_kernel<IFmtQ8_0, 1, 1, 1024, 8, false>(const GemvParams);
template __global__ void gemv_gated_kernel<1024, WGML_Q8_0>(const GatedParams);
// (the output matrix of a token loop)
template __global__ void gemv_quant_i8_kernel<IFmtQ6K, 1, 1, 1024, 4, false, EXTRA_MAXIMA>(const GemvParams);
template __global__ void gemv_quant_i8_kernel<IFmtQ8_0, 2, 1, 1024, 4, false, EXTRA_MAXIMA>(const GemvParams);
template __global__ void gemv_quant_i8_kernel<IFmtQ8_0, 1, 1, 1024, 8, false, EXTRA_MAXIMA>(const GemvParams);
template __global__ void gemv_quant_i8_kernel<IFmtQ4K, 1, 1, 1024, 8, false, EXTRA_MAXIMA>(const GemvParams);

// ------------------------------------------------------------- dense f32 ----
// out = A v, A row-major f32 (p.p0).  One wave per row, float4 loads, x from LDS.  For what the
// shared body does not take -- f32 tensors as operator arguments (any width and alignment) and
// matrices whose rows are not a multiple of 16 floats -- and for what it takes longer for
// (dense_f32_general_faster).
__global__ __launch_bounds__(256) void gemv_f32_kernel(const GemvParams p, int vec4) {
    extern __shared__ float4 smem[];
    __shared__ float red[16];
    float *xs = reinterpret_cast<float *>(smem);
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nwaves = blockDim.x >> 6;
    const uint32_t nrows = p.nrows, ncols = p.ncols;
    float rms = 1.f;
    if (p.norm_w) rms = block_rms_scale(p, red);  // needs ncols % 4 == 0 and aligned x
    for (uint32_t i = tid; i < ncols; i += blockDim.x)
        xs[i] = p.norm_w ? (p.x[i] * rms) * p.norm_w[i] : p.x[i];
    __syncthreads();
    const uint32_t row = blockIdx.x * nwaves + wave;
    if (row >= nrows) return;
    const float *ar = reinterpret_cast<const float *>(p.p0) + (size_t)row * ncols;
    float acc = 0.f;
    if (vec4) {
        const float4 *a4 = reinterpret_cast<const float4 *>(ar);
        const uint32_t n4 = ncols >> 2;
        for (uint32_t g = lane; g < n4; g += 64) {
            const float4 av = a4[g];
            const float4 xv = smem[g];
            acc = fmaf(av.x, xv.x, acc);
            acc = fmaf(av.y, xv.y, acc);
            acc = fmaf(av.z, xv.z, acc);
            acc = fmaf(av.w, xv.w, acc);
        }
    } else {
        for (uint32_t j = lane; j < ncols; j += 64) acc = fmaf(ar[j], xs[j], acc);
    }
    const float total = wave_sum(acc);
    if (lane == 0) {
        float *out = p.out;
        if (p.dyn_pos) out += (size_t)(*p.dyn_pos) * p.out_pos_stride;
        float v = total;
        if (p.bias) v += p.bias[row];
        if (p.accumulate) v += out[row];
        out[row] = v;
    }
}

// out = A^T v: thread per output column, coalesced across columns.
__global__ __launch_bounds__(256) void gemv_tr_f32_kernel(const float *__restrict__ a,
                                                          const float *__restrict__ v,
                                                          float *__restrict__ out, uint32_t nrows,
                                                          uint32_t ncols) {
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= ncols) return;
    float acc = 0.f;
    for (uint32_t i = 0; i < nrows; ++i) acc = fmaf(a[(size_t)i * ncols + j], v[i], acc);
    out[j] = acc;
}

constexpr size_t kMaxLds = 128 * 1024;

// Workgroups of `fn` that fit a CU with `lds` bytes of dynamic LDS (opting in to more than
// 64 KB first); remembered per context and kernel.
int blocks_per_cu(wgml_ctx *ctx, const void *fn, int threads, size_t lds, int *blocks) {
    wgml_kernel_info &ki = ctx->kernel_info[fn];
    if (lds > 64 * 1024 && !ki.opted_in) {
        // gfx950 has 160 KB of LDS per CU; above 64 KB a kernel must opt in once.
        WGML_CHECK_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)kMaxLds));
        ki.opted_in = true;
    }
    if (ki.lds != lds) {
        int nb = 0;
        WGML_CHECK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, fn, threads, lds));
        ki.blocks_per_cu = nb > 0 ? nb : 1;
        ki.lds = lds;
    }
    *blocks = ki.blocks_per_cu;
    const int cap = ctx->tuning[WGML_TUNE_GEMV_WG_PER_CU];
    if (cap > 0 && cap < *blocks) *blocks = cap;
    return WGML_OK;
}

// Shares `ngroups` row-groups out over at most `max_wgs` workgroups of up to
// `max_waves` waves: every workgroup gets the same count c (the last one the
// remainder), and the fewest waves are active that still give every wave at most
// ceil(c / max_waves) groups, so that the waves of a workgroup finish together.
// A wave parks one result per lane, so it takes at most `max_per_wave` groups (64 results
// divided by the results of a group): very tall matrices get more workgroups than the
// machine holds at once.
struct WgPlan {
    uint32_t groups_per_wg, active_waves, wgs;
};
WgPlan plan_groups(uint32_t ngroups, uint32_t max_wgs, uint32_t max_waves, uint32_t max_per_wave,
                   uint32_t min_c = 1) {
    if (ngroups == 0) return {1, 1, 1};
    if (max_wgs < 1) max_wgs = 1;
    uint32_t c = (ngroups + max_wgs - 1) / max_wgs;
    if (c > max_per_wave * max_waves) c = max_per_wave * max_waves;
    // small matrices: a few groups per workgroup rather than one wave per workgroup
    const uint32_t floor_c = max_waves < 4 ? max_waves : 4;
    if (c < floor_c) c = floor_c;
    if (c < min_c) c = min_c;
    if (c > ngroups) c = ngroups;
    const uint32_t wgs = (ngroups + c - 1) / c;
    c = (ngroups + wgs - 1) / wgs;
    const uint32_t k = (c + max_waves - 1) / max_waves;
    const uint32_t nw = (c + k - 1) / k;
    return {c, nw, wgs};
}

// LDS a workgroup of the shared body needs for x: two int8 planes + per-tile scales and sums
// (integer dot), or the floats themselves + per-tile sums (fp32 activations).
template <class F>
size_t lds_bytes_of(uint32_t ncols) {
    const uint32_t ntiles = ncols / F::TILE;
    const size_t ntiles_pad = ((ntiles + 63) / 64) * 64;
    if (F::F32X) return ntiles_pad * (F::TILE / 4) * 16 + ntiles_pad * F::NSUM * 4;
    return ntiles_pad * 2 * (F::TILE / 16) * 16 + ntiles_pad * (F::NXB + F::NSUM) * 4;
}
// `fn`: a gemv_quant_i8_kernel with R rows per group and workgroups of `maxt` threads.
// `n_maxima`: fn leaves maxima (EXTRA_MAXIMA); receives how many, 0 (and none are left) if they are more than kMaxRowMaxima.
// `cap`: workgroups per compute unit at most.
int launch_plain(wgml_ctx *ctx, const void *fn, uint32_t R, uint32_t maxt, GemvParams p, size_t lds,
                 uint32_t *n_maxima = nullptr, int cap = 8) {
    int per_cu = 1;
    WGML_TRY(blocks_per_cu(ctx, fn, (int)maxt, lds, &per_cu));
    if (per_cu > cap) per_cu = cap;
    const uint32_t cu = ctx->n_cu > 0 ? (uint32_t)ctx->n_cu : 256u;
    // One workgroup per CU with all its waves at work rather than two half-empty ones
    // (each would stage x), as long as that still gives every CU a workgroup (min_c).
    const uint32_t ngroups = (p.nrows + R - 1) / R;
    uint32_t min_c = (ngroups + cu - 1) / cu;
    if (min_c > maxt / 64) min_c = maxt / 64;
    const WgPlan plan = plan_groups(ngroups, cu * (uint32_t)per_cu, maxt / 64, 64 / R, min_c);
    p.active_waves = plan.active_waves;
    if (n_maxima) {
        // a wave's number is that of its first row-group
        const uint32_t waves = plan.wgs * plan.active_waves, n = waves < ngroups ? waves : ngroups;
        *n_maxima = n <= kMaxRowMaxima ? n : 0;
        if (!*n_maxima) p.maxima = nullptr;
    }
    void *args[] = {&p};
    WGML_CHECK_HIP(hipLaunchKernel(fn, dim3(plan.wgs), dim3(maxt), args, lds, ctx->stream));
    WGML_CHECK_LAUNCH();
    ctx->launches++;
    return WGML_OK;
}

template <class F, int R, int D, int MAXT, int MINW = MAXT / 256, bool XPART = false>
int launch_variant_i8(wgml_ctx *ctx, const GemvParams &p, size_t lds, int cap = 8) {
    return launch_plain(ctx, (const void *)gemv_quant_i8_kernel<F, R, D, MAXT, MINW, XPART>, R, MAXT, p, lds, nullptr, cap);
}

// Workgroups per compute unit, at most, of a plain product with fp32 activations.  Two share the loads of a tall matrix better as long
// as its rows fill the lanes of their steps (f32: 1024 columns a step); below 40 rows per compute unit the second ones are too few to
// come out even.  us, two / one: f32 50257x272 14.4 / 13.3, x512 19.0 / 17.6, x768 26.5 / 25.6, x896 30.5 / 30.7, x1008 35.2 / 36.4,
// x1280 44.3 / 42.2, x2048 70.1 / 71.5; 16384x1024 12.7 / 13.0, 8200x1024 7.9 / 7.7, 6000x2048 11.8 / 10.2; Q6_K 50257x768 22.5 / 23.8,
// 32000x2048 14.9 / 16.5, x4096 21.1 / 20.6, 11008x4096 9.4 / 9.2, 8192x3072 6.8 / 6.7, 6144x1024 5.9 / 5.3, 5000x4096 6.9 / 6.1.
template <class WF>
int f32_wgs_per_cu(const wgml_ctx *ctx, const GemvParams &p) {
    const uint32_t cu = ctx->n_cu > 0 ? (uint32_t)ctx->n_cu : 256u, steps = (p.ncols + 1023) / 1024;
    if (std::is_same_v<WF, FmtF32>) return p.nrows >= 40 * cu && p.ncols >= steps * 896 ? 2 : 1;
    if (std::is_same_v<WF, FmtQ6K>) return p.nrows >= 40 * cu && p.ncols <= 2048 ? 2 : 1;
    return 8;
}

bool legacy_format(int type) {
    return type == WGML_Q4_0 || type == WGML_Q4_1 || type == WGML_Q5_0 || type == WGML_Q5_1;
}
// Tiles of two blocks instead of one: a lane asks for twice the bytes, and a row of up to 4096 columns is one step.  Up to
// 2048 columns the lanes' blocks are one step as it is, and tiles of two would leave half of them idle.  us per launch, blocks as
// in the file / planes, tiles of one block / of two: Q4_0 3072x3072 4.8 / 4.6 / 3.9, gate and up 8192x3072 11.8 / 9.0 / 8.2,
// 3072x8192 7.1 / 6.7 / 6.1, 32000x3072 18.7 / 17.2 / 12.3, 4096x2112 4.4 / 4.4 / 4.2; gate and up 5632x2048 6.8 / 5.9 / -;
// Q5_0 gate and up 8192x3072 13.7 / 10.9 / 10.5; Q5_1 3072x8192 7.4 / 7.6 / 7.4.
int legacy_kernel_format(int type, uint32_t ncols) {
    return ncols > 2048 && ncols % 64 == 0 ? kLegacyWide + type : type;
}

// Workgroups per compute unit, at most.  Q5_1 matrices of more than 256 MB whose rows fill the lanes are faster with one (the file's
// blocks, of 24 bytes, streamed better than three planes do).  us, blocks as in the file / planes, two workgroups / one: 128256x4096 68.2 /
// 69.3 / 67.2, 64000x8192 68.1 / 71.6 / 70.0, 256000x2048 64.4 / 67.9 / 66.4, 151936x3584 75.6 / 72.8 / 70.6; 64000x4096 36.3 / 34.6 / 35.2,
// 128256x5120 92.9 / 92.3 / 94.1.
int legacy_wgs_per_cu(int type, const GemvParams &p) {
    if (type != WGML_Q5_1 || (uint64_t)p.nrows * (p.ncols / 32) * 24 <= (uint64_t(256) << 20)) return 8;
    const uint32_t tiles = p.ncols / (legacy_kernel_format(type, p.ncols) == type ? 32 : 64), steps = (tiles + 63) / 64;
    return tiles >= steps * 48 ? 1 : 8;
}

size_t lds_bytes_legacy(int type, uint32_t ncols) {
    return legacy_kernel_format(type, ncols) == type ? lds_bytes_of<IFmtLegacy<false, false, 1>>(ncols)
                                                     : lds_bytes_of<IFmtLegacy<false, false, 2>>(ncols);
}

int launch_legacy(wgml_ctx *ctx, int type, const GemvParams &p) {
    if (p.part_n) return set_error(WGML_E_UNSUPPORTED, "gemv_quant: no merging kernel for this format");
    const size_t lds = lds_bytes_legacy(type, p.ncols);
    if (lds > kMaxLds)
        return set_error(WGML_E_UNSUPPORTED, "gemv_quant: %u columns need %zu bytes of LDS (limit %zu)", p.ncols, lds,
                         kMaxLds);
    return launch_plain(ctx, gemv_legacy_kernels(legacy_kernel_format(type, p.ncols)).plain, 1, 1024, p, lds, nullptr,
                        legacy_wgs_per_cu(type, p));
}

template <class F, int R, int D>
int launch_rd_i8(wgml_ctx *ctx, const GemvParams &p, size_t lds, int waves) {
    switch (waves) {
    case 16: return launch_variant_i8<F, R, D, 1024>(ctx, p, lds);
    case 8: return launch_variant_i8<F, R, D, 512>(ctx, p, lds);
    default: return launch_variant_i8<F, R, D, 256>(ctx, p, lds);
    }
}

// GPT-2 124M's shapes, Q8_0 rows of 768 columns: 16-wave workgroups are as fast as 8-wave
// ones or faster -- 3072x768 3.3 against 3.6 us, 50257x768 11.1 against 13.4 -- and the
// tall output projection gains again from two rows per wave, 10.7 us.
int rows_per_wave_q8(const GemvParams &p) { return p.ncols <= 1024 && p.nrows >= 16384 ? 2 : 1; }

// SWEEP: the variants the tuning keys select (rows per wave, waves per workgroup, depth) exist
// for this format; otherwise only the default one.
template <class F, bool SWEEP = true>
int launch_fmt_i8(wgml_ctx *ctx, const GemvParams &p) {
    constexpr int PCH = F::TILE / 16, MF = F::NXB + F::NSUM;
    const uint32_t ntiles = p.ncols / F::TILE;
    const uint32_t ntiles_pad = ((ntiles + 63) / 64) * 64;
    const size_t lds = (size_t)ntiles_pad * 2 * PCH * 16 + (size_t)ntiles_pad * MF * 4;
    if (lds > kMaxLds)
        return set_error(WGML_E_UNSUPPORTED,
                         "gemv_quant: %u columns need %zu bytes of LDS (limit %zu)", p.ncols, lds,
                         kMaxLds);
    // Defaults from a sweep over the Llama-2-7B shapes on MI355X: one row per
    // wave and 16-wave workgroups (x is staged once per 16 rows in flight), and
    // no register ring for Q4_K and Q6_K: a deeper pipeline measured slower at every
    // shape, also with exact waits (11008x4096 Q4_K: 7.7 us at depth 1, 8.1 at 2, 8.8
    // at 3; Q6_K spills from depth 2 on).
    int R = ctx->tuning[WGML_TUNE_GEMV_ROWS_PER_WAVE], waves = ctx->tuning[WGML_TUNE_GEMV_WAVES_PER_WG],
        depth = ctx->tuning[WGML_TUNE_GEMV_DEPTH];
    const bool q8 = F::TILE == 32;
    if (!R) R = q8 && SWEEP ? rows_per_wave_q8(p) : 1;
    if (!waves) waves = 16;
    if (waves == 12) waves = 16;  // 12-wave workgroups exist for the fused launches only
    // Q8_0 rows of five and more steps (over 8192 columns): four tiles in flight per wave
    // (4096x11008: 11.0 us against 13.4); everywhere else one tile is as fast or faster
    if (!depth) depth = (q8 && ntiles > 256 && SWEEP) ? 4 : 1;
    if (p.part_n) {
        // the input is merged from attention partial results: one configuration (16-wave
        // workgroups with room for the partial results in registers)
        if constexpr (SWEEP) return launch_variant_i8<F, 1, 1, 1024, 4, true>(ctx, p, lds);
        return set_error(WGML_E_UNSUPPORTED, "gemv_quant: no merging kernel for this format");
    }
    if constexpr (SWEEP) {
        if (R == 2) {
            if (depth >= 2) return launch_rd_i8<F, 2, 2>(ctx, p, lds, waves);
            return launch_rd_i8<F, 2, 1>(ctx, p, lds, waves);
        }
        if (depth >= 4) return launch_rd_i8<F, 1, 4>(ctx, p, lds, waves);
        if (depth == 3) return launch_rd_i8<F, 1, 3>(ctx, p, lds, waves);
        if (depth == 2) return launch_rd_i8<F, 1, 2>(ctx, p, lds, waves);
        if constexpr (std::is_same_v<F, IFmtQ4K> || std::is_same_v<F, IFmtQ8_0>) {
            // these fit 64 vector registers without spilling: two workgroups per CU
            if (waves == 16) return launch_variant_i8<F, 1, 1, 1024, 8>(ctx, p, lds);
        }
        return launch_rd_i8<F, 1, 1>(ctx, p, lds, waves);
    } else {
        return launch_variant_i8<F, 1, 1, 1024>(ctx, p, lds);
    }
}

// fp32-activation path: the same body with x staged as floats.  16-wave workgroups, or 8-wave workgroups with two tiles in flight
// per wave when WGML_TUNE_GEMV_WAVES_PER_WG is 8.
template <class WF>
int launch_fmt_f32(wgml_ctx *ctx, const GemvParams &p) {
    using F = FFmt<WF>;
    const uint32_t ntiles = p.ncols / F::TILE;
    const uint32_t ntiles_pad = ((ntiles + 63) / 64) * 64;
    const size_t lds = (size_t)ntiles_pad * F::CHUNKS * 16 + (size_t)ntiles_pad * F::NSUM * 4;
    if (lds > kMaxLds)
        return set_error(WGML_E_UNSUPPORTED,
                         "gemv_quant: %u columns need %zu bytes of LDS (limit %zu)", p.ncols, lds,
                         kMaxLds);
    if constexpr (!std::is_same_v<WF, FmtF32>) {
        if (p.part_n) return launch_variant_i8<F, 1, 1, 1024, 4, true>(ctx, p, lds);
    }
    // (the workgroup size is selectable for the quantized formats only)
    const int waves = std::is_same_v<WF, FmtF32> ? 16 : ctx->tuning[WGML_TUNE_GEMV_WAVES_PER_WG];
    if constexpr (!std::is_same_v<WF, FmtF32>) {
        if (waves == 8) return launch_variant_i8<F, 1, 2, 512, 2>(ctx, p, lds);
    }
    return launch_variant_i8<F, 1, 1, 1024, 4>(ctx, p, lds, f32_wgs_per_cu<WF>(ctx, p));
}

}  // namespace

namespace wgml {

int launch_gemv_f32(wgml_ctx *ctx, float *out, const float *a, uint32_t nrows, uint32_t ncols,
                    int transposed, const float *v) {
    if (transposed) {
        gemv_tr_f32_kernel<<<dim3((ncols + 255) / 256), dim3(256), 0, ctx->stream>>>(a, v, out,
                                                                                     nrows, ncols);
    } else {
        const size_t lds = (((size_t)ncols + 3) / 4) * 16;
        if (lds > kMaxLds)
            return set_error(WGML_E_UNSUPPORTED, "gemv_f32: %u columns exceed the LDS limit", ncols);
        int unused = 0;  // opts in to more than 64 KB of LDS when the row needs it
        WGML_TRY(blocks_per_cu(ctx, (const void *)gemv_f32_kernel, 256, lds, &unused));
        const int vec4 = (ncols % 4 == 0) && ((uintptr_t)a % 16 == 0);
        GemvParams p{};
        p.p0 = reinterpret_cast<const uint8_t *>(a);
        p.x = v;
        p.out = out;
        p.nrows = nrows;
        p.ncols = ncols;
        gemv_f32_kernel<<<dim3((nrows + 3) / 4), dim3(256), lds, ctx->stream>>>(p, vec4);
    }
    WGML_CHECK_LAUNCH();
    ctx->launches++;
    return WGML_OK;
}

// Dense f32 in the shared body.  Defined behind everything else in this file, so that its kernels
// come last in the code object: between the others they moved those by 10 to 30 KB, and decoding the
// 7B shape took 22.82 ms for 16 tokens instead of 22.69, with the same instructions.
static int launch_dense_f32(wgml_ctx *ctx, const GemvParams &p);
static GemvKernels dense_f32_kernels();

// Dense f32 matrices that run in the shared body: whole tiles, and x within the LDS limit.
static bool dense_f32_in_shared_body(const wgml_qmat *m) {
    return m->type == WGML_F32 && m->ncols % FmtF32::TILE == 0 && (size_t)m->ncols * 4 <= kMaxLds;
}

// Products of such matrices (without LayerNorm or activation) that gemv_f32_kernel does faster.
// In the shared body a lane takes 16 columns of a row, there 4, so rows of few columns leave most of
// a wave idle here; but the body requests its weights ahead of x, which the general kernel does
// behind it, a memory round trip that shows where x comes from the launch before.  Beyond 64
// results in each of the machine's waves the body needs a second round of workgroups.  General /
// shared, us, each with x at rest and as part of a chain of dependent products (with the product
// that leads back to x):
//     4096x64     2.0 /  3.0    5.9 /  6.7        8192x512    4.6 /  4.8    9.0 /  9.0
//     4096x256    2.4 /  3.3    6.5 /  6.9        768x768     2.3 /  2.5    6.5 /  5.8
//     768x512     2.1 /  2.5    5.8 /  5.7        4096x1024   4.7 /  4.8    9.8 /  9.2 (1008)
//     32768x256   7.7 /  8.3   12.0 / 12.2        50257x256  13.9 / 13.5
//     50000x128   9.1 /  9.8   13.8 / 14.9        262160x256  69 / 100 (300001)  47 / 82
// A folded RMSNorm makes the general kernel pass over x twice: up to 128 columns it is the faster one
// still (a Llama of dimension 128 at fusion level 2, 40 tokens: 4.29 / 4.40 ms; of 288: 8.0 / 7.0).
static bool dense_f32_general_faster(const wgml_ctx *ctx, uint32_t nrows, uint32_t ncols, bool norm) {
    const uint32_t cu = ctx->n_cu > 0 ? (uint32_t)ctx->n_cu : 256u;
    if (ncols <= 128) return true;
    if (norm) return false;
    if (ncols <= 512 && nrows <= 8192) return true;
    return ncols <= 256 && (nrows <= 32768 || nrows > cu * 16 * 64);
}

// F16 tensors stay 16 bits wide where the shared body always takes their products (dense_f32_general_faster: never beyond
// 512 columns); narrower or ragged rows are expanded to f32 when the matrix is created.
bool gemv_keeps_f16(uint32_t ncols) {
    return ncols > 512 && ncols % FmtF16::TILE == 0 && (size_t)ncols * 4 <= kMaxLds;
}
static int dense_format(const wgml_qmat *m) { return m->half ? kFusedDenseF16 : kFusedDenseF32; }

bool gemv_partials_supported(const wgml_ctx *, const wgml_qmat *m) {
    return m && (m->type == WGML_Q4_K || m->type == WGML_Q6_K || m->type == WGML_Q8_0);
}

static size_t lds_bytes_fused(int type, uint32_t ncols, bool f32) {
    switch (type) {
    case WGML_F32: return lds_bytes_of<FFmt<FmtF32>>(ncols);
    case WGML_Q4_K: return f32 ? lds_bytes_of<FFmt<FmtQ4K>>(ncols) : lds_bytes_of<IFmtQ4K>(ncols);
    case WGML_Q6_K: return f32 ? lds_bytes_of<FFmt<FmtQ6K>>(ncols) : lds_bytes_of<IFmtQ6K>(ncols);
    case WGML_Q8_0: return f32 ? lds_bytes_of<FFmt<FmtQ8_0>>(ncols) : lds_bytes_of<IFmtQ8_0>(ncols);
    case WGML_Q5_K: return lds_bytes_of<IFmtQ5K>(ncols);
    case WGML_Q8_K: return lds_bytes_of<IFmtQ8K>(ncols);
    default: return lds_bytes_legacy(type, ncols);
    }
}

static bool main_format(int type) { return type == WGML_Q4_K || type == WGML_Q6_K || type == WGML_Q8_0; }

// With LayerNorm or activation (gemv_full.hip): one variant per format, Q8_0 in one or two rows per wave; the overrides of rows, waves and
// depth do not reach these.  (Q8_0 rows of more than 8192 columns with four tiles in flight, as without LayerNorm: a GPT-2 of 8448 columns
// with 50257 logits 264 us per token, with one tile 259.)
static int launch_full(wgml_ctx *ctx, const wgml_qmat *m, const GemvParams &p, uint32_t *n_maxima) {
    if (m->type == WGML_F32 && !dense_f32_in_shared_body(m))
        return set_error(WGML_E_UNSUPPORTED, "gemv_quant: LayerNorm / activation folding needs rows of a "
                                             "multiple of 16 elements");
    if (p.part_n) return set_error(WGML_E_UNSUPPORTED, "gemv_quant: no merging kernel with an activation");
    const bool f32 = m->type == WGML_F32 || (main_format(m->type) && ctx->tuning[WGML_TUNE_GEMV_F32_ACTIVATIONS]);
    if (p.ln_g && (p.ncols >> 2) > 3u * 1024u)  // XP float4 per thread
        return set_error(WGML_E_UNSUPPORTED, "gemv_quant: %u columns are too many for the folded LayerNorm", p.ncols);
    const size_t lds = lds_bytes_fused(m->type, p.ncols, f32);
    if (lds > kMaxLds)
        return set_error(WGML_E_UNSUPPORTED, "gemv_quant: %u columns need %zu bytes of LDS (limit %zu)", p.ncols, lds,
                         kMaxLds);
    const int fmt = m->type == WGML_F32 ? dense_format(m)
                    : legacy_format(m->type) ? legacy_kernel_format(m->type, p.ncols)
                                             : m->type;
    const int rows = m->type == WGML_Q8_0 && !f32 ? rows_per_wave_q8(p) : 1;
    return launch_plain(ctx, gemv_full_kernels(fmt, f32, rows).plain, (uint32_t)rows, 1024, p, lds, n_maxima);
}

// The kernel that leaves maxima for a plain product (gemv_maxima.hip: one row per wave, one tile in flight, workgroups of 16
// waves), or null where the product runs in another shape: launch-shape overrides, Q8_0 rows that have four tiles in
// flight, dense rows that the general kernel takes, rows beyond the LDS limit (the caller's own path refuses them).
static const void *maxima_kernel_for(const wgml_ctx *ctx, const wgml_qmat *m, const GemvParams &p, uint32_t *rows,
                                     size_t *lds) {
    for (int key : {WGML_TUNE_GEMV_ROWS_PER_WAVE, WGML_TUNE_GEMV_WAVES_PER_WG, WGML_TUNE_GEMV_DEPTH})
        if (ctx->tuning[key]) return nullptr;
    const bool dense = m->type == WGML_F32;
    if (p.part_n || (dense && (!dense_f32_in_shared_body(m) ||
                               dense_f32_general_faster(ctx, p.nrows, p.ncols, p.norm_w != nullptr))))
        return nullptr;
    const bool f32 = dense || (main_format(m->type) && ctx->tuning[WGML_TUNE_GEMV_F32_ACTIVATIONS]);
    if (m->type == WGML_Q8_0 && !f32 && p.ncols > 8192) return nullptr;
    *lds = lds_bytes_fused(m->type, p.ncols, f32);
    if (*lds > kMaxLds) return nullptr;
    *rows = m->type == WGML_Q8_0 && !f32 ? (uint32_t)rows_per_wave_q8(p) : 1u;
    if (!f32) {
        switch (m->type) {
        case WGML_Q6_K: return (const void *)gemv_quant_i8_kernel<IFmtQ6K, 1, 1, 1024, 4, false, EXTRA_MAXIMA>;
        case WGML_Q4_K: return (const void *)gemv_quant_i8_kernel<IFmtQ4K, 1, 1, 1024, 8, false, EXTRA_MAXIMA>;
        case WGML_Q8_0:
            if (*rows == 2) return (const void *)gemv_quant_i8_kernel<IFmtQ8_0, 2, 1, 1024, 4, false, EXTRA_MAXIMA>;
            return (const void *)gemv_quant_i8_kernel<IFmtQ8_0, 1, 1, 1024, 8, false, EXTRA_MAXIMA>;
        default: break;
        }
    }
    return gemv_maxima_kernel(dense                     ? dense_format(m)
                              : legacy_format(m->type) ? legacy_kernel_format(m->type, p.ncols)
                                                       : m->type,
                              f32);
}

int launch_gemv_quant(wgml_ctx *ctx, float *out, const wgml_qmat *m, const float *v,
                      const GemvEpilogue &ep) {
    GemvParams p{};
    p.p0 = m->p0;
    p.p1 = m->p1;
    p.p2 = m->p2;
    p.p3 = m->p3;
    p.x = v;
    p.out = out;
    p.bias = ep.bias;
    p.nrows = m->nrows;
    p.ncols = m->ncols;
    p.accumulate = ep.accumulate;
    p.dyn_pos = ep.dyn_pos;
    p.out_pos_stride = ep.out_pos_stride;
    p.norm_w = ep.norm_w;
    p.norm_eps = ep.norm_eps;
    p.ln_g = ep.ln_gamma;
    p.ln_b = ep.ln_beta;
    p.act = ep.act;
    if (ep.partials.n) {
        const AttnPartials &a = ep.partials;
        if (!gemv_partials_supported(ctx, m) || a.n > 16 || !a.o || !a.ml || a.head_size == 0 ||
            a.head_size % 4 != 0 || a.hsp < a.head_size || a.hsp % 4 != 0 ||
            m->ncols % a.head_size != 0 || m->ncols >= (1u << 20) || a.head_size > 4096 || ep.ln_gamma)
            return set_error(WGML_E_INVALID, "gemv_quant: these attention partial results cannot "
                                             "be merged by this product");
        p.part_o = a.o;
        p.part_ml = a.ml;
        p.part_n = a.n;
        p.part_hsp = a.hsp;
        p.part_hs = a.head_size;
        p.part_hs_inv = (uint32_t)(((uint64_t(1) << 32) + a.head_size - 1) / a.head_size);
        p.x = nullptr;
    } else if ((uintptr_t)v % 16 != 0) {
        return set_error(WGML_E_INVALID, "gemv_quant: the input vector must be 16-byte aligned");
    }
    p.maxima = ep.maxima;
    if (ep.n_maxima) *ep.n_maxima = 0;
    if (p.ln_g || p.act) return launch_full(ctx, m, p, ep.n_maxima);
    if (ep.n_maxima) {
        uint32_t rows = 1;
        size_t lds = 0;
        if (const void *fn = maxima_kernel_for(ctx, m, p, &rows, &lds)) {
            const int cap = m->type == WGML_F32 && !m->half                                          ? f32_wgs_per_cu<FmtF32>(ctx, p)
                            : m->type == WGML_Q6_K && ctx->tuning[WGML_TUNE_GEMV_F32_ACTIVATIONS] ? f32_wgs_per_cu<FmtQ6K>(ctx, p)
                                                                                                  : legacy_wgs_per_cu(m->type, p);
            return launch_plain(ctx, fn, rows, 1024, p, lds, ep.n_maxima, cap);
        }
    }
    if (m->half) return launch_plain(ctx, gemv_f16_kernels().plain, 1, 1024, p, lds_bytes_of<FFmt<FmtF16>>(p.ncols));
    if (dense_f32_in_shared_body(m) && !dense_f32_general_faster(ctx, p.nrows, p.ncols, p.norm_w != nullptr))
        return launch_dense_f32(ctx, p);
    if (m->type == WGML_F32) {
        const size_t lds = (size_t)m->ncols * 4;
        if (lds > kMaxLds)
            return set_error(WGML_E_UNSUPPORTED, "gemv_f32: %u columns exceed the LDS limit",
                             m->ncols);
        int unused = 0;  // opts in to more than 64 KB of LDS when the row needs it
        WGML_TRY(blocks_per_cu(ctx, (const void *)gemv_f32_kernel, 256, lds, &unused));
        gemv_f32_kernel<<<dim3((m->nrows + 3) / 4), dim3(256), lds, ctx->stream>>>(p, 1);
        WGML_CHECK_LAUNCH();
        ctx->launches++;
        return WGML_OK;
    }
    switch (m->type) {  // formats that exist as integer-dot kernels only
    case WGML_Q4_0: case WGML_Q4_1: case WGML_Q5_0: case WGML_Q5_1: return launch_legacy(ctx, m->type, p);
    case WGML_Q5_K: return launch_fmt_i8<IFmtQ5K, false>(ctx, p);
    case WGML_Q8_K: return launch_fmt_i8<IFmtQ8K, false>(ctx, p);
    default: break;
    }
    if (!ctx->tuning[WGML_TUNE_GEMV_F32_ACTIVATIONS]) {
        switch (m->type) {
        case WGML_Q4_K: return launch_fmt_i8<IFmtQ4K>(ctx, p);
        case WGML_Q6_K: return launch_fmt_i8<IFmtQ6K>(ctx, p);
        case WGML_Q8_0: return launch_fmt_i8<IFmtQ8_0>(ctx, p);
        default: break;
        }
    }
    switch (m->type) {
    case WGML_Q4_K: return launch_fmt_f32<FmtQ4K>(ctx, p);
    case WGML_Q6_K: return launch_fmt_f32<FmtQ6K>(ctx, p);
    case WGML_Q8_0: return launch_fmt_f32<FmtQ8_0>(ctx, p);
    default: return set_error(WGML_E_UNSUPPORTED, "gemv_quant: unsupported type %d", m->type);
    }
}

bool gemv_fused_supported(const wgml_qmat *m) {
    if (!m) return false;
    switch (m->type) {
    case WGML_F32: return dense_f32_in_shared_body(m);
    case WGML_Q4_K: case WGML_Q6_K: case WGML_Q8_0: case WGML_Q5_K: case WGML_Q8_K: case WGML_Q4_0:
    case WGML_Q4_1: case WGML_Q5_0: case WGML_Q5_1: return true;
    default: return false;
    }
}

// One launch takes matrices of one format (any of the nine, or dense f32), or a mix of Q4_K / Q6_K
// / Q8_0; with fp32 activations only those three, or dense f32.
bool gemv_fused_set_supported(const wgml_ctx *ctx, const wgml_qmat *const *mats, int n) {
    bool same = true, all_main = true;
    for (int i = 0; i < n; ++i) {
        if (!gemv_fused_supported(mats[i])) return false;
        same = same && mats[i]->type == mats[0]->type;
        all_main = all_main && main_format(mats[i]->type);
    }
    if (ctx->tuning[WGML_TUNE_GEMV_F32_ACTIVATIONS]) return all_main || (same && mats[0]->type == WGML_F32);
    return same || all_main;
}

// The format number of a fused launch's kernel: that of its matrices, kFusedDenseMix for F16 beside F32, or 0 for a mix of the
// main ones.  (us per token of six layers with K and up in F32 and the rest in F16: a launch per operation, as any other mix takes, 187
// for 640 columns and 225 for 1024; in one launch 119 and 150.)
static int fused_format(const FusedGemv &f, uint32_t ncols) {
    const int type = f.jobs[0].a->type;
    bool mix = false;
    for (int i = 0; i < f.njobs; ++i) {
        if (f.jobs[i].a->type != type) return 0;
        mix = mix || f.jobs[i].a->half != f.jobs[0].a->half || (f.jobs[i].mode == FUSED_SILU && f.jobs[i].b->half != f.jobs[0].a->half);
    }
    if (mix) return kFusedDenseMix;
    return type == WGML_F32 ? dense_format(f.jobs[0].a) : legacy_format(type) ? legacy_kernel_format(type, ncols) : type;
}
static GemvKernels fused_kernels(int fmt, bool f32) {
    if (fmt == kFusedDenseF32) return dense_f32_kernels();
    if (fmt == kFusedDenseF16) return gemv_f16_kernels();
    if (fmt == kFusedDenseMix) return gemv_dense_mix_kernels();
    if (f32) {
        switch (fmt) {
        case WGML_Q4_K: return gemv_kernels_of<WGML_Q4_K, true, false>();
        case WGML_Q6_K: return gemv_kernels_of<WGML_Q6_K, true, false>();
        case WGML_Q8_0: return gemv_kernels_of<WGML_Q8_0, true, false>();
        default:
            return {nullptr, (const void *)gemv_fused_kernel<1, 1024, 1, 0, true>,
                    (const void *)gemv_fused_kernel<1, 768, 1, 0, true>, nullptr, nullptr};
        }
    }
    switch (fmt) {
    // the mixed-format kernel is held to 96 registers (5 waves per SIMD): it fits without
    // spilling, and the waves of a workgroup start sooner the fewer registers they take
    case 0:
        return {nullptr, (const void *)gemv_fused_kernel<1, 1024, 5, 0>, (const void *)gemv_fused_kernel<1, 768, 1, 0>,
                nullptr, nullptr};
    case WGML_Q4_K: return gemv_kernels_of<WGML_Q4_K, false, false>();
    case WGML_Q6_K: return gemv_kernels_of<WGML_Q6_K, false, false>();
    case WGML_Q8_0: return gemv_kernels_of<WGML_Q8_0, false, false>();
    case WGML_Q5_K: return gemv_kernels_of<WGML_Q5_K, false, false>();
    case WGML_Q8_K: return gemv_kernels_of<WGML_Q8_K, false, false>();
    default: return gemv_legacy_kernels(fmt);
    }
}

// Workgroups a fused launch is shared out over: one per compute unit, or as many as the machine holds at once where it streams
// more than 64 MB.  A second workgroup on a compute unit stages x again, and the waves' row pairs are fewer and less even.  us
// per launch, as many as fit (two of 64 registers) / one per compute unit: gate and up 8192x3072 in Q4_0 9.2 / 7.8, Q4_1 9.7 / 8.2,
// Q8_0 (53 MB) 11.8 / 11.6, 9216x3072 rows in pairs in Q8_0 9.2 / 8.8, 2304x768 3.8 / 3.4; gate and up 11008x4096 in Q8_0 (96 MB)
// 19.0 / 19.5; F16 2304x4096 9.4 / 8.8, 5120x3072 (63 MB) 12.8 / 12.4, rows in pairs 9216x3072 12.2 / 11.6, 5120x4096 9.95 / 10.1.
static uint32_t fused_workgroups(const wgml_ctx *ctx, int per_cu, uint64_t bytes) {
    const uint32_t cu = ctx->n_cu > 0 ? (uint32_t)ctx->n_cu : 256u;
    return bytes <= (uint64_t(64) << 20) ? cu : cu * (uint32_t)per_cu;
}

// Plane p1 as a kernel gets it: FmtDenseMix tells F32 tensors by their having none.
static const uint8_t *plane1(const wgml_qmat *m) { return m->type == WGML_F32 && !m->half ? nullptr : m->p1; }

static int launch_gated(wgml_ctx *ctx, const FusedGemv &f, const FusedGemvJob &s, uint32_t threads) {
    const uint32_t ncols = s.a->ncols;
    const bool f32 = ctx->tuning[WGML_TUNE_GEMV_F32_ACTIVATIONS] != 0;
    if (!s.b || s.b->type != s.a->type || s.b->nrows != s.a->nrows || s.b->ncols != ncols || s.row0 || s.nrows)
        return set_error(WGML_E_INVALID, "gemv_fused: gate/up matrices differ");
    if (f.ln_gamma) return set_error(WGML_E_UNSUPPORTED, "gemv_fused: a gated job behind a LayerNorm");
    FusedGemv one = f;
    one.jobs[0] = s;
    one.njobs = 1;
    const GemvKernels k = fused_kernels(fused_format(one, ncols), f32);
    const void *kern = threads == 768 ? k.gated768 : k.gated1024;
    const size_t lds = lds_bytes_fused(s.a->type, ncols, f32);
    if (lds > kMaxLds)
        return set_error(WGML_E_UNSUPPORTED, "gemv_fused: %u columns need %zu bytes of LDS", ncols, lds);
    GatedParams P{s.a->p0, plane1(s.a), s.a->p2, s.a->p3, s.b->p0, plane1(s.b), s.b->p2, s.b->p3, f.x, f.norm_w, s.out,
                  f.norm_eps, s.a->nrows, ncols, 0};
    int per_cu = 1;
    WGML_TRY(blocks_per_cu(ctx, kern, (int)threads, lds, &per_cu));
    const uint32_t nwaves = threads / 64;
    const WgPlan plan = plan_groups(P.nrows, fused_workgroups(ctx, per_cu, s.a->gguf_bytes + s.b->gguf_bytes), nwaves, 32);
    P.active_waves = plan.active_waves;
    void *args[] = {&P};
    WGML_CHECK_HIP(hipLaunchKernel(kern, dim3(plan.wgs), dim3(threads), args, lds, ctx->stream));
    WGML_CHECK_LAUNCH();
    ctx->launches++;
    return WGML_OK;
}

// The jobs in PLAIN and ROPE mode.
static int launch_jobs(wgml_ctx *ctx, const FusedGemv &f, uint32_t threads) {
    const uint32_t nwaves = threads / 64, ncols = f.jobs[0].a->ncols;
    FusedParams P{};
    P.njobs = f.njobs;
    P.x = f.x;
    P.norm_w = f.norm_w;
    P.norm_eps = f.norm_eps;
    P.ln_g = f.ln_gamma;
    P.ln_b = f.ln_beta;
    P.pos = f.pos;
    P.head_size = f.head_size ? f.head_size : 2;
    P.rope_base = f.rope_base;
    P.rope_cs = reinterpret_cast<const float2 *>(f.rope_cs);
    P.ncols = ncols;
    const bool f32 = ctx->tuning[WGML_TUNE_GEMV_F32_ACTIVATIONS] != 0;
    size_t lds = 0;
    uint64_t bytes[3] = {0, 0, 0};
    uint32_t ngroups[3];
    for (int i = 0; i < f.njobs; ++i) {
        const FusedGemvJob &s = f.jobs[i];
        GemvJob &j = P.jobs[i];
        j.a0 = s.a->p0; j.a1 = plane1(s.a); j.a2 = s.a->p2; j.a3 = s.a->p3;
        j.out = s.out;
        j.bias = s.bias;
        j.nrows = s.a->nrows;
        if (s.row0 || s.nrows) {  // a slice of the rows: move the plane pointers to its first row
            const uint32_t n = s.nrows ? s.nrows : s.a->nrows - s.row0;
            if ((uint64_t)s.row0 + n > s.a->nrows)
                return set_error(WGML_E_INVALID, "gemv_fused: job %d: bad row slice", i);
            const uint64_t r = s.row0, nb = r * (ncols / 256), nb32 = r * (ncols / 32);
            switch (s.a->type) {
            case WGML_F32: j.a0 += r * ncols * (s.a->half ? 2 : 4); break;
            case WGML_Q4_K: j.a0 += nb * 144; break;
            case WGML_Q5_K: j.a0 += nb * 176; break;
            case WGML_Q8_K: j.a0 += nb * 292; break;
            case WGML_Q6_K: j.a0 += nb * 128; j.a1 += nb * 64; j.a2 += nb * 16; j.a3 += nb * 2; break;
            case WGML_Q8_0: j.a0 += r * ncols; j.a1 += nb32 * 2; break;
            default: {  // the 32-element formats
                const bool has_m = s.a->type == WGML_Q4_1 || s.a->type == WGML_Q5_1;
                j.a0 += nb32 * 16; j.a1 += nb32 * (has_m ? 4 : 2); j.a2 += nb32 * 4;
            }
            }
            j.nrows = n;
        }
        j.kind = gemv_kind(s.a->type, s.mode, s.accumulate);
        j.out_pos_stride = s.out_pos_stride;
        bytes[i] = s.a->gguf_bytes / s.a->nrows * j.nrows;
        if (s.mode == JOB_ROPE && (j.nrows % 2 != 0 || P.head_size % 2 != 0))
            return set_error(WGML_E_INVALID, "gemv_fused: RoPE needs even row counts");
        ngroups[i] = (j.nrows + 1) / 2;
        const size_t l = lds_bytes_fused(s.a->type, ncols, f32);
        if (l > lds) lds = l;
    }
    if (lds > kMaxLds)
        return set_error(WGML_E_UNSUPPORTED, "gemv_fused: %u columns need %zu bytes of LDS", ncols,
                         lds);
    if (P.ln_g && (ncols >> 2) > 3u * threads)  // XP float4 per thread
        return set_error(WGML_E_UNSUPPORTED,
                         "gemv_fused: %u columns are too many for the folded LayerNorm", ncols);
    const int fmt = fused_format(f, ncols);
    // (heads of two elements: both RoPE variants rotate the same pairs)
    const bool neox = f.rope_neox && P.head_size > 2;
    const bool dense = fmt == kFusedDenseF32 || fmt == kFusedDenseF16 || fmt == kFusedDenseMix;
    if (neox && (f32 || dense))
        return set_error(WGML_E_UNSUPPORTED, "gemv_fused: Neox RoPE takes the integer-dot formats only");
    if (P.ln_g && (neox || fmt == 0 || fmt == kFusedDenseMix))
        return set_error(WGML_E_UNSUPPORTED, "gemv_fused: LayerNorm before Neox RoPE or mixed formats");
    const GemvKernels k = P.ln_g ? gemv_full_kernels(fmt, f32 || dense, 1) : fused_kernels(fmt, f32);
    const void *const kern = neox ? gemv_neox_kernel(fmt, (int)threads) : threads == 768 ? k.fused768 : k.fused1024;
    int per_cu = 1;
    WGML_TRY(blocks_per_cu(ctx, kern, (int)threads, lds, &per_cu));
    const uint32_t resident = fused_workgroups(ctx, per_cu, bytes[0] + bytes[1] + bytes[2]);
    // Every workgroup streams about the same number of bytes: the smallest per-
    // workgroup budget T is searched for which the matrices together need no more
    // workgroups than the machine holds at once.
    double bpg[3], lo = 0.0, hi = 0.0;
    for (int i = 0; i < f.njobs; ++i) {
        bpg[i] = (double)bytes[i] / (double)ngroups[i];
        hi += (double)bytes[i];
    }
    auto wgs_needed = [&](double T) {
        uint64_t n = 0;
        for (int i = 0; i < f.njobs; ++i) {
            uint64_t c = (uint64_t)(T / bpg[i]);
            if (c < 1) c = 1;
            n += (ngroups[i] + c - 1) / c;
        }
        return n;
    };
    for (int it = 0; it < 50; ++it) {
        const double mid = 0.5 * (lo + hi);
        if (wgs_needed(mid) <= resident) hi = mid; else lo = mid;
    }
    uint32_t begin = 0;
    for (int i = 0; i < f.njobs; ++i) {
        uint32_t c = (uint32_t)(hi / bpg[i]);
        if (c < 1) c = 1;
        const WgPlan plan = plan_groups(ngroups[i], (ngroups[i] + c - 1) / c, nwaves, 32);
        P.jobs[i].wg_begin = begin;
        P.jobs[i].wg_count = plan.wgs;
        P.jobs[i].active_waves = plan.active_waves;
        begin += plan.wgs;
    }
    const uint32_t half = P.head_size / 2;
    NeoxPairs neox_pairs{half, half ? (uint32_t)(((uint64_t(1) << 32) + half - 1) / half) : 0};
    void *args[] = {&P, &neox_pairs};  // (the others take the first only)
    WGML_CHECK_HIP(hipLaunchKernel(kern, dim3(begin), dim3(threads), args, lds, ctx->stream));
    WGML_CHECK_LAUNCH();
    ctx->launches++;
    return WGML_OK;
}

int launch_gemv_fused(wgml_ctx *ctx, const FusedGemv &f) {
    if (f.njobs < 1 || f.njobs > 3)
        return set_error(WGML_E_INVALID, "gemv_fused: %d jobs", f.njobs);
    if ((uintptr_t)f.x % 16 != 0)
        return set_error(WGML_E_INVALID, "gemv_fused: the input vector must be 16-byte aligned");
    const bool f32 = ctx->tuning[WGML_TUNE_GEMV_F32_ACTIVATIONS] != 0;
    bool gated = false, mixed = false, all_main = true;
    uint32_t pairs = 0;
    for (int i = 0; i < f.njobs; ++i) {
        const FusedGemvJob &s = f.jobs[i];
        if (!gemv_fused_supported(s.a) || s.a->ncols != f.jobs[0].a->ncols)
            return set_error(WGML_E_INVALID, "gemv_fused: job %d has an unsupported matrix", i);
        if (f32 && !main_format(s.a->type) && s.a->type != WGML_F32)
            return set_error(WGML_E_UNSUPPORTED, "gemv_fused: fp32 activations exist for Q4_K, Q6_K "
                                                 "and Q8_0 only");
        gated = gated || s.mode == FUSED_SILU;
        mixed = mixed || s.a->type != f.jobs[0].a->type;
        all_main = all_main && main_format(s.a->type);
        const uint32_t rows = s.nrows ? s.nrows : s.a->nrows - s.row0;
        pairs += s.mode == FUSED_SILU ? rows : (rows + 1) / 2;
    }
    if (mixed && !all_main)
        return set_error(WGML_E_UNSUPPORTED, "gemv_fused: formats can be mixed among Q4_K, Q6_K and Q8_0 only");
    if (gated && f.rope_neox && f.head_size > 2)
        return set_error(WGML_E_INVALID, "gemv_fused: a gated job beside Neox RoPE");
    // 12-wave workgroups for launches with a little less than one row pair per wave of a
    // machine full of 16-wave workgroups (Q/K/V of 4096/1024/1024 rows: 8.6 us against 9.6;
    // small launches are better off with the 16-wave kernel: GPT-2's Q/K/V 5.1 us against 7.1)
    const int waves = ctx->tuning[WGML_TUNE_GEMV_WAVES_PER_WG];
    const uint32_t cu = ctx->n_cu > 0 ? (uint32_t)ctx->n_cu : 256u;
    const uint32_t threads = waves == 12 || (waves != 16 && pairs > cu * 8 && pairs <= cu * 16) ? 768 : 1024;
    if (!gated) return launch_jobs(ctx, f, threads);
    // gated jobs are a launch each
    FusedGemv rest = f;
    rest.njobs = 0;
    for (int i = 0; i < f.njobs; ++i) {
        if (f.jobs[i].mode == FUSED_SILU)
            WGML_TRY(launch_gated(ctx, f, f.jobs[i], threads));
        else
            rest.jobs[rest.njobs++] = f.jobs[i];
    }
    return rest.njobs ? launch_jobs(ctx, rest, threads) : WGML_OK;
}

}  // namespace wgml

extern "C" {

int wgml_gemv_quant(wgml_ctx *ctx, wgml_view out, const wgml_qmat *m, wgml_view v) {
    WGML_REQUIRE(ctx && m, "wgml_gemv_quant: null argument");
    WGML_TRY(check_view(out, "wgml_gemv_quant: out"));
    WGML_TRY(check_view(v, "wgml_gemv_quant: v"));
    WGML_REQUIRE(v.len == m->ncols, "Gemv: dimension mismatch (v has %u, matrix has %u columns)",
                 v.len, m->ncols);
    WGML_REQUIRE(out.len == m->nrows, "Gemv: dimension mismatch (out has %u, matrix has %u rows)",
                 out.len, m->nrows);
    return launch_gemv_quant(ctx, view_ptr(out), m, view_ptr(v), GemvEpilogue{});
}

int wgml_gemv_f32(wgml_ctx *ctx, wgml_view out, wgml_view a, uint32_t nrows, uint32_t ncols,
                  int transposed, wgml_view v) {
    WGML_REQUIRE(ctx != nullptr, "wgml_gemv_f32: null context");
    WGML_TRY(check_view(out, "wgml_gemv_f32: out"));
    WGML_TRY(check_view(a, "wgml_gemv_f32: a"));
    WGML_TRY(check_view(v, "wgml_gemv_f32: v"));
    WGML_REQUIRE((uint64_t)a.len == (uint64_t)nrows * ncols,
                 "wgml_gemv_f32: matrix view has %u elements, expected %llu", a.len,
                 (unsigned long long)nrows * ncols);
    if (transposed) {
        WGML_REQUIRE(v.len == nrows && out.len == ncols, "GemvTr: dimension mismatch");
    } else {
        WGML_REQUIRE(v.len == ncols && out.len == nrows, "Gemv: dimension mismatch");
    }
    return launch_gemv_f32(ctx, view_ptr(out), view_ptr(a), nrows, ncols, transposed, view_ptr(v));
}

}  // extern "C"

namespace wgml {

static int launch_dense_f32(wgml_ctx *ctx, const GemvParams &p) { return launch_fmt_f32<FmtF32>(ctx, p); }

static GemvKernels dense_f32_kernels() { return gemv_kernels_of<kFusedDenseF32, true, false>(); }

}  // namespace wgml
