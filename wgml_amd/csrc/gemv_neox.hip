#include "gemv_kernels.h"

namespace {

// The Q/K/V launch of the Neox variant (ops/rope.wgsl:60-78): pair g of a job in ROPE mode is the rows i and
// i + head_size / 2 of a head.  A policy and kernels of its own, in a code object of their own: with the pair
// arithmetic as a case of JobPolicy, or these kernels behind the others, a decode step without them took 0.5-1.3 %
// longer (in the second case with the same instructions).
// Against a rope launch per layer it saves 2.5 us per layer and token (eight layers of 2048 x 5632 in Q5_K, 12 tokens
// and 20 sampled ones: 8.10 ms -> 7.65).
struct NeoxPolicy {
    static constexpr int S = 1;
    const GemvJob &j;
    const GemvParams &p;
    DynPos dpos;
    const float2 *rope_cs;
    uint32_t head_size;
    float rope_base;
    NeoxPairs pairs;  // zeros: the pairs are neighbours (a job in PLAIN mode)
    __device__ uint32_t row_of(uint32_t g) const {
        return pairs.magic ? g + __umulhi(g, pairs.magic) * pairs.half : 2 * g;
    }
    __device__ uint32_t step() const { return pairs.magic ? pairs.half : 1u; }
    template <class WF, int R>
    __device__ void load(typename WF::Row (&w)[R], uint32_t g, uint32_t, uint32_t tile, bool ok) const {
        static_assert(R == 2, "fused launches work on row pairs");
        const uint32_t r0 = row_of(ok ? g : 0u);
        WF::load(w[0], WF::row_base(p, r0), tile);
        WF::load(w[1], WF::row_base(p, min(r0 + step(), j.nrows - 1)), tile);
    }
    float pre_bias, pre_out;
    float2 pre_cs;
    uint32_t pos;
    __device__ const uint32_t *pos_ptr() const { return dpos.ptr; }
    __device__ void set_pos(uint32_t fetched) { pos = dpos.ptr ? fetched : dpos.val; }
    __device__ float2 entry(uint32_t g) const {
        const uint32_t k = g % (head_size / 2);
        if (rope_cs) return rope_cs[k];
        const float theta = powf(rope_base, -(float)(2 * k) / (float)head_size);
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
        const uint32_t g = g0 + (lane >> 1) * GW, row = row_of(g) + (lane & 1) * step();
        if (!(lane < 2 * my_groups && row < j.nrows)) return;
        const bool out_needs_pos = dpos.ptr && j.out_pos_stride;
        const bool cs_needs_pos = dpos.ptr && !rope_cs;
        if (!late && j.bias) pre_bias = j.bias[row];
        if (!late) pos = dpos.val;
        if (j.accumulate() && late == out_needs_pos) pre_out = (j.out + (size_t)pos * j.out_pos_stride)[row];
        if (j.mode() == JOB_ROPE && late == cs_needs_pos) pre_cs = entry(g);
    }
    template <int R>
    __device__ void finish(float mine, uint32_t n, uint32_t g0, uint32_t GW, uint32_t lane) {
        const uint32_t sub = lane & 1, row = row_of(g0 + (lane >> 1) * GW) + sub * step();
        float *out = j.out + (size_t)pos * j.out_pos_stride;
        float t = mine + pre_bias;
        if (j.mode() == JOB_ROPE) {
            const float other = dpp_f32<0xB1>(t);
            // (x, y) = (first row, second row):  x' = cs x - sn y,  y' = sn x + cs y
            t = sub ? pre_cs.y * other + pre_cs.x * t : pre_cs.x * t - pre_cs.y * other;
        }
        if (lane < n && row < j.nrows) out[row] = j.accumulate() ? pre_out + t : t;
    }
};

template <class F>
__device__ __forceinline__ void neox_job_body(const FusedParams &P, const GemvJob &j, NeoxPairs pairs) {
    GemvParams p{};
    p.x = P.x;
    p.ncols = P.ncols;
    p.norm_w = P.norm_w;
    p.norm_eps = P.norm_eps;
    p.nrows = j.nrows;
    p.p0 = j.a0;
    p.p1 = j.a1;
    p.p2 = j.a2;
    p.p3 = j.a3;
    if (j.mode() != JOB_ROPE) pairs = {};
    NeoxPolicy pol{j, p, P.pos, P.rope_cs, P.head_size, P.rope_base, pairs, 0.f, 0.f, make_float2(1.f, 0.f), 0};
    const uint32_t ngroups = (j.nrows + 1) / 2, wg = blockIdx.x - j.wg_begin;
    if (P.ncols <= 64 * F::TILE)
        gemv_i8_body<F, 2, 1, true>(p, pol, wg, j.wg_count, j.active_waves, ngroups);
    else
        gemv_i8_body<F, 2, 1, false>(p, pol, wg, j.wg_count, j.active_waves, ngroups);
}

template <int MAXT, int MINW, int FMT>
__global__ __launch_bounds__(MAXT, MINW) void gemv_fused_neox_kernel(const FusedParams P, const NeoxPairs pairs) {
    // the workgroup's job field by field, as in gemv_fused_kernel
    const bool is1 = P.njobs > 1 && blockIdx.x >= P.jobs[1].wg_begin;
    const bool is2 = P.njobs > 2 && blockIdx.x >= P.jobs[2].wg_begin;
    const GemvJob &j0 = P.jobs[0], &j1 = P.jobs[1], &j2 = P.jobs[2];
    const GemvJob j{WGML_PICK(a0), WGML_PICK(a1), WGML_PICK(a2), WGML_PICK(a3),
                    WGML_PICK(out), WGML_PICK(bias), WGML_PICK(nrows), WGML_PICK(kind),
                    WGML_PICK(out_pos_stride), WGML_PICK(wg_begin), WGML_PICK(wg_count),
                    WGML_PICK(active_waves)};
    if constexpr (FMT != 0) {
        neox_job_body<typename FusedFmt<FMT, false>::T>(P, j, pairs);
    } else {
        switch (j.type()) {
        case WGML_Q4_K: neox_job_body<IFmtQ4K>(P, j, pairs); break;
        case WGML_Q6_K: neox_job_body<IFmtQ6K>(P, j, pairs); break;
        default: neox_job_body<IFmtQ8_0>(P, j, pairs); break;
        }
    }
}

template <int MAXT>
void (*neox_kernel_of(int fmt))(const FusedParams, const NeoxPairs) {
    switch (fmt) {
    case WGML_Q4_K: return gemv_fused_neox_kernel<MAXT, 1, WGML_Q4_K>;
    case WGML_Q6_K: return gemv_fused_neox_kernel<MAXT, 1, WGML_Q6_K>;
    case WGML_Q8_0: return gemv_fused_neox_kernel<MAXT, 1, WGML_Q8_0>;
    case WGML_Q5_K: return gemv_fused_neox_kernel<MAXT, 1, WGML_Q5_K>;
    case WGML_Q8_K: return gemv_fused_neox_kernel<MAXT, 1, WGML_Q8_K>;
    case WGML_Q4_0: return gemv_fused_neox_kernel<MAXT, 1, WGML_Q4_0>;
    case WGML_Q4_1: return gemv_fused_neox_kernel<MAXT, 1, WGML_Q4_1>;
    case WGML_Q5_0: return gemv_fused_neox_kernel<MAXT, 1, WGML_Q5_0>;
    case WGML_Q5_1: return gemv_fused_neox_kernel<MAXT, 1, WGML_Q5_1>;
    case kLegacyWide + WGML_Q4_0: return gemv_fused_neox_kernel<MAXT, 1, kLegacyWide + WGML_Q4_0>;
    case kLegacyWide + WGML_Q4_1: return gemv_fused_neox_kernel<MAXT, 1, kLegacyWide + WGML_Q4_1>;
    case kLegacyWide + WGML_Q5_0: return gemv_fused_neox_kernel<MAXT, 1, kLegacyWide + WGML_Q5_0>;
    case kLegacyWide + WGML_Q5_1: return gemv_fused_neox_kernel<MAXT, 1, kLegacyWide + WGML_Q5_1>;
    default: return gemv_fused_neox_kernel<MAXT, (MAXT == 1024 ? 5 : 1), 0>;
    }
}

}  // namespace

const void *wgml::gemv_neox_kernel(int fmt, int threads) {
    return (const void *)(threads == 768 ? neox_kernel_of<768>(fmt) : neox_kernel_of<1024>(fmt));
}
