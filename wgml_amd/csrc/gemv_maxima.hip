// Matrix-vector kernels whose waves leave the largest of their results, for the output matrix of a token loop, in a code
// object of their own (see gemv_neox.hip); those of Q4_K, Q6_K and Q8_0 stand beside the step's other kernels (gemv.hip: here
// the 7B step took 21.46 ms for 16 tokens, there 21.35).
#include "gemv_kernels.h"

namespace {
template <class F>
const void *kernel_of() {
    return (const void *)gemv_quant_i8_kernel<F, 1, 1, 1024, 4, false, EXTRA_MAXIMA>;
}
template <int FMT>
const void *kernel_of_format() {
    return kernel_of<typename FusedFmt<FMT, false>::T>();
}
}  // namespace

const void *wgml::gemv_maxima_kernel(int fmt, bool f32) {
    if (f32) {
        switch (fmt) {
        case WGML_Q4_K: return kernel_of<FFmt<FmtQ4K>>();
        case WGML_Q6_K: return kernel_of<FFmt<FmtQ6K>>();
        case WGML_Q8_0: return kernel_of<FFmt<FmtQ8_0>>();
        case kFusedDenseF16: return kernel_of<FFmt<FmtF16>>();
        default: return kernel_of<FFmt<FmtF32>>();
        }
    }
    switch (fmt) {
    case WGML_Q5_K: return kernel_of_format<WGML_Q5_K>();
    case WGML_Q8_K: return kernel_of_format<WGML_Q8_K>();
    case WGML_Q4_0: return kernel_of_format<WGML_Q4_0>();
    case WGML_Q4_1: return kernel_of_format<WGML_Q4_1>();
    case WGML_Q5_0: return kernel_of_format<WGML_Q5_0>();
    case WGML_Q5_1: return kernel_of_format<WGML_Q5_1>();
    case kLegacyWide + WGML_Q4_0: return kernel_of_format<kLegacyWide + WGML_Q4_0>();
    case kLegacyWide + WGML_Q4_1: return kernel_of_format<kLegacyWide + WGML_Q4_1>();
    case kLegacyWide + WGML_Q5_0: return kernel_of_format<kLegacyWide + WGML_Q5_0>();
    default: return kernel_of_format<kLegacyWide + WGML_Q5_1>();
    }
}
