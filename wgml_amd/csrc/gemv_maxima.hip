// Matrix-vector kernels whose waves leave the largest of their results, for the output matrix of a token loop, in a code
// object of their own (see gemv_neox.hip).
#include "gemv_kernels.h"

namespace {
template <class F, int R, int MINW>
const void *kernel_of() {
    return (const void *)gemv_quant_i8_kernel<F, R, 1, 1024, MINW, false, EXTRA_MAXIMA>;
}
template <int FMT>
const void *kernel_of_format() {
    return kernel_of<typename FusedFmt<FMT, false>::T, 1, 4>();
}
}  // namespace

const void *wgml::gemv_maxima_kernel(int fmt, bool f32, int rows) {
    if (f32) {
        switch (fmt) {
        case WGML_Q4_K: return kernel_of<FFmt<FmtQ4K>, 1, 4>();
        case WGML_Q6_K: return kernel_of<FFmt<FmtQ6K>, 1, 4>();
        case WGML_Q8_0: return kernel_of<FFmt<FmtQ8_0>, 1, 4>();
        default: return kernel_of<FFmt<FmtF32>, 1, 4>();
        }
    }
    switch (fmt) {
    case WGML_Q8_0: return rows == 2 ? kernel_of<IFmtQ8_0, 2, 4>() : kernel_of<IFmtQ8_0, 1, 8>();
    case WGML_Q4_K: return kernel_of<IFmtQ4K, 1, 8>();
    case WGML_Q6_K: return kernel_of_format<WGML_Q6_K>();
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
