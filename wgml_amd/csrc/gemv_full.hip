// Matrix-vector kernels with LayerNorm and activation (GPT-2's), in a code object of their own.
#include "gemv_kernels.h"

GemvKernels wgml::gemv_full_kernels(int fmt, bool f32, int rows) {
    if (f32) {
        switch (fmt) {
        case WGML_Q4_K: return gemv_kernels_of<WGML_Q4_K, true, true>();
        case WGML_Q6_K: return gemv_kernels_of<WGML_Q6_K, true, true>();
        case WGML_Q8_0: return gemv_kernels_of<WGML_Q8_0, true, true>();
        case kFusedDenseF16: return gemv_kernels_of<kFusedDenseF16, true, true>();
        default: return gemv_kernels_of<kFusedDenseF32, true, true>();
        }
    }
    switch (fmt) {
    case WGML_Q8_0: {
        GemvKernels k = gemv_kernels_of<WGML_Q8_0, false, true>();
        if (rows == 2) k.plain = (const void *)gemv_quant_i8_kernel<IFmtQ8_0, 2, 1, 1024, 4, false, EXTRA_FULL | EXTRA_MAXIMA>;
        return k;
    }
    case WGML_Q4_K: return gemv_kernels_of<WGML_Q4_K, false, true>();
    case WGML_Q6_K: return gemv_kernels_of<WGML_Q6_K, false, true>();
    case WGML_Q5_K: return gemv_kernels_of<WGML_Q5_K, false, true>();
    case WGML_Q8_K: return gemv_kernels_of<WGML_Q8_K, false, true>();
    case WGML_Q4_0: return gemv_kernels_of<WGML_Q4_0, false, true>();
    case WGML_Q4_1: return gemv_kernels_of<WGML_Q4_1, false, true>();
    case WGML_Q5_0: return gemv_kernels_of<WGML_Q5_0, false, true>();
    case WGML_Q5_1: return gemv_kernels_of<WGML_Q5_1, false, true>();
    case kLegacyWide + WGML_Q4_0: return gemv_kernels_of<kLegacyWide + WGML_Q4_0, false, true>();
    case kLegacyWide + WGML_Q4_1: return gemv_kernels_of<kLegacyWide + WGML_Q4_1, false, true>();
    case kLegacyWide + WGML_Q5_0: return gemv_kernels_of<kLegacyWide + WGML_Q5_0, false, true>();
    default: return gemv_kernels_of<kLegacyWide + WGML_Q5_1, false, true>();
    }
}
