// Matrix-vector kernels of the 32-element formats Q4_0, Q4_1, Q5_0 and Q5_1, in a code object of their own (behind the
// other kernels they would move those apart, see gemv_neox.hip).
#include "gemv_kernels.h"

namespace {

template <int TYPE>
GemvKernels kernels_of() {
    using F = typename FusedFmt<TYPE, false>::T;
    return {(const void *)gemv_quant_i8_kernel<F, 1, 1, 1024>, (const void *)gemv_fused_kernel<1, 1024, 1, TYPE>,
            (const void *)gemv_fused_kernel<1, 768, 1, TYPE>};
}

}  // namespace

GemvKernels wgml::gemv_legacy_kernels(int fmt) {
    switch (fmt) {
    case WGML_Q4_0: return kernels_of<WGML_Q4_0>();
    case WGML_Q4_1: return kernels_of<WGML_Q4_1>();
    case WGML_Q5_0: return kernels_of<WGML_Q5_0>();
    case WGML_Q5_1: return kernels_of<WGML_Q5_1>();
    case kLegacyWide + WGML_Q4_0: return kernels_of<kLegacyWide + WGML_Q4_0>();
    case kLegacyWide + WGML_Q4_1: return kernels_of<kLegacyWide + WGML_Q4_1>();
    case kLegacyWide + WGML_Q5_0: return kernels_of<kLegacyWide + WGML_Q5_0>();
    default: return kernels_of<kLegacyWide + WGML_Q5_1>();
    }
}
