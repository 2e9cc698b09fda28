// Matrix-vector kernels of the 32-element formats Q4_0, Q4_1, Q5_0 and Q5_1, in a code object of their own (behind the
// other kernels they would move those apart, see gemv_neox.hip).
#include "gemv_kernels.h"

GemvKernels wgml::gemv_legacy_kernels(int fmt) {
    switch (fmt) {
    case WGML_Q4_0: return gemv_kernels_of<WGML_Q4_0, false, false>();
    case WGML_Q4_1: return gemv_kernels_of<WGML_Q4_1, false, false>();
    case WGML_Q5_0: return gemv_kernels_of<WGML_Q5_0, false, false>();
    case WGML_Q5_1: return gemv_kernels_of<WGML_Q5_1, false, false>();
    case kLegacyWide + WGML_Q4_0: return gemv_kernels_of<kLegacyWide + WGML_Q4_0, false, false>();
    case kLegacyWide + WGML_Q4_1: return gemv_kernels_of<kLegacyWide + WGML_Q4_1, false, false>();
    case kLegacyWide + WGML_Q5_0: return gemv_kernels_of<kLegacyWide + WGML_Q5_0, false, false>();
    default: return gemv_kernels_of<kLegacyWide + WGML_Q5_1, false, false>();
    }
}
