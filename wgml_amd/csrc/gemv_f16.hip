// Matrix-vector kernels of F16 tensors, alone and beside F32 ones, in a code object of their own (see gemv_neox.hip).
#include "gemv_kernels.h"

GemvKernels wgml::gemv_f16_kernels() { return gemv_kernels_of<kFusedDenseF16, true, false>(); }

GemvKernels wgml::gemv_dense_mix_kernels() {
    return {nullptr, (const void *)gemv_fused_kernel<1, 1024, 1, kFusedDenseMix, true>,
            (const void *)gemv_fused_kernel<1, 768, 1, kFusedDenseMix, true>,
            (const void *)gemv_gated_kernel<1024, kFusedDenseMix, true>, (const void *)gemv_gated_kernel<768, kFusedDenseMix, true>};
}
