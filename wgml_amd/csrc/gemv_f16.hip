// Matrix-vector kernels of F16 tensors, in a code object of their own (see gemv_neox.hip).
#include "gemv_kernels.h"

GemvKernels wgml::gemv_f16_kernels() { return gemv_kernels_of<kFusedDenseF16, true, false>(); }
