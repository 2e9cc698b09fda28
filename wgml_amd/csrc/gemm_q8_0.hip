#include "gemm_kernel.h"

int wgml::launch_gemm_q8_0(wgml_ctx *ctx, const GemmArgs &a, uint32_t tiles) { return launch_gemm_fmt<GemmQ8_0>(ctx, a, tiles); }
