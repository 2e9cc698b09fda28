#include "gemm_kernel.h"

int wgml::launch_gemm_q5_1(wgml_ctx *ctx, const GemmArgs &a, uint32_t tiles) { return launch_gemm_fmt<GemmQ5_1>(ctx, a, tiles); }
