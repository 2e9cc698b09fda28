#include "gemm_kernel.h"

int wgml::launch_gemm_q4_k(wgml_ctx *ctx, const GemmArgs &a, uint32_t tiles) { return launch_gemm_fmt<GemmQ4K>(ctx, a, tiles); }
