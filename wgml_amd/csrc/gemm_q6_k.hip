#include "gemm_kernel.h"

int wgml::launch_gemm_q6_k(wgml_ctx *ctx, const GemmArgs &a, uint32_t tiles) { return launch_gemm_fmt<GemmQ6K>(ctx, a, tiles); }
