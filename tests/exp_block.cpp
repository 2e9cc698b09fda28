// The sampler's blocks of exp, both bodies, for test_sampler.py.
#include "../wgml_amd/csrc/sampler.cpp"

namespace wgml {
int set_error(int code, const char *, ...) { return code; }
}  // namespace wgml

extern "C" {
// what the sampler takes for exp(x[i] - 0): the block's value, or std::exp where that is marked
void take_exp(const float *x, uint32_t n, int avx2, float *out, uint32_t *asked) {
    *asked = 0;
    for (uint32_t i0 = 0; i0 < n; i0 += kExpBlock) {
        uint32_t ask[kExpBlock];
        const uint32_t m = std::min(kExpBlock, n - i0);
        (avx2 ? exp_block_avx2 : exp_block)(x + i0, 0.0f, m, out + i0, ask);
        for (uint32_t i = 0; i < m; ++i)
            if (ask[i]) {
                out[i0 + i] = std::exp(x[i0 + i]);
                ++*asked;
            }
    }
}
void std_exp(const float *x, uint32_t n, float *out) {
    for (uint32_t i = 0; i < n; ++i) out[i] = std::exp(x[i]);
}
int cpu_has_avx2(void) { return have_avx2(); }
}
