// CPU-side sampler of the reference (models/sampler.rs:14-130): greedy for
// temperature 0, else temperature scaling, softmax, and multinomial or top-p
// (nucleus) sampling.  The random number is an argument (`coin` in [0, 1)), so a
// caller with a seeded generator gets reproducible text.  Host only.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <numeric>
#include <vector>

#include "common.h"

using namespace wgml;

namespace {

// Sampler::sample_mult (models/sampler.rs:58-76)
uint32_t sample_mult(const float *p, uint32_t n, float coin) {
    float cdf = 0.0f;
    for (uint32_t i = 0; i < n; ++i) {
        cdf += p[i];
        if (coin < cdf) return i;
    }
    return n - 1;
}

// Sampler::sample_topp (models/sampler.rs:78-130)
uint32_t sample_topp(const float *p, uint32_t n, float topp, float coin) {
    // values below (1 - topp) / (n - 1) cannot be part of the nucleus
    const float cutoff = (1.0f - topp) / ((float)n - 1.0f);
    std::vector<uint32_t> idx;
    idx.reserve(256);
    for (uint32_t i0 = 0; i0 < n; i0 += 64) {  // few are: blocks without one are passed over
        const uint32_t i1 = std::min(n, i0 + 64);
        int any = 0;
        for (uint32_t i = i0; i < i1; ++i) any |= p[i] >= cutoff;
        if (!any) continue;
        for (uint32_t i = i0; i < i1; ++i)
            if (p[i] >= cutoff) idx.push_back(i);
    }
    if (idx.empty()) return n - 1;
    // decreasing probability; ties keep their index order (the reference's sort is stable)
    std::stable_sort(idx.begin(), idx.end(), [p](uint32_t a, uint32_t b) { return p[a] > p[b]; });
    float cumulative = 0.0f;
    size_t last = idx.size() - 1;  // in case of rounding errors consider all elements
    for (size_t i = 0; i < idx.size(); ++i) {
        cumulative += p[idx[i]];
        if (cumulative > topp) {
            last = i;
            break;
        }
    }
    const float r = coin * cumulative;
    float cdf = 0.0f;
    for (size_t i = 0; i <= last; ++i) {
        cdf += p[idx[i]];
        if (r < cdf) return idx[i];
    }
    return idx[last];
}

// exp(x) for a block of x = logits - maximum, the same floats as std::exp.  y is e^x in double to
// about 1e-11 (x = k ln 2 + r with |r| <= ln 2 / 2, the Taylor polynomial of degree 9 in r, times
// 2^k): far closer than float, so rounding it gives the correctly rounded result, which is also
// what std::exp returns unless e^x lies almost half way between two floats.  `ask` marks those (4 %
// of all, within 0.02 of the last place of a half way point) and what is outside the range of
// normal results; the caller takes std::exp there.  32000 logits took 306 us with a call for each,
// most of a small model's step; the loop below is vectorised.
constexpr uint32_t kExpBlock = 256;
inline __attribute__((always_inline)) void exp_block_body(const float *logits, float max_val, uint32_t n,
                                                          float *out, uint32_t *ask) {
    constexpr double kLog2E = 1.4426950408889634, kLn2 = 0.6931471805599453, kRound = 6755399441055744.0;
    for (uint32_t i = 0; i < n; ++i) {
        const float xf = logits[i] - max_val;
        const double x = (double)xf, kr = x * kLog2E + kRound, k = kr - kRound, r = x - k * kLn2;
        double p = 1.0 / 362880;
        p = p * r + 1.0 / 40320;
        p = p * r + 1.0 / 5040;
        p = p * r + 1.0 / 720;
        p = p * r + 1.0 / 120;
        p = p * r + 1.0 / 24;
        p = p * r + 1.0 / 6;
        p = p * r + 0.5;
        p = p * r + 1.0;
        p = p * r + 1.0;
        uint64_t kb, yb;
        std::memcpy(&kb, &kr, 8);  // the low bits of kr hold k
        kb = (kb + 1023) << 52;
        double scale;
        std::memcpy(&scale, &kb, 8);
        const double y = p * scale;
        out[i] = (float)y;
        std::memcpy(&yb, &y, 8);
        // a float keeps the upper 23 of y's 52 fraction bits: 2^28 in the others is half way
        constexpr uint32_t kNear = 10737418;  // 0.02 * 2^29
        const uint32_t low = (uint32_t)yb & 0x1fffffffu;
        ask[i] = (uint32_t)(low - (0x10000000u - kNear) < 2 * kNear) | (uint32_t)!(xf >= -87.0f);
    }
}
void exp_block(const float *logits, float max_val, uint32_t n, float *out, uint32_t *ask) {
    exp_block_body(logits, max_val, n, out, ask);
}
#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
__attribute__((target("avx2"))) void exp_block_avx2(const float *logits, float max_val, uint32_t n, float *out,
                                                    uint32_t *ask) {
    exp_block_body(logits, max_val, n, out, ask);
}
bool have_avx2() { return __builtin_cpu_supports("avx2"); }
#else
void exp_block_avx2(const float *logits, float max_val, uint32_t n, float *out, uint32_t *ask) {
    exp_block_body(logits, max_val, n, out, ask);
}
bool have_avx2() { return false; }
#endif

}  // namespace

extern "C" {

int wgml_sample(float *logits, uint32_t n, float temperature, float topp, float coin,
                uint32_t *out_token) {
    WGML_REQUIRE(logits && out_token && n > 0, "wgml_sample: bad argument");
    WGML_REQUIRE(temperature >= 0.0f, "wgml_sample: negative temperature %g", (double)temperature);
    WGML_REQUIRE(coin >= 0.0f && coin < 1.0f, "wgml_sample: coin %g outside [0, 1)", (double)coin);
    if (temperature == 0.0f) {  // Sampler::sample_argmax: first index of the maximum
        uint32_t best = 0;
        for (uint32_t i = 1; i < n; ++i)
            if (logits[i] > logits[best]) best = i;
        *out_token = best;
        return WGML_OK;
    }
    for (uint32_t i = 0; i < n; ++i) logits[i] /= temperature;
    // SoftMax::run_cpu (ops/softmax.rs:36-49)
    float maxes[16];  // sixteen chains of comparisons instead of one
    for (float &v : maxes) v = logits[0];
    uint32_t j = 0;
    for (; j + 16 <= n; j += 16)
        for (uint32_t k = 0; k < 16; ++k) maxes[k] = std::max(maxes[k], logits[j + k]);
    for (; j < n; ++j) maxes[0] = std::max(maxes[0], logits[j]);
    float max_val = maxes[0];
    for (float v : maxes) max_val = std::max(max_val, v);
    float sum = 0.0f;
    const auto block = have_avx2() ? exp_block_avx2 : exp_block;
    for (uint32_t i0 = 0; i0 < n; i0 += kExpBlock) {
        float e[kExpBlock];
        uint32_t ask[kExpBlock];
        const uint32_t m = std::min(kExpBlock, n - i0);
        block(logits + i0, max_val, m, e, ask);
        for (uint32_t i = 0; i < m; ++i) {
            const float v = ask[i] ? std::exp(logits[i0 + i] - max_val) : e[i];
            logits[i0 + i] = v;
            sum += v;  // in index order, as the reference adds them
        }
    }
    for (uint32_t i = 0; i < n; ++i) logits[i] /= sum;
    *out_token = (topp <= 0.0f || topp >= 1.0f) ? sample_mult(logits, n, coin)
                                                : sample_topp(logits, n, topp, coin);
    return WGML_OK;
}

}  // extern "C"
