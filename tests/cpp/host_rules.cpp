// Dispatch rules and workspace sizes: host code of the library, run without a GPU.  One check per argument
// (tests/test_host_rules.py); a check that fails prints what it found and ends with status 1.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>

#include "tq_device.h"
#include "tq_prefill_common.h"
#include "turboquant_c/tq_quantizer.h"

namespace {

int failures = 0;
void expect(bool ok, const char* what, unsigned long long value) {
    if (!ok) { std::printf("failed: %s (%llu)\n", what, value); ++failures; }
}

// The codebook fit walks the samples of one value cell, all of them where every sample lies in it, with counters of 32
// bits and strides of up to 2^19: the largest number of samples it takes must leave them room.
void fit_limit() {
    unsigned long long lo = 1, hi = 1ull << 33;            // supported at lo, not at hi
    expect(tq::fit_supported(lo), "one sample is supported", lo);
    expect(!tq::fit_supported(hi), "2^33 samples are not", hi);
    while (hi - lo > 1) {
        const unsigned long long mid = lo + (hi - lo) / 2;
        (tq::fit_supported(mid) ? lo : hi) = mid;
    }
    const uint32_t n = (uint32_t)lo, stride = 1u << 19;
    uint32_t at = 0, rounds = 0;
    for (; (at == 0 || at < n) && rounds <= 8192; at += stride) ++rounds;
    expect(rounds <= 8192, "the walk over one cell ends at the largest number of samples", lo);
    expect(lo + stride < (1ull << 32), "a stride beyond the last sample is still a 32-bit number", lo);
}

tq::LayerView layer(int mode, int in, int out) {
    tq::LayerView v{};
    v.mode = mode;
    v.in_features = in; v.out_features = out;
    v.block_size = 512;
    v.fp16_centroids_ok = 1;
    v.compose_scale = 0.75f;
    return v;
}

// Planes are composed where there are two of them; the modes without are refused whatever the view's fields say.
void compose_modes() {
    for (int mode = tq::kPrimaryOnly; mode <= tq::kDual5; ++mode) {
        const bool two = mode == tq::kDual || mode == tq::kDual5 || mode == tq::kShared5;
        const bool got = tq::prefill_compose_supported(layer(mode, 5120, 27648), 2048, 256, ~(size_t)0);
        expect(got == two, "composed planes by mode", mode);
    }
}

// Planes are composed where the rounding of the sum to fp16 is no larger than that of the centroids: never where these are
// fp16 numbers already (and in range), and the scale is a plain factor.
void compose_precision() {
    float analytic[32], exact[32], wide[32];
    const int n = tq_generate_codebook(4, analytic, nullptr);
    for (int i = 0; i < n; ++i) {
        exact[i] = std::nearbyint(analytic[i] * 256.0f) / 256.0f;        // (fp16 holds them, and sums of two)
        wide[i] = analytic[i] * 20000.0f;
    }
    const float s = tq::compose_scale(tq::kDual, 512, analytic, n, analytic, n);
    expect(s > 0.5f && s <= 1.0f, "the analytic codebooks are composed", (unsigned long long)(s * 1000));
    expect(tq::compose_scale(tq::kDual, 512, exact, n, exact, n) == 0.0f, "exact centroids are not", 0);
    expect(tq::compose_scale(tq::kShared5, 512, exact, n, exact, n) > 0.0f, "but their sum in one rotation is as exact", 0);
    expect(tq::compose_scale(tq::kDual, 512, wide, n, wide, n) == 0.0f, "nor sums beyond the range of fp16", 0);
    expect(tq::compose_scale(tq::kDual, 1024, analytic, n, analytic, n) == 0.0f, "nor blocks of 1024", 0);
    wide[3] = NAN;
    expect(tq::compose_scale(tq::kDual, 512, wide, n, analytic, n) == 0.0f, "nor what is no number", 0);
}

}  // namespace

int main(int argc, char** argv) {
    const struct { const char* name; void (*run)(); } checks[] = {{"fit_limit", fit_limit}, {"compose_modes", compose_modes},
                                                                    {"compose_precision", compose_precision}};
    for (const auto& c : checks)
        if (argc == 2 && std::strcmp(argv[1], c.name) == 0) {
            c.run();
            if (!failures) std::printf("ok\n");
            return failures ? 1 : 0;
        }
    std::fprintf(stderr, "usage: host_rules <check>\n");
    return 2;
}
