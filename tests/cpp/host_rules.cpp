// Dispatch rules and workspace sizes: host code of the library, run without a GPU.  One check per argument
// (tests/test_host_rules.py); a check that fails prints what it found and ends with status 1.
#include <cstdint>
#include <cstdio>
#include <cstring>

#include "tq_device.h"
#include "tq_prefill_common.h"

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
    v.compose_ok = 1;
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

}  // namespace

int main(int argc, char** argv) {
    const struct { const char* name; void (*run)(); } checks[] = {{"fit_limit", fit_limit}, {"compose_modes", compose_modes}};
    for (const auto& c : checks)
        if (argc == 2 && std::strcmp(argv[1], c.name) == 0) {
            c.run();
            if (!failures) std::printf("ok\n");
            return failures ? 1 : 0;
        }
    std::fprintf(stderr, "usage: host_rules <check>\n");
    return 2;
}
