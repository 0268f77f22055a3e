// Which kernels the forward calls launch and what they do where memory is short: all of the library's host code on a
// faked runtime (fake_hip.h), without a GPU.  One check per argument (tests/test_host_rules.py).
#include "fake_hip.h"
#include "tq_device.h"
#include "turboquant_c/tq_linear.h"
#include "turboquant_c/tq_quantizer.h"

using fake::dev;
using fake::expect;

namespace {

struct Layer {
    int in, out;
    std::vector<unsigned char> x, y;
    tq_linear_t h = nullptr;
    explicit Layer(int in_, int out_, int rows) : in(in_), out(out_), x((size_t)rows * in_ * 4), y((size_t)rows * out_ * 4) {
        float cb[16];
        tq_generate_codebook(4, cb, nullptr);
        std::vector<uint8_t> p((size_t)out * in / 2, 0x5a), r(p.size(), 0xa5);
        std::vector<float> norms(out, 1.0f);
        const uint32_t seeds[3] = {99, 1234, 256};
        h = tq_linear_create(in, out, p.data(), in / 2, r.data(), in / 2, norms.data(), seeds, cb, 16, cb, 16, 256);
        expect(h != nullptr, tq_last_error());
    }
    ~Layer() { tq_linear_free(h); }
    int forward(int rows) {
        dev.launched.clear();
        return tq_linear_forward(h, x.data(), TQ_DTYPE_F32, rows, y.data(), TQ_DTYPE_F32, reinterpret_cast<void*>(&dev));
    }
    static bool ran(const char* kernel) {
        for (const std::string& k : dev.launched)
            if (k.find(kernel) != std::string::npos) return true;
        return false;
    }
};

constexpr int kIn = 1792, kOut = 8322, kRows = 600;        // composes where there is room: 34 MB
constexpr size_t kPlaneByPlane = (size_t)30 << 20;

// No room for the slab of composed weights: the call is done plane by plane, as it was before there were any.
void compose_without_memory() {
    Layer layer(kIn, kOut, kRows);
    expect(layer.forward(kRows) == 0 && Layer::ran("tq_compose_kernel"), "composed where there is room");
    Layer other(kIn, kOut, kRows);
    dev.size = dev.live + kPlaneByPlane;
    expect(other.forward(kRows) == 0, tq_last_error());
    expect(!dev.launched.empty() && !Layer::ran("tq_compose_kernel"), "plane by plane where there is none", dev.launched.size());
}

// The same for tq_linear_reserve, and captured calls afterwards.
void reserve_without_memory() {
    Layer layer(kIn, kOut, kRows);
    dev.size = dev.live + kPlaneByPlane;
    expect(tq_linear_reserve(layer.h, kRows) == 0, tq_last_error());
    dev.capturing = true;
    for (int rows : {40, 128, 257, 513, kRows}) expect(layer.forward(rows) == 0, tq_last_error(), rows);
    expect(!Layer::ran("tq_compose_kernel"), "plane by plane");
}

}  // namespace

int main(int argc, char** argv) {
    const fake::Check checks[] = {{"compose_without_memory", compose_without_memory},
                                  {"reserve_without_memory", reserve_without_memory}};
    return fake::run(checks, argc, argv);
}
