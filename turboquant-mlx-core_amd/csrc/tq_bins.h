// Bin of a value among sorted boundaries, for the codebook fit.
//
// std::lower_bound over the boundaries (reference src/codebook.cpp:295-297) is the number of boundaries strictly below
// the value.  Comparing with each of them is two vector instructions per boundary and value (30 for 4 bits; the
// quantizer bisects a tree of them, 12 and two LDS reads); here 256 equally wide cells over the boundaries' range say how many boundaries lie
// in the cells below, and only the boundaries of the value's own cell (one at most for any codebook whose
// boundaries are 1/253 of the range apart) are compared.  The cell is a monotone function of the value, rounding included,
// and the boundaries' own cells come from the same function, so the result is the exact count.
#pragma once

#include "tq_device.h"

namespace tq {

struct BinTable {                    // in LDS
    float bound[32];                 // the boundaries, then +inf
    float scale, bias;
    int steps;                       // boundaries in the fullest cell; -1: not sorted, compare with all of them
    uint8_t below[256];              // boundaries in the cells below
};

__device__ __forceinline__ int bin_cell(float v, float scale, float bias) {
    const float c = __builtin_fminf(__builtin_fmaxf(__builtin_fmaf(v, scale, bias), 0.0f), 255.0f);
    return (int)c;                   // (NaN: the maximum gives 0)
}

// All threads of a workgroup of at least 256 threads; two barriers inside, the table is complete after them.
__device__ __forceinline__ void bin_table_build(BinTable& t, const float* bounds, int nb, int tid) {
    if (tid < 32) t.bound[tid] = tid < nb ? bounds[tid] : __builtin_inff();
    __syncthreads();
    const float lo = t.bound[0], hi = t.bound[nb - 1];
    const float scale = hi > lo ? 253.0f / (hi - lo) : 0.0f;
    const float bias = hi > lo ? __builtin_fmaf(-lo, scale, 1.0f) : 1.0f;
    if (tid < 256) {
        int n = 0;
        for (int k = 0; k < nb; ++k) n += bin_cell(t.bound[k], scale, bias) < tid ? 1 : 0;
        t.below[tid] = (uint8_t)n;
    }
    if (tid == 0) {
        int most = 0, run = 0, last = -1;
        bool sorted = true;
        for (int k = 0; k < nb; ++k) {
            const int c = bin_cell(t.bound[k], scale, bias);
            run = c == last ? run + 1 : 1;
            last = c;
            most = most > run ? most : run;
            if (k > 0 && !(t.bound[k - 1] <= t.bound[k])) sorted = false;
        }
        t.scale = scale; t.bias = bias;
        t.steps = sorted && scale > 0.0f && scale < 1e30f ? most : -1;
    }
    __syncthreads();
}

// Number of boundaries strictly below v.  `steps` / `scale` / `bias`: the table's, read once by the caller.
__device__ __forceinline__ uint32_t bin_find(const BinTable& t, float scale, float bias, int steps, int nb, float v) {
    if (steps < 0) {
        uint32_t n = 0;
        for (int k = 0; k < nb; ++k) n += (t.bound[k] < v) ? 1u : 0u;
        return n;
    }
    uint32_t g = t.below[bin_cell(v, scale, bias)];
    g += (t.bound[g] < v) ? 1u : 0u;
    for (int s = 1; s < steps; ++s) g += (t.bound[g] < v) ? 1u : 0u;       // (an inf ends it: nothing is above)
    return g;
}

}  // namespace tq
