// One row of 5-bit layers that keep two planes (own residual rotation, or a 4-bit residual), for gfx950: metal/turboquant_dequant_mm.metal:240-248, 277-292; src/dequantizer.cpp:625-626, 657.
//
//   y[r] = norm[r] / sqrt(in * bs) * ( sum_i cP[p(r,i)] x~p[i]  +  sum_i cR[q(r,i)] x~r[i] )
//
// A workgroup holds the whole activation row: each wave takes a segment of 512 columns, eight columns per lane, rotates it
// (blocks of at most 512 columns lie inside a segment) and keeps the rotated fp32 values in registers while rows go by,
// four at a time and the next four on their way.  A row's sums meet in LDS.  fp32 throughout.
//
// The generic kernel (tq_generic.hip) read both rotated rows again for every weight row, 8 bytes of them per weight from
// the L1 against 1.5 of indices, and needed a launch for the rotation.  us per call, dual rotation, bf16, before -> now, in x
// out: 5120 x 13824 44.4 -> 29.2 (3.6 TB/s), 5120 x 27648 78.9 -> 52.3 (4.1 TB/s), 3584 x 18944 41.3 -> 29.9, 8192 x 8192 41.8
// -> 29.3, 2048 x 2048 9.8 -> 7.2.  What bounds it: ten vector instructions per weight with both planes (the vector
// units are busy 82 % of the time) and two table reads, and the rotation every workgroup repeats (a few us, hence few
// workgroups: 20 waves per CU; 28 measured the same).  Two rows
// at a time took 38.0 us for 5120 x 13824.  Rows beyond 8192 columns would give a wave two segments and twice the rotation:
// 13824 x 5120 45.4 -> 37.2, but 9728 x 3584 26.3 -> 30.6, so they stay with the generic kernel.
#include "tq_device.h"

namespace tq {

namespace {

constexpr int kFiveMaxWaves = 16;
constexpr int kFiveMaxCols = kFiveMaxWaves * 512;
constexpr int kFiveRows = 4;                               // rows that go by at a time
constexpr int kFiveWavesPerCu = 20;

struct FiveArgs {
    const uint8_t* primary;    // [out, in] bytes
    const uint8_t* residual;   // [out, in / 2] nibbles
    const float* tables;       // [0..31] primary centroids, [32..47] residual centroids (build_tables)
    const float* norms;
    const void* x;
    void* y;
    const float* gate;         // optional fp32 [out]
    int x_dtype, y_dtype;
    int in, out, groups;       // groups of kFiveRows rows
    uint32_t seed0, seed1, bs;
    float out_scale;
};

// Eight consecutive activations in fp32.
__device__ __forceinline__ void load_eight(const void* x, int dtype, int col, float (&v)[8]) {
    if (dtype == kF32) {
        const float4* p = reinterpret_cast<const float4*>(static_cast<const float*>(x) + col);
        const float4 a = p[0], b = p[1];
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
        return;
    }
    const uint4 t = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(x) + col);
    const uint32_t w[4] = {t.x, t.y, t.z, t.w};
    if (dtype == kBF16) {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = bf16_bits_to_float((w[j >> 1] >> (16 * (j & 1))) & 0xffffu);
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = (float)__builtin_bit_cast(_Float16, (uint16_t)(w[j >> 1] >> (16 * (j & 1))));
    }
}

// Sums over the 64 lanes of four values at once: lane l ends with the sum of value row_of_lane(l).
__device__ __forceinline__ float reduce_rows(float (&v)[kFiveRows], int lane) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const float keep = (lane & 1) ? v[j + 2] : v[j], send = (lane & 1) ? v[j] : v[j + 2];
        v[j] = keep + lane_xor<1>(send);
    }
    const float keep = (lane & 2) ? v[1] : v[0], send = (lane & 2) ? v[0] : v[1];
    float t = keep + lane_xor<2>(send);
    t += lane_xor<4>(t); t += lane_xor<8>(t); t += lane_xor<16>(t); t += lane_xor<32>(t);
    return t;
}
__device__ __forceinline__ int row_of_lane(int lane) { return (lane & 1) * 2 + ((lane >> 1) & 1); }

}  // namespace

template <int MODE>
__global__ __launch_bounds__(64 * kFiveMaxWaves) void tq_gemv_five_kernel(FiveArgs a) {
    constexpr bool dual = (MODE == kDual5);
    constexpr int R = kFiveRows;
    __shared__ float tabp[256];                              // (a byte plane may hold more than 31: src/dequantizer.cpp:94)
    __shared__ float tabr[16];
    __shared__ float part[2][kFiveMaxWaves][R];
    const int lane = threadIdx.x & 63, waves = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool active = (wave * 64 + lane) * 8 < a.in;
    const int col = active ? (wave * 64 + lane) * 8 : 0;     // (beyond the row: column 0 loaded again and not used)

    uint2 p[R], pn[R];
    uint32_t q[R], qn[R];
    auto load = [&](int group, uint2 (&pp)[R], uint32_t (&qq)[R]) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int row = group * R + r < a.out ? group * R + r : a.out - 1;
            pp[r] = *reinterpret_cast<const uint2*>(a.primary + (size_t)row * a.in + col);
            qq[r] = *reinterpret_cast<const uint32_t*>(a.residual + (size_t)row * (a.in >> 1) + (col >> 1));
        }
    };
    load((int)blockIdx.x, p, q);

    for (int i = threadIdx.x; i < 256; i += blockDim.x) tabp[i] = a.tables[i < 31 ? i : 31];
    if (threadIdx.x < 16) tabr[threadIdx.x] = a.tables[32 + threadIdx.x];
    float x0[8], x1[8];
    load_eight(a.x, a.x_dtype, col, x0);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const uint32_t c = (uint32_t)(col + j) & (a.bs - 1);
        if constexpr (dual) x1[j] = x0[j] * sign_of(a.seed1, c);
        x0[j] *= sign_of(a.seed0, c);
    }
    // (the width is a multiple of 32 and of the block: no block has both active lanes and others)
    fwht_lanes<8>(x0, a.bs, lane);
    if constexpr (dual) fwht_lanes<8>(x1, a.bs, lane);
    __syncthreads();

    int turn = 0, buf = 0;
    for (int group = (int)blockIdx.x; group < a.groups; group += (int)gridDim.x) {      // the same for all waves
        const bool more = group + (int)gridDim.x < a.groups;
        if (more) load(group + (int)gridDim.x, pn, qn);
        float acc[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            float t = 0.0f, u = 0.0f;
            const uint32_t lo = q[r] & 0x0f0f0f0fu, hi = (q[r] >> 4) & 0x0f0f0f0fu;     // even, odd columns
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float cp = tabp[((j < 4 ? p[r].x : p[r].y) >> (8 * (j & 3))) & 255u];
                const float cr = tabr[((j & 1 ? hi : lo) >> (8 * (j >> 1))) & 15u];
                if constexpr (dual) {
                    t = __builtin_fmaf(cp, x0[j], t);
                    u = __builtin_fmaf(cr, x1[j], u);
                } else {
                    t = __builtin_fmaf(cp + cr, x0[j], t);                      // (src/dequantizer.cpp:186-212)
                }
            }
            if constexpr (dual) t += u;
            acc[r] = active ? t : 0.0f;
        }
        const float sum = reduce_rows(acc, lane);
        if (lane < R) part[buf][wave][row_of_lane(lane)] = sum;
        __syncthreads();
        // One wave in turn adds the waves' sums; the buffer is written again after the next barrier but one.
        const int row = group * R + lane;
        if (wave == turn && lane < R && row < a.out) {
            float t = 0.0f;
            for (int w = 0; w < waves; ++w) t += part[buf][w][lane];
            t *= a.out_scale * a.norms[row];
            if (a.gate) { const float g = a.gate[row]; t = g / (1.0f + expf(-g)) * t; }
            store_scalar(a.y, a.y_dtype, (size_t)row, t);
        }
        buf ^= 1;
        if (++turn == waves) turn = 0;
        if (more) {
#pragma unroll
            for (int r = 0; r < R; ++r) { p[r] = pn[r]; q[r] = qn[r]; }
        }
    }
}

bool gemv_five_supported(const LayerView& L) {
    if (L.mode != kShared5 && L.mode != kDual5) return false;          // (byte primaries alone run as a one-byte-per-weight layer)
    return L.block_size >= 2 && L.block_size <= 512 && L.in_features % 32 == 0 && L.in_features % (int)L.block_size == 0 &&
           L.in_features <= kFiveMaxCols;
}

hipError_t launch_gemv_five(const LayerView& L, const void* x, int x_dtype, void* y, int y_dtype, int num_cus,
                            hipStream_t stream, const float* gate) {
    const int waves = (L.in_features + 511) / 512;
    FiveArgs a{};
    a.primary = L.packed_primary;
    a.residual = L.packed_residual;
    a.tables = L.tables;
    a.norms = L.norms;
    a.x = x; a.x_dtype = x_dtype;
    a.y = y; a.y_dtype = y_dtype;
    a.gate = gate;
    a.in = L.in_features; a.out = L.out_features;
    a.seed0 = L.seed_primary; a.seed1 = L.seed_residual; a.bs = L.block_size;
    a.out_scale = L.inv_scale * L.inv_sqrt_bs;
    a.groups = (a.out + kFiveRows - 1) / kFiveRows;
    int grid = num_cus * (kFiveWavesPerCu / waves > 1 ? kFiveWavesPerCu / waves : 1);
    if (grid > a.groups) grid = a.groups;
    const dim3 g((unsigned)grid), t((unsigned)(64 * waves));
    switch (L.mode) {
        case kShared5: hipLaunchKernelGGL(tq_gemv_five_kernel<kShared5>, g, t, 0, stream, a); break;
        default: hipLaunchKernelGGL(tq_gemv_five_kernel<kDual5>, g, t, 0, stream, a); break;
    }
    return hipGetLastError();
}

}  // namespace tq
