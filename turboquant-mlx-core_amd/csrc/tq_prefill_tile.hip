// TQ8 prefill of calls with few output tiles (33 rows and more of small layers, ragged widths), for gfx950.
//
// Same contraction as tq_prefill.hip (Y = X~ L^T, fp16 operands of v_mfma_f32_32x32x16_f16, fp32 accumulation) on small
// output tiles: where 256 x 256 or 512 x 128 tiles leave most of the chip idle, 32 x 32 to 128 x 128 tiles fill it, and
// the length of a row is shared out among the waves of one workgroup instead of among workgroups.
//   * every wave decodes the weights of its own K range straight into the matrix operand (lane -> weight row; one dword
//     of a nibble plane, or two of the combined plane, is one operand): no weight tile in LDS and no barrier in the
//     loop.  A lane takes 32 SUB consecutive columns at a time, so that the two halves of a wave ask for whole cache
//     lines of 32 rows with neighbouring instructions where the width allows it;
//   * the activations are fragment images of 32 rows (tq_rotate_panel_kernel); the two halves of a wave
//     take different 16-column steps of the image so that the operand's columns are those of the weights' loads;
//   * the sums of the KS waves that share an output tile meet in LDS at the end: no partial products in memory and
//     no second kernel.
// A call is the rotation and this kernel.  The loop is a ring of D 64-column tiles of activations per wave (D = 4 for one
// row block of 32 rows, 2 for two and four) and of BR weight tiles; what bounds it is said at prefill_tile_shape.
#include "tq_prefill_common.h"

#include <type_traits>

namespace tq {

namespace {

struct TileArgs {
    const char* xt;            // fragment images [planes][row blocks of 32][K / 16][1 KB]
    const uint8_t* plane0;     // combined bytes [N, K] (shared rotation) or primary nibbles [N, K / 2]
    const uint8_t* plane1;     // residual nibbles [N, K / 2] (dual rotation) or NULL
    const float* tables;
    const float* norms;
    void* y;
    int y_dtype;
    int M, N, K;
    int m_tiles, n_tiles;
    float out_scale;
};

}  // namespace

// MB x NB blocks of 32 x 32 outputs per wave; KS waves share them along K, WN such groups stand side by side along N.
// SUB: 64-column tiles that a lane's weights are loaded for at once (a whole number of them in a row).
template <int MODE, int SUB, int MB, int NB, int KS, int WN>
__global__ __launch_bounds__(64 * KS * WN) void tq_prefill_tile_kernel(TileArgs a) {
    constexpr bool combined = (MODE == kSharedLut);
    constexpr int kPlanes = (MODE == kDual) ? 2 : 1;
    constexpr int kWaves = KS * WN;
    constexpr int kBlocks = MB * NB;
    constexpr int kLut = 256 * 256;                        // lane-private table, 256 entries x 64 lanes x 4 bytes
    constexpr int kExchange = kWaves * kBlocks * 4096;     // [wave][block][register][lane] floats, over the table
    constexpr int D = MB == 1 ? 4 : 2;
    constexpr int PV = combined ? 2 : 1;                   // 16-byte pieces of 32 columns
    constexpr int BV = SUB * PV;
    constexpr int BR = D / SUB > 2 ? D / SUB : 2;
    __shared__ __align__(16) char smem[kExchange > kLut ? kExchange : kLut];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wn = wave % WN, ks = wave / WN;
    const int l = lane & 31, g = lane >> 5;

    // Workgroup ids go round the XCDs (id % 8): the row tiles that share a tile of weights run on one XCD.
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const int n_tile = (slot / a.m_tiles) * 8 + xcd, m_tile = slot % a.m_tiles;
    if (n_tile >= a.n_tiles) return;                       // whole workgroup leaves together
    const int n0 = n_tile * (32 * NB * WN), m0 = m_tile * (32 * MB);

    // Weight tiles (64 SUB columns) of this wave, the second plane's after the first's.
    const int T = (a.K >> 6) / SUB, total = T * kPlanes;
    const int t_begin = total * ks / KS, t_end = total * (ks + 1) / KS;

    const size_t plane_stride = (size_t)((a.M + 31) >> 5) * (a.K >> 4) * 1024;
    // (uniform base addresses and 32-bit lane offsets throughout: with a 64-bit address per lane a third of the loop's
    // instructions computed addresses)
    const uint32_t aoff = (uint32_t)(g * (SUB * 2048) + l * 16);
    const char* ap[MB];
#pragma unroll
    for (int i = 0; i < MB; ++i) {
        int rb = m_tile * MB + i;                          // row block; past the call: the last one again, never stored
        if (rb * 32 >= a.M) rb = (a.M - 1) >> 5;
        ap[i] = a.xt + (size_t)rb * (a.K >> 4) * 1024;
    }
    uint32_t boff[NB];                                     // (prefill_supported: planes below 4 GB)
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        int n = n0 + (wn * NB + j) * 32 + l;
        if (n >= a.N) n = a.N - 1;
        boff[j] = combined ? (uint32_t)n * (uint32_t)a.K + g * (32 * SUB) : (uint32_t)n * (uint32_t)(a.K >> 1) + g * (16 * SUB);
    }

    f16x8 A[D][MB][4];
    u32x4v B[BR][NB][BV];
    auto request_b = [&](u32x4v (&bv)[NB][BV], int st) {
        if (st >= t_end) st = t_end - 1;                   // (past the range: the last tile again, not used)
        if (st < 0) st = 0;                                // (a wave without tiles)
        const int p = (kPlanes == 2 && st >= T) ? 1 : 0;
        const uint8_t* const w = (p ? a.plane1 : a.plane0) + (size_t)(st - p * T) * (combined ? 64 * SUB : 32 * SUB);
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int q = 0; q < BV; ++q) bv[j][q] = *reinterpret_cast<const u32x4v*>(w + q * 16 + boff[j]);
    };
    // Activations of piece q (32 columns of either half of the wave) of weight tile st.
    auto request_a = [&](f16x8 (&av)[MB][4], int st, int q) {
        if (st >= t_end) st = t_end - 1;
        if (st < 0) st = 0;
        const int p = (kPlanes == 2 && st >= T) ? 1 : 0;
        const size_t at = p * plane_stride + (size_t)(st - p * T) * (SUB * 4096) + q * 2048;
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int s = 0; s < 4; ++s)
                av[i][s] = *reinterpret_cast<const f16x8*>(ap[i] + at + ((s >> 1) * 1024 + (s & 1) * 512) + aoff);
    };
#pragma unroll
    for (int b = 0; b < BR; ++b) request_b(B[b], t_begin + b);
#pragma unroll
    for (int d = 0; d < D; ++d) request_a(A[d], t_begin + d / SUB, d % SUB);

    // The table, while those travel.  Shared rotation: fp16(lut[b]) in the upper half.  Nibble planes: the fp16 centroids
    // of both nibbles of byte b; with two planes lanes 0..31 of an entry hold the primary's and lanes 32..63 the
    // residual's, and lanes l and l + 32 read the same column (the LDS serves a wave's reads in two halves).
    {
        typedef const __attribute__((address_space(4))) float cfloat;
        cfloat* const src = (cfloat*)a.tables;
        uint32_t* const dst = reinterpret_cast<uint32_t*>(smem) + lane;
#pragma unroll 8
        for (int e = 0; e < 256 / kWaves; ++e) {
            const int entry = wave * (256 / kWaves) + e;
            uint32_t v;
            if constexpr (combined) {
                v = (uint32_t)float_to_f16_bits(src[entry]) << 16;
            } else {
                v = (uint32_t)float_to_f16_bits(src[entry & 15]) | ((uint32_t)float_to_f16_bits(src[entry >> 4]) << 16);
                if constexpr (kPlanes == 2) {
                    const uint32_t r = (uint32_t)float_to_f16_bits(src[16 + (entry & 15)]) |
                                       ((uint32_t)float_to_f16_bits(src[16 + (entry >> 4)]) << 16);
                    v = g ? r : v;
                }
            }
            dst[entry * 64] = v;
        }
    }
    __syncthreads();

    f32x16 acc[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    auto compute = [&](const f16x8 (&av)[MB][4], const u32x4v (&bv)[NB][BV], auto Qc, int st) {
        constexpr int q = decltype(Qc)::value;
        const uint32_t off = kPlanes == 2 ? (uint32_t)l * 4 + (st >= T ? 128u : 0u) : (uint32_t)lane * 4;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            f16x8 bf[NB];
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                u32x4v o;
                if constexpr (combined) {
                    const u32x4v& piece = bv[j][q * PV + (s >> 1)];
                    const uint32_t w0 = piece[(s & 1) * 2], w1 = piece[(s & 1) * 2 + 1];
                    uint32_t lv[8];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        lv[k] = *reinterpret_cast<const uint32_t*>(smem + gemm_entry_addr(w0, off, k));
                        lv[4 + k] = *reinterpret_cast<const uint32_t*>(smem + gemm_entry_addr(w1, off, k));
                    }
                    o.x = pack_half2(lv[0], lv[1]); o.y = pack_half2(lv[2], lv[3]);
                    o.z = pack_half2(lv[4], lv[5]); o.w = pack_half2(lv[6], lv[7]);
                } else {
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        o[k] = *reinterpret_cast<const uint32_t*>(smem + gemm_entry_addr(bv[j][q][s], off, k));
                }
                bf[j] = __builtin_bit_cast(f16x8, o);
            }
            // (weights as the first operand: a lane's 16 results are 4 x 4 consecutive output columns of one token)
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int j = 0; j < NB; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(bf[j], av[i][s], acc[i][j], 0, 0, 0);
        }
    };
    // Weight tile st + b with the activations that were requested D pieces ago; the slot of each piece is filled again.
    auto tile = [&](auto Bc, int st) {
        constexpr int b = decltype(Bc)::value;
        auto piece = [&](auto Qc) {
            constexpr int q = decltype(Qc)::value;
            if constexpr (q < SUB) {
                constexpr int at = b * SUB + q, next = at + D;
                compute(A[at % D], B[b], Qc, st + b);
                request_a(A[at % D], st + next / SUB, next % SUB);
                if constexpr (q == SUB - 1) request_b(B[b], st + BR + b);
                // (left alone the compiler gathers the requests of the whole iteration at its end)
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        piece(std::integral_constant<int, 0>{});
        piece(std::integral_constant<int, 1>{});
    };
    static_assert(SUB <= 2 && BR <= 4 && (BR * SUB) % D == 0, "ring positions repeat with the loop");
    int st = t_begin;
    for (; st + BR <= t_end; st += BR) {
        tile(std::integral_constant<int, 0>{}, st);
        tile(std::integral_constant<int, 1>{}, st);
        if constexpr (BR > 2) {
            tile(std::integral_constant<int, 2>{}, st);
            tile(std::integral_constant<int, 3>{}, st);
        }
    }
    if (st < t_end) tile(std::integral_constant<int, 0>{}, st);
    if constexpr (BR > 2) {
        if (st + 1 < t_end) tile(std::integral_constant<int, 1>{}, st);
        if (st + 2 < t_end) tile(std::integral_constant<int, 2>{}, st);
    }

    // Sum over the waves of a K group, in their order; * norm / sqrt(in); store.
    __syncthreads();                                       // the table has been read for the last time
    float* const ex = reinterpret_cast<float*>(smem);
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) ex[((wave * kBlocks + i * NB + j) * 16 + r) * 64 + lane] = acc[i][j][r];
    __syncthreads();
    const bool vec = (a.N & 3) == 0;
    for (int u = wave; u < WN * kBlocks * 4; u += kWaves) {
        const int q = u & 3, b = (u >> 2) % kBlocks, w = (u >> 2) / kBlocks;
        const int row = m0 + (b / NB) * 32 + l, col = n0 + (w * NB + b % NB) * 32 + 8 * q + 4 * g;
        float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < KS; ++k)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += ex[(((k * WN + w) * kBlocks + b) * 16 + 4 * q + e) * 64 + lane];
        if (row >= a.M) continue;
        const size_t at = (size_t)row * a.N + col;
        if (vec) {
            if (col >= a.N) continue;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] *= a.out_scale * a.norms[col + e];
            if (a.y_dtype == kF32) {
                const u32x4v o = {__builtin_bit_cast(uint32_t, v[0]), __builtin_bit_cast(uint32_t, v[1]),
                                  __builtin_bit_cast(uint32_t, v[2]), __builtin_bit_cast(uint32_t, v[3])};
                *reinterpret_cast<u32x4v*>(static_cast<float*>(a.y) + at) = o;
            } else {
                uint32_t h[4];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    h[e] = a.y_dtype == kBF16 ? (uint32_t)float_to_bf16_bits(v[e]) : (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v[e]);
                const u32x2v o = {h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
                *reinterpret_cast<u32x2v*>(static_cast<uint16_t*>(a.y) + at) = o;
            }
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (col + e < a.N) store_scalar(a.y, a.y_dtype, at + e, v[e] * (a.out_scale * a.norms[col + e]));
        }
    }
}

namespace {

struct TileShape { int mb, nb, ks, wn; };
constexpr TileShape kTileShapes[] = {{1, 1, 8, 1}, {1, 2, 8, 1}, {2, 2, 8, 1}, {4, 2, 2, 2}};

template <int MODE, int SUB>
void launch_shape(int shape, const TileArgs& a, dim3 grid, hipStream_t stream) {
    switch (shape) {
        case 0: hipLaunchKernelGGL((tq_prefill_tile_kernel<MODE, SUB, 1, 1, 8, 1>), grid, dim3(512), 0, stream, a); break;
        case 1: hipLaunchKernelGGL((tq_prefill_tile_kernel<MODE, SUB, 1, 2, 8, 1>), grid, dim3(512), 0, stream, a); break;
        case 2: hipLaunchKernelGGL((tq_prefill_tile_kernel<MODE, SUB, 2, 2, 8, 1>), grid, dim3(512), 0, stream, a); break;
        default: hipLaunchKernelGGL((tq_prefill_tile_kernel<MODE, SUB, 4, 2, 2, 2>), grid, dim3(256), 0, stream, a); break;
    }
}

}  // namespace

size_t prefill_tile_workspace_bytes(const LayerView& L, int batch) {
    const size_t planes = (L.mode == kDual) ? 2 : 1;
    return planes * (((size_t)batch + 31) / 32) * 32 * L.in_features * sizeof(uint16_t);
}

// The shape with the shortest estimate, in us without the rotation, fitted to seven layer shapes x five row counts
// (40 to 1024) per mode: rounds of workgroups on the CUs, each a fixed cost (table, first requests, sum over the waves,
// stores) and a cost per 64-column tile of the row, which is what a CU's loads deliver (20 to 36 bytes per clock; the
// matrix units are busy 6 to 12 % of the time with 32-row tiles, 19 % with 64 x 64, the vector units 16 to 33 %).  The 256 x 256 tiles of
// tq_prefill.hip: 0.8 us per 32-column step of a range, and the ranges' products written and read again.  Where
// 512 x 128 tiles fill the chip (prefill_panel_supported) they are faster throughout.
//   us per call before -> now, bf16:  dual rotation, in x out: 896 x 4864 at 77 rows 57.7 -> 17.9, at 512 rows 60.3 -> 36.2;
//   4864 x 896 at 77 rows 72.7 -> 25.3; 7680 x 565 at 160 rows 82.2 -> 37.2; 5120 x 5120 at 77 rows 68.2 -> 34.6, at 1024 rows
//   138.6 (not taken).  Shared rotation: 896 x 4864 at 77 rows 34.9 -> 13.5; 2048 x 2048 at 512 rows 43.2 -> 22.4.
int prefill_tile_shape(const LayerView& L, int batch, int num_cus) {
    if (!prefill_supported(L, kBF16, batch)) return -1;    // (up to 32 rows: what the small-batch kernels leave)
    if (prefill_panel_supported(L, batch, num_cus, ~(size_t)0)) return -1;
    static constexpr double kFirst[4] = {5.0, 5.0, 5.0, 12.0}, kMore[4] = {2.4, 6.5, 7.0, 16.0};
    static constexpr double kPerTile[3][4] = {{0.094, 0.125, 0.17, 0.45}, {0.107, 0.164, 0.24, 0.60}, {0.07, 0.12, 0.17, 0.45}};
    const double* const per_tile = kPerTile[L.mode == kDual ? 0 : (L.mode == kSharedLut ? 1 : 2)];
    const int planes = L.mode == kDual ? 2 : 1;
    const double tiles64 = (double)planes * (L.in_features / 64);
    const PrefillPlan p = prefill_plan(L, batch, num_cus, ~(size_t)0);
    const long long big = (long long)((batch + 255) / 256) * ((L.out_features + 255) / 256) * p.splits;
    double best = (double)((big + num_cus - 1) / num_cus) * 0.8 * planes * p.steps_per_split;
    if (p.splits > 1) best += 5.0 + (double)p.splits * batch * L.out_features * 8.0 / 5.0e6;
    best *= 0.95;
    int shape = -1;
    for (int s = 0; s < 4; ++s) {
        const TileShape t = kTileShapes[s];
        const long long wgs = (long long)((batch + 32 * t.mb - 1) / (32 * t.mb)) * ((L.out_features + 32 * t.nb * t.wn - 1) / (32 * t.nb * t.wn));
        const double rounds = (double)((wgs + num_cus - 1) / num_cus);
        const double cost = kFirst[s] + (rounds - 1.0) * kMore[s] + rounds * per_tile[s] * tiles64;
        if (cost < best) { best = cost; shape = s; }
    }
    return shape;
}

hipError_t launch_prefill_tile(const LayerView& L, int shape, const void* x, int x_dtype, int batch, void* y, int y_dtype,
                               void* workspace, hipStream_t stream) {
    hipError_t e = launch_rotate_tiles(L, x, x_dtype, batch, workspace, stream, kBlockImage);
    if (e != hipSuccess) return e;
    const TileShape t = kTileShapes[shape];
    TileArgs a{};
    a.xt = static_cast<const char*>(workspace);
    a.plane0 = (L.mode == kSharedLut) ? L.packed_combined : L.packed_primary;
    a.plane1 = L.packed_residual;
    a.tables = L.tables;
    a.norms = L.norms;
    a.y = y; a.y_dtype = y_dtype;
    a.M = batch; a.N = L.out_features; a.K = L.in_features;
    a.m_tiles = (batch + 32 * t.mb - 1) / (32 * t.mb);
    a.n_tiles = (a.N + 32 * t.nb * t.wn - 1) / (32 * t.nb * t.wn);
    a.out_scale = L.inv_scale;                             // (1 / sqrt(bs) is in the rotated activations)
    const dim3 grid((unsigned)((a.n_tiles + 7) / 8 * 8 * a.m_tiles));
    // Two 64-column tiles of a nibble plane at a time where the width allows it: 64 bytes of a row per pair of requests
    // instead of 32 (4864 x 896 at 512 rows 40.6 -> 38.0 us, 7680 x 565 55.0 -> 49.6; four tiles cost registers: 58).  The
    // combined plane's tile is 64 bytes already (two tiles at a time: 5 to 30 % slower).
    const bool pairs = a.K % 128 == 0;
    auto go = [&](auto Mode) {
        constexpr int M = decltype(Mode)::value;
        if constexpr (M != kSharedLut) { if (pairs) { launch_shape<M, 2>(shape, a, grid, stream); return; } }
        launch_shape<M, 1>(shape, a, grid, stream);
    };
    switch (L.mode) {
        case kSharedLut: go(std::integral_constant<int, kSharedLut>{}); break;
        case kDual: go(std::integral_constant<int, kDual>{}); break;
        default: go(std::integral_constant<int, kPrimaryOnly>{}); break;
    }
    return hipGetLastError();
}

}  // namespace tq
