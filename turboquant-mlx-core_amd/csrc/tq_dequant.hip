// Materialising dequantiser and stand-alone block rotation for gfx950.
//
// tq_dequant_kernel rebuilds the fp32 weight [out, in] from the packed indices and
// follows the reference CPU dequantiser operation by operation
// (src/dequantizer.cpp:52-256 with the inverse rotation of src/rotation.cpp:323-350):
// lookup, * 1/sqrt(in), butterfly, * (1/sqrt(bs) * sign), [+ residual plane], * norm.
// Every step is a single fp32 operation in the reference's order (this file is
// compiled with -ffp-contract=off), so the output is bit-identical to the CPU path.
//
// A wave takes 64 consecutive 32-column chunks of the row-major matrix (whole blocks: a row holds a whole number of
// them, and 2048 columns are a multiple of every block), one chunk per lane, and walks the matrix with the stride of the
// grid: the position of a lane's columns in their block is the same in every step, so the signs are hashed once per wave.
// The butterfly runs inside the lanes: five stages on the 32 columns of a chunk, then the 16 chunks of 512 columns change
// places through LDS (lane p of 16 receives columns 2 p and 2 p + 1 of all 16 chunks) and four stages on those; only
// blocks of 1024 and 2048 columns have stages across lanes.  Stage order and operations are the reference's.
#include "tq_device.h"

#include <type_traits>

namespace tq {

constexpr int kDqWaves = 4;   // waves per workgroup

// Exchange area of a wave: [4 groups of 512 columns][16 column pairs][16 chunks] x 8 bytes.  A group is padded so that two
// of them lie on different halves of the banks; the 16-byte slots of a pair's 128 bytes are permuted by the pair, so that
// the 16 lanes that read 16 bytes together find them on different banks.
constexpr int kDqGroup = 16 * 128 + 128;
constexpr int kDqExchange = 4 * kDqGroup;

// v: 32 consecutive columns of a lane's chunk -> column pair p = lane % 16 of all 16 chunks of its 512 columns
// (v[2 j], v[2 j + 1]: chunk j).  `area`: this wave's exchange area.
__device__ __forceinline__ void chunks_to_pairs(float (&v)[kChunk], char* area, int lane) {
    char* const base = area + (lane >> 4) * kDqGroup;
    const int c = lane & 15, wr = ((c >> 1) << 4) | ((c & 1) << 3);
#pragma unroll
    for (int p = 0; p < 16; ++p)
        *reinterpret_cast<float2*>(base + p * 128 + (wr ^ (((p >> 1) & 7) << 4))) = make_float2(v[2 * p], v[2 * p + 1]);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const char* const rd = base + c * 128;
    const int sw = ((c >> 1) & 7) << 4;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        const float4 t = *reinterpret_cast<const float4*>(rd + ((s << 4) ^ sw));
        v[4 * s] = t.x; v[4 * s + 1] = t.y; v[4 * s + 2] = t.z; v[4 * s + 3] = t.w;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();                       // (the area is written again)
}

// The way back.
__device__ __forceinline__ void pairs_to_chunks(float (&v)[kChunk], char* area, int lane) {
    char* const base = area + (lane >> 4) * kDqGroup;
    const int c = lane & 15, wr = ((c >> 1) << 4) | ((c & 1) << 3), sw = ((c >> 1) & 7) << 4;
#pragma unroll
    for (int s = 0; s < 8; ++s)
        *reinterpret_cast<float4*>(base + c * 128 + ((s << 4) ^ sw)) = make_float4(v[4 * s], v[4 * s + 1], v[4 * s + 2], v[4 * s + 3]);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int p = 0; p < 16; ++p) {
        const float2 t = *reinterpret_cast<const float2*>(base + p * 128 + (wr ^ (((p >> 1) & 7) << 4)));
        v[2 * p] = t.x; v[2 * p + 1] = t.y;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Stages 1 .. 16 of the butterfly on a lane's chunk, and 32 .. 1024 on its pairs.
__device__ __forceinline__ void fwht_chunk(float (&v)[kChunk], uint32_t bs) {
#pragma unroll
    for (int h = 1; h < kChunk; h <<= 1) {
        if ((uint32_t)h < bs) {
#pragma unroll
            for (int i = 0; i < kChunk; i += 2 * h)
#pragma unroll
                for (int j = i; j < i + h; ++j) { const float a = v[j], b = v[j + h]; v[j] = a + b; v[j + h] = a - b; }
        }
    }
}
__device__ __forceinline__ void fwht_pairs(float (&v)[kChunk], uint32_t bs, int lane) {
#pragma unroll
    for (int h = 2; h < kChunk; h <<= 1) {                 // (chunk j at 2 j: stage 16 h of the block)
        if ((uint32_t)h * 16 < bs) {
#pragma unroll
            for (int i = 0; i < kChunk; i += 2 * h)
#pragma unroll
                for (int j = i; j < i + h; ++j) { const float a = v[j], b = v[j + h]; v[j] = a + b; v[j + h] = a - b; }
        }
    }
    if (bs > 512) butterfly_lanes<16, kChunk>(v, lane);
    if (bs > 1024) butterfly_lanes<32, kChunk>(v, lane);
}

// Index bytes of a chunk: 16 (nibbles) or 32.
template <bool BYTES> struct ChunkBytes { uint4 v[BYTES ? 2 : 1]; };
template <bool BYTES>
__device__ __forceinline__ ChunkBytes<BYTES> load_chunk_bytes(const uint8_t* plane, long long chunk) {
    ChunkBytes<BYTES> r;
    const uint4* p = reinterpret_cast<const uint4*>(plane + (size_t)chunk * (BYTES ? 32 : 16));
    r.v[0] = p[0];
    if constexpr (BYTES) r.v[1] = p[1];
    return r;
}
__device__ __forceinline__ uint32_t chunk_word(const ChunkBytes<false>& r, int d) {
    return d == 0 ? r.v[0].x : d == 1 ? r.v[0].y : d == 2 ? r.v[0].z : r.v[0].w;
}
__device__ __forceinline__ uint32_t chunk_word(const ChunkBytes<true>& r, int d) {
    const uint4& t = r.v[d >> 2];
    const int e = d & 3;
    return e == 0 ? t.x : e == 1 ? t.y : e == 2 ? t.z : t.w;
}
// tab[nibble k] of a chunk; the 16 entries of a table lie on 16 different banks.  Byte offsets 4 n straight from the word.
__device__ __forceinline__ void lookup_nibbles(const ChunkBytes<false>& r, const char* tab, float (&v)[kChunk]) {
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const uint32_t w = chunk_word(r, d), lo = (w << 2) & 0x3c3c3c3cu, hi = (w >> 2) & 0x3c3c3c3cu;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[8 * d + 2 * j] = *reinterpret_cast<const float*>(tab + ((lo >> (8 * j)) & 0xffu));       // lo nibble = even column (src/dequantizer.cpp:46)
            v[8 * d + 2 * j + 1] = *reinterpret_cast<const float*>(tab + ((hi >> (8 * j)) & 0xffu));   // hi nibble = odd column  (src/dequantizer.cpp:47)
        }
    }
}

// Which planes a layer has and how a centroid is found.
template <int MODE> struct DequantMode {
    static constexpr bool five = MODE == kShared5 || MODE == kPrimaryOnly5 || MODE == kDual5;
    static constexpr bool dual = MODE == kDual || MODE == kDual5;
};

// COMBINED: the layer's one-byte-per-weight plane (kSharedLut; kShared5 and kPrimaryOnly5 where the residual index fits
// the byte's top three bits).
//
// Bound by its vector instructions (39 per weight in dual rotation: two butterflies of 9, lookups and exchange,
// signs, sum, norm and conversion) and by three waves per SIMD (registers, 11 KB of LDS per wave).
// 27648 x 5120 to bf16: dual 364 -> 152 us (2.8 TB/s of planes and weights), shared 104.  Before, a lane kept 32 consecutive
// columns throughout: four more stages across lanes at two to three instructions per value, two sign hashes per weight,
// 64-byte pieces per lane in every store, and idle lanes behind the last 2048 columns of a row.
template <int MODE, bool COMBINED>
__global__ __launch_bounds__(kDqWaves* kWave, 3) void tq_dequant_kernel(LayerView L, void* __restrict__ Wout, int w_dtype,
                                                                         int chunks_per_row, long long chunks) {
    using M = DequantMode<MODE>;
    constexpr bool bytes = COMBINED || M::five;            // of the primary plane
    constexpr bool residual_plane = M::dual || (MODE == kShared5 && !COMBINED);
    constexpr int kCopies = 8;                             // of the 256-entry table: a lane reads the copy lane % 8
    __shared__ float tab[MODE == kSharedLut ? 256 * kCopies : 64];
    __shared__ __align__(16) char exchange[kDqWaves * kDqExchange];
    __shared__ __align__(16) float row_norm[kDqWaves * kWave];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
    // (every centroid, or sum of two, is multiplied by 1/sqrt(in) before the butterfly: one fp32 product, whether formed
    // here or per weight)
    if constexpr (MODE == kSharedLut) {
        for (int i = threadIdx.x; i < 256 * kCopies; i += blockDim.x) tab[i] = L.tables[i / kCopies] * L.inv_scale;
    } else {
        for (int i = threadIdx.x; i < 64; i += blockDim.x) tab[i] = MODE == kShared5 ? L.tables[i] : L.tables[i] * L.inv_scale;
    }
    // Signs of the residual's rotation over 2048 columns (a second set of 32 registers per lane does not fit).
    __shared__ __align__(16) float signs_r[M::dual ? kSlab : 4];
    if constexpr (M::dual)
        for (int i = threadIdx.x; i < kSlab; i += blockDim.x)
            signs_r[i] = L.inv_sqrt_bs * sign_of(L.seed_residual, (uint32_t)i & (L.block_size - 1));
    __syncthreads();
    const char* const tab_p = reinterpret_cast<const char*>(tab);
    const char* const tab_r = reinterpret_cast<const char*>(tab + (M::five ? 32 : 16));
    char* const area = exchange + wave * kDqExchange;
    float* const nrm_of = row_norm + wave * kWave;

    const uint32_t bs = L.block_size;
    // Signs of this lane's 32 values after the exchange: columns 32 j + 2 p + (0, 1) of its 512.
    float sp[kChunk];
#pragma unroll
    for (int k = 0; k < kChunk; ++k) {
        const uint32_t col = (uint32_t)((lane >> 4) * 512 + (k >> 1) * 32 + 2 * (lane & 15) + (k & 1)) & (bs - 1);
        sp[k] = L.inv_sqrt_bs * sign_of(L.seed_primary, col);
    }

    const long long step = (long long)gridDim.x * (kDqWaves * kWave);
    long long base = ((long long)blockIdx.x * kDqWaves + wave) * kWave;
    if (base >= chunks) return;                            // whole wave leaves together; no workgroup barrier below
    auto mine = [&](long long b) { return b + lane < chunks ? b + lane : chunks - 1; };     // (past the end: the last chunk again, not stored)
    const uint8_t* const plane_p = COMBINED ? L.packed_combined : L.packed_primary;
    ChunkBytes<bytes> P = load_chunk_bytes<bytes>(plane_p, mine(base));
    ChunkBytes<false> R{};
    if constexpr (residual_plane) R = load_chunk_bytes<false>(L.packed_residual, mine(base));
    for (; base < chunks; base += step) {
        const ChunkBytes<bytes> pb = P;
        const ChunkBytes<false> rb = R;
        const long long ahead = base + step < chunks ? base + step : base;
        P = load_chunk_bytes<bytes>(plane_p, mine(ahead));
        if constexpr (residual_plane) R = load_chunk_bytes<false>(L.packed_residual, mine(ahead));
        nrm_of[lane] = L.norms[mine(base) / chunks_per_row];

        float v[kChunk];
        if constexpr (MODE == kSharedLut) {
            // path A: 256-entry table of centroid sums (src/dequantizer.cpp:136-184)
#pragma unroll
            for (int d = 0; d < 8; ++d)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    v[4 * d + j] = tab[((chunk_word(pb, d) >> (8 * j)) & 0xffu) * kCopies + (lane & (kCopies - 1))];
        } else if constexpr (bytes) {
            float t[kChunk];
            if constexpr (MODE == kShared5 && !COMBINED) lookup_nibbles(rb, tab_r, t);
#pragma unroll
            for (int d = 0; d < 8; ++d)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t c = (chunk_word(pb, d) >> (8 * j)) & 0xffu;
                    // (combined: residual index in the top three bits, both clamped when the plane was built)
                    const uint32_t pi = COMBINED ? (c & 31u) : (c > 31u ? 31u : c);
                    float x = tab[pi];
                    if constexpr (MODE == kShared5)                                          // path B (src/dequantizer.cpp:186-212)
                        x = (x + (COMBINED ? tab[32 + (c >> 5)] : t[4 * d + j])) * L.inv_scale;
                    v[4 * d + j] = x;
                }
        } else {
            lookup_nibbles(pb, tab_p, v);
        }
        fwht_chunk(v, bs);
        chunks_to_pairs(v, area, lane);
        fwht_pairs(v, bs, lane);
#pragma unroll
        for (int k = 0; k < kChunk; ++k) v[k] *= sp[k];
        if constexpr (M::dual) {
            // path C second plane (src/dequantizer.cpp:220-245)
            float u[kChunk];
            lookup_nibbles(rb, tab_r, u);
            fwht_chunk(u, bs);
            chunks_to_pairs(u, area, lane);
            fwht_pairs(u, bs, lane);
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const float2 sr = *reinterpret_cast<const float2*>(signs_r + (lane >> 4) * 512 + j * 32 + 2 * (lane & 15));
                u[2 * j] *= sr.x; u[2 * j + 1] *= sr.y;
                v[2 * j] = v[2 * j] + u[2 * j]; v[2 * j + 1] = v[2 * j + 1] + u[2 * j + 1];
            }
        }

        const long long chunk0 = base + (lane >> 4) * 16;  // of the 16 chunks whose pair this lane holds
        const float4* const np = reinterpret_cast<const float4*>(nrm_of + (lane >> 4) * 16);
        const size_t elem = (size_t)chunk0 * kChunk + 2 * (lane & 15);
        const int have = chunks - chunk0 < 16 ? (int)(chunks - chunk0) : 16;
        auto store = [&](auto Tc) {
            constexpr int T = decltype(Tc)::value;
            typedef float f32x2_t __attribute__((ext_vector_type(2)));
            typedef __bf16 b16x2_t __attribute__((ext_vector_type(2)));
            typedef _Float16 h16x2_t __attribute__((ext_vector_type(2)));
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 n4 = np[q];
                const float n[4] = {n4.x, n4.y, n4.z, n4.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int j = 4 * q + e;
                    const f32x2_t f = {v[2 * j] * n[e], v[2 * j + 1] * n[e]};
                    if (j >= have) continue;
                    // 16-bit: the fp32 weight rounded to nearest-even, the cast src/turboquant_c_dequant.cpp:166 applies.
                    if constexpr (T == kF32) *reinterpret_cast<f32x2_t*>(static_cast<float*>(Wout) + elem + j * kChunk) = f;
                    else if constexpr (T == kBF16)
                        *reinterpret_cast<uint32_t*>(static_cast<uint16_t*>(Wout) + elem + j * kChunk) =
                            __builtin_bit_cast(uint32_t, __builtin_convertvector(f, b16x2_t));
                    else
                        *reinterpret_cast<uint32_t*>(static_cast<uint16_t*>(Wout) + elem + j * kChunk) =
                            __builtin_bit_cast(uint32_t, __builtin_convertvector(f, h16x2_t));
                }
            }
        };
        if (w_dtype == kF32) store(std::integral_constant<int, kF32>{});
        else if (w_dtype == kBF16) store(std::integral_constant<int, kBF16>{});
        else store(std::integral_constant<int, kF16>{});
    }
}

hipError_t launch_dequant(const LayerView& L, void* w, int w_dtype, hipStream_t stream) {
    const int per_row = L.in_features / kChunk;
    const long long chunks = (long long)L.out_features * per_row;
    const long long groups = (chunks + kDqWaves * kWave - 1) / (kDqWaves * kWave);
    const dim3 grid((unsigned)(groups < 768 ? groups : 768)), block(kDqWaves * kWave);     // three workgroups per CU
    auto go = [&](auto Mode, auto Combined) {
        hipLaunchKernelGGL((tq_dequant_kernel<decltype(Mode)::value, decltype(Combined)::value>), grid, block, 0, stream, L, w,
                           w_dtype, per_row, chunks);
    };
    const bool combined = L.packed_combined != nullptr;
    switch (L.mode) {
        case kSharedLut: go(std::integral_constant<int, kSharedLut>{}, std::true_type{}); break;
        case kDual: go(std::integral_constant<int, kDual>{}, std::false_type{}); break;
        case kPrimaryOnly: go(std::integral_constant<int, kPrimaryOnly>{}, std::false_type{}); break;
        case kShared5:
            if (combined) go(std::integral_constant<int, kShared5>{}, std::true_type{});
            else go(std::integral_constant<int, kShared5>{}, std::false_type{});
            break;
        case kPrimaryOnly5:
            if (combined) go(std::integral_constant<int, kPrimaryOnly5>{}, std::true_type{});
            else go(std::integral_constant<int, kPrimaryOnly5>{}, std::false_type{});
            break;
        default: go(std::integral_constant<int, kDual5>{}, std::false_type{}); break;
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Two planes with rotations of their own as ONE fp16 weight in the primary's rotation, for prefill of many rows:
//   sum_k cP[k] x~p[k] + cR[k] x~r[k]  =  sum_k (cP + H (s_p s_r (.) H cR) / bs)[k] x~p[k],     x~ = H (s (.) x)
// so that the contraction runs once instead of once per plane.  The sum is formed in fp32 and rounded to fp16 once; the
// planes multiplied one after the other round each centroid by itself (compose_scale() looks at which of the two is
// closer).  kShared5: both planes in one rotation, a plain sum.
// Rows [row0, row0 + rows) of the layer (row0 a multiple of 128), in the order in which tq_prefill_panel_kernel's threads
// load them: [row / 128][K / 64][4 pieces of 8 columns][row % 128 / 32][half of the 64 columns][row % 32] x 16 bytes.
// Bound by its vector instructions (38 per weight); 27648 x 5120 in two slabs of 76 us, a quarter of the contraction at 2048
// rows.
// Four waves per SIMD (128 registers) spill and are 10 % slower.
// A wave takes 512 columns (whole blocks: at most 512) of four rows, 16 lanes each, and eight waves in a row the same
// columns of 32 rows; exchange as above.
// ---------------------------------------------------------------------------
template <int MODE>
__global__ __launch_bounds__(kDqWaves* kWave, 3) void tq_compose_kernel(LayerView L, char* __restrict__ out, int row0, int rows,
                                                                         int segs, int tasks) {
    constexpr bool bytes = DequantMode<MODE>::five, rotate = DequantMode<MODE>::dual;
    __shared__ float tab[64];
    __shared__ __align__(16) char exchange[rotate ? kDqWaves * kDqExchange : 16];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
    if (threadIdx.x < 64) tab[threadIdx.x] = L.tables[threadIdx.x] * L.compose_scale;
    __syncthreads();
    const char* const tab_p = reinterpret_cast<const char*>(tab);
    const char* const tab_r = reinterpret_cast<const char*>(tab + (bytes ? 32 : 16));
    char* const area = exchange + (rotate ? wave * kDqExchange : 0);
    const uint32_t bs = L.block_size;
    float sg[rotate ? kChunk : 1];
    if constexpr (rotate) {
        const float scale = 1.0f / (float)bs;              // (a power of two)
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
            const uint32_t col = (uint32_t)((k >> 1) * 32 + 2 * (lane & 15) + (k & 1)) & (bs - 1);
            sg[k] = scale * sign_of(L.seed_primary, col) * sign_of(L.seed_residual, col);
        }
    }
    const int per_row = L.in_features / kChunk, step = gridDim.x * kDqWaves;
    int task = blockIdx.x * kDqWaves + wave;               // (32 rows, 512 columns, four of the rows)
    if (task >= tasks) return;                             // whole wave leaves together; no workgroup barrier below
    int r = 0, c = 0;                                      // this lane's row of the slab and chunk of the row
    auto place = [&](int t) {
        const int unit = t >> 3, rb = unit / segs;
        r = rb * 32 + (t & 7) * 4 + (lane >> 4);
        c = (unit - rb * segs) * 16 + (lane & 15);
    };
    // (past the last row or column: the last row, chunk 0 .. 15, not stored)
    auto mine = [&]() { return (long long)(row0 + (r < rows ? r : rows - 1)) * per_row + (c < per_row ? c : 0); };
    place(task);
    ChunkBytes<bytes> P = load_chunk_bytes<bytes>(L.packed_primary, mine());
    ChunkBytes<false> R = load_chunk_bytes<false>(L.packed_residual, mine());
    for (; task < tasks; task += step) {
        const ChunkBytes<bytes> pb = P;
        const ChunkBytes<false> rb = R;
        const int row = r, chunk = c;
        place(task + step < tasks ? task + step : task);
        P = load_chunk_bytes<bytes>(L.packed_primary, mine());
        R = load_chunk_bytes<false>(L.packed_residual, mine());
        float u[kChunk], v[kChunk];
        lookup_nibbles(rb, tab_r, u);
        if constexpr (rotate) {
            fwht_chunk(u, bs);
            chunks_to_pairs(u, area, lane);
            fwht_pairs(u, bs, lane);
#pragma unroll
            for (int k = 0; k < kChunk; ++k) u[k] *= sg[k];
            fwht_pairs(u, bs, lane);
            pairs_to_chunks(u, area, lane);
            fwht_chunk(u, bs);
        }
        if constexpr (bytes) {
#pragma unroll
            for (int d = 0; d < 8; ++d)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t c = (chunk_word(pb, d) >> (8 * j)) & 0xffu;
                    v[4 * d + j] = tab[c > 31u ? 31u : c];
                }
        } else {
            lookup_nibbles(pb, tab_p, v);
        }
        if (row >= rows || chunk >= per_row) continue;
        char* const dst = out + ((size_t)(row >> 7) * (per_row >> 1) + (chunk >> 1)) * 16384 +
                          (((row & 127) >> 5) * 64 + (chunk & 1) * 32 + (row & 31)) * 16;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            typedef float f32x8_t __attribute__((ext_vector_type(8)));
            typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
            f32x8_t f;
#pragma unroll
            for (int j = 0; j < 8; ++j) f[j] = v[8 * i + j] + u[8 * i + j];
            *reinterpret_cast<f16x8_t*>(dst + i * 4096) = __builtin_convertvector(f, f16x8_t);      // (in range: compose_scale)
        }
    }
}

hipError_t launch_compose(const LayerView& L, int row0, int rows, void* out, hipStream_t stream) {
    const int segs = (L.in_features / kChunk + 15) / 16;
    const long long tasks = (long long)((rows + 31) / 32) * segs * 8, groups = tasks / kDqWaves;
    if (tasks > 0x3fffffff || (row0 & 127) || L.in_features % 64 || L.block_size > 512) return hipErrorInvalidValue;
    const dim3 grid((unsigned)(groups < 768 ? groups : 768)), block(kDqWaves * kWave);
    char* const o = static_cast<char*>(out);
    switch (L.mode) {
        case kDual: hipLaunchKernelGGL(tq_compose_kernel<kDual>, grid, block, 0, stream, L, o, row0, rows, segs, (int)tasks); break;
        case kDual5: hipLaunchKernelGGL(tq_compose_kernel<kDual5>, grid, block, 0, stream, L, o, row0, rows, segs, (int)tasks); break;
        case kShared5: hipLaunchKernelGGL(tq_compose_kernel<kShared5>, grid, block, 0, stream, L, o, row0, rows, segs, (int)tasks); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Block rotation of an fp32 matrix (reference src/rotation.cpp:291-350).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kDqWaves* kWave) void tq_wht_kernel(const float* __restrict__ in, float* __restrict__ out,
                                                                  int rows, int cols, int chunks, int slabs,
                                                                  uint32_t seed, uint32_t bs, float inv_sqrt_bs,
                                                                  int inverse) {
    const int lane = threadIdx.x & (kWave - 1);
    const long long wid = (long long)blockIdx.x * kDqWaves + (threadIdx.x >> 6);
    const int row = (int)(wid / slabs);
    const int slab = (int)(wid % slabs);
    if (row >= rows) return;
    const int chunk = slab * kWave + lane;
    const bool active = chunk < chunks;
    const uint32_t col0 = ((uint32_t)chunk * kChunk) & (bs - 1);

    float v[kChunk];
    if (active) {
        load_chunk(in, kF32, (size_t)row * cols + (size_t)chunk * kChunk, v);
    } else {
#pragma unroll
        for (int k = 0; k < kChunk; ++k) v[k] = 0.0f;
    }
    if (!inverse) {
#pragma unroll
        for (int k = 0; k < kChunk; ++k) v[k] *= sign_of(seed, (col0 + k) & (bs - 1));
    }
    fwht_lane32(v, bs, lane);
    if (!inverse) {
#pragma unroll
        for (int k = 0; k < kChunk; ++k) v[k] *= inv_sqrt_bs;
    } else {
#pragma unroll
        for (int k = 0; k < kChunk; ++k) v[k] *= inv_sqrt_bs * sign_of(seed, (col0 + k) & (bs - 1));
    }
    if (active) {
        float4* dst = reinterpret_cast<float4*>(out + (size_t)row * cols + (size_t)chunk * kChunk);
#pragma unroll
        for (int i = 0; i < 8; ++i) dst[i] = make_float4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
    }
}

hipError_t launch_wht(const float* in, float* out, int rows, int cols, uint32_t seed,
                      uint32_t block_size, float inv_sqrt_bs, int inverse, hipStream_t stream) {
    const int chunks = cols / kChunk;
    const int slabs = (chunks + kWave - 1) / kWave;
    const long long waves = (long long)rows * slabs;
    const long long grid = (waves + kDqWaves - 1) / kDqWaves;
    if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
    hipLaunchKernelGGL(tq_wht_kernel, dim3((unsigned)grid), dim3(kDqWaves * kWave), 0, stream,
                       in, out, rows, cols, chunks, slabs, seed, block_size, inv_sqrt_bs, inverse);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// "Does the residual plane hold any non-zero byte" (src/dequantizer.cpp:118-128)
// for tensors that already live on the GPU.
// ---------------------------------------------------------------------------
__global__ void tq_any_nonzero_kernel(const uint8_t* __restrict__ data, size_t n, int* flag) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    uint32_t acc = 0;
    const size_t n16 = n / 16;
    const uint4* p = reinterpret_cast<const uint4*>(data);
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += stride) {
        const uint4 t = p[i];
        acc |= t.x | t.y | t.z | t.w;
    }
    for (size_t i = n16 * 16 + (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) acc |= data[i];
    if (acc) atomicOr(flag, 1);
}

// Interleave the two nibble planes into one byte per weight (residual high, primary low),
// the layout the shared-rotation GEMV streams.  One thread per packed byte pair.
__global__ void tq_combine_planes_kernel(const uint8_t* __restrict__ primary, const uint8_t* __restrict__ residual,
                                         uint16_t* __restrict__ combined, size_t plane_bytes) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < plane_bytes; i += stride) {
        const uint32_t pb = primary[i], rb = residual[i];
        const uint32_t even = (pb & 0x0fu) | ((rb & 0x0fu) << 4);   // src/dequantizer.cpp:163
        const uint32_t odd = (pb >> 4) | (rb & 0xf0u);              // src/dequantizer.cpp:168
        combined[i] = (uint16_t)(even | (odd << 8));
    }
}

hipError_t launch_combine_planes(const uint8_t* primary, const uint8_t* residual, uint8_t* combined,
                                 size_t plane_bytes, hipStream_t stream) {
    hipLaunchKernelGGL(tq_combine_planes_kernel, dim3(2048), dim3(256), 0, stream, primary, residual,
                       reinterpret_cast<uint16_t*>(combined), plane_bytes);
    return hipGetLastError();
}

// 5-bit primary (one index per byte) + residual nibbles of at most 3 significant bits -> one byte
// per weight: min(r, n_residual - 1) << 5 | min(p, n_primary - 1)  (clamps of src/dequantizer.cpp:94,103).
__global__ void tq_combine_planes5_kernel(const uint8_t* __restrict__ primary, const uint8_t* __restrict__ residual,
                                          uint16_t* __restrict__ combined, size_t residual_bytes, uint32_t pmax,
                                          uint32_t rmax) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < residual_bytes; i += stride) {
        const uint32_t rb = residual[i];
        const uint32_t p0 = min((uint32_t)primary[2 * i], pmax), p1 = min((uint32_t)primary[2 * i + 1], pmax);
        const uint32_t r0 = min(rb & 0x0fu, rmax), r1 = min(rb >> 4, rmax);
        combined[i] = (uint16_t)((r0 << 5) | p0 | (((r1 << 5) | p1) << 8));
    }
}

hipError_t launch_combine_planes5(const uint8_t* primary, const uint8_t* residual, uint8_t* combined,
                                  size_t residual_bytes, int n_primary, int n_residual, hipStream_t stream) {
    hipLaunchKernelGGL(tq_combine_planes5_kernel, dim3(2048), dim3(256), 0, stream, primary, residual,
                       reinterpret_cast<uint16_t*>(combined), residual_bytes, (uint32_t)(n_primary - 1),
                       (uint32_t)(n_residual - 1));
    return hipGetLastError();
}

__global__ void tq_silu_mul_kernel(const float* __restrict__ gate, const float* __restrict__ up, void* __restrict__ out,
                                   int out_dtype, size_t n) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        const float g = gate[i];
        store_scalar(out, out_dtype, i, g / (1.0f + expf(-g)) * up[i]);
    }
}

hipError_t launch_silu_mul(const float* gate, const float* up, void* out, int out_dtype, size_t n, hipStream_t stream) {
    const size_t blocks = (n + 255) / 256;
    hipLaunchKernelGGL(tq_silu_mul_kernel, dim3((unsigned)(blocks < 1 ? 1 : (blocks > 4096 ? 4096 : blocks))), dim3(256), 0,
                       stream, gate, up, out, out_dtype, n);
    return hipGetLastError();
}

// out[i] = a[i] + b[i] over n fp32 values, written as out_dtype; out may be a itself.
__global__ void tq_add_kernel(const float* a, const float* __restrict__ b, void* out, int out_dtype, size_t n) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        store_scalar(out, out_dtype, i, a[i] + b[i]);
}

hipError_t launch_add(const float* a, const float* b, void* out, int out_dtype, size_t n, hipStream_t stream) {
    const size_t blocks = (n + 255) / 256;
    hipLaunchKernelGGL(tq_add_kernel, dim3((unsigned)(blocks < 1 ? 1 : (blocks > 4096 ? 4096 : blocks))), dim3(256), 0,
                       stream, a, b, out, out_dtype, n);
    return hipGetLastError();
}

hipError_t launch_any_nonzero(const uint8_t* data, size_t n, int* flag_dev, hipStream_t stream) {
    hipLaunchKernelGGL(tq_any_nonzero_kernel, dim3(1024), dim3(256), 0, stream, data, n, flag_dev);
    return hipGetLastError();
}

}  // namespace tq
