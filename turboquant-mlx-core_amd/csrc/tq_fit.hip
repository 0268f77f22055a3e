// Lloyd-Max codebook fit on the GPU (reference src/codebook.cpp:99-143; per layer src/converter.cpp:291-372).
//
// A Lloyd-Max step needs, for every bin, how many samples lie in it and what they add up to.  Reading all samples once
// per step costs 200 passes for the two codebooks of a layer.  Here the samples are put in coarse value order once and
// a step looks at the few thousand samples around each boundary only:
//
//   tq_fit_absmax_kernel    largest |sample|: fixes the scale of the value cells (the kernel that makes a layer's samples knows it)
//   tq_fit_hist_kernel      per tile of the samples: how many fall into each of kFitCells value cells, and the sum of
//                           their offsets inside the cell
//   tq_fit_offsets_kernel   the tiles' counts become positions; the cells' totals
//   tq_fit_scan_kernel      prefix sums over the cells
//   tq_fit_predict_kernel   all steps on the cells alone (a boundary splits its cell in proportion): which cells the
//                           boundaries will visit
//   tq_fit_scatter_kernel   the samples of those cells written cell by cell
//   tq_fit_refine_kernel    every such cell put in the order of 64 equal parts
//   tq_fit_iterate_kernel   all steps: one workgroup per codebook, one wave per boundary; the samples below a boundary
//                           are the cells below it, the parts of its cell below it (prefix sums) and the samples of its
//                           own part that compare below it
//
// Cells are a monotone function of the value (about 10 bits of mantissa), so a boundary splits one cell only and bins
// are exactly those of the comparison `boundary < value`.  Sums are integers in units of 2^-38 of the scale, exact whatever
// the order the samples arrive in and rounded once, where the reference adds doubles one after the other.  Samples from
// 2^-15 of the scale on are whole numbers of units; those below lose what is smaller than one.  Where that could
// reach a quarter of the rounding of a centroid (samples that are tiny beside the largest: no rotated weight does
// that) the fit says so and is left to the pass per step.
//
// 18944 x 3584 (68 M samples, 2 x 100 steps).  One pass over all samples per step took 230 ms, 1.1 ms each (thread-private
// bins in 96 KB of LDS, one wave per SIMD) and a copy of the partial sums to the host; the kernels here take 0.95 ms:
// scatter 260 to 320 us, iterate 246, hist 140, refine 115, predict 84, offsets 45, scan 23.  What bounds them is
// said at each.  Sorting every sample instead of the expected 15 % took 1840 us in the scatter kernel and 870 in refine.
#include "tq_bins.h"
#include "tq_device.h"

namespace tq {

typedef __int128 i128;

constexpr int kFitLin = 1024;                         // cells of [0, 2^-6) of the scale, all equally wide
constexpr int kFitHalf = kFitLin * 7;                 // ... and 1024 per octave from 2^-6 to 1
constexpr int kFitCells = 2 * kFitHalf;               // negative values mirrored below
constexpr int kFitThreads = 1024;
constexpr int kFitMaxExp = 8;                         // of the scale: the pass per step takes samples of 2^8 and more
constexpr int kFitCut = 2;                            // cells on either side of zero whose samples may be no whole number of units
constexpr uint32_t kFitLinEnd = 0x3c800000u;          // 2^-6
constexpr int kFitMaxTile = 1 << 19;                  // samples per tile: offset sums (22 bits each) stay below 2^41

struct FitParams {                                    // written by tq_fit_absmax_fold_kernel
    float scale[2];                                   // 2^-E, 2^E above every |sample| of the problem
    double unit[2];                                   // 2^(E - 38)
    int bad;                                          // samples that are no finite numbers or beyond 2^8 (a normalised row
                                                      // of 32768 columns times sqrt(32768) stays below it)
};

struct FitProblem {                                   // what a sample of problem p is
    const float* data;
    size_t n;
    const float* gtab[2];                             // NULL, or the global codebook: [0..31] centroids, [32..62] boundaries
    int ngc;
};

// Cell of a value and its offset inside the cell: 22 bits in units of 2^-38 below 2^-6 of the scale, the 13 low
// mantissa bits above (units of 2^-29 and up, one octave after the other).
__device__ __forceinline__ void fit_cell(float v, float scale, uint32_t& cell, uint32_t& off) {
    const float t = __builtin_fabsf(v) * scale;
    const uint32_t bits = __builtin_bit_cast(uint32_t, t);
    const float s = t * 65536.0f;
    const uint32_t li = (uint32_t)s;
    const uint32_t lo = (uint32_t)((s - (float)li) * 4194304.0f);
    const uint32_t d = bits - kFitLinEnd;
    const bool lin = bits < kFitLinEnd;
    uint32_t i = lin ? li : (uint32_t)kFitLin + (d >> 13);
    off = lin ? lo : (d & 0x1fffu);
    if (i >= (uint32_t)kFitHalf) { i = (uint32_t)kFitHalf - 1; off = 0x1fffu; }   // (a boundary beyond all samples)
    cell = v < 0.0f ? (uint32_t)kFitHalf - 1u - i : (uint32_t)kFitHalf + i;
}

// The offset of a sample whose cell is known, one or four instructions: the scale is a power of two and leaves the mantissa
// as it is.  `whole`: the linear cell's number.
__device__ __forceinline__ uint32_t fit_log_offset(float v) { return __builtin_bit_cast(uint32_t, v) & 0x1fffu; }
__device__ __forceinline__ uint32_t fit_linear_offset(float v, float scale, float whole) {
    return (uint32_t)((__builtin_fabsf(v) * scale * 65536.0f - whole) * 4194304.0f);
}
__device__ __forceinline__ float fit_cell_whole(uint32_t cell) {
    return (float)(cell < (uint32_t)kFitHalf ? (uint32_t)kFitHalf - 1u - cell : cell - (uint32_t)kFitHalf);
}

// Magnitude of a cell's lower end, and how far its offsets are shifted, in units of 2^-38 of the scale.
__device__ __forceinline__ void fit_cell_base(uint32_t cell, uint64_t& base, int& shift, bool& neg) {
    neg = cell < (uint32_t)kFitHalf;
    const uint32_t i = neg ? (uint32_t)kFitHalf - 1u - cell : cell - (uint32_t)kFitHalf;
    if (i < (uint32_t)kFitLin) { base = (uint64_t)i << 22; shift = 0; return; }
    const uint32_t o = (i - kFitLin) >> 10, f = (i - kFitLin) & 1023u;
    base = (uint64_t)(1024u + f) << (22 + o);
    shift = 9 + (int)o;
}

// The residual of a sample: its distance from the global codebook's centroid (src/converter.cpp:348-356).
struct FitResidual { BinTable bins; float cent[32]; };
__device__ __forceinline__ void fit_residual_build(FitResidual& r, const float* gtab, int ngc) {
    if (threadIdx.x < 32) r.cent[threadIdx.x] = (int)threadIdx.x < ngc ? gtab[threadIdx.x] : 0.0f;
    bin_table_build(r.bins, gtab + 32, ngc - 1, threadIdx.x);
}

// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void tq_fit_absmax_kernel(const float* __restrict__ data, size_t n,
                                                            uint32_t* __restrict__ part) {
    __shared__ uint32_t s[4];
    uint32_t m = 0;
    const size_t n4 = n / 4, stride = (size_t)gridDim.x * 256;
    const uint4* p = reinterpret_cast<const uint4*>(data);
    size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    for (; i + 3 * stride < n4; i += 4 * stride) {
        uint4 v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = p[i + k * stride];
#pragma unroll
        for (int k = 0; k < 4; ++k)
            m = max(max(max(m, v[k].x & 0x7fffffffu), max(v[k].y & 0x7fffffffu, v[k].z & 0x7fffffffu)), v[k].w & 0x7fffffffu);
    }
    for (; i < n4; i += stride) {
        const uint4 v = p[i];
        m = max(max(max(m, v.x & 0x7fffffffu), max(v.y & 0x7fffffffu, v.z & 0x7fffffffu)), v.w & 0x7fffffffu);
    }
    for (size_t j = n4 * 4 + (size_t)blockIdx.x * 256 + threadIdx.x; j < n; j += stride)
        m = max(m, __builtin_bit_cast(uint32_t, data[j]) & 0x7fffffffu);
    for (int k = 32; k >= 1; k >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, k, kWave));
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = max(max(s[0], s[1]), max(s[2], s[3]));
}

__device__ void fit_scale(float biggest, FitParams* P, int p) {
    const uint32_t b = __builtin_bit_cast(uint32_t, biggest);
    int e = (int)(b >> 23) - 127 + 1;                             // 2^e > biggest
    if (e > kFitMaxExp) { P->bad = 1; e = kFitMaxExp; }           // infinities and NaN among them
    if (e < -100) e = -100;
    P->scale[p] = __builtin_bit_cast(float, (uint32_t)(127 - e) << 23);
    P->unit[p] = __builtin_bit_cast(double, (uint64_t)(1023 + e - 38) << 52);
}

// One workgroup: the largest |sample| and the scales.  A residual is at most half a gap of the global codebook, or
// what lies beyond its last centroid, where that codebook is sorted.
__global__ __launch_bounds__(256) void tq_fit_absmax_fold_kernel(const uint32_t* __restrict__ part, int parts, FitProblem fp,
                                                                 int problems, FitParams* __restrict__ P, FitCodebooks cb,
                                                                 FitResult* __restrict__ state) {
    __shared__ uint32_t s[4];
    uint32_t m = 0;
    for (int i = threadIdx.x; i < parts; i += 256) m = max(m, part[i]);
    for (int k = 32; k >= 1; k >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, k, kWave));
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x < 64) state->cent[threadIdx.x >> 5][threadIdx.x & 31] = cb.init[threadIdx.x >> 5][threadIdx.x & 31];
    if (threadIdx.x != 0) return;
    state->steps[0] = state->steps[1] = 0;
    m = max(max(s[0], s[1]), max(s[2], s[3]));
    const float big = __builtin_bit_cast(float, m);
    P->bad = 0;
    for (int p = 0; p < problems; ++p) {
        float b = big;
        if (fp.gtab[p]) {
            const float* c = fp.gtab[p];
            const float* g = c + 32;
            b = fmaxf(fabsf(big - c[fp.ngc - 1]), fabsf(-big - c[0]));
            bool sorted = true;
            float far = 0.0f;
            for (int k = 0; k < fp.ngc; ++k) {
                if (!(fabsf(c[k]) < 1e30f)) P->bad = 1;           // infinities and NaN: no residual is a number
                far = fmaxf(far, fabsf(c[k]));
                if (k + 1 == fp.ngc) break;
                b = fmaxf(b, fmaxf(fabsf(g[k] - c[k]), fabsf(c[k + 1] - g[k])));
                if (!(c[k] <= c[k + 1])) sorted = false;
            }
            if (!sorted) b = big + far;                           // (a bin may have any centroid)
            b *= 1.0001f;
            if (!(m < 0x7f800000u)) P->bad = 1;
        }
        fit_scale(b, P, p);
    }
}

// Calls f(value) for every sample of tile `w` of `tiles`: 16 bytes per lane and load, four loads in flight.
template <typename F>
__device__ __forceinline__ void fit_tile(const float* data, size_t n, size_t tile, F&& f) {
    const size_t lo = (size_t)blockIdx.x * tile;                  // (tile is a multiple of 4)
    if (lo >= n) return;
    const size_t hi = lo + tile < n ? lo + tile : n;
    const size_t h4 = lo / 4 + (hi - lo) / 4;
    const float4* p = reinterpret_cast<const float4*>(data);
    size_t i = lo / 4 + threadIdx.x;
    for (; i + 3 * kFitThreads < h4; i += 4 * kFitThreads) {
        float4 v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = p[i + k * kFitThreads];
#pragma unroll
        for (int k = 0; k < 4; ++k) { f(v[k].x); f(v[k].y); f(v[k].z); f(v[k].w); }
    }
    for (; i < h4; i += kFitThreads) { const float4 v = p[i]; f(v.x); f(v.y); f(v.z); f(v.w); }
    for (size_t j = h4 * 4 + threadIdx.x; j < hi; j += kFitThreads) f(data[j]);
}

// Counts (upper 23 bits) and offset sums (lower 41) of one tile, in LDS: one 64-bit LDS atomic per sample.  The cells fill
// 112 KB, so a workgroup of 16 waves has the CU to itself.  140 us for both codebooks: 2 x 272 MB at 3.9 TB/s, bound by
// the 27 vector instructions per sample (busy 77 % of the time) and the LDS atomics (64 random 8-byte cells per wave
// instruction; 47 %).
__global__ __launch_bounds__(kFitThreads) void tq_fit_hist_kernel(FitProblem fp, const FitParams* __restrict__ P, size_t tile,
                                                                  unsigned long long* __restrict__ hist) {
    __shared__ unsigned long long h[kFitCells];
    __shared__ FitResidual res;
    if (P->bad) return;
    const int p = blockIdx.y;
    for (int i = threadIdx.x; i < kFitCells; i += kFitThreads) h[i] = 0;
    if (fp.gtab[p]) fit_residual_build(res, fp.gtab[p], fp.ngc);
    __syncthreads();
    const float scale = P->scale[p];
    auto count = [&](float v) {
        uint32_t cell, off;
        fit_cell(v, scale, cell, off);
        atomicAdd(&h[cell], (1ull << 41) | (unsigned long long)off);
    };
    if (fp.gtab[p]) {
        const float bs = res.bins.scale, bb = res.bins.bias;
        const int steps = res.bins.steps;
        fit_tile(fp.data, fp.n, tile, [&](float v) { count(v - res.cent[bin_find(res.bins, bs, bb, steps, fp.ngc - 1, v)]); });
    } else {
        fit_tile(fp.data, fp.n, tile, count);
    }
    __syncthreads();
    unsigned long long* dst = hist + ((size_t)p * gridDim.x + blockIdx.x) * kFitCells;
    for (int i = threadIdx.x; i < kFitCells; i += kFitThreads) dst[i] = h[i];
}

// One thread per cell: the counts of the tiles become first positions inside the cell, totals per cell.  88 MB of traffic in
// 45 us: 448 waves with eight loads in flight.
__global__ __launch_bounds__(256) void tq_fit_offsets_kernel(const FitParams* __restrict__ P, int tiles,
                                                             const unsigned long long* __restrict__ hist,
                                                             uint32_t* __restrict__ first, unsigned long long* __restrict__ cell_n,
                                                             i128* __restrict__ cell_q) {
    if (P->bad) return;
    const int p = blockIdx.y;
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= kFitCells) return;
    const unsigned long long* src = hist + (size_t)p * tiles * kFitCells + c;
    uint32_t* dst = first + (size_t)p * tiles * kFitCells + c;
    unsigned long long cnt = 0, off = 0;
#pragma unroll 8
    for (int w = 0; w < tiles; ++w) {
        const unsigned long long t = src[(size_t)w * kFitCells];
        dst[(size_t)w * kFitCells] = (uint32_t)cnt;
        cnt += t >> 41;
        off += t & ((1ull << 41) - 1);
    }
    uint64_t base; int shift; bool neg;
    fit_cell_base((uint32_t)c, base, shift, neg);
    const i128 q = (i128)cnt * (i128)base + ((i128)off << shift);
    cell_n[(size_t)p * kFitCells + c] = cnt;
    cell_q[(size_t)p * kFitCells + c] = neg ? -q : q;
}

// One workgroup per problem: exclusive prefix sums over the cells (start[kFitCells] = n).
constexpr int kFitOwn = kFitCells / kFitThreads;
static_assert(kFitOwn * kFitThreads == kFitCells, "cells per thread");
__global__ __launch_bounds__(kFitThreads) void tq_fit_scan_kernel(const FitParams* __restrict__ P,
                                                                  const unsigned long long* __restrict__ cell_n,
                                                                  const i128* __restrict__ cell_q,
                                                                  uint32_t* __restrict__ start, i128* __restrict__ below) {
    __shared__ unsigned long long sn[kFitThreads];
    __shared__ i128 sq[kFitThreads];
    if (P->bad) return;
    const int p = blockIdx.x, tid = threadIdx.x;
    const unsigned long long* n = cell_n + (size_t)p * kFitCells + (size_t)tid * kFitOwn;
    const i128* q = cell_q + (size_t)p * kFitCells + (size_t)tid * kFitOwn;
    unsigned long long tn = 0;
    i128 tq = 0;
    for (int i = 0; i < kFitOwn; ++i) { tn += n[i]; tq += q[i]; }
    sn[tid] = tn; sq[tid] = tq;
    __syncthreads();
    for (int d = 1; d < kFitThreads; d <<= 1) {
        const unsigned long long an = tid >= d ? sn[tid - d] : 0;
        const i128 aq = tid >= d ? sq[tid - d] : (i128)0;
        __syncthreads();
        sn[tid] += an; sq[tid] += aq;
        __syncthreads();
    }
    unsigned long long en = sn[tid] - tn;
    i128 eq = sq[tid] - tq;
    uint32_t* st = start + (size_t)p * (kFitCells + 1);
    i128* be = below + (size_t)p * (kFitCells + 1);
    for (int i = 0; i < kFitOwn; ++i) {
        st[tid * kFitOwn + i] = (uint32_t)en;
        be[tid * kFitOwn + i] = eq;
        en += n[i]; eq += q[i];
    }
    if (tid == kFitThreads - 1) { st[kFitCells] = (uint32_t)en; be[kFitCells] = eq; }
}

__device__ __forceinline__ double i128_to_double(i128 q) {
    const bool neg = q < 0;
    const unsigned __int128 a = neg ? -(unsigned __int128)q : (unsigned __int128)q;      // below 2^71
    const double d = (double)(uint64_t)(a >> 32) * 4294967296.0 + (double)(uint32_t)a;   // one rounding
    return neg ? -d : d;
}

// All steps with the cells alone, one workgroup per problem: a boundary splits its cell in proportion to where it lies in
// it.  Writes which cells the boundaries touch (and their neighbours) as first positions in `sorted`; kFitAbsent:
// not among them.  Cells of few samples are all kept: they hold little, and nothing can be said about where in them
// a boundary will have its samples.  `everything`: all cells.
constexpr uint32_t kFitAbsent = 0xffffffffu;
constexpr int kFitMargin = 8;        // neighbours on either side that a visited cell takes along, as long as they hold few samples

// The kept samples of all problems lie one behind the other in one buffer of `capacity` samples.
__device__ __forceinline__ bool fit_room(const uint32_t* kept, int problems, size_t capacity) {
    return (size_t)kept[0] + (problems > 1 ? kept[1] : 0u) <= capacity;
}
__device__ __forceinline__ size_t fit_region(const uint32_t* kept, int p) { return p ? kept[0] : 0; }
__global__ __launch_bounds__(kFitThreads) void tq_fit_predict_kernel(const FitParams* __restrict__ P, int iterations,
                                                                     const uint32_t* __restrict__ start_all,
                                                                     const i128* __restrict__ below_all, FitCodebooks cb,
                                                                     const FitResult* __restrict__ state, int everything, uint32_t* __restrict__ place_all,
                                                                     uint32_t* __restrict__ kept) {
    __shared__ uint32_t start[kFitCells + 1];
    __shared__ float sum[kFitCells];                                  // of the samples below a cell; from the middle on, minus
                                                                      // those in and above it: small where the samples are few
    __shared__ uint8_t mark[kFitCells];
    __shared__ uint32_t scan[kFitThreads];
    if (P->bad) return;
    const int p = blockIdx.x, tid = threadIdx.x;
    const float scale = P->scale[p];
    const double unit = P->unit[p];
    for (int i = tid; i <= kFitCells; i += kFitThreads) {
        start[i] = start_all[(size_t)p * (kFitCells + 1) + i];
        if (i < kFitCells) {
            const i128* below = below_all + (size_t)p * (kFitCells + 1);
            sum[i] = (float)(i128_to_double(i < kFitHalf ? below[i] : below[i] - below[kFitCells]) * unit);
        }
    }
    __syncthreads();
    const uint32_t few = start[kFitCells] >> 16, near = start[kFitCells] >> 14;
    const bool done = state->steps[p] >= iterations;                  // (an earlier round finished this codebook)
    for (int i = tid; i < kFitCells; i += kFitThreads)
        mark[i] = !done && (everything || start[i + 1] - start[i] <= few) ? 1 : 0;
    __syncthreads();
    if (!everything && tid < kWave) {
        const int lane = tid, nc = cb.nc[p];
        float c = lane < nc ? state->cent[p][lane] : 0.0f;
        const float total = (float)(i128_to_double(below_all[(size_t)p * (kFitCells + 1) + kFitCells]) * unit);
        for (int iter = state->steps[p]; iter < iterations; ++iter) {
            const float next = __shfl(c, (lane + 1) & 63, kWave);
            uint32_t lo = start[kFitCells];                           // samples below boundary `lane`: lo + part
            float part = 0.0f, ls = 0.0f, side = 1.0f;                // their sum: ls + side * total
            if (lane < nc - 1) {
                const float b = (c + next) * 0.5f;
                uint32_t cell, off;
                fit_cell(b, scale, cell, off);
                mark[cell] = 2;                                       // (one of the few cells kept, or not)
                uint64_t base; int shift; bool neg;
                fit_cell_base(cell, base, shift, neg);
                const float width = (float)(shift ? 8192u << shift : 1u << 22);
                float f = (float)((unsigned long long)off << shift) / width;
                const float edge = (float)unit * (neg ? -((float)base + width) : (float)base);
                f = neg ? 1.0f - f : f;
                lo = start[cell];
                part = f * (float)(start[cell + 1] - lo);
                ls = sum[cell] + part * 0.5f * (edge + b);
                side = cell >= (uint32_t)kFitHalf ? 1.0f : 0.0f;
            }
            const uint32_t plo = (uint32_t)__shfl_up((int)lo, 1, kWave);
            const float pp = __shfl_up(part, 1, kWave), ps = __shfl_up(ls, 1, kWave), pside = __shfl_up(side, 1, kWave);
            const float bn = lane == 0 ? (float)lo + part : (float)(int)(lo - plo) + (part - pp);
            const float bsum = lane == 0 ? ls + side * total : (ls - ps) + (side - pside) * total;
            float move = 0.0f;
            if (lane < nc && bn > 0.0f) {
                const float nv = bsum / bn;
                move = fabsf(nv - c);
                c = nv;
            }
            if (__ballot(move >= 1e-7f) == 0) break;                  // (a maximum over the wave: six LDS latencies a step)
        }
    }
    __syncthreads();
    for (int i = 0; i < kFitOwn; ++i) {                               // visited cells take their neighbours along
        const int c = tid * kFitOwn + i;
        if (mark[c] != 2) continue;
        uint32_t acc = 0;
        for (int d = c + 1; d < kFitCells && d <= c + kFitMargin && acc <= near; ++d) {
            if (mark[d] == 0) mark[d] = 1;
            acc += start[d + 1] - start[d];
        }
        acc = 0;
        for (int d = c - 1; d >= 0 && d >= c - kFitMargin && acc <= near; --d) {
            if (mark[d] == 0) mark[d] = 1;
            acc += start[d + 1] - start[d];
        }
    }
    __syncthreads();
    uint32_t own = 0;
    for (int i = 0; i < kFitOwn; ++i) {
        const int c = tid * kFitOwn + i;
        own += mark[c] ? start[c + 1] - start[c] : 0u;
    }
    scan[tid] = own;
    __syncthreads();
    for (int d = 1; d < kFitThreads; d <<= 1) {
        const uint32_t a = tid >= d ? scan[tid - d] : 0u;
        __syncthreads();
        scan[tid] += a;
        __syncthreads();
    }
    uint32_t at = scan[tid] - own;
    for (int i = 0; i < kFitOwn; ++i) {
        const int c = tid * kFitOwn + i;
        place_all[(size_t)p * kFitCells + c] = mark[c] ? at : kFitAbsent;
        at += mark[c] ? start[c + 1] - start[c] : 0u;
    }
    if (tid == kFitThreads - 1) kept[p] = at;
}

// Samples of the kept cells written cell by cell; the position inside a cell is whatever the LDS counter hands out.  Bound
// by the stores: neighbouring lanes write to different lines (64 address cycles per wave store), which is why
// only cells that a boundary is expected to visit are written at all.
__global__ __launch_bounds__(kFitThreads) void tq_fit_scatter_kernel(FitProblem fp, const FitParams* __restrict__ P, size_t tile,
                                                                     const uint32_t* __restrict__ first,
                                                                     const uint32_t* __restrict__ place,
                                                                     const uint32_t* __restrict__ kept, size_t capacity,
                                                                     float* __restrict__ sorted) {
    __shared__ uint32_t pos[kFitCells];
    __shared__ uint32_t keep[kFitCells / 32];
    __shared__ FitResidual res;
    const int p = blockIdx.y;
    if (P->bad || kept[p] == 0 || !fit_room(kept, gridDim.y, capacity)) return;
    const uint32_t* fi = first + ((size_t)p * gridDim.x + blockIdx.x) * kFitCells;
    const uint32_t* pl = place + (size_t)p * kFitCells;
    for (int i = threadIdx.x; i < kFitCells; i += kFitThreads) {      // (kFitCells and kFitThreads: whole waves)
        const uint32_t at = pl[i];
        pos[i] = at + fi[i];
        const unsigned long long m = __ballot(at != kFitAbsent);
        if ((threadIdx.x & 31) == 0) keep[i >> 5] = (uint32_t)(m >> (threadIdx.x & 32));
    }
    if (fp.gtab[p]) fit_residual_build(res, fp.gtab[p], fp.ngc);
    __syncthreads();
    const float scale = P->scale[p];
    float* dst = sorted + fit_region(kept, p);
    const uint32_t n_kept = kept[p];
    auto put = [&](float v) {
        uint32_t cell, off;
        fit_cell(v, scale, cell, off);
        if ((keep[cell >> 5] >> (cell & 31u)) & 1u) {
            const uint32_t at = atomicAdd(&pos[cell], 1u);
            if (at < n_kept) dst[at] = v;
        }
    };
    if (fp.gtab[p]) {
        const float bs = res.bins.scale, bb = res.bins.bias;
        const int steps = res.bins.steps;
        fit_tile(fp.data, fp.n, tile, [&](float v) { put(v - res.cent[bin_find(res.bins, bs, bb, steps, fp.ngc - 1, v)]); });
    } else {
        fit_tile(fp.data, fp.n, tile, put);
    }
}

// Part of a cell by its offset: 64 parts.
constexpr int kFitParts = 64;
__device__ __forceinline__ uint32_t fit_part(uint32_t off, int shift) { return shift ? off >> 7 : off >> 16; }

// One workgroup per (cell, problem): its samples in the order of the parts, from `sorted` to `fine`, and the parts'
// first positions and offset sums.  A cell is a chain of latencies (its entries, its samples, the counters, its samples again),
// so four workgroups share a CU.  Cells of up to kRefineLds samples are put in order in LDS and written in whole lines: written
// where they belong one by one, every sample is a request to the L2 of its own, 20 M of them in 18944 x 3584 (138 us -> 115).
constexpr int kRefineThreads = 512, kRefineLds = 8192;
__global__ __launch_bounds__(kRefineThreads) void tq_fit_refine_kernel(const FitParams* __restrict__ P,
                                                                    const uint32_t* __restrict__ start_all,
                                                                    const uint32_t* __restrict__ place,
                                                                    const uint32_t* __restrict__ kept, size_t capacity,
                                                                    const float* __restrict__ sorted, float* __restrict__ fine,
                                                                    uint32_t* __restrict__ part_n,
                                                                    unsigned long long* __restrict__ part_o) {
    __shared__ unsigned long long both[kFitParts];                    // counts (upper 23 bits) and offset sums, as in the tiles
    __shared__ uint32_t pos[kFitParts];
    __shared__ float ordered[kRefineLds];
    const int p = blockIdx.y, cell = blockIdx.x, tid = threadIdx.x;
    if (P->bad || !fit_room(kept, gridDim.y, capacity)) return;
    const uint32_t at = place[(size_t)p * kFitCells + cell];
    if (at == kFitAbsent) return;
    const uint32_t* start = start_all + (size_t)p * (kFitCells + 1);
    const uint32_t n = start[cell + 1] - start[cell];
    const float scale = P->scale[p];
    const float* src = sorted + fit_region(kept, p) + at;
    float* dst = fine + fit_region(kept, p) + at;
    uint64_t base; int shift; bool neg;
    fit_cell_base((uint32_t)cell, base, shift, neg);
    const float whole = fit_cell_whole((uint32_t)cell);
    auto part_of = [&](float v, uint32_t& o) {
        o = shift ? fit_log_offset(v) : fit_linear_offset(v, scale, whole);
        return fit_part(o, shift);
    };
    uint32_t cnt = 0;                                                 // wave 0: of part `tid`
    unsigned long long off = 0;
    for (uint32_t lo = 0; lo == 0 || lo < n; lo += kFitMaxTile) {     // (more than one round only where a cell is that full)
        const uint32_t hi = lo + kFitMaxTile < n ? lo + kFitMaxTile : n;
        if (tid < kFitParts) both[tid] = 0;
        __syncthreads();
        for (uint32_t i = lo + tid; i < hi; i += 4 * kRefineThreads) {
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = src[i + j * kRefineThreads < hi ? i + j * kRefineThreads : i];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                uint32_t o;
                const uint32_t k = part_of(v[j], o);
                if (i + j * kRefineThreads < hi) atomicAdd(&both[k], (1ull << 41) | (unsigned long long)o);
            }
        }
        __syncthreads();
        if (tid < kFitParts) {
            cnt += (uint32_t)(both[tid] >> 41);
            off += both[tid] & ((1ull << 41) - 1);
        }
        __syncthreads();
    }
    if (tid < kWave) {
        uint32_t a = cnt;
        unsigned long long b = off;
        for (int d = 1; d < kWave; d <<= 1) {
            const uint32_t x = (uint32_t)__shfl_up((int)a, d, kWave);
            const unsigned long long y = (unsigned long long)__shfl_up((long long)b, d, kWave);
            if (tid >= d) { a += x; b += y; }
        }
        const size_t q = ((size_t)p * kFitCells + cell) * (kFitParts + 1);
        part_n[q + tid + 1] = a; part_o[q + tid + 1] = b;
        if (tid == 0) { part_n[q] = 0; part_o[q] = 0; }
        pos[tid] = a - cnt;
    }
    __syncthreads();
    const bool in_lds = n <= (uint32_t)kRefineLds;
    for (uint32_t i = tid; i < n; i += 4 * kRefineThreads) {
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = src[i + j * kRefineThreads < n ? i + j * kRefineThreads : i];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            uint32_t o;
            const uint32_t k = part_of(v[j], o);
            if (i + j * kRefineThreads < n) {
                const uint32_t to = atomicAdd(&pos[k], 1u);
                if (to >= n) continue;
                if (in_lds) ordered[to] = v[j];
                else dst[to] = v[j];
            }
        }
    }
    if (!in_lds) return;
    __syncthreads();
    for (uint32_t i = tid; i < n; i += kRefineThreads) dst[i] = ordered[i];
}

// All Lloyd-Max steps of one codebook (src/codebook.cpp:105-136): one workgroup, a wave per boundary.  out->missed[p]:
// a boundary came to a cell that was not kept; out->cent and out->steps say how far the fit has come.  A step is a chain
// of latencies (the cell's entries, its samples, the workgroup's sums).  The entries stay in the wave's registers, a part per
// lane, as long as the boundary stays in its cell; a sample's offset comes from its mantissa, the cell being known; no more
// rounds of 64 samples run than there are samples for (four waves share a SIMD: what a wave issues counts), and sums over a
// wave go through DPP operands, whether a centroid moved is a ballot: 3.0 us a step -> 2.5.
struct FitCut {                                       // a boundary's cell
    uint32_t cell, at, s0;
    i128 q0;                                          // of the samples below the cell
    uint32_t n_part, n_all;                           // lane l: samples and offset sums below part l; of all
    unsigned long long o_part, o_all;
    uint64_t base; int shift; bool neg;
};
__device__ __forceinline__ uint32_t wave_sum_u32(uint32_t v) {
    auto step = [&](auto other) { v += __builtin_bit_cast(uint32_t, other(__builtin_bit_cast(float, v))); };
    step([](float x) { return lane_xor<1>(x); });
    step([](float x) { return lane_xor<2>(x); });
    step([](float x) { return lane_xor<4>(x); });
    step([](float x) { return lane_xor<8>(x); });
    step([](float x) { return lane_xor<16>(x); });
    step([](float x) { return lane_xor<32>(x); });
    return v;
}
__device__ __forceinline__ unsigned long long lane_value(unsigned long long v, int l) {
    return (unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(v >> 32), l) << 32 |
           (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, l);
}
__global__ __launch_bounds__(kFitThreads) void tq_fit_iterate_kernel(const FitParams* __restrict__ P, size_t n, int iterations,
                                                                     const uint32_t* __restrict__ start_all,
                                                                     const i128* __restrict__ below_all,
                                                                     const uint32_t* __restrict__ place_all,
                                                                     const uint32_t* __restrict__ kept, size_t capacity,
                                                                     const float* __restrict__ fine_all,
                                                                     const uint32_t* __restrict__ part_n,
                                                                     const unsigned long long* __restrict__ part_o,
                                                                     FitCodebooks cb, FitResult* out) {
    __shared__ float cent[32];
    __shared__ unsigned long long left_n[33];
    __shared__ i128 left_q[33];
    __shared__ int stop, missed, coarse;
    const int p = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nc = cb.nc[p];
    const bool bad = P->bad != 0;
    if (tid == 0) {
        if (p == 0) out->bad = bad ? 1 : 0;
        out->kept[p] = bad ? 0 : kept[p];
        out->missed[p] = !bad && !fit_room(kept, gridDim.x, capacity) ? 1 : 0;
        out->coarse[p] = 0;
        stop = 0; missed = 0; coarse = 0;
    }
    if (bad || !fit_room(kept, gridDim.x, capacity)) return;
    if (tid < nc) cent[tid] = out->cent[p][tid];
    const float scale = P->scale[p];
    const double unit = P->unit[p];
    const uint32_t* start = start_all + (size_t)p * (kFitCells + 1);
    const i128* below = below_all + (size_t)p * (kFitCells + 1);
    const uint32_t* place = place_all + (size_t)p * kFitCells;
    const float* fine = fine_all + fit_region(kept, p);
    if (tid == 0) { left_n[0] = 0; left_q[0] = 0; left_n[nc] = n; left_q[nc] = below[kFitCells]; }
    __syncthreads();
    const unsigned long long cut_lo = start[kFitHalf - kFitCut], cut_hi = start[kFitHalf + kFitCut];
    int iter = out->steps[p];
    constexpr int kCuts = 2;                                          // boundaries of a wave: 31 of them, 16 waves
    FitCut cuts[kCuts];
#pragma unroll
    for (int u = 0; u < kCuts; ++u) cuts[u].cell = kFitAbsent;
    for (; iter < iterations; ++iter) {
#pragma unroll
        for (int u = 0; u < kCuts; ++u) {
            const int k = wave + u * (kFitThreads / kWave);
            if (k >= nc - 1) continue;
            FitCut& c = cuts[u];
            const float b = (cent[k] + cent[k + 1]) * 0.5f;
            uint32_t cell, boff;
            fit_cell(b, scale, cell, boff);
            cell = (uint32_t)__builtin_amdgcn_readfirstlane((int)cell);
            boff = (uint32_t)__builtin_amdgcn_readfirstlane((int)boff);
            if (cell != c.cell) {
                const size_t q = ((size_t)p * kFitCells + cell) * (kFitParts + 1);
                c.cell = cell;
                c.at = place[cell];
                c.s0 = start[cell];
                c.q0 = below[cell];
                c.n_part = part_n[q + lane];
                c.n_all = part_n[q + kFitParts];
                c.o_part = part_o[q + lane];
                c.o_all = part_o[q + kFitParts];
                fit_cell_base(cell, c.base, c.shift, c.neg);
            }
            if (c.at == kFitAbsent) { if (lane == 0) missed = 1; continue; }
            const int part = (int)fit_part(boff, c.shift);
            const uint32_t n0 = (uint32_t)__builtin_amdgcn_readlane((int)c.n_part, part);
            const uint32_t n1 = part + 1 < kFitParts ? (uint32_t)__builtin_amdgcn_readlane((int)c.n_part, (part + 1) & 63) : c.n_all;
            // larger magnitudes are smaller values below zero: the parts above are the ones to the left there
            uint32_t cnt = 0;
            unsigned long long off = 0;
            const float whole = fit_cell_whole(cell);
            for (uint32_t i = n0; i < n1; i += kWave * 8) {                               // eight loads at once: a step is a chain of latencies
                const float* src = fine + c.at + i;
                const uint32_t left = n1 - i;                                            // (no more rounds of 64 than samples fill)
                float v[8];
                uint32_t own = 0;                                                        // (8 offsets of 22 bits, 64 lanes: below 2^31)
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    if (j * kWave < left) v[j] = src[j * kWave + lane < left ? j * kWave + lane : 0];
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    if (j * kWave < left) {
                        const bool below_b = j * kWave + lane < left && !(b < v[j]);
                        const uint32_t o = c.shift ? fit_log_offset(v[j]) : fit_linear_offset(v[j], scale, whole);
                        cnt += (uint32_t)__popcll(__ballot(below_b));
                        own += below_b ? o : 0u;
                    }
                off += wave_sum_u32(own);
            }
            if (c.neg) {
                cnt += c.n_all - n1;
                off += c.o_all - (part + 1 < kFitParts ? lane_value(c.o_part, (part + 1) & 63) : c.o_all);
            } else {
                cnt += n0;
                off += lane_value(c.o_part, part);
            }
            if (lane == 0) {
                const i128 t = (i128)cnt * (i128)c.base + ((i128)off << c.shift);
                left_n[k + 1] = c.s0 + (unsigned long long)cnt;
                left_q[k + 1] = c.q0 + (c.neg ? -t : t);
            }
        }
        __syncthreads();
        if (missed) break;
        if (wave == 0) {
            float shift = 0.0f;
            if (lane < nc) {
                const unsigned long long c = left_n[lane + 1] - left_n[lane];
                if (c > 0) {                                                         // src/codebook.cpp:124-129
                    const double s = i128_to_double(left_q[lane + 1] - left_q[lane]) * unit;
                    const float nv = (float)(s / (double)c);
                    shift = fabsf(nv - cent[lane]);
                    cent[lane] = nv;
                }
            }
            const bool moves = __ballot(shift >= 1e-6f) != 0;                        // src/codebook.cpp:132
            if (lane == 0) stop = moves ? 0 : 1;
        } else if (wave == 1 && lane < nc) {
            // each of a bin's samples around zero may have lost up to one unit; the centroid again, beside wave 0
            const unsigned long long from = max(left_n[lane], cut_lo), to = min(left_n[lane + 1], cut_hi);
            if (from < to && (double)(to - from) > fabs(i128_to_double(left_q[lane + 1] - left_q[lane])) * 0x1p-26) coarse = 1;
        }
        __syncthreads();
        if (stop || coarse) break;
    }
    if (tid == 0) {
        out->missed[p] = missed;
        out->coarse[p] = coarse;
        out->steps[p] = stop ? iterations : iter;
    }
    if (tid < nc) out->cent[p][tid] = cent[tid];
}

// ---------------------------------------------------------------------------
static size_t fit_align(size_t b) { return (b + 255) & ~(size_t)255; }

// Tiles: 16384 samples or more each, one tile per CU until they reach 2^19 samples, then rounds of 256.
static size_t fit_tiles(size_t n) {
    const size_t per_cu = (n + 256 * (size_t)kFitMaxTile - 1) / (256 * (size_t)kFitMaxTile);
    const size_t small = (n + 16383) / 16384;
    return small < 256 ? (small < 1 ? 1 : small) : 256 * per_cu;
}

// Samples the kept cells may hold.  `everything`: all.  Otherwise half of them: on normally distributed weights the 4-bit
// codebook's boundaries visit 1 % of the samples and the residual's, which start from a far too wide codebook, a quarter.
static size_t fit_capacity(size_t n, int problems, bool everything) { return everything ? problems * n : n / 2; }

// (positions and counters of 32 bits: tq_fit_refine_kernel walks a cell in strides of kFitMaxTile samples, and a cell may
// hold all of them)
bool fit_supported(size_t n) { return n >= 1 && n < ((size_t)1 << 32) - 2 * (size_t)kFitMaxTile; }
bool fit_predicts(size_t n) { return n >= ((size_t)1 << 22); }

size_t fit_workspace_bytes(size_t n, int problems, bool everything) {
    const size_t cells = (size_t)problems * fit_tiles(n) * kFitCells, pc = (size_t)problems * kFitCells;
    return fit_align(4096) + fit_align(sizeof(FitParams)) + fit_align(cells * 8) + fit_align(cells * 4) +
           fit_align(pc * 8) + fit_align(pc * 16) + fit_align((pc + problems) * 4) + fit_align((pc + problems) * 16) +
           fit_align(pc * 4) + fit_align(8) + fit_align(pc * (kFitParts + 1) * 4) + fit_align(pc * (kFitParts + 1) * 8) +
           2 * fit_align(fit_capacity(n, problems, everything) * 4);
}

hipError_t launch_fit(const float* samples, size_t n, int problems, const float* gtab_dev, int ngc, const FitCodebooks& cb,
                      int iterations, bool first_round, bool everything, void* workspace, FitResult* state, hipStream_t stream) {
    if (!fit_supported(n) || problems < 1 || problems > 2) return hipErrorInvalidValue;
    const size_t tiles = fit_tiles(n);
    const size_t tile = (((n + tiles - 1) / tiles) + 3) & ~(size_t)3;
    if (tile > (size_t)kFitMaxTile) return hipErrorInvalidValue;
    const size_t cells = (size_t)problems * tiles * kFitCells, pc = (size_t)problems * kFitCells;
    const size_t cap = fit_capacity(n, problems, everything);
    unsigned char* w = static_cast<unsigned char*>(workspace);
    auto take = [&](size_t bytes) { void* p = w; w += fit_align(bytes); return p; };
    uint32_t* part = static_cast<uint32_t*>(take(4096));
    FitParams* P = static_cast<FitParams*>(take(sizeof(FitParams)));
    unsigned long long* hist = static_cast<unsigned long long*>(take(cells * 8));
    uint32_t* first = static_cast<uint32_t*>(take(cells * 4));
    unsigned long long* cell_n = static_cast<unsigned long long*>(take(pc * 8));
    i128* cell_q = static_cast<i128*>(take(pc * 16));
    uint32_t* start = static_cast<uint32_t*>(take((pc + problems) * 4));
    i128* below = static_cast<i128*>(take((pc + problems) * 16));
    uint32_t* place = static_cast<uint32_t*>(take(pc * 4));
    uint32_t* kept = static_cast<uint32_t*>(take(8));
    uint32_t* part_n = static_cast<uint32_t*>(take(pc * (kFitParts + 1) * 4));
    unsigned long long* part_o = static_cast<unsigned long long*>(take(pc * (kFitParts + 1) * 8));
    float* sorted = static_cast<float*>(take(cap * 4));
    float* fine = static_cast<float*>(take(cap * 4));

    FitProblem fp{};
    fp.data = samples; fp.n = n; fp.ngc = ngc;
    fp.gtab[0] = nullptr; fp.gtab[1] = gtab_dev;                    // problem 0: the samples; problem 1: their residuals
    const dim3 grid((unsigned)tiles, (unsigned)problems);
    if (first_round) {
        const unsigned parts = (unsigned)(n / 16384 < 1 ? 1 : (n / 16384 > 1024 ? 1024 : n / 16384));
        if (!cb.absmax) hipLaunchKernelGGL(tq_fit_absmax_kernel, dim3(parts), dim3(256), 0, stream, samples, n, part);
        hipLaunchKernelGGL(tq_fit_absmax_fold_kernel, dim3(1), dim3(256), 0, stream, cb.absmax ? cb.absmax : part,
                           cb.absmax ? cb.absmax_parts : (int)parts, fp, problems, P, cb, state);
        hipLaunchKernelGGL(tq_fit_hist_kernel, grid, dim3(kFitThreads), 0, stream, fp, P, tile, hist);
        hipLaunchKernelGGL(tq_fit_offsets_kernel, dim3(kFitCells / 256, problems), dim3(256), 0, stream, P, (int)tiles, hist, first,
                           cell_n, cell_q);
        hipLaunchKernelGGL(tq_fit_scan_kernel, dim3(problems), dim3(kFitThreads), 0, stream, P, cell_n, cell_q, start, below);
    }
    hipLaunchKernelGGL(tq_fit_predict_kernel, dim3(problems), dim3(kFitThreads), 0, stream, P, iterations, start, below, cb,
                       state, everything ? 1 : 0, place, kept);
    hipLaunchKernelGGL(tq_fit_scatter_kernel, grid, dim3(kFitThreads), 0, stream, fp, P, tile, first, place, kept, cap, sorted);
    hipLaunchKernelGGL(tq_fit_refine_kernel, dim3(kFitCells, problems), dim3(kRefineThreads), 0, stream, P, start, place, kept, cap, sorted,
                       fine, part_n, part_o);
    hipLaunchKernelGGL(tq_fit_iterate_kernel, dim3(problems), dim3(kFitThreads), 0, stream, P, n, iterations, start, below, place,
                       kept, cap, fine, part_n, part_o, cb, state);
    return hipGetLastError();
}

}  // namespace tq
