// full_chunks.hip -- the full pair histogram over spatially sorted chunks of 64
// atoms.
//
// Most pairs of a box are out of the histogram's range, and a pair whose
// distance is known to be out of range need not be evaluated.  The atoms are
// sorted into columns along the third cell axis and along it within each
// column; 64 consecutive atoms are a chunk, one per lane of a wave.  A wave
// holds one chunk as rows, tests the bounding boxes of 64 other chunks at once
// against its own, then the 64 atoms of each surviving chunk against its own
// box, and evaluates its rows against the surviving atoms only.
//
// What bounds it: the float32 arithmetic of the evaluated pairs.  Chunks of 64
// atoms keep the evaluated pairs near 2.5 times the pairs in range at 20 A and
// 0.066 atoms/A^3 (a cell list with cells of the range evaluates 7 times, whole
// tiles of chunks 5 times).  The bin of a pair comes from the hardware's
// approximate square root and one multiplication when it is farther from a
// bin edge than their error bound; the rest (about one in a thousand) go to
// a queue that a full wave evaluates exactly.
//
// Measured (MI355X, whole calls): 200,000 atoms, 2 elements, 2,000 bins: 648 us
// against 3,260 with the cell list this replaced; 13,500 atoms in 45 x 45 x 90 A,
// 1,000 bins: 99 us against 312 (all pairs); the binary64 recompute of 40,000
// atoms in a triclinic cell: 249 us against 3,000 (all pairs); 1,000 atoms: 52
// us against 160.  Of the 648 us, 633 are the pair loop: 5.5e8 pairs for the
// 2.2e8 in range, about 40 vector instructions each, at 180 cycles per wave
// and listed atom of a SIMD.  Reading the next four atoms ahead measured no
// faster (664 us).
#include <math.h>
#include <stddef.h>

#include <algorithm>
#include <type_traits>

#include "chunks.h"
#include "full_hist.h"

namespace frmc {

namespace {

constexpr int kListPad = 4;         // a list is padded to the unrolled loop's step
constexpr int kQueue = 128;         // queued pairs per wave: drained from 64 on
constexpr int kWaveLds = (64 + kListPad) * 32 + kQueue * 4;
constexpr int32_t kSelfKey = 1 << 30;

struct FastBin {
    float inv;            // 1 / bin
    float half;           // 0.5 - error bound of the approximate bin, or below 0: every pair is queued
    float thi;            // bins below it are inside the range and the row of H bins
    float tie;            // binary64 mode: largest |b| whose image is certain
};

__device__ void make_plan(const float *__restrict__ dbasis, const Basis &hB, int isPBC, int32_t n, ChunkPlan &P) {
    double b[9], h[3] = {1.0, 1.0, 1.0};
    for (int q = 0; q < 9; q++) {
        P.B.b[q] = !isPBC ? 0.0f : dbasis ? load_dev(dbasis + q) : hB.b[q];
        b[q] = P.B.b[q];
    }
    P.ortho = P.B.b[1] == 0.f && P.B.b[2] == 0.f && P.B.b[3] == 0.f && P.B.b[5] == 0.f && P.B.b[6] == 0.f &&
              P.B.b[7] == 0.f;
    P.C = ChunkCut{1.f, 0.f, 1.f, 0.f, 0.f, 1.f, 1.f};
    if (isPBC) {
        const double vol = fabs(b[0] * (b[4] * b[8] - b[5] * b[7]) - b[1] * (b[3] * b[8] - b[5] * b[6]) +
                                b[2] * (b[3] * b[7] - b[4] * b[6]));
        double g[3][3], rows = 0.0;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const double *u = b + 3 * ((i + 1) % 3), *v = b + 3 * ((i + 2) % 3);
            const double cx = u[1] * v[2] - u[2] * v[1], cy = u[2] * v[0] - u[0] * v[2],
                         cz = u[0] * v[1] - u[1] * v[0];
            h[i] = vol / sqrt(cx * cx + cy * cy + cz * cz);  // spacing of the planes across axis i
#pragma unroll
            for (int j = 0; j < 3; j++) {
                rows += fabs(b[3 * i + j]);
                g[i][j] = b[3 * i] * b[3 * j] + b[3 * i + 1] * b[3 * j + 1] + b[3 * i + 2] * b[3 * j + 2];
            }
        }
        // the Cholesky factor; a vanishing pivot ends it (fewer rows only lower the bound)
        const double tiny = 1e-9 * (g[0][0] + g[1][1] + g[2][2]);
        double L0 = 0, L1 = 0, L2 = 0, L3 = 0, L4 = 0, L5 = 0;
        if (g[0][0] > tiny) {
            L0 = sqrt(g[0][0]);
            L1 = g[1][0] / L0;
            L3 = g[2][0] / L0;
            const double p1 = g[1][1] - L1 * L1;
            if (p1 > tiny) {
                L2 = sqrt(p1);
                L4 = (g[2][1] - L3 * L1) / L2;
                const double p2 = g[2][2] - L3 * L3 - L4 * L4;
                if (p2 > tiny) L5 = sqrt(p2);
            }
        }
        P.C = ChunkCut{(float)L0, (float)L1, (float)L2, (float)L3, (float)L4, (float)L5, (float)rows};
    }
    P.m0 = P.m1 = 1;
    const double s = cbrt(h[0] * h[1] * h[2] * 64.0 / (n > 1 ? n : 1));
    const double f0 = h[0] / s, f1 = h[1] / s;
    if (f0 > 0.0 && f1 > 0.0 && f0 < 1e6 && f1 < 1e6) {
        P.m0 = max(1, (int32_t)(f0 + 0.5));
        P.m1 = max(1, (int32_t)(f1 + 0.5));
        while ((int64_t)P.m0 * P.m1 > columns_most(n)) {
            if (P.m0 >= P.m1) P.m0 = max(1, P.m0 * 3 / 4);
            else P.m1 = max(1, P.m1 * 3 / 4);
        }
    }
}

// zeroes the scratch header, the sort's counters and (if own) the counts, and makes the plan
__global__ void __launch_bounds__(256) k_chunk_setup(const float *__restrict__ dbasis, Basis hB, int isPBC, int32_t n,
                                                     uint32_t *__restrict__ meta, int32_t *__restrict__ cellcnt,
                                                     int64_t cells, int32_t *__restrict__ counts, int64_t ncounts) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x, stride = (int64_t)gridDim.x * 256;
    for (int64_t i = t; i < M_WORDS; i += stride)
        if (i < M_PLAN || i >= M_SUM) meta[i] = 0;
    for (int64_t i = t; i < cells; i += stride) cellcnt[i] = 0;
    for (int64_t i = t; i < ncounts; i += stride) counts[i] = 0;
    if (t == 0) {
        ChunkPlan P;
        make_plan(dbasis, hB, isPBC, n, P);
        uint32_t w[kPlanWords];
        __builtin_memcpy(w, &P, sizeof(P));
#pragma unroll
        for (int k = 0; k < kPlanWords; k++) meta[M_PLAN + k] = w[k];
    }
}

// Open boundaries: the sort's cells cover mean +- 1.8 standard deviations along
// each axis, within the extent (a uniform box entirely, at 1.74); atoms past
// them fall into the cells at the ends.  Over the extent alone one atom far away puts
// all others into one cell: 50,000 atoms and one at a thousand times their extent
// 1,312 us a call against 436 (874 for all pairs).
struct Window {
    float from, wide;
};
__device__ Window sort_window(float lo, float hi, double sum, double squares, int32_t n) {
    const double mean = sum / n, d = 1.8 * sqrt(fmax(squares / n - mean * mean, 0.0));
    const float a = fmaxf(lo, (float)(mean - d)), b = fminf(hi, (float)(mean + d));
    return b > a ? Window{a, b - a} : Window{lo, hi - lo};
}

__device__ __forceinline__ void add_finite(float x, double &sum, double &squares) {
    const double v = fabsf(x) < 1e30f ? x : 0.0;
    sum += v;
    squares += v * v;
}

// open boundaries: the coordinates' extent (maxima of the ordered bits and of their
// complements), and the sums of the sort's window
__global__ void __launch_bounds__(256) k_chunk_extent(const float *__restrict__ coords, int32_t n,
                                                      uint32_t *__restrict__ meta) {
    __shared__ uint32_t ext[6];
    __shared__ double sums[6];
    if (threadIdx.x < 6) {
        ext[threadIdx.x] = 0;
        sums[threadIdx.x] = 0.0;
    }
    __syncthreads();
    uint32_t hi[3] = {0, 0, 0}, lo[3] = {0, 0, 0};
    double sum[3] = {0.0, 0.0, 0.0}, squares[3] = {0.0, 0.0, 0.0};
    for (int32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256)
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const float x = coords[3 * (int64_t)i + k];
            const uint32_t u = ordered_bits(x);
            hi[k] = max(hi[k], u);
            lo[k] = max(lo[k], ~u);
            add_finite(x, sum[k], squares[k]);
        }
#pragma unroll
    for (int k = 0; k < 3; k++) {
        for (int o = 32; o > 0; o >>= 1) {
            hi[k] = max(hi[k], (uint32_t)__shfl_xor((int)hi[k], o));
            lo[k] = max(lo[k], (uint32_t)__shfl_xor((int)lo[k], o));
            sum[k] += __shfl_xor(sum[k], o);
            squares[k] += __shfl_xor(squares[k], o);
        }
        if ((threadIdx.x & 63) == 0) {
            atomicMax(&ext[k], lo[k]);
            atomicMax(&ext[3 + k], hi[k]);
            atomicAdd(&sums[k], sum[k]);
            atomicAdd(&sums[3 + k], squares[k]);
        }
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        atomicMax(&meta[M_LO + threadIdx.x], ext[threadIdx.x]);
        atomicAdd(reinterpret_cast<double *>(meta + M_SUM) + threadIdx.x, sums[threadIdx.x]);
    }
}

// fraction of coordinate x along an axis, in [0, 1] where a window covers it
template <bool PBC>
__device__ __forceinline__ float sort_fraction(float x, const Window &W) {
    if (PBC) return x - floorf(x);
    return W.wide > 0.0f ? (x - W.from) / W.wide : 0.0f;
}

// counting-sort cell of a position's fractions: its column, then its bin along the column
__device__ __forceinline__ int32_t cell_of(float f0, float f1, float fz, int32_t m0, int32_t m1) {
    const int32_t c0 = max(0, min(m0 - 1, (int32_t)(f0 * (float)m0))), c1 = max(0, min(m1 - 1, (int32_t)(f1 * (float)m1)));
    return (c0 * m1 + c1) * kNZ + max(0, min(kNZ - 1, (int32_t)(fz * (float)kNZ)));
}

// counting-sort cell of every atom, its rank there, and the largest |coordinate|
template <bool PBC>
__global__ void __launch_bounds__(256) k_chunk_count(const float *__restrict__ coords, int32_t n,
                                                     uint32_t *__restrict__ meta, int32_t *__restrict__ cellcnt,
                                                     int2 *__restrict__ where) {
    const int32_t i = blockIdx.x * 256 + threadIdx.x;
    const int32_t m0 = (int32_t)load_dev(meta + M_PLAN + offsetof(ChunkPlan, m0) / 4),
                  m1 = (int32_t)load_dev(meta + M_PLAN + offsetof(ChunkPlan, m1) / 4);
    __shared__ Window W[3];
    if (!PBC) {
        const int k = threadIdx.x;
        const double *sums = reinterpret_cast<const double *>(meta + M_SUM);
        if (k < 3)
            W[k] = sort_window(from_ordered(~load_dev(meta + M_LO + k)), from_ordered(load_dev(meta + M_HI + k)),
                               load_dev(sums + k), load_dev(sums + 3 + k), n);
        __syncthreads();
    }
    float a = 0.0f;
    if (i < n) {
        const float x = coords[3 * (int64_t)i], y = coords[3 * (int64_t)i + 1], z = coords[3 * (int64_t)i + 2];
        if (PBC) a = fmaxf(fmaxf(abs_or_inf(x), abs_or_inf(y)), abs_or_inf(z));
        const int32_t cell = cell_of(sort_fraction<PBC>(x, W[0]), sort_fraction<PBC>(y, W[1]),
                                     sort_fraction<PBC>(z, W[2]), m0, m1);
        where[i] = make_int2(cell, atomicAdd(&cellcnt[cell], 1));
    }
    if (!PBC) return;  // the extent gives it
    // boxes within [-1, 1], the usual ones, need no atomics: cut_squared takes at least 1
    __shared__ float wmax[4];
    for (int o = 32; o > 0; o >>= 1) a = fmaxf(a, __shfl_xor(a, o));
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = a;
    __syncthreads();
    a = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
    if (threadIdx.x == 0 && a > 1.0f && __float_as_uint(a) > load_dev(meta + M_AMAX))
        atomicMax(&meta[M_AMAX], __float_as_uint(a));
}

__device__ __forceinline__ int32_t wave_scan(int32_t v, int lane) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int32_t u = __shfl_up(v, o);
        if (lane >= o) v += u;
    }
    return v;
}

// One workgroup: cells' starts within their column, columns' starts (each a
// multiple of 64), the number of chunks, and the columns' padding atoms (NaN
// coordinates: never in range; id -1).
__global__ void __launch_bounds__(1024) k_chunk_scan(const int2 *__restrict__ cellcnt,
                                                     int2 *__restrict__ cellstart, int32_t *__restrict__ coltot,
                                                     int32_t *__restrict__ colbase, uint32_t *__restrict__ meta,
                                                     float4 *__restrict__ sx, int32_t *__restrict__ smol) {
    __shared__ int32_t wsum[16];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int32_t ncol = (int32_t)(load_dev(meta + M_PLAN + offsetof(ChunkPlan, m0) / 4) *
                                   load_dev(meta + M_PLAN + offsetof(ChunkPlan, m1) / 4));
    for (int32_t c = wave; c < ncol; c += 16) {
        const int2 v = cellcnt[c * 64 + lane];
        const int32_t s = v.x + v.y, incl = wave_scan(s, lane);
        cellstart[c * 64 + lane] = make_int2(incl - s, incl - v.y);
        if (lane == 63) coltot[c] = incl;
    }
    __syncthreads();
    int32_t carry = 0;
    for (int32_t base = 0; base < ncol; base += 1024) {
        const int32_t c = base + tid;
        const int32_t t = c < ncol ? coltot[c] : 0, p = (t + 63) & ~63;
        const int32_t incl = wave_scan(p, lane);
        if (lane == 63) wsum[wave] = incl;
        __syncthreads();
        int32_t before = 0, total = 0;
        for (int w = 0; w < 16; w++) {
            const int32_t v = wsum[w];
            before += w < wave ? v : 0;
            total += v;
        }
        const int32_t start = carry + before + incl - p;
        if (c < ncol) {
            colbase[c] = start;
            for (int32_t j = t; j < p; j++) {
                const float nan = __uint_as_float(0x7fc00000u);
                sx[start + j] = make_float4(nan, nan, nan, __int_as_float(-1));
                smol[start + j] = -1;
            }
        }
        carry += total;
        __syncthreads();
    }
    if (tid == 0) meta[M_NCHUNK] = (uint32_t)(carry / 64);
}

// id * 64 + element; an element outside the arrays, which the callers exclude, stays inside the bins
__device__ __forceinline__ int32_t packed_id(int32_t i, int32_t e, int32_t nel) {
    return i * 64 + max(0, min(nel - 1, e));
}

// sorted copies: (x, y, z, id * 64 + element), molecule
__global__ void __launch_bounds__(256) k_chunk_scatter(const float *__restrict__ coords, int32_t n,
                                                       const int32_t *__restrict__ mol,
                                                       const int32_t *__restrict__ elem, int32_t nel,
                                                       const int2 *__restrict__ where,
                                                       const int32_t *__restrict__ cellstart,
                                                       const int32_t *__restrict__ colbase,
                                                       float4 *__restrict__ sx, int32_t *__restrict__ smol) {
    const int32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int2 w = where[i];
    const int32_t pos = colbase[w.x / kNZ] + cellstart[w.x] + w.y;
    sx[pos] = make_float4(coords[3 * (int64_t)i], coords[3 * (int64_t)i + 1], coords[3 * (int64_t)i + 2],
                          __int_as_float(packed_id(i, elem[i], nel)));
    smol[pos] = mol[i];
}

// The setup, count, scan and scatter of up to kSmallSort atoms in one workgroup,
// the cells' counters in LDS: four launches less, which is most of a small
// call's time: 1,000 atoms in 52 us against 62, 4,000 in 64 against 67; at 13,500
// the one workgroup would take longer than the launches it saves.
constexpr int32_t kSmallSort = 4096;
// Words of counts that the one workgroup clears besides; beyond, the launches that
// clear with the whole chip: 1,000 atoms of 64 elements, 1,000 bins (8.2 million words)
// 114 us a call against 540, of 20 elements, 2,000 bins 97 against 167.
constexpr int64_t kSmallClear = 1 << 16;

template <bool PBC>
__global__ void __launch_bounds__(1024) k_chunk_sort_small(const float *__restrict__ dbasis, Basis hB,
                                                           const float *__restrict__ coords, int32_t n,
                                                           const int32_t *__restrict__ mol,
                                                           const int32_t *__restrict__ elem, int32_t nel,
                                                           uint32_t *__restrict__ meta, int2 *__restrict__ where,
                                                           float4 *__restrict__ sx, int32_t *__restrict__ smol,
                                                           int32_t *__restrict__ counts, int64_t ncounts) {
    constexpr int kCols = kSmallSort / 96 + 1;
    __shared__ __align__(8) int32_t cell[kCols * kNZ];  // read as pairs below
    __shared__ int32_t tot[kCols], base[kCols];
    __shared__ uint32_t amax, ext[6];
    __shared__ ChunkPlan P;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    for (int32_t i = tid; i < kCols * kNZ; i += 1024) cell[i] = 0;
    for (int64_t i = tid; i < ncounts; i += 1024) counts[i] = 0;
    if (tid < 6) ext[tid] = 0;
    if (tid == 64) amax = 0;
    if (tid == 128) make_plan(dbasis, hB, PBC, n, P);
    __syncthreads();
    // the largest |coordinate|, or the extent
    uint32_t hi[3] = {0, 0, 0}, lo[3] = {0, 0, 0};
    float a = 0.0f;
    for (int32_t i = tid; i < n; i += 1024)
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const float x = coords[3 * i + k];
            if (PBC) {
                a = fmaxf(a, abs_or_inf(x));
            } else {
                const uint32_t u = ordered_bits(x);
                hi[k] = max(hi[k], u);
                lo[k] = max(lo[k], ~u);
            }
        }
    if (PBC) {
        for (int o = 32; o > 0; o >>= 1) a = fmaxf(a, __shfl_xor(a, o));
        if (lane == 0) atomicMax(&amax, __float_as_uint(a));
    } else {
#pragma unroll
        for (int k = 0; k < 3; k++) {
            for (int o = 32; o > 0; o >>= 1) {
                hi[k] = max(hi[k], (uint32_t)__shfl_xor((int)hi[k], o));
                lo[k] = max(lo[k], (uint32_t)__shfl_xor((int)lo[k], o));
            }
            if (lane == 0) {
                atomicMax(&ext[k], lo[k]);
                atomicMax(&ext[3 + k], hi[k]);
            }
        }
    }
    __syncthreads();
    if (tid < M_WORDS - M_PAIRS) meta[M_PAIRS + tid] = 0;
    if (tid < M_PLAN) {
        uint32_t v = 0;
        if (tid == M_AMAX) v = amax;
        if (!PBC && tid >= M_LO && tid < M_LO + 6) v = ext[tid - M_LO];
        meta[tid] = v;
    }
    if (tid >= 64 && tid < 64 + kPlanWords) {
        uint32_t w;
        __builtin_memcpy(&w, reinterpret_cast<const char *>(&P) + 4 * (tid - 64), 4);
        meta[M_PLAN + tid - 64] = w;
    }
    const int32_t m0 = P.m0, m1 = P.m1, ncol = m0 * m1;
    // (over the extent: the sums of the large sort's window would cost 5 us more than they save here)
    Window W[3] = {{0.f, 1.f}, {0.f, 1.f}, {0.f, 1.f}};
    if (!PBC)
#pragma unroll
        for (int k = 0; k < 3; k++) {
            W[k].from = from_ordered(~ext[k]);
            W[k].wide = from_ordered(ext[3 + k]) - W[k].from;
        }
    auto frac = [&](float x, int k) { return sort_fraction<PBC>(x, W[k]); };
    for (int32_t i = tid; i < n; i += 1024) {
        const int32_t c = cell_of(frac(coords[3 * i], 0), frac(coords[3 * i + 1], 1), frac(coords[3 * i + 2], 2), m0, m1);
        where[i] = make_int2(c, atomicAdd(&cell[c], 1));
    }
    __syncthreads();
    for (int32_t c = wave; c < ncol; c += 16) {
        int2 *v = reinterpret_cast<int2 *>(cell) + c * 64 + lane;
        const int2 n2 = *v;
        const int32_t sum = n2.x + n2.y, incl = wave_scan(sum, lane);
        *v = make_int2(incl - sum, incl - n2.y);
        if (lane == 63) tot[c] = incl;
    }
    __syncthreads();
    if (wave == 0) {  // at most 64 columns
        const int32_t t = lane < ncol ? tot[lane] : 0, p = (t + 63) & ~63, incl = wave_scan(p, lane);
        if (lane < ncol) base[lane] = incl - p;
        if (lane == 63) meta[M_NCHUNK] = (uint32_t)(incl / 64);
    }
    __syncthreads();
    for (int32_t c = wave; c < ncol; c += 16) {
        const int32_t j = tot[c] + lane;
        if (j < ((tot[c] + 63) & ~63)) {
            const float nan = __uint_as_float(0x7fc00000u);
            sx[base[c] + j] = make_float4(nan, nan, nan, __int_as_float(-1));
            smol[base[c] + j] = -1;
        }
    }
    for (int32_t i = tid; i < n; i += 1024) {
        const int2 w = where[i];
        const int32_t pos = base[w.x / kNZ] + cell[w.x] + w.y;
        sx[pos] = make_float4(coords[3 * i], coords[3 * i + 1], coords[3 * i + 2],
                              __int_as_float(packed_id(i, elem[i], nel)));
        smol[pos] = mol[i];
    }
}

// Box of every chunk's atoms, kBox float4 each: centre and half-width (of
// wrapped fractions when periodic), then the coordinates' own ends.
template <bool PBC>
__global__ void __launch_bounds__(256) k_chunk_boxes(const float4 *__restrict__ sx,
                                                     const uint32_t *__restrict__ meta,
                                                     float4 *__restrict__ cbox) {
    const int32_t c = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (c >= (int32_t)load_dev(meta + M_NCHUNK)) return;
    const float4 v = sx[(int64_t)c * 64 + lane];
    const float p[3] = {v.x, v.y, v.z};
    const float inf = __uint_as_float(0x7f800000u);
    float mid[3], half[3], from[3], to[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        float lo = p[k] == p[k] ? p[k] : inf, hi = p[k] == p[k] ? p[k] : -inf;
        const float f = PBC ? p[k] - floorf(p[k]) : p[k];
        float flo = f == f ? f : inf, fhi = f == f ? f : -inf;
        for (int o = 32; o > 0; o >>= 1) {
            lo = fminf(lo, __shfl_xor(lo, o));
            hi = fmaxf(hi, __shfl_xor(hi, o));
            flo = fminf(flo, __shfl_xor(flo, o));
            fhi = fmaxf(fhi, __shfl_xor(fhi, o));
        }
        from[k] = lo;
        to[k] = hi;
        mid[k] = 0.5f * (flo + fhi);
        half[k] = 0.5f * (fhi - flo);
    }
    if (lane == 0) {
        float4 *b = cbox + kBox * (int64_t)c;
        b[0] = make_float4(mid[0], mid[1], mid[2], 0.0f);
        b[1] = make_float4(half[0], half[1], half[2], 0.0f);
        b[2] = make_float4(from[0], from[1], from[2], 0.0f);
        b[3] = make_float4(to[0], to[1], to[2], 0.0f);
    }
}

struct ChunkArgs {
    const float4 *sx;
    const int32_t *smol;
    const float4 *cbox;
    uint32_t *meta;
    int32_t nsub;         // items per row chunk
    float range;          // end of the histogram's range
    HistArgs A;
    FastBin F;
    int32_t lds_intra;    // bins in LDS: both halves, or the inter-molecular one
    int32_t count_pairs;
    int32_t *partial, *counts;
};

template <bool PBC, bool ORTHO, bool LDS_HIST, bool EDGE>
__device__ __forceinline__ void full_chunks(const ChunkArgs &K, const Basis &B, const ChunkCut &C, const Edge64 &E) {
    const float4 *__restrict__ sx = K.sx, *__restrict__ cbox = K.cbox;
    const int32_t *__restrict__ smol = K.smol;
    uint32_t *__restrict__ meta = K.meta;
    const HistArgs &A = K.A;
    const FastBin &F = K.F;
    const int32_t lds_intra = K.lds_intra;
    int32_t *__restrict__ counts = K.counts;
    extern __shared__ float4 lds4[];
    __shared__ int32_t next;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nwave = blockDim.x >> 6;
    char *mine = reinterpret_cast<char *>(lds4) + wave * kWaveLds;
    float4 *lxyz = reinterpret_cast<float4 *>(mine);
    int4 *linfo = reinterpret_cast<int4 *>(mine + (64 + kListPad) * 16);
    uint32_t *queue = reinterpret_cast<uint32_t *>(mine + (64 + kListPad) * 32);
    int32_t *hist = reinterpret_cast<int32_t *>(reinterpret_cast<char *>(lds4) + nwave * kWaveLds);
    const int32_t size = (int32_t)A.size, H = A.g.H, nel = A.nel;
    const int32_t nbins = LDS_HIST ? (lds_intra ? 2 * size : size) : 0;  // inter-molecular bins first
    for (int32_t s = tid; s < nbins; s += blockDim.x) hist[s] = 0;
    if (tid == 0) next = 0;
    __syncthreads();

    const int32_t N = (int32_t)load_dev(meta + M_NCHUNK);
    const float cut2 = cut_squared(C, K.range, coord_max<PBC>(meta));
    const int32_t ndist = N / 2 + 1, per = (ndist + K.nsub - 1) / K.nsub;
    const int64_t items = (int64_t)N * K.nsub;
    int32_t lost = 0;
    uint32_t nre = 0;
    unsigned long long evaluated = 0;

    // intra-molecular bins, in bytes: size after the inter-molecular ones in LDS, size before in counts
    const int32_t same_at = LDS_HIST ? 4 * size : -4 * size;

    // Workgroup b takes items b, b + gridDim, ...: every row chunk's first part
    // comes before its second, so its items mix the parts' uneven shares of
    // near chunks; its waves take them from a counter in LDS.  (One counter in
    // memory for all waves: 563 us at 13,500 atoms against 61, the atomics on one
    // address; items dealt to the waves in turn: 1,002 us at 200,000 against 778.)
    for (;;) {
        int32_t turn = 0;
        if (lane == 0) turn = atomicAdd(&next, 1);
        const int64_t it = (int64_t)__builtin_amdgcn_readfirstlane(turn) * gridDim.x + blockIdx.x;
        if (it >= items) break;
        const int32_t sub = (int32_t)((uint32_t)it / (uint32_t)N), i = (int32_t)((uint32_t)it - (uint32_t)sub * (uint32_t)N);
        const int32_t e0 = sub * per, e1 = min(ndist, e0 + per);
        const float4 r = sx[(int64_t)i * 64 + lane];
        const int32_t rm = smol[(int64_t)i * 64 + lane];
        // the row chunk's box: a lane-varying load (see load_dev), then one value per lane broadcast
        const int bx = __float_as_int(reinterpret_cast<const float *>(cbox + kBox * (int64_t)i)[lane & 15]);
        auto of = [&](int k) { return __int_as_float(__builtin_amdgcn_readlane(bx, k)); };
        const float3 bm = make_float3(of(0), of(1), of(2)), bh = make_float3(of(4), of(5), of(6)),
                     blo = make_float3(of(8), of(9), of(10)), bhi = make_float3(of(12), of(13), of(14));
        const int32_t rmeta = __float_as_int(r.w), rid = rmeta >> 6;
        // byte offsets of the row atom's bins, as the later and as the earlier atom
        const int32_t rH = (rmeta & 63) * H * 4, rNH = rH * nel;
        const int32_t rowpos = i * 64 + lane;
        int32_t qn = 0;

        auto drain = [&](int32_t from, int32_t len) {
            if (lane < len) {
                const uint32_t q = queue[from + lane];
                const int64_t pr = (int64_t)i * 64 + (q >> 26), pc = q & 0x3ffffffu;
                float4 a = sx[pr], c = sx[pc];
                const bool same = smol[pr] == smol[pc];
                if (__float_as_int(c.w) < __float_as_int(a.w)) {  // the earlier atom first
                    const float4 t = a;
                    a = c;
                    c = t;
                }
                const int32_t off = ((__float_as_int(a.w) & 63) * nel + (__float_as_int(c.w) & 63)) * H;
                int64_t b;
                const float s = pair_s<PBC, ORTHO>(a.x, a.y, a.z, c.x, c.y, c.z, B);
                if (EDGE) {
                    bool re64 = false;
                    b = edge_bin<PBC>(s, a.x, a.y, a.z, c.x, c.y, c.z, B, E, re64);
                    nre += re64;
                } else {
                    b = bin_of(s, A.g);
                }
                if (b >= 0) {
                    if (b >= size - off)
                        lost++;
                    else if (LDS_HIST && (lds_intra || !same))
                        atomicAdd(&hist[off + (int32_t)b + (same ? size : 0)], 1);
                    else
                        atomicAdd(&counts[(same ? 0 : A.size) + off + b], 1);
                }
            }
        };

        // the rows against the wave's list of cnt atoms; ONE: image (kx, ky, kz) for every pair
        auto walk = [&](auto ONE, int32_t cnt, float kx, float ky, float kz) {
            for (int32_t t0 = 0; t0 < cnt; t0 += kListPad) {
                float4 q[kListPad];
                int4 w[kListPad];
#pragma unroll
                for (int u = 0; u < kListPad; u++) {
                    q[u] = lxyz[t0 + u];
                    w[u] = linfo[t0 + u];
                }
                // no branch on a pair's range or bin: the four pairs' arithmetic
                // interleaves, lanes out of range only leave the add
                uint32_t exact = 0;
#pragma unroll
                for (int u = 0; u < kListPad; u++) {
                    float bx = r.x - q[u].x, by = r.y - q[u].y, bz = r.z - q[u].z;
                    if (PBC && decltype(ONE)::value) {
                        bx -= kx;
                        by -= ky;
                        bz -= kz;
                    } else if (PBC && ORTHO) {  // signs fall out of the squares
                        bx = min_image_pm(bx);
                        by = min_image_pm(by);
                        bz = min_image_pm(bz);
                    } else if (PBC) {
                        bx = min_image(bx);
                        by = min_image(by);
                        bz = min_image(bz);
                    }
                    float x = bx, y = by, z = bz;
                    if (PBC && ORTHO) {
                        x = bx * B.b[0];
                        y = by * B.b[4];
                        z = bz * B.b[8];
                    } else if (PBC) {
                        x = bx * B.b[0] + by * B.b[3] + bz * B.b[6];
                        y = bx * B.b[1] + by * B.b[4] + bz * B.b[7];
                        z = bx * B.b[2] + by * B.b[5] + bz * B.b[8];
                    }
                    const float s = norm2(x, y, z);
                    const bool in = (EDGE ? (s >= E.s_lo && s < E.s_hi) : in_range(s, A.g)) && w[u].y > rowpos;
                    const float t = (__builtin_amdgcn_sqrtf(s) - A.g.minD) * F.inv;
                    bool fast = fabsf(__builtin_amdgcn_fractf(t) - 0.5f) < F.half && t < F.thi;
                    if (EDGE) fast = fast && t >= 0.0f;
                    if (EDGE && PBC) fast = fast && fmaxf(fmaxf(fabsf(bx), fabsf(by)), fabsf(bz)) <= F.tie;
                    const bool same = w[u].x == rm;
                    if (LDS_HIST) fast = fast && (lds_intra || !same);
                    const int32_t off = (rid < w[u].z ? rNH + __float_as_int(q[u].w) : w[u].w + rH) +
                                        (same ? same_at : 0) + ((int32_t)t << 2);
                    if (in && fast) {
                        char *bins = reinterpret_cast<char *>(LDS_HIST ? hist : counts + A.size);
                        atomicAdd(reinterpret_cast<int32_t *>(bins + off), 1);
                    }
                    exact |= in && !fast ? 1u << u : 0u;
                }
                if (!__ballot(exact != 0)) continue;
                for (int u = 0; u < kListPad; u++) {
                    const bool ex = (exact >> u) & 1;
                    const uint64_t sm = __ballot(ex);
                    if (!sm) continue;
                    if (ex)
                        queue[qn + __builtin_amdgcn_mbcnt_hi((uint32_t)(sm >> 32),
                                                             __builtin_amdgcn_mbcnt_lo((uint32_t)sm, 0))] =
                            ((uint32_t)lane << 26) | (uint32_t)(linfo[t0 + u].y & (kSelfKey - 1));
                    qn += __popcll(sm);
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                    if (qn >= 64) {
                        qn -= 64;
                        drain(qn, 64);
                        __builtin_amdgcn_wave_barrier();
                    }
                }
            }
        };

        for (int32_t e = e0; e < e1; e += 64) {
            // the offset N/2 of an even N joins each pair of chunks from both sides: taken from the first half
            const int32_t el = e + lane;
            const bool mineok = el < e1 && (2 * el != N || i < el || el == 0);
            int32_t j = i + el;
            j = j >= N ? j - N : j;
            bool near = false;
            if (mineok) {
                const float4 m = cbox[kBox * (int64_t)j], h = cbox[kBox * (int64_t)j + 1];
                near = !(lower_bound2<PBC, ORTHO>(m.x - bm.x, m.y - bm.y, m.z - bm.z, h.x + bh.x, h.y + bh.y,
                                                  h.z + bh.z, C) > cut2);
            }
            uint64_t todo = __ballot(near);
            float4 cn = make_float4(0.f, 0.f, 0.f, 0.f);
            int32_t mn = 0, jn = 0;
            if (todo) {
                jn = i + e + __builtin_ctzll(todo);
                jn = jn >= N ? jn - N : jn;
                cn = sx[(int64_t)jn * 64 + lane];
                mn = smol[(int64_t)jn * 64 + lane];
            }
            while (todo) {
                todo &= todo - 1;
                const float4 c = cn;
                const int32_t cm = mn, jc = jn;
                if (todo) {  // the next chunk's atoms load while this one is evaluated
                    jn = i + e + __builtin_ctzll(todo);
                    jn = jn >= N ? jn - N : jn;
                    cn = sx[(int64_t)jn * 64 + lane];
                    mn = smol[(int64_t)jn * 64 + lane];
                }
                const int32_t cmeta = __float_as_int(c.w);
                bool keep = cmeta >= 0;
                if (PBC)
                    keep = keep && !(lower_bound2<PBC, ORTHO>(c.x - floorf(c.x) - bm.x, c.y - floorf(c.y) - bm.y,
                                                              c.z - floorf(c.z) - bm.z, bh.x, bh.y, bh.z, C) > cut2);
                else
                    keep = keep && !(lower_bound2<PBC, ORTHO>(c.x - bm.x, c.y - bm.y, c.z - bm.z, bh.x, bh.y, bh.z,
                                                              C) > cut2);
                const uint64_t km = __ballot(keep);
                const int32_t cnt = __popcll(km);
                const int32_t at = __builtin_amdgcn_mbcnt_hi((uint32_t)(km >> 32),
                                                             __builtin_amdgcn_mbcnt_lo((uint32_t)km, 0));
                __builtin_amdgcn_wave_barrier();
                if (keep) {
                    const int32_t cH = (cmeta & 63) * H * 4;
                    lxyz[at] = make_float4(c.x, c.y, c.z, __int_as_float(cH));
                    linfo[at] = make_int4(cm, (jc * 64 + lane) | (jc == i ? 0 : kSelfKey), cmeta >> 6, cH * nel);
                }
                if (lane < kListPad) {
                    const float nan = __uint_as_float(0x7fc00000u);
                    lxyz[cnt + lane] = make_float4(nan, nan, nan, 0.0f);
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
                evaluated += (unsigned)cnt;
                // The image of a difference never falls as the difference grows: where it
                // is the same at both ends of the row chunk, and for every listed atom, it
                // is the same for every pair, and subtracting it is all of min_image.
                if (PBC) {
                    const float kx = image_of(blo.x - c.x), ky = image_of(blo.y - c.y), kz = image_of(blo.z - c.z);
                    const int first = km ? __builtin_ctzll(km) : 0;
                    auto at_first = [&](float x) {
                        return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), first));
                    };
                    const float ux = at_first(kx), uy = at_first(ky), uz = at_first(kz);
                    const bool other = !(kx == ux && ky == uy && kz == uz && image_of(bhi.x - c.x) == ux &&
                                         image_of(bhi.y - c.y) == uy && image_of(bhi.z - c.z) == uz);
                    if (__ballot(keep && other))
                        walk(std::false_type{}, cnt, 0.f, 0.f, 0.f);
                    else
                        walk(std::true_type{}, cnt, ux, uy, uz);
                } else {
                    walk(std::false_type{}, cnt, 0.f, 0.f, 0.f);
                }
            }
        }
        drain(0, qn);
        __builtin_amdgcn_wave_barrier();
    }
    if (lost) atomicAdd(&counts[2 * A.size], lost);
    if (EDGE && nre)
        atomicAdd(reinterpret_cast<unsigned long long *>(&counts[2 * A.size + 2]), (unsigned long long)nre);
    if (K.count_pairs && lane == 0)
        atomicAdd(reinterpret_cast<unsigned long long *>(&meta[M_PAIRS + kPairStep * (blockIdx.x % kPairWords)]),
                  evaluated * 64ull);
    if (LDS_HIST) {
        __syncthreads();
        int32_t *dst = K.partial + (int64_t)blockIdx.x * nbins;
        for (int32_t s = tid; s < nbins; s += blockDim.x) dst[s] = hist[s];
    }
}

// Orthorhombic cells take their shorter arithmetic.
template <bool PBC, bool LDS_HIST, bool EDGE>
__global__ void __launch_bounds__(1024, EDGE ? 4 : 8) k_full_chunks(ChunkArgs K, Edge64 E) {
    const ChunkPlan P = plan_of(K.meta);
    if (PBC && P.ortho)
        full_chunks<PBC, true, LDS_HIST, EDGE>(K, P.B, P.C, E);
    else
        full_chunks<PBC, false, LDS_HIST, EDGE>(K, P.B, P.C, E);
}

// Slot s of the result: counts[s] plus the partials of s (stored with the
// inter-molecular half first; len 0, size or 2 size slots each).  64 slots per
// workgroup, sixteen waves each adding every sixteenth partial.  With hintra:
// written there as float32; else added into counts.  overflow: host word for
// the lost pairs.
__global__ void __launch_bounds__(1024) k_chunk_finish(const int32_t *__restrict__ partial, int32_t nparts,
                                                       int64_t len, int64_t size, int32_t *__restrict__ counts,
                                                       float *__restrict__ hintra, float *__restrict__ hinter,
                                                       int64_t *overflow) {
    __shared__ int32_t part[16][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t s = (int64_t)blockIdx.x * 64 + lane;
    const int64_t from = s >= size ? s - size : s + size;
    int32_t acc = 0;
    if (s < 2 * size && from < len) {
        int32_t p = w;
        for (; p + 112 < nparts; p += 128) {
            int32_t v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = partial[(int64_t)(p + 16 * u) * len + from];
#pragma unroll
            for (int u = 0; u < 8; u++) acc += v[u];
        }
        for (; p < nparts; p += 16) acc += partial[(int64_t)p * len + from];
    }
    part[w][lane] = acc;
    __syncthreads();
    if (w == 0 && s < 2 * size) {
        for (int q = 1; q < 16; q++) acc += part[q][lane];
        if (hintra) {
            const float f = (float)(counts[s] + acc);
            if (s < size) hintra[s] = f;
            else hinter[s - size] = f;
        } else if (acc) {
            counts[s] += acc;
        }
    }
    if (overflow && blockIdx.x == 0 && threadIdx.x == 0) *overflow = load_dev(counts + 2 * size);
}

// k_chunk_finish without partials: counts made by atomics, as float32.  Bound by
// its reads and writes (16 waves per 64 slots, as for partials, took about 150 us
// more at 8.2 million slots).
__global__ void __launch_bounds__(256) k_chunk_convert(const int32_t *__restrict__ counts, int64_t size,
                                                       float *__restrict__ hintra, float *__restrict__ hinter,
                                                       int64_t *overflow) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *overflow = load_dev(counts + 2 * size);
    for (int64_t s = (int64_t)blockIdx.x * 256 + threadIdx.x; s < 2 * size; s += (int64_t)gridDim.x * 256) {
        const float f = (float)counts[s];
        if (s < size) hintra[s] = f;
        else hinter[s - size] = f;
    }
}

// the number of evaluated pairs to a host word
__global__ void k_chunk_pairs(const uint32_t *__restrict__ meta, int64_t *pairs) {
    int64_t sum = 0;
    for (int w = 0; w < kPairWords; w++)
        sum += load_dev(reinterpret_cast<const int64_t *>(meta + M_PAIRS + kPairStep * w));
    if (threadIdx.x == 0) *pairs = sum;
}

// Bounds of the approximate bin t = (v_sqrt(s) - min) * (1/bin) against the
// reference's t = fl(fl(fl(sqrt(s)) - min) / bin): v_sqrt is within 1 ulp, each
// rounding within 2^-24 relative.  |difference| <= u (4 d + 3 |d - min|) / bin
// + 3 u |t|, u = 2^-24, taken at the range's end and half as much again.  In
// the binary64 mode d differs from the double distance by the per-pair bound
// of edge_bin, here at its largest over all pairs.
FastBin fast_bin(const HistArgs &A, const Edge64 *E, int isPBC) {
    const double u = 5.9604644775390625e-08, bin = A.g.bin, mx = A.g.maxD, mn = A.g.minD;
    const double t = fabs((mx - mn) / bin);
    double eps = 1.5 * u * ((4.0 * fabs(mx) + 3.0 * (fabs(mx) + fabs(mn))) / fabs(bin) + 3.0 * t + 4.0);
    FastBin F;
    F.inv = (float)(1.0 / bin);
    F.thi = (float)A.g.H;
    F.tie = INFINITY;
    if (E) {
        const double amax = E->amax;
        double bound = fabs(mx);
        for (int m = 0; m < 3; m++) bound += E->rowsum[m] * (2.0 * amax + 1.0);
        eps += 1.01 * 8.0 * u * 1.001 * bound / bin;
        F.thi = (float)std::min((double)A.g.H, t - eps - 1e-6 * t);
        if (isPBC) F.tie = (float)(0.5 - 5.0e-7 * (2.0 * amax + 1.0));
    }
    // not usable: bins near the distances' own rounding, or a grid that is not finite and increasing
    F.half = eps < 0.2 && bin > 0.0 && mx > mn && std::isfinite(F.inv) ? (float)(0.5 - eps) : -1.0f;
    return F;
}

}  // namespace

ChunkSort chunk_layout(int32_t n) {
    ChunkSort S;
    memset(&S, 0, sizeof(S));
    S.ncol = columns_most(n);
    S.cells = S.ncol * kNZ;
    S.maxchunks = (n + 63) / 64 + S.ncol;
    const size_t np = (size_t)S.maxchunks * 64;
    size_t off = 4 * M_WORDS;
    auto take = [&](size_t bytes) {
        const size_t at = off;
        off = (off + bytes + 255) & ~(size_t)255;
        return at;
    };
    S.o_cnt = take(4 * (size_t)S.cells);
    S.o_start = take(4 * (size_t)S.cells);
    S.o_tot = take(4 * (size_t)S.ncol);
    S.o_base = take(4 * (size_t)S.ncol);
    S.o_where = take(8 * (size_t)n);
    S.o_sx = take(16 * np);
    S.o_mol = take(4 * np);
    S.o_box = take(sizeof(float4) * kBox * (size_t)S.maxchunks);
    S.bytes = off;
    return S;
}

void launch_chunk_sort(ChunkSort &S, char *scr, const float *coords, int32_t n, const float *dbasis, const Basis &hB,
                       int isPBC, const int32_t *mol, const int32_t *elem, int32_t nel, int32_t *zero, int64_t nzero,
                       hipStream_t st) {
    uint32_t *meta = S.meta = (uint32_t *)scr;
    float4 *sx = S.sx = (float4 *)(scr + S.o_sx), *cbox = S.cbox = (float4 *)(scr + S.o_box);
    int32_t *smol = S.smol = (int32_t *)(scr + S.o_mol);
    int32_t *cnt = (int32_t *)(scr + S.o_cnt), *start = (int32_t *)(scr + S.o_start), *tot = (int32_t *)(scr + S.o_tot),
            *base = (int32_t *)(scr + S.o_base);
    int2 *where = (int2 *)(scr + S.o_where);
    const unsigned nb = blocks_for(n, 256), cb = (unsigned)((S.maxchunks + 3) / 4);
    const bool small = n <= kSmallSort && nzero <= kSmallClear;
    if (small && isPBC) {
        k_chunk_sort_small<true><<<1, 1024, 0, st>>>(dbasis, hB, coords, n, mol, elem, nel, meta, where, sx, smol, zero,
                                                     nzero);
    } else if (small) {
        k_chunk_sort_small<false><<<1, 1024, 0, st>>>(dbasis, hB, coords, n, mol, elem, nel, meta, where, sx, smol, zero,
                                                      nzero);
    } else {
        k_chunk_setup<<<std::min(512u, blocks_for(S.cells + nzero, 256)), 256, 0, st>>>(dbasis, hB, isPBC, n, meta, cnt,
                                                                                        S.cells, zero, nzero);
        if (!isPBC) k_chunk_extent<<<std::min(nb, 64u), 256, 0, st>>>(coords, n, meta);
        if (isPBC)
            k_chunk_count<true><<<nb, 256, 0, st>>>(coords, n, meta, cnt, where);
        else
            k_chunk_count<false><<<nb, 256, 0, st>>>(coords, n, meta, cnt, where);
        k_chunk_scan<<<1, 1024, 0, st>>>((const int2 *)cnt, (int2 *)start, tot, base, meta, sx, smol);
        k_chunk_scatter<<<nb, 256, 0, st>>>(coords, n, mol, elem, nel, where, start, base, sx, smol);
    }
    if (isPBC)
        k_chunk_boxes<true><<<cb, 256, 0, st>>>(sx, meta, cbox);
    else
        k_chunk_boxes<false><<<cb, 256, 0, st>>>(sx, meta, cbox);
}

bool chunks_take(int32_t n, const HistArgs &A) { return A.nel <= 64 && n < (1 << 25) && A.size < (1 << 27); }

int add_partials(const int32_t *partial, int64_t nparts, int64_t size, int32_t *counts, hipStream_t st) {
    k_chunk_finish<<<(unsigned)((2 * size + 63) / 64), 1024, 0, st>>>(partial, (int32_t)nparts, 2 * size, size, counts,
                                                                      nullptr, nullptr, nullptr);
    FRMC_CHECK_LAUNCH();
    return FRMC_OK;
}

int run_chunks(const ChunkRun &R, const float *coords, int32_t n, const float *dbasis, const Basis &hB, int isPBC,
               const int32_t *mol, const int32_t *elem, const HistArgs &A, const Edge64 *E, int ncu, hipStream_t st) {
    ChunkSort S = chunk_layout(n);
    const int64_t maxchunks = S.maxchunks;
    // bins in LDS: both halves, else the inter-molecular half, else none
    const size_t kMaxHist = 112 * 1024;  // leaves sixteen waves' lists (42 KB) of the 160 KB
    const int64_t size = A.size;
    const int64_t nbins = sizeof(int32_t) * 2 * size <= kMaxHist ? 2 * size
                          : sizeof(int32_t) * size <= kMaxHist   ? size
                                                                 : 0;
    const size_t hist_bytes = sizeof(int32_t) * (size_t)nbins;
    auto lds_of = [&](int32_t t) { return hist_bytes + (size_t)(t / 64) * kWaveLds; };
    // workgroups per CU by LDS and by the kernels' registers (8 waves a SIMD, 5 in the binary64 mode)
    auto fit_of = [&](int32_t t) {
        return (int32_t)std::min<size_t>((E ? 1280 : 2048) / t, (160 * 1024) / (lds_of(t) + 64));
    };
    // Threads per workgroup: the most resident waves, the fewest partials among
    // equals; in the binary64 mode the smallest workgroups among equals (40,000
    // atoms: 250 us with 512 threads, 257 with 1,024; 80,000 atoms with 256: 247
    // against 277 and 308).  200,000 atoms with 64 KB of bins: 1,024 threads 633
    // us, 512 (one workgroup per CU either way) 966.
    int32_t nt = R.nt, per_cu = R.per_cu;
    if (!nt) {
        nt = 1024;
        for (int32_t t = 512; t >= 256; t /= 2)
            if (fit_of(t) * t > fit_of(nt) * nt || (E && fit_of(t) * t == fit_of(nt) * nt)) nt = t;
    }
    while (nt > 256 && fit_of(nt) < 1) nt /= 2;
    const size_t shm = lds_of(nt);
    const int32_t fit = std::max(1, fit_of(nt));
    if (per_cu <= 0) per_cu = fit;
    const int64_t ndist = maxchunks / 2 + 1, tiles = maxchunks * ndist;
    const int64_t waves = (int64_t)ncu * fit * (nt / 64);
    // about 32 items per resident wave, so that the last ones are short (6: 905 us
    // against 848 at 200,000 atoms, before the pair loop lost its branches)
    const int64_t per = std::max<int64_t>(1, tiles / (32 * waves));
    ChunkArgs K;
    K.nsub = (int32_t)((ndist + per - 1) / per);
    const int64_t items = maxchunks * K.nsub;
    int64_t blocks = std::min<int64_t>((int64_t)ncu * per_cu, (items + nt / 64 - 1) / (nt / 64));
    if (blocks < 1) blocks = 1;
    if (R.blocks) *R.blocks = blocks;
    if (R.used_nt) *R.used_nt = nt;

    const int64_t ncounts = R.counts ? 0 : 2 * size + 4;
    const size_t o_counts = S.bytes, o_part = (o_counts + 4 * (size_t)ncounts + 255) & ~(size_t)255,
                 bytes = o_part + hist_bytes * (size_t)blocks;
    char *scr = nullptr;
    hipError_t e = pool_malloc((void **)&scr, bytes, st);
    if (e != hipSuccess) {
        set_error("hipMallocAsync of %zu bytes for the full histogram failed: %s", bytes, hipGetErrorString(e));
        return FRMC_ENOMEM;
    }
    int32_t *counts = R.counts ? R.counts : (int32_t *)(scr + o_counts);
    launch_chunk_sort(S, scr, coords, n, dbasis, hB, isPBC, mol, elem, A.nel, counts, ncounts, st);
    Edge64 none;
    memset(&none, 0, sizeof(none));
    const Edge64 &EE = E ? *E : none;
    K.sx = S.sx;
    K.smol = S.smol;
    K.cbox = S.cbox;
    K.meta = S.meta;
    K.range = E ? (float)sqrt((double)E->s_hi) : A.g.maxD;
    K.A = A;
    K.F = fast_bin(A, E, isPBC);
    K.lds_intra = nbins == 2 * size;
    K.count_pairs = R.pairs != nullptr;
    K.partial = (int32_t *)(scr + o_part);
    K.counts = counts;
#define FRMC_CHUNKS(P, L, ED)                                                                                     \
    do {                                                                                                          \
        if (shm > 48 * 1024)                                                                                      \
            (void)hipFuncSetAttribute((const void *)k_full_chunks<P, L, ED>,                                      \
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);                      \
        k_full_chunks<P, L, ED><<<(unsigned)blocks, nt, shm, st>>>(K, EE);                                        \
    } while (0)
#define FRMC_CHUNKS_ED(P, L)                \
    do {                                    \
        if (E) FRMC_CHUNKS(P, L, true);     \
        else FRMC_CHUNKS(P, L, false);      \
    } while (0)
    if (isPBC) {
        if (nbins) FRMC_CHUNKS_ED(true, true);
        else FRMC_CHUNKS_ED(true, false);
    } else {
        if (nbins) FRMC_CHUNKS_ED(false, true);
        else FRMC_CHUNKS_ED(false, false);
    }
#undef FRMC_CHUNKS_ED
#undef FRMC_CHUNKS
    if (!nbins && !R.counts)
        k_chunk_convert<<<std::min(2048u, blocks_for(2 * size, 256)), 256, 0, st>>>(counts, size, R.hintra, R.hinter,
                                                                                    R.overflow);
    else if (nbins)
        k_chunk_finish<<<(unsigned)((2 * size + 63) / 64), 1024, 0, st>>>(
            K.partial, (int32_t)blocks, nbins, size, counts, R.counts ? nullptr : R.hintra,
            R.counts ? nullptr : R.hinter, R.overflow);
    if (R.pairs) k_chunk_pairs<<<1, 64, 0, st>>>(S.meta, R.pairs);
    e = hipGetLastError();
    (void)hipFreeAsync(scr, st);
    if (e != hipSuccess) {
        set_error("full histogram launch failed: %s", hipGetErrorString(e));
        return FRMC_EHIP;
    }
    return FRMC_OK;
}

}  // namespace frmc
