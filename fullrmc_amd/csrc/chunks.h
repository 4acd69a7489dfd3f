// chunks.h -- atoms sorted into chunks of 64 (full_chunks.hip makes them): layout,
// and the tests that skip what is out of range.  Used by the full histogram
// (full_chunks.hip) and the atomic distances (atomic_distances.hip).
#pragma once
#include "frmc_device.h"
#include "frmc_host.h"

namespace frmc {

constexpr int kNZ = 128;            // counting-sort bins along a column
constexpr int kBox = 4;             // float4 per chunk box

// words of the scratch header (zeroed before the sort, then the plan; six 64-bit
// sums of open boundaries; then the
// evaluated pairs while they are counted, over kPairWords cache lines: the waves'
// atomics took 60 us at 13,500 atoms on one word, 20 on 32 words of two lines)
constexpr int kPairWords = 32, kPairStep = 32;
enum { M_AMAX = 0, M_NCHUNK = 1, M_LO = 8, M_HI = 11, M_PLAN = 16, M_SUM = 46, M_PAIRS = 64, M_WORDS = M_PAIRS + kPairStep * kPairWords };

// Lower bound of a squared distance from fractional differences known up to
// half-widths: |b B|^2 = |b L|^2 with B B^T = L L^T (L lower triangular).
struct ChunkCut {
    float L00, L10, L11, L20, L21, L22;
    float rows;           // sum of |B| (periodic), 1 otherwise
};

// What follows from the cell, computed on the device: the basis is device
// memory, and reading it back first cost a synchronisation per call (20 us).
struct ChunkPlan {
    Basis B;
    ChunkCut C;
    int32_t m0, m1;       // columns across the first two axes
    int32_t ortho;        // the off-diagonal entries are zero
};
constexpr int kPlanWords = sizeof(ChunkPlan) / 4;
static_assert(M_WORDS <= 1024 + M_PAIRS, "the small sort clears the pair words with 1,024 threads");
static_assert(sizeof(ChunkPlan) % 4 == 0 && kPlanWords <= 64 && kPlanWords <= M_SUM - M_PLAN && M_SUM + 12 <= M_PAIRS, "plan size");

// Columns across the first two axes, for n atoms: cross-sections of about the
// side of a cube of 64 atoms, so that 64 consecutive atoms of a column fill
// about a cube; at most columns_most(n), or the columns' padding outweighs the
// atoms (flat cells).
__host__ __device__ __forceinline__ int32_t columns_most(int32_t n) { return n / 96 > 1 ? n / 96 : 1; }

__device__ __forceinline__ uint32_t ordered_bits(float x) {
    const uint32_t b = __float_as_uint(x);
    return b ^ ((b >> 31) ? 0xffffffffu : 0x80000000u);
}
__device__ __forceinline__ float from_ordered(uint32_t u) {
    return __uint_as_float(u ^ ((u >> 31) ? 0x80000000u : 0xffffffffu));
}

__device__ __forceinline__ float abs_or_inf(float x) {
    const float a = fabsf(x);
    return a == a ? a : __uint_as_float(0x7f800000u);
}

// the largest |coordinate| (at least 1), infinite if one is not a number
template <bool PBC>
__device__ __forceinline__ float coord_max(const uint32_t *__restrict__ meta) {
    if (PBC) return fmaxf(1.0f, __uint_as_float(load_dev(meta + M_AMAX)));
    float a = 1.0f;
#pragma unroll
    for (int k = 0; k < 3; k++)
        a = fmaxf(a, fmaxf(abs_or_inf(from_ordered(~load_dev(meta + M_LO + k))),
                           abs_or_inf(from_ordered(load_dev(meta + M_HI + k)))));
    return a;
}

// Squared lower bound of the distance of any pair whose wrapped differences
// lie within w of d.  Per row of L: |b_k L_kk| is at least L_kk (|d_k| - w_k)
// whatever image is taken; where no axis of the row can cross +-1/2, the
// row's interval is used instead.
template <bool PBC, bool ORTHO>
__device__ __forceinline__ float lower_bound2(float d0, float d1, float d2, float w0, float w1, float w2,
                                              const ChunkCut &C) {
    if (PBC) {
        d0 -= rintf(d0);
        d1 -= rintf(d1);
        d2 -= rintf(d2);
    }
    float x = (fabsf(d0) - w0) * C.L00, y = (fabsf(d1) - w1) * C.L11, z = (fabsf(d2) - w2) * C.L22;
    if (PBC && !ORTHO) {
        const float M0 = fabsf(d0) + w0, M1 = fabsf(d1) + w1, M2 = fabsf(d2) + w2;
        const float a10 = fabsf(C.L10), a20 = fabsf(C.L20), a21 = fabsf(C.L21);
        const bool s12 = fmaxf(M1, M2) < 0.5f, s012 = fmaxf(M0, fmaxf(M1, M2)) < 0.5f;
        y -= a21 * fminf(M2, 0.5f);
        x -= a10 * fminf(M1, 0.5f) + a20 * fminf(M2, 0.5f);
        const float ys = fabsf(d1 * C.L11 + d2 * C.L21) - (w1 * C.L11 + w2 * a21);
        const float xs = fabsf(d0 * C.L00 + d1 * C.L10 + d2 * C.L20) - (w0 * C.L00 + w1 * a10 + w2 * a20);
        y = s12 ? fmaxf(y, ys) : y;
        x = s012 ? fmaxf(x, xs) : x;
    }
    x = fmaxf(x, 0.0f);
    y = fmaxf(y, 0.0f);
    z = fmaxf(z, 0.0f);
    return x * x + y * y + z * z;
}

// The range with a margin for every rounding between the bound above and the
// float32 distance: differences of coordinates up to amax (2^-24 each, times
// sum |B|), the image, the product with the basis, norm and sqrt (1e-5).
// Squared; infinite when a coordinate is not finite (then nothing is skipped).
__device__ __forceinline__ float cut_squared(const ChunkCut &C, float range, float amax) {
    const float w = range * 1.00001f + C.rows * 9.5367431640625e-07f * (amax + 1.0f);
    const float w2 = w * w * 1.00001f;
    return w2 == w2 ? w2 : __uint_as_float(0x7f800000u);
}

// x - min_image(x): the image taken, which never falls as x grows
__device__ __forceinline__ float image_of(float x) { return copysignf(floorf(fabsf(x) + 0.5f), x); }

// The plan reaches a wave through one lane-varying load and broadcasts (see load_dev).
__device__ __forceinline__ ChunkPlan plan_of(const uint32_t *meta) {
    const uint32_t v = meta[M_PLAN + min((int)(threadIdx.x & 63), kPlanWords - 1)];
    uint32_t w[kPlanWords];
#pragma unroll
    for (int k = 0; k < kPlanWords; k++) w[k] = (uint32_t)__builtin_amdgcn_readlane((int)v, k);
    ChunkPlan P;
    __builtin_memcpy(&P, w, sizeof(P));
    return P;
}

// The sorted atoms of one call, in the caller's scratch.
struct ChunkSort {
    int64_t cells, ncol, maxchunks;
    size_t bytes;         // of scratch, from its (256-byte aligned) start
    size_t o_cnt, o_start, o_tot, o_base, o_where, o_sx, o_mol, o_box;
    uint32_t *meta;       // header: chunks, plan, extent
    float4 *sx;           // (x, y, z, id * 64 + element), 64 per chunk; id -1 and NaN: padding
    int32_t *smol;
    float4 *cbox;
};
ChunkSort chunk_layout(int32_t n);
// Queues the sort into scr (scr + S.bytes may be used by the caller); zero:
// nzero words cleared before anything else of the sort runs.
void launch_chunk_sort(ChunkSort &S, char *scr, const float *coords, int32_t n, const float *dbasis, const Basis &hB,
                       int isPBC, const int32_t *mol, const int32_t *elem, int32_t nel, int32_t *zero, int64_t nzero,
                       hipStream_t st);

}  // namespace frmc
