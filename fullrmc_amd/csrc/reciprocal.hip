// reciprocal.hip -- the G(r) -> S(Q) sine transform as a standalone entry
// (the transform the S(Q) constraints apply, StructureFactorConstraints.py:
// 772-773, 1255-1256) and the reciprocal_space extension
// (Extensions/reciprocal_space.pyx).
//
//   k_sq_exact   S[p][q] = sum_r G[p][r]*M[r][q] (+1), the float32 product
//                rounded, then summed sequentially over r from +0 -- the
//                order of NumPy's axis-0 sum, so bit-identical to the
//                constraint's S(Q).  One lane per (p, q); some waves of a
//                workgroup stage M and G in LDS, the others sum.
//   k_sq_mfma, k_sq_tiles  the same contraction for k curves at once on the
//                matrix cores (v_mfma_f32_16x16x4_f32, float32 inputs, float32
//                accumulation): 32x16 tiles, the r range split over a
//                workgroup's waves, or, for large products, 64x64 tiles with the
//                range split over blocks.  Not bit-identical to the sequential sum; its error against a
//                float64 transform is measured.
//   k_Gr_to_sq / k_gr_to_sq   reciprocal_space.pyx:89-122 / :42-80: one lane
//                per Q; each term in double (sin of the float32 product q*r,
//                then the reference's operand order) added to the float32
//                accumulator in double and rounded back, as the Cython loop's
//                Python-float arithmetic does.
//   k_sq_to_Gr   the transform of reciprocal_space.pyx:131-162 (which
//                raises for any input there), in double, rounded once.
#include <algorithm>
#include <mutex>

#include "frmc_device.h"
#include "frmc_host.h"

namespace frmc {

namespace {

constexpr int kGChunk = 2048;  // values staged in LDS per pass

typedef float floatx4 __attribute__((ext_vector_type(4)));

// A workgroup barrier for LDS alone: __syncthreads also waits for the global
// loads in flight, which here are chunks ahead.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Exact transform.  A workgroup takes 64 Q points (one per lane) and 4 P curves.
// Four waves only load: matrix rows and G rows, kSqRows at a time, chunks ahead in
// registers, into LDS.  The other four only sum, P curves each: a value of the
// matrix read from LDS serves P curves, and each row's product is made between
// two dependent adds.  Bound by the vector issue of one wave per SIMD, a product
// and an add per curve, row and Q (about 9 cycles), and with one curve per wave by
// the LDS reads (17 cycles a row in all).  2,000 r x 1,000 Q, a call: 64 curves
// 19 us against 34, 128 curves 27 against 44 to 56, 256 curves 41 against 88 (one
// lane per curve and Q, each wave reading the matrix from L2 by itself).
constexpr int kSqRows = 64;
constexpr int kSqLoaders = 4;  // loading waves (eight, and six or eight chunks ahead, measured no faster)
constexpr int kSqAhead = 4;    // chunks of loads in flight

// Sixteen rows of P curves: acc += x[row], the product of sixteen rows before, then
// x[row] = (lane `row` of each sixteen lanes of g) * m[row].  Written out so that
// the products stand between the chain's dependent adds: an add issues 9 cycles
// after the one it waits for, and the compiler puts each product right before its
// own add (32 cycles a row).  G's value comes by a DPP row broadcast: reading it
// from LDS as a broadcast took half of the LDS time.  The leading s_nop covers a
// g written by the instruction before.
#define FRMC_SQ_ROW(A, X, G, M, L)                \
    "v_add_f32 %[" A "], %[" A "], %[" X "]\n\t" \
    "v_mul_f32_dpp %[" X "], %[" G "], %[" M "] row_newbcast:" L " row_mask:0xf bank_mask:0xf\n\t"
#define FRMC_X(P_, J_) [x##P_##J_] "+v"(x[P_][r + J_])
#define FRMC_M(J_) [m##J_] "v"(m[r + J_])

// acc, x and g of curve 0, rows r..r+7
#define FRMC_SQ_ROWS1(r_, L0, L1, L2, L3, L4, L5, L6, L7)                                                         \
    {                                                                                                             \
        constexpr int r = r_;                                                                                     \
        asm volatile("s_nop 1\n\t" FRMC_SQ_ROW("a0", "x00", "g0", "m0", L0) FRMC_SQ_ROW("a0", "x01", "g0", "m1", L1)    \
                         FRMC_SQ_ROW("a0", "x02", "g0", "m2", L2) FRMC_SQ_ROW("a0", "x03", "g0", "m3", L3)        \
                             FRMC_SQ_ROW("a0", "x04", "g0", "m4", L4) FRMC_SQ_ROW("a0", "x05", "g0", "m5", L5)    \
                                 FRMC_SQ_ROW("a0", "x06", "g0", "m6", L6) FRMC_SQ_ROW("a0", "x07", "g0", "m7", L7) \
                     : [a0] "+v"(acc[0]), FRMC_X(0, 0), FRMC_X(0, 1), FRMC_X(0, 2), FRMC_X(0, 3), FRMC_X(0, 4),   \
                       FRMC_X(0, 5), FRMC_X(0, 6), FRMC_X(0, 7)                                                   \
                     : [g0] "v"(g[0]), FRMC_M(0), FRMC_M(1), FRMC_M(2), FRMC_M(3), FRMC_M(4), FRMC_M(5),          \
                       FRMC_M(6), FRMC_M(7));                                                                     \
    }
// two curves, rows r..r+3
#define FRMC_SQ_ROWS2(r_, L0, L1, L2, L3)                                                                         \
    {                                                                                                             \
        constexpr int r = r_;                                                                                     \
        asm volatile("s_nop 1\n\t" FRMC_SQ_ROW("a0", "x00", "g0", "m0", L0) FRMC_SQ_ROW("a1", "x10", "g1", "m0", L0)    \
                         FRMC_SQ_ROW("a0", "x01", "g0", "m1", L1) FRMC_SQ_ROW("a1", "x11", "g1", "m1", L1)        \
                             FRMC_SQ_ROW("a0", "x02", "g0", "m2", L2) FRMC_SQ_ROW("a1", "x12", "g1", "m2", L2)    \
                                 FRMC_SQ_ROW("a0", "x03", "g0", "m3", L3) FRMC_SQ_ROW("a1", "x13", "g1", "m3", L3) \
                     : [a0] "+v"(acc[0]), [a1] "+v"(acc[1]), FRMC_X(0, 0), FRMC_X(0, 1), FRMC_X(0, 2),            \
                       FRMC_X(0, 3), FRMC_X(1, 0), FRMC_X(1, 1), FRMC_X(1, 2), FRMC_X(1, 3)                       \
                     : [g0] "v"(g[0]), [g1] "v"(g[1]), FRMC_M(0), FRMC_M(1), FRMC_M(2), FRMC_M(3));               \
    }
// four curves, rows r and r+1
#define FRMC_SQ_ROWS4(r_, L0, L1)                                                                                 \
    {                                                                                                             \
        constexpr int r = r_;                                                                                     \
        asm volatile("s_nop 1\n\t" FRMC_SQ_ROW("a0", "x00", "g0", "m0", L0) FRMC_SQ_ROW("a1", "x10", "g1", "m0", L0)    \
                         FRMC_SQ_ROW("a2", "x20", "g2", "m0", L0) FRMC_SQ_ROW("a3", "x30", "g3", "m0", L0)        \
                             FRMC_SQ_ROW("a0", "x01", "g0", "m1", L1) FRMC_SQ_ROW("a1", "x11", "g1", "m1", L1)    \
                                 FRMC_SQ_ROW("a2", "x21", "g2", "m1", L1) FRMC_SQ_ROW("a3", "x31", "g3", "m1", L1) \
                     : [a0] "+v"(acc[0]), [a1] "+v"(acc[1]), [a2] "+v"(acc[2]), [a3] "+v"(acc[3]), FRMC_X(0, 0),  \
                       FRMC_X(0, 1), FRMC_X(1, 0), FRMC_X(1, 1), FRMC_X(2, 0), FRMC_X(2, 1), FRMC_X(3, 0),        \
                       FRMC_X(3, 1)                                                                               \
                     : [g0] "v"(g[0]), [g1] "v"(g[1]), [g2] "v"(g[2]), [g3] "v"(g[3]), FRMC_M(0), FRMC_M(1));     \
    }

__device__ __forceinline__ void add_then_mul(float (&acc)[1], float (&x)[1][16], const float (&g)[1],
                                             const float (&m)[16]) {
    FRMC_SQ_ROWS1(0, "0", "1", "2", "3", "4", "5", "6", "7")
    FRMC_SQ_ROWS1(8, "8", "9", "10", "11", "12", "13", "14", "15")
}
__device__ __forceinline__ void add_then_mul(float (&acc)[2], float (&x)[2][16], const float (&g)[2],
                                             const float (&m)[16]) {
    FRMC_SQ_ROWS2(0, "0", "1", "2", "3")
    FRMC_SQ_ROWS2(4, "4", "5", "6", "7")
    FRMC_SQ_ROWS2(8, "8", "9", "10", "11")
    FRMC_SQ_ROWS2(12, "12", "13", "14", "15")
}
__device__ __forceinline__ void add_then_mul(float (&acc)[4], float (&x)[4][16], const float (&g)[4],
                                             const float (&m)[16]) {
    FRMC_SQ_ROWS4(0, "0", "1")
    FRMC_SQ_ROWS4(2, "2", "3")
    FRMC_SQ_ROWS4(4, "4", "5")
    FRMC_SQ_ROWS4(6, "6", "7")
    FRMC_SQ_ROWS4(8, "8", "9")
    FRMC_SQ_ROWS4(10, "10", "11")
    FRMC_SQ_ROWS4(12, "12", "13")
    FRMC_SQ_ROWS4(14, "14", "15")
}
#undef FRMC_SQ_ROWS4
#undef FRMC_SQ_ROWS2
#undef FRMC_SQ_ROWS1
#undef FRMC_M
#undef FRMC_X
#undef FRMC_SQ_ROW

template <int P>
__global__ void __launch_bounds__(256 + 64 * kSqLoaders) k_sq_exact(const float *__restrict__ G, int32_t k, int32_t H,
                                                  const float *__restrict__ M, int32_t nQ, int32_t addOne,
                                                  float *__restrict__ S) {
    // three chunks: the sums read ahead into the next one while the loads fill the third
    // (a float4 of the matrix is four rows of one Q point)
    __shared__ float4 ms[3][kSqRows / 4][64];
    __shared__ float gs[3][4 * P][kSqRows];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int32_t q0 = blockIdx.x * 64, p0 = blockIdx.y * 4 * P;
    const int32_t chunks = (H + kSqRows - 1) / kSqRows;
    if (wave >= 4) {
        const int w = wave - 4;
        constexpr int NM = kSqRows / kSqLoaders, NG = (4 * P + kSqLoaders - 1) / kSqLoaders;
        const int32_t qc = min(q0 + lane, nQ - 1);  // lanes past nQ run the chain on the last column, store nothing
        float mr[kSqAhead][NM], gr[kSqAhead][NG];
        // uniform row addresses, one offset per lane; rows past H are zero in both matrices
        // (their products add +0, which changes no sum that started from +0)
        auto load = [&](int32_t c0, float *m, float *g) {
            if (c0 + kSqRows <= H) {
                const float *row = M + (int64_t)(c0 + 4 * w) * nQ;
#pragma unroll
                for (int i = 0; i < NM; i++) m[i] = row[(int64_t)(i / 4 * 4 * kSqLoaders + i % 4) * nQ + qc];
            } else if (c0 < H) {
#pragma unroll
                for (int i = 0; i < NM; i++)
                    m[i] = M[(int64_t)min(c0 + i / 4 * 4 * kSqLoaders + 4 * w + i % 4, H - 1) * nQ + qc];
            } else {
                return;
            }
            const int32_t r = min(c0 + lane, H - 1);
#pragma unroll
            for (int i = 0; i < NG; i++) g[i] = G[(int64_t)min(p0 + min(kSqLoaders * i + w, 4 * P - 1), k - 1) * H + r];
        };
        auto store = [&](int32_t c0, const float *m, const float *g, int which) {
#pragma unroll
            for (int i = 0; i < NM; i += 4) {
                const int r = i * kSqLoaders + 4 * w;
                ms[which][r / 4][lane] = make_float4(c0 + r < H ? m[i] : 0.0f, c0 + r + 1 < H ? m[i + 1] : 0.0f,
                                                     c0 + r + 2 < H ? m[i + 2] : 0.0f, c0 + r + 3 < H ? m[i + 3] : 0.0f);
            }
#pragma unroll
            for (int i = 0; i < NG; i++)
                if (kSqLoaders * i + w < 4 * P) gs[which][kSqLoaders * i + w][lane] = c0 + lane < H ? g[i] : 0.0f;
        };
#pragma unroll
        for (int u = 0; u < kSqAhead; u++) load(u * kSqRows, mr[u], gr[u]);
        int which = 0;
        for (int32_t c = 0; c < chunks; c += kSqAhead)
#pragma unroll
            for (int u = 0; u < kSqAhead; u++) {
                if (c + u >= chunks) break;
                store((c + u) * kSqRows, mr[u], gr[u], which);
                which = which == 2 ? 0 : which + 1;
                load((c + u + kSqAhead) * kSqRows, mr[u], gr[u]);
                // barrier c + u - 1: chunk c + u is in LDS, chunk c + u - 2 is summed
                if (c + u > 0) lds_barrier();
            }
        if (chunks == 1) lds_barrier();
        return;
    }
    float acc[P];
#pragma unroll
    for (int p = 0; p < P; p++) acc[p] = 0.0f;  // NumPy's add reduction starts from +0 (a sum of -0 terms is +0)
    // sixteen rows: the lane's matrix values, and per curve the sixteen G values,
    // one per lane of each sixteen lanes
    struct Rows {
        float m[16], g[P];
    };
    auto fetch = [&](Rows &R, int which, int i) {
#pragma unroll
        for (int j = 0; j < 16; j += 4) {
            const float4 m = ms[which][(i + j) / 4][lane];
            R.m[j] = m.x;
            R.m[j + 1] = m.y;
            R.m[j + 2] = m.z;
            R.m[j + 3] = m.w;
        }
#pragma unroll
        for (int p = 0; p < P; p++) R.g[p] = gs[which][wave * P + p][i + (lane & 15)];
    };
    // products not yet added: none at first (adding +0 changes no sum that started from +0)
    float x[P][16];
#pragma unroll
    for (int p = 0; p < P; p++)
#pragma unroll
        for (int j = 0; j < 16; j++) x[p][j] = 0.0f;
    // before chunk c: barrier c, after which chunks c and c + 1 are in LDS (the
    // last chunk has none: it came with the barrier before)
    lds_barrier();
    Rows R[2];
    fetch(R[0], 0, 0);
    int which = 0;
    for (int32_t c = 0; c + 1 < chunks; c++) {
        const int ahead = which == 2 ? 0 : which + 1;
#pragma unroll
        for (int i = 0; i < kSqRows / 16; i++) {
            if (i + 1 < kSqRows / 16) fetch(R[(i + 1) & 1], which, 16 * (i + 1));
            else fetch(R[0], ahead, 0);
            add_then_mul(acc, x, R[i & 1].g, R[i & 1].m);
        }
        which = ahead;
        if (c + 2 < chunks) lds_barrier();
    }
    // the last chunk: only the sixteens that hold rows (8 rows, 1,000 curves, 4,000 Q:
    // 30 us with all of them)
    const int32_t left = H - (chunks - 1) * kSqRows;
#pragma unroll
    for (int i = 0; i < kSqRows / 16; i++) {
        if (16 * i >= left) break;
        if (i + 1 < kSqRows / 16) fetch(R[(i + 1) & 1], which, 16 * (i + 1));
        add_then_mul(acc, x, R[i & 1].g, R[i & 1].m);
    }
#pragma unroll
    for (int j = 0; j < 16; j++)
#pragma unroll
        for (int p = 0; p < P; p++) acc[p] = acc[p] + x[p][j];
    if (q0 + lane < nQ)
#pragma unroll
        for (int p = 0; p < P; p++) {
            const int32_t pp = p0 + wave * P + p;
            if (pp < k) S[(int64_t)pp * nQ + q0 + lane] = addOne ? acc[p] + 1.0f : acc[p];
        }
}

// A few rows: one lane per (curve, Q), the row loop as it stands.  Bound by the
// result's stores; the staging above costs more than sixteen rows save (1,000
// curves x 4,000 Q: 8 rows 15 us against 23, 32 rows 22 against 25, 40 rows 27 against 28).
constexpr int kSqShort = 32, kSqT = 256;

__global__ void __launch_bounds__(kSqT) k_sq_short(const float *__restrict__ G, int32_t H, const float *__restrict__ M,
                                                   int32_t nQ, int32_t addOne, float *__restrict__ S) {
    __shared__ float gs[kSqShort];
    const int32_t q = blockIdx.x * kSqT + threadIdx.x;
    if ((int32_t)threadIdx.x < H) gs[threadIdx.x] = G[(int64_t)blockIdx.y * H + threadIdx.x];
    __syncthreads();
    if (q >= nQ) return;
    const float *m = M + q;
    float acc = 0.0f;  // as in k_sq_exact
    int32_t i = 0;
    // batches of 16 rows: the loads issue together, then the dependent adds
    for (; i + 16 <= H; i += 16) {
        float mv[16];
#pragma unroll
        for (int j = 0; j < 16; j++) mv[j] = m[(int64_t)(i + j) * nQ];
#pragma unroll
        for (int j = 0; j < 16; j++) mv[j] = gs[i + j] * mv[j];
#pragma unroll
        for (int j = 0; j < 16; j++) acc = acc + mv[j];
    }
    for (; i < H; i++) {
        const float pr = gs[i] * m[(int64_t)i * nQ];
        acc = acc + pr;
    }
    S[(int64_t)blockIdx.y * nQ + q] = addOne ? acc + 1.0f : acc;
}

// Matrix-core transform: C (k x nQ) = G (k x H) . M (H x nQ).  A workgroup
// takes a 32 x 16 tile of C; its waves split the r range and add their tiles
// through LDS, so one launch writes the result (a split over workgroups wrote
// and read 16 MB of partials and needed a second kernel).  Fragments come
// straight from memory, 16 rows ahead in registers: in a step of 16 rows, lane
// group g = lane / 16 holds rows 4g..4g+3, one float4 of G and four values of
// M, and the four products of the step pair row 4g + j of both (any order of
// rows is a sum).  Each product has its own accumulators, which shortens the
// chains (and their rounding: 8.1e-8 of the norm against float64 at 2,000 r, 1.3e-7
// for the split over workgroups; smaller over 200 to 2,000 r).  Bound by the loads
// from L2 and one launch: 128 curves x 2,000 r x 1,000 Q 13.2 us against 21 to
// 25, 64 x 1,001 x 500 7.6 against 20.8.
//
// v_mfma_f32_16x16x4_f32 operand layout (64 lanes): lane l supplies
// A[l%16][l/16] and B[l/16][l%16] of a 16x4 by 4x16 product and holds
// D[4*(l/16)+i][l%16], i = 0..3, of the 16x16 accumulator.
constexpr int kTP = 32, kTQ = 16;

template <int W>
__global__ void __launch_bounds__(64 * W) k_sq_mfma(const float *__restrict__ G, int32_t k, int32_t H,
                                                    const float *__restrict__ M, int32_t nQ, int32_t addOne,
                                                    float *__restrict__ S) {
    __shared__ float part[W][kTP][kTQ + 1];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, g = lane >> 4, l = lane & 15;
    const int32_t p0 = blockIdx.y * kTP, q0 = blockIdx.x * kTQ;
    const int32_t steps = (H + 15) / 16, per = (steps + W - 1) / W;
    const int32_t s0 = min(steps, w * per), s1 = min(steps, s0 + per);
    const float *ga = G + (int64_t)min(p0 + l, k - 1) * H, *gb = G + (int64_t)min(p0 + 16 + l, k - 1) * H;
    const float *mq = M + min(q0 + l, nQ - 1);
    floatx4 acc[4][2];
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
        for (int i = 0; i < 2; i++) acc[j][i] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    struct Frag {
        float a[2][4], b[4];
    };
    // four values of G in one load, at the alignment of a float (rows of any H);
    // in the last step, rows past H: index clamped, values not used
    typedef floatx4 __attribute__((aligned(4))) row4;
    auto load = [&](int32_t s, Frag &f) {
        const int32_t r0 = 16 * s + 4 * g;
        if (16 * s + 16 <= H) {
            const floatx4 x = *reinterpret_cast<const row4 *>(ga + r0), y = *reinterpret_cast<const row4 *>(gb + r0);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                f.a[0][j] = x[j];
                f.a[1][j] = y[j];
                f.b[j] = mq[(int64_t)(r0 + j) * nQ];
            }
            return;
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int32_t r = min(r0 + j, H - 1);
            f.a[0][j] = ga[r];
            f.a[1][j] = gb[r];
            f.b[j] = mq[(int64_t)r * nQ];
        }
    };
    auto use = [&](int32_t s, const Frag &f) {
        const int32_t r0 = 16 * s + 4 * g;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const bool in = r0 + j < H;
#pragma unroll
            for (int i = 0; i < 2; i++)
                acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? f.a[i][j] : 0.0f, in ? f.b[j] : 0.0f, acc[j][i],
                                                                 0, 0, 0);
        }
    };
    constexpr int kAhead = 4;
    Frag f[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; u++) load(min(s0 + u, steps - 1), f[u]);
    for (int32_t s = s0; s < s1; s += kAhead)
#pragma unroll
        for (int u = 0; u < kAhead; u++) {
            if (s + u < s1) use(s + u, f[u]);
            load(min(s + u + kAhead, steps - 1), f[u]);
        }
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const floatx4 x = (acc[0][i] + acc[1][i]) + (acc[2][i] + acc[3][i]);
#pragma unroll
        for (int v = 0; v < 4; v++) part[w][16 * i + 4 * g + v][l] = x[v];
    }
    __syncthreads();
    for (int e = t; e < kTP * kTQ; e += 64 * W) {
        const int32_t p = p0 + e / kTQ, q = q0 + e % kTQ;
        float x = part[0][e / kTQ][e % kTQ];
#pragma unroll
        for (int v = 1; v < W; v++) x = x + part[v][e / kTQ][e % kTQ];
        if (addOne) x = x + 1.0f;
        if (p < k && q < nQ) S[(int64_t)p * nQ + q] = x;
    }
}

// Large products: a 64 x 64 tile of C per block of four waves (each a 32 x 32 quarter
// as 2 x 2 MFMA tiles), the r range in chunks of kKC staged through LDS, the next
// chunk's global loads in flight while the current one is multiplied.  The r range
// is split over gridDim.z blocks (enough blocks to fill the chip at small k);
// their partial tiles go to a buffer that k_sq_splitsum adds in split order.  Each
// value loaded is used 64 times, in the 32 x 16 tiles above 16 to 32 times, and
// a long r range spreads over the chip.
constexpr int kLP = 64, kLQ = 64, kKC = 64;
constexpr int kLA = kKC + 2;   // As row stride: fragment reads and row stores hit distinct banks
constexpr int kLB = kLQ + 16;  // Bs row stride: the two rows a half-wave reads land in disjoint banks
constexpr int kNA = kLP * kKC / 256, kNB = kKC * kLQ / 256;  // chunk elements per thread

__global__ void __launch_bounds__(256) k_sq_tiles(const float *__restrict__ G, int32_t k, int32_t H,
                                                 const float *__restrict__ M, int32_t nQ, int32_t kPerSplit,
                                                 int32_t addOne, float *__restrict__ out, int32_t direct) {
    __shared__ float As[kLP * kLA];
    __shared__ float Bs[kKC * kLB];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int wp = w >> 1, wq = w & 1;
    const int32_t p0 = blockIdx.y * kLP, q0 = blockIdx.x * kLQ;
    const int32_t kb0 = blockIdx.z * kPerSplit;
    const int32_t kend = min(H, kb0 + kPerSplit);
    float ar[kNA], br[kNB];
    // chunk loads: A 64 rows (p) x kKC r, B kKC r x 64 q; indexes clamped into
    // the arrays, values past the split's r range (or past k / nQ) unused or zero
    auto load = [&](int32_t kc0) {
#pragma unroll
        for (int i = 0; i < kNA; i++) {
            const int idx = t + 256 * i;
            const int32_t ra = kc0 + idx % kKC;
            const float va = G[(int64_t)min(p0 + idx / kKC, k - 1) * H + min(ra, kend - 1)];
            ar[i] = ra < kend ? va : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < kNB; i++) {
            const int idx = t + 256 * i;
            const int32_t rb = kc0 + idx / kLQ;
            const float vb = M[(int64_t)min(rb, kend - 1) * nQ + min(q0 + idx % kLQ, nQ - 1)];
            br[i] = rb < kend ? vb : 0.0f;
        }
    };
    floatx4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    if (kb0 < kend) load(kb0);
    for (int32_t kc0 = kb0; kc0 < kend; kc0 += kKC) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kNA; i++) {
            const int idx = t + 256 * i;
            As[(idx / kKC) * kLA + idx % kKC] = ar[i];
        }
#pragma unroll
        for (int i = 0; i < kNB; i++) {
            const int idx = t + 256 * i;
            Bs[(idx / kLQ) * kLB + idx % kLQ] = br[i];
        }
        __syncthreads();
        if (kc0 + kKC < kend) load(kc0 + kKC);
#pragma unroll
        for (int kb = 0; kb < kKC; kb += 4) {
            float af[2], bf[2];
#pragma unroll
            for (int i = 0; i < 2; i++) af[i] = As[(wp * 32 + 16 * i + (lane & 15)) * kLA + kb + (lane >> 4)];
#pragma unroll
            for (int j = 0; j < 2; j++) bf[j] = Bs[(kb + (lane >> 4)) * kLB + wq * 32 + 16 * j + (lane & 15)];
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[i], bf[j], acc[i][j], 0, 0, 0);
        }
    }
    float *dst = direct ? out : out + (int64_t)blockIdx.z * k * nQ;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int32_t q = q0 + wq * 32 + 16 * j + (lane & 15);
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int32_t p = p0 + wp * 32 + 16 * i + 4 * (lane >> 4) + v;
                float x = acc[i][j][v];
                if (direct && addOne) x = x + 1.0f;
                if (p < k && q < nQ) dst[(int64_t)p * nQ + q] = x;
            }
        }
}

// S = sum over the splits of the partial products, in split order (+1)
__global__ void __launch_bounds__(256) k_sq_splitsum(const float *__restrict__ part, int32_t nsplit, int64_t len,
                                                     int32_t addOne, float *__restrict__ S) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < len; i += (int64_t)gridDim.x * blockDim.x) {
        float x = 0.0f;
        // eight independent loads in flight, then their adds in order
        for (int32_t z0 = 0; z0 < nsplit; z0 += 8) {
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = part[(int64_t)min(z0 + j, nsplit - 1) * len + i];
#pragma unroll
            for (int j = 0; j < 8; j++)
                if (z0 + j < nsplit) x = x + v[j];
        }
        S[i] = addOne ? x + 1.0f : x;
    }
}

// Curves per wave, by the chains (64 Q of a curve each): one up to two chains per
// SIMD (128 curves of 1,000 Q: 27.6 us with one, 27.4 with two, and 64 curves
// 19.3 against 27.3), two up to four (256 curves: 51, 41 and 43 us with one, two
// and four), four beyond.
void launch_sq_exact(const float *G, int32_t k, int32_t H, const float *M, int32_t nQ, int32_t addOne, float *S,
                     hipStream_t st) {
    const unsigned bq = (unsigned)((nQ + 63) / 64);
    const int64_t chains = (int64_t)bq * k;
    const int threads = 64 * (4 + kSqLoaders);
    if (H <= kSqShort && nQ > 128)  // (at 100 Q most lanes of a block would idle: 60,000 curves x 24 rows 68 us against 43)
        k_sq_short<<<dim3((unsigned)((nQ + kSqT - 1) / kSqT), (unsigned)k), kSqT, 0, st>>>(G, H, M, nQ, addOne, S);
    else if (chains <= 2048)
        k_sq_exact<1><<<dim3(bq, (unsigned)((k + 3) / 4)), threads, 0, st>>>(G, k, H, M, nQ, addOne, S);
    else if (chains <= 4096)
        k_sq_exact<2><<<dim3(bq, (unsigned)((k + 7) / 8)), threads, 0, st>>>(G, k, H, M, nQ, addOne, S);
    else
        k_sq_exact<4><<<dim3(bq, (unsigned)((k + 15) / 16)), threads, 0, st>>>(G, k, H, M, nQ, addOne, S);
}

// Waves per workgroup: eight while the tiles do not fill the chip by themselves
// (2,000 r, 1,000 Q: 64 curves 12.0 us against 13.5 with four and with sixteen),
// four beyond (256 curves: 22.4 us against 24.3).  A launch takes the curves of as
// many tiles as a grid has rows; more curves take more launches.
constexpr int32_t kTileRows = 65535;
constexpr int64_t kMaxCurves = 64 * 65535;  // of a call

void launch_sq_mfma(const float *G, int32_t k, int32_t H, const float *M, int32_t nQ, int32_t addOne, float *S,
                    hipStream_t st) {
    for (int64_t p = 0; p < k; p += (int64_t)kTileRows * kTP) {
        const int32_t kp = (int32_t)std::min<int64_t>(k - p, (int64_t)kTileRows * kTP);
        const dim3 grid((unsigned)((nQ + kTQ - 1) / kTQ), (unsigned)((kp + kTP - 1) / kTP));
        if ((int64_t)grid.x * grid.y > 256)
            k_sq_mfma<4><<<grid, 256, 0, st>>>(G + p * H, kp, H, M, nQ, addOne, S + p * nQ);
        else
            k_sq_mfma<8><<<grid, 512, 0, st>>>(G + p * H, kp, H, M, nQ, addOne, S + p * nQ);
    }
}

// Which matrix-core kernel takes a shape, and the split of the r range over
// blocks in the large tiles.  The 32 x 16 tiles, without a second kernel, are better
// where they nearly fill the chip once and r is neither one chunk nor longer
// than a workgroup's waves hide (us, 32 x 16 against 64 x 64): 128 curves x 2,000
// r x 1,000 Q 13.6 and 24, 256 x 2,000 x 1,000 25.0 and 29.6, 16,384 x 2,000 x 16
// 25.4 and 61.9; and worse elsewhere: 1,000 x 2,000 x 1,000 84 and 69, 512 x 2,000 x
// 4,000 176 and 126, 4,096 x 200 x 1,000 108 and 35, 2,000 x 8 x 1,000 76 and 10, 64 x
// 8,000 x 300 43 and 27, 1 x 60,000 x 100 241 and 49.
struct SqPlan {
    bool tiles;        // k_sq_tiles
    int64_t bq, bp;    // its tiles
    int64_t nsplit;    // parts of the r range, about 1,024 blocks in all
    int32_t per;       // rows of a part
};

SqPlan sq_plan(int32_t k, int32_t H, int32_t nQ) {
    SqPlan P;
    const int64_t t = (int64_t)((k + kTP - 1) / kTP) * ((nQ + kTQ - 1) / kTQ);
    P.tiles = H <= 64 || H > 5000 || (nQ > kTQ && (t > 700 || t * H > 1050000));
    P.bq = (nQ + kLQ - 1) / kLQ;
    P.bp = (k + kLP - 1) / kLP;
    const int64_t chunks = (H + kKC - 1) / kKC;
    P.nsplit = std::max<int64_t>(1, std::min<int64_t>((1024 + P.bq * P.bp - 1) / (P.bq * P.bp), chunks));
    P.per = (int32_t)(((chunks + P.nsplit - 1) / P.nsplit) * kKC);
    P.nsplit = (H + P.per - 1) / P.per;
    return P;
}

// part: nsplit * k * nQ floats if the r range is split
void launch_sq_tiles(const SqPlan &P, const float *G, int32_t k, int32_t H, const float *M, int32_t nQ, int32_t addOne,
                     float *part, float *S, hipStream_t st) {
    const bool direct = P.nsplit == 1;
    k_sq_tiles<<<dim3((unsigned)P.bq, (unsigned)P.bp, (unsigned)P.nsplit), 256, 0, st>>>(
        G, k, H, M, nQ, P.per, addOne, direct ? S : part, direct);
    const int64_t len = (int64_t)k * nQ;
    if (!direct)
        k_sq_splitsum<<<(unsigned)std::min<int64_t>(blocks_for(len, 256), 4096), 256, 0, st>>>(part, (int32_t)P.nsplit,
                                                                                              len, addOne, S);
}

// reciprocal_space.pyx:89-122: sq = ones; sq[q] += dr*(sin(q*r)/q)*Gr[r]
// (Cython: q*r a float32 product; sin, the division and the products in
// double; the += in double, rounded to the float32 element).
__global__ void __launch_bounds__(256) k_Gr_to_sq(const float *__restrict__ dist, const float *__restrict__ Gr,
                                                  int32_t n, const float *__restrict__ qr, int32_t m,
                                                  float *__restrict__ sq) {
    __shared__ float rs[kGChunk], gs[kGChunk];
    const int32_t qi = blockIdx.x * blockDim.x + threadIdx.x;
    const float q = qr[min(qi, m - 1)];
    const float dr = load_dev(dist + 1) - load_dev(dist);
    float acc = 1.0f;
    for (int32_t c0 = 0; c0 < n; c0 += kGChunk) {
        const int32_t len = min(kGChunk, n - c0);
        __syncthreads();
        for (int32_t i = threadIdx.x; i < len; i += blockDim.x) {
            rs[i] = dist[c0 + i];
            gs[i] = Gr[c0 + i];
        }
        __syncthreads();
        for (int32_t i = 0; i < len; i++) {
            const float x = q * rs[i];
            double t = sin((double)x) / (double)q;
            t = (double)dr * t;
            t = t * (double)gs[i];
            acc = (float)((double)acc + t);
        }
    }
    if (qi < m) sq[qi] = acc;
}

// reciprocal_space.pyx:42-80: fact = 4*PI*rho (float32, PI = 3.1415927);
// sq[q] += fact*(dr*r*(sin(q*r)/q)*(gr[r]-1)) with dr*r and gr[r]-1 in
// float32 and the rest as above.
__global__ void __launch_bounds__(256) k_gr_to_sq(const float *__restrict__ dist, const float *__restrict__ gr,
                                                  int32_t n, const float *__restrict__ qr, int32_t m, float rho,
                                                  float *__restrict__ sq) {
    __shared__ float rs[kGChunk], gs[kGChunk];
    const int32_t qi = blockIdx.x * blockDim.x + threadIdx.x;
    const float q = qr[min(qi, m - 1)];
    const float dr = load_dev(dist + 1) - load_dev(dist);
    float fact = 4.0f * 3.1415927f;
    fact = fact * rho;
    float acc = 1.0f;
    for (int32_t c0 = 0; c0 < n; c0 += kGChunk) {
        const int32_t len = min(kGChunk, n - c0);
        __syncthreads();
        for (int32_t i = threadIdx.x; i < len; i += blockDim.x) {
            rs[i] = dist[c0 + i];
            gs[i] = gr[c0 + i];
        }
        __syncthreads();
        for (int32_t i = 0; i < len; i++) {
            const float r = rs[i];
            const float drr = dr * r;
            const float x = q * r;
            double t = sin((double)x) / (double)q;
            t = (double)drr * t;
            const float g1 = gs[i] - 1.0f;
            t = t * (double)g1;
            t = (double)fact * t;
            acc = (float)((double)acc + t);
        }
    }
    if (qi < m) sq[qi] = acc;
}

// G(r) = (2/PI) * sum_q Q (S(Q)-1) dq sin(Q r), dq = qValues[1]-qValues[0],
// evaluated in double and rounded once.
__global__ void __launch_bounds__(256) k_sq_to_Gr(const float *__restrict__ qv, const float *__restrict__ rv,
                                                  int32_t nr, const float *__restrict__ sq, int32_t m,
                                                  float *__restrict__ Gr) {
    __shared__ float qs[kGChunk], ss[kGChunk];
    const int32_t ri = blockIdx.x * blockDim.x + threadIdx.x;
    const double r = (double)rv[min(ri, nr - 1)];
    const double dq = (double)load_dev(qv + 1) - (double)load_dev(qv);
    double acc = 0.0;
    for (int32_t c0 = 0; c0 < m; c0 += kGChunk) {
        const int32_t len = min(kGChunk, m - c0);
        __syncthreads();
        for (int32_t i = threadIdx.x; i < len; i += blockDim.x) {
            qs[i] = qv[c0 + i];
            ss[i] = sq[c0 + i];
        }
        __syncthreads();
        for (int32_t i = 0; i < len; i++) {
            const double q = (double)qs[i];
            acc += q * ((double)ss[i] - 1.0) * sin(q * r);
        }
    }
    if (ri < nr) Gr[ri] = (float)(2.0 / 3.141592653589793 * dq * acc);
}

}  // namespace

}  // namespace frmc

using namespace frmc;

namespace {

// HIP events around the transform kernels when per-thread timing is on
// (frmc_set_timing); the stop synchronises and sets frmc_last_kernel_ms.
struct KernelTimer {
    hipEvent_t a = nullptr, b = nullptr;
    bool on = false;
    hipError_t start(hipStream_t st) {
        on = timing_enabled();
        if (!on) return hipSuccess;
        hipError_t e = hipEventCreate(&a);
        if (e == hipSuccess) e = hipEventCreate(&b);
        if (e == hipSuccess) e = hipEventRecord(a, st);
        return e;
    }
    hipError_t stop(hipStream_t st) {
        if (!on) return hipSuccess;
        float ms = 0.f;
        hipError_t e = hipEventRecord(b, st);
        if (e == hipSuccess) e = hipEventSynchronize(b);
        if (e == hipSuccess) e = hipEventElapsedTime(&ms, a, b);
        set_last_kernel_ms(ms);
        return e;
    }
    ~KernelTimer() {
        if (a) (void)hipEventDestroy(a);
        if (b) (void)hipEventDestroy(b);
    }
};

}  // namespace

extern "C" int frmc_sq_transform(const float *Gr, int32_t k, int32_t H, const float *sqMatrix, int32_t nQ,
                                 int addOne, int mode, float *Sq, void *stream) {
    FRMC_REQUIRE(k >= 0 && H >= 1 && nQ >= 0, "sq_transform: bad sizes k=%d H=%d nQ=%d", k, H, nQ);
    FRMC_REQUIRE(mode == FRMC_SQ_EXACT || mode == FRMC_SQ_MFMA, "sq_transform: unknown mode %d", mode);
    if (k == 0 || nQ == 0) return FRMC_OK;
    FRMC_REQUIRE(Gr && sqMatrix && Sq, "sq_transform: NULL array");
    FRMC_REQUIRE((int64_t)H * nQ < ((int64_t)1 << 40), "sq_transform: matrix too large");
    hipStream_t st = as_stream(stream);
    KernelTimer timer;
    if (mode == FRMC_SQ_EXACT)
        FRMC_REQUIRE(k <= 65535, "sq_transform: at most 65535 curves per call");
    else
        FRMC_REQUIRE(k <= kMaxCurves, "sq_transform: too many curves per call");
    const SqPlan P = sq_plan(k, H, nQ);
    float *part = nullptr;
    if (mode == FRMC_SQ_MFMA && P.tiles && P.nsplit > 1) {
        const hipError_t e = pool_malloc((void **)&part, sizeof(float) * P.nsplit * k * nQ, st);
        if (e != hipSuccess) {
            set_error("hipMallocAsync of the split partials failed: %s", hipGetErrorString(e));
            return FRMC_ENOMEM;
        }
    }
    hipError_t le = timer.start(st);
    if (le == hipSuccess) {
        if (mode == FRMC_SQ_EXACT) launch_sq_exact(Gr, k, H, sqMatrix, nQ, addOne != 0, Sq, st);
        else if (P.tiles) launch_sq_tiles(P, Gr, k, H, sqMatrix, nQ, addOne != 0, part, Sq, st);
        else launch_sq_mfma(Gr, k, H, sqMatrix, nQ, addOne != 0, Sq, st);
        le = hipGetLastError();
    }
    if (le == hipSuccess) le = timer.stop(st);
    if (part) (void)hipFreeAsync(part, st);
    if (le != hipSuccess) {
        set_error("sq_transform failed: %s", hipGetErrorString(le));
        return FRMC_EHIP;
    }
    return FRMC_OK;
}

// ------------------------------------------------- no-allocation variant
//
// The large matrix-core tiles' split partials in a file-scope device array
// instead of stream-ordered pool memory, for callers that cannot allocate
// (code under HIP graph capture, allocation-free serving loops).  Each GPU
// the library runs on holds its own copy (16 MiB) until the process ends.
// Every call on a GPU shares that GPU's copy, and the next call overwrites
// it: calls of such shapes that overlap on one GPU (other streams, other threads)
// race.
// k_sq_tiles stores every partial element it owns, so nothing needs clearing.
constexpr int64_t kSqScratchFloats = (int64_t)1 << 22;
static __device__ __align__(256) float scratch[kSqScratchFloats];

static std::mutex g_sq_scratch_mu;
static float *g_sq_scratch[64] = {nullptr};  // device address of scratch, per device

// This device's copy of scratch: its address is taken once per device
// (with that device current), then reused; host code never uses the
// symbol itself, which is only a host-side stand-in.
static int sq_scratch_of_current_device(float **out) {
    int dev = 0;
    FRMC_CHECK_HIP(hipGetDevice(&dev));
    FRMC_REQUIRE(dev >= 0 && dev < 64, "sq_transform_noalloc: device %d out of range", dev);
    std::lock_guard<std::mutex> lock(g_sq_scratch_mu);
    if (!g_sq_scratch[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            set_error("sq_transform_noalloc: hipGetSymbolAddress of the scratch array failed: %s",
                      hipGetErrorString(e));
            return FRMC_EHIP;
        }
        g_sq_scratch[dev] = (float *)p;
    }
    *out = g_sq_scratch[dev];
    return FRMC_OK;
}

extern "C" int frmc_sq_transform_noalloc(const float *Gr, int32_t k, int32_t H, const float *sqMatrix, int32_t nQ,
                                         int addOne, int mode, float *Sq, void *stream) {
    FRMC_REQUIRE(k >= 0 && H >= 1 && nQ >= 0, "sq_transform_noalloc: bad sizes k=%d H=%d nQ=%d", k, H, nQ);
    FRMC_REQUIRE(mode == FRMC_SQ_EXACT || mode == FRMC_SQ_MFMA, "sq_transform_noalloc: unknown mode %d", mode);
    if (k == 0 || nQ == 0) return FRMC_OK;
    FRMC_REQUIRE(Gr && sqMatrix && Sq, "sq_transform_noalloc: NULL array");
    FRMC_REQUIRE((int64_t)H * nQ < ((int64_t)1 << 40), "sq_transform_noalloc: matrix too large");
    hipStream_t st = as_stream(stream);
    if (mode == FRMC_SQ_EXACT) {
        FRMC_REQUIRE(k <= 65535, "sq_transform_noalloc: at most 65535 curves per call");
        launch_sq_exact(Gr, k, H, sqMatrix, nQ, addOne != 0, Sq, st);
        FRMC_CHECK_LAUNCH();
        return FRMC_OK;
    }
    FRMC_REQUIRE(k <= kMaxCurves, "sq_transform_noalloc: too many curves per call");
    const SqPlan P = sq_plan(k, H, nQ);
    // the limit of the split partials holds for every shape, also those whose tiles need none
    const int64_t need = P.nsplit * k * nQ;
    FRMC_REQUIRE(P.nsplit == 1 || need <= kSqScratchFloats,
                 "sq_transform_noalloc: k=%d, H=%d, nQ=%d is past this entry's limit of matrix-core shapes "
                 "(%lld parts of the r range, %lld results in all, at most %lld): use frmc_sq_transform",
                 k, H, nQ, (long long)P.nsplit, (long long)need, (long long)kSqScratchFloats);
    float *part = nullptr;
    if (P.tiles && P.nsplit > 1)
        if (int rc = sq_scratch_of_current_device(&part)) return rc;
    if (P.tiles) launch_sq_tiles(P, Gr, k, H, sqMatrix, nQ, addOne != 0, part, Sq, st);
    else launch_sq_mfma(Gr, k, H, sqMatrix, nQ, addOne != 0, Sq, st);
    FRMC_CHECK_LAUNCH();
    return FRMC_OK;
}

extern "C" int frmc_Gr_to_sq(const float *distances, const float *Gr, int32_t n, const float *qrange, int32_t m,
                             float *sq, void *stream) {
    FRMC_REQUIRE(n >= 2 && m >= 0, "Gr_to_sq: need at least two distances (n=%d)", n);
    if (m == 0) return FRMC_OK;
    FRMC_REQUIRE(distances && Gr && qrange && sq, "Gr_to_sq: NULL array");
    hipLaunchKernelGGL(k_Gr_to_sq, dim3(blocks_for(m, 256)), dim3(256), 0, as_stream(stream), distances, Gr, n,
                       qrange, m, sq);
    FRMC_CHECK_LAUNCH();
    return FRMC_OK;
}

extern "C" int frmc_gr_to_sq(const float *distances, const float *gr, int32_t n, const float *qrange, int32_t m,
                             float rho, float *sq, void *stream) {
    FRMC_REQUIRE(n >= 2 && m >= 0, "gr_to_sq: need at least two distances (n=%d)", n);
    if (m == 0) return FRMC_OK;
    FRMC_REQUIRE(distances && gr && qrange && sq, "gr_to_sq: NULL array");
    hipLaunchKernelGGL(k_gr_to_sq, dim3(blocks_for(m, 256)), dim3(256), 0, as_stream(stream), distances, gr, n,
                       qrange, m, rho, sq);
    FRMC_CHECK_LAUNCH();
    return FRMC_OK;
}

extern "C" int frmc_sq_to_Gr(const float *qValues, const float *rValues, int32_t nr, const float *sq, int32_t m,
                             float *Gr, void *stream) {
    FRMC_REQUIRE(m >= 2 && nr >= 0, "sq_to_Gr: need at least two Q values (m=%d)", m);
    if (nr == 0) return FRMC_OK;
    FRMC_REQUIRE(qValues && rValues && sq && Gr, "sq_to_Gr: NULL array");
    hipLaunchKernelGGL(k_sq_to_Gr, dim3(blocks_for(nr, 256)), dim3(256), 0, as_stream(stream), qValues, rValues,
                       nr, sq, m, Gr);
    FRMC_CHECK_LAUNCH();
    return FRMC_OK;
}
