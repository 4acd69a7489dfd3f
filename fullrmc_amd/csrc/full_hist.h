// full_hist.h -- shared by the two full-histogram kernels: the binary64 bin of a
// pair (histograms.hip, k_full_pairs; full_chunks.hip, k_full_chunks) and the
// chunk-pruned pass's host entry.
#pragma once
#include "frmc_device.h"
#include "frmc_host.h"

namespace frmc {

// Float64 edge re-check (EDGE mode): the histogram of the binary64 recompute
// (every pair's distance evaluated in double from the float32 coordinates,
// range and bin in double).  The float32 distance d32 of a pair is within
// eps = 8u*(sum_m (|dx_m|+1)*rowsum_m + d32) of the double one (u = 2^-24;
// error analysis of the float32 difference, the exact minimum-image
// subtraction, the 3-term basis product, the squared norm and the rounded
// sqrt, with a factor > 2 to spare); a pair whose d32 lies farther than eps
// from every bin edge and range end, and whose fractional components are not
// within a rounding tie of +-1/2, takes its bin from d32; every other pair is
// recomputed in double.
struct Edge64 {
    double mn, mx, bn;      // the grid in double
    float s_lo, s_hi;       // candidate window of float32 squared norms
    float rowsum[3];        // sum_k |B[m][k]| per basis row (PBC), 1 otherwise
    float amax;             // largest |coordinate|
};

__device__ __forceinline__ double round64(double x) { return x > 0.0 ? floor(x + 0.5) : ceil(x - 0.5); }

template <bool PBC>
__device__ __forceinline__ double pair_d64(float ax, float ay, float az, float cx, float cy, float cz,
                                           const Basis &B) {
    const double dx = (double)ax - (double)cx, dy = (double)ay - (double)cy, dz = (double)az - (double)cz;
    double rx = dx, ry = dy, rz = dz;
    if (PBC) {
        const double bx = dx - round64(dx), by = dy - round64(dy), bz = dz - round64(dz);
        rx = (bx * (double)B.b[0] + by * (double)B.b[3]) + bz * (double)B.b[6];
        ry = (bx * (double)B.b[1] + by * (double)B.b[4]) + bz * (double)B.b[7];
        rz = (bx * (double)B.b[2] + by * (double)B.b[5]) + bz * (double)B.b[8];
    }
    return __builtin_sqrt((rx * rx + ry * ry) + rz * rz);
}

// Bin of a candidate pair in the binary64 recompute, or -1 out of range;
// *rechecked is set when the pair needed the double evaluation.
template <bool PBC>
__device__ __forceinline__ int64_t edge_bin(float s, float ax, float ay, float az, float cx, float cy, float cz,
                                            const Basis &B, const Edge64 &E, bool &rechecked) {
    const float dx = ax - cx, dy = ay - cy, dz = az - cz;
    const float d32 = cr_sqrt(s);
    const float bound = (fabsf(dx) + 1.0f) * E.rowsum[0] + (fabsf(dy) + 1.0f) * E.rowsum[1] +
                        (fabsf(dz) + 1.0f) * E.rowsum[2] + d32;
    const double eps = 8.0 * 5.9604644775390625e-08 * 1.001 * (double)bound;
    bool tie = false;
    if (PBC) {
        // fractional differences near +-1/2: float and double may pick different images
        tie = fabsf(0.5f - fabsf(min_image(dx))) <= 4.8e-7f * (fabsf(dx) + 1.0f) ||
              fabsf(0.5f - fabsf(min_image(dy))) <= 4.8e-7f * (fabsf(dy) + 1.0f) ||
              fabsf(0.5f - fabsf(min_image(dz))) <= 4.8e-7f * (fabsf(dz) + 1.0f);
    }
    const double t = ((double)d32 - E.mn) / E.bn;
    const double kf = floor(t);
    const double margin = fmin(t - kf, kf + 1.0 - t) * E.bn;
    rechecked = tie || margin <= eps || fabs((double)d32 - E.mn) <= eps || fabs((double)d32 - E.mx) <= eps;
    if (rechecked) {
        const double d = pair_d64<PBC>(ax, ay, az, cx, cy, cz, B);
        if (d < E.mn || d >= E.mx) return -1;
        return (int64_t)((d - E.mn) / E.bn);
    }
    if ((double)d32 < E.mn || (double)d32 >= E.mx) return -1;
    return (int64_t)kf;
}

// A chunk-pruned pass over all unordered pairs (full_chunks.hip).
struct ChunkRun {
    int32_t nt = 0;             // threads per workgroup: 256, 512 or 1024 (fewer if LDS does not hold them), 0: by rule
    int32_t *used_nt = nullptr; // threads launched
    int32_t per_cu = 0;         // workgroups per CU, 0: as many as fit
    int64_t *blocks = nullptr;  // workgroups launched
    int64_t *pairs = nullptr;   // host word for the pairs evaluated, or null: not counted
    // the result: added into counts ([2][nel][nel][H], overflow, re-checks),
    // or written as the float32 histograms, the lost pairs to a host word
    int32_t *counts = nullptr;
    float *hintra = nullptr, *hinter = nullptr;
    int64_t *overflow = nullptr;
};
// whether run_chunks takes these inputs (packed atom ids and elements, 32-bit offsets of bins)
bool chunks_take(int32_t n, const HistArgs &A);
// every unordered pair's bin; the basis from dbasis (device memory), else hB
int run_chunks(const ChunkRun &R, const float *coords, int32_t n, const float *dbasis, const Basis &hB, int isPBC,
               const int32_t *mol, const int32_t *elem, const HistArgs &A, const Edge64 *E, int ncu, hipStream_t st);
// counts += the sum over nparts partials of 2 size slots each, stored with the
// inter-molecular half first
int add_partials(const int32_t *partial, int64_t nparts, int64_t size, int32_t *counts, hipStream_t st);

}  // namespace frmc
