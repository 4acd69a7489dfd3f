// distances.hip -- pairs_distances entry points on gfx950.
//
// One kernel family computes "point vs all atoms" distances or differences
// for k points at once; the point is either an atom of the array (index mode) or
// an explicit (3,k) column (point mode).  The basis is read from device memory
// by every thread (scalar loads, uniform), so no host synchronisation is needed
// per call.
#include "frmc_device.h"
#include "frmc_host.h"

namespace frmc {

enum PointMode { PM_INDEX = 0, PM_POINTS = 1 };

__device__ __forceinline__ void load_basis_dev(const float *__restrict__ basis, Basis &B) {
#pragma unroll
    for (int k = 0; k < 9; k++) B.b[k] = basis[k];
}

// out layout: distances (n,k) -> out[i*k+c]; differences (n,3,k) -> out[(i*3+d)*k+c]
//
// A workgroup takes `rows` atoms and up to kVsCols points, both staged in LDS,
// and walks the tile's elements in output order, so a wave's stores are
// contiguous.  Bound by those stores and the launch; with a point per workgroup
// row and stores k floats apart, 64 points x 20,000 atoms took 17.8 us a call
// against 7.4.
constexpr int kVsCols = 256, kVsRows = 256;

template <bool PBC, bool DIFF>
__global__ void __launch_bounds__(256) k_vs_all(const float *__restrict__ coords, int32_t n,
                                                const float *__restrict__ basis, int mode,
                                                const int32_t *__restrict__ indexes, int32_t atomIndex,
                                                const float *__restrict__ points, int32_t k, int allAtoms, int32_t rows,
                                                float *__restrict__ out) {
    __shared__ float px[3][kVsCols], cx[3][kVsRows];
    __shared__ int32_t first[kVsCols];  // first row of the column that is written
    const int32_t t = threadIdx.x, i0 = blockIdx.x * rows, c0 = blockIdx.y * kVsCols;
    const int32_t ni = min(rows, n - i0), nc = min(kVsCols, k - c0);
    if (t < nc) {
        const int32_t c = c0 + t;
        int32_t from = 0;
        if (mode == PM_INDEX) {
            const int32_t a = indexes ? indexes[c] : atomIndex;
            const bool ok = a >= 0 && a < n;  // out-of-range index: nothing written (host shim rejects it)
            // reference leaves [0,atomIndex) uninitialised
            from = !ok ? 0x7fffffff : allAtoms ? 0 : a;
#pragma unroll
            for (int d = 0; d < 3; d++) px[d][t] = ok ? coords[3 * (int64_t)a + d] : 0.0f;
        } else {
#pragma unroll
            for (int d = 0; d < 3; d++) px[d][t] = points[(int64_t)d * k + c];
        }
        first[t] = from;
    }
    for (int32_t e = t; e < 3 * ni; e += 256) cx[e % 3][e / 3] = coords[3 * (int64_t)i0 + e];
    Basis B;
    if (PBC) load_basis_dev(basis, B);
    __syncthreads();
    const int32_t di = 256 / nc, dc = 256 % nc;
    int32_t i = t / nc, c = t % nc;
    while (i < ni) {
        if (i0 + i >= first[c]) {
            // pairs_distances.pyx:373-375 / 461-463: diff = point - coords[i]
            const float dx = px[0][c] - cx[0][i], dy = px[1][c] - cx[1][i], dz = px[2][c] - cx[2][i];
            float rx = dx, ry = dy, rz = dz;
            if (PBC) pbc_real(dx, dy, dz, B, rx, ry, rz);
            const int64_t row = i0 + i, col = c0 + c;
            if (DIFF) {
                out[(row * 3 + 0) * k + col] = rx;
                out[(row * 3 + 1) * k + col] = ry;
                out[(row * 3 + 2) * k + col] = rz;
            } else {
                out[row * k + col] = cr_sqrt(norm2(rx, ry, rz));
            }
        }
        i += di;
        c += dc;
        if (c >= nc) {
            c -= nc;
            i++;
        }
    }
}

// One point against all atoms (k = 1): `per` atoms a thread.  Bound by the
// coordinates' reads and the results' stores; staged as above, 8,000,000 atoms took 47 us
// against 21.  The point comes through lane-varying loads (see load_dev; uniform
// coherent loads past the L1 cache: 30 us).
constexpr int32_t kPointRows = 1 << 20;  // four atoms a thread beyond

template <bool PBC, bool DIFF>
__global__ void __launch_bounds__(256) k_point_vs_all(const float *__restrict__ coords, int32_t n,
                                                      const float *__restrict__ basis, int mode,
                                                      const int32_t *__restrict__ indexes, int32_t atomIndex,
                                                      const float *__restrict__ points, int32_t k, int allAtoms,
                                                      int32_t per, float *__restrict__ out) {
    const int32_t c = min((int32_t)(threadIdx.x & 63), k - 1);  // 0
    int32_t from = 0;
    const float *point = points + c;
    if (mode == PM_INDEX) {
        const int32_t a = indexes ? indexes[c] : atomIndex + c;
        if (a < 0 || a >= n) return;  // out-of-range index: nothing written (host shim rejects it)
        point = coords + 3 * (int64_t)a;
        from = allAtoms ? 0 : a;  // reference leaves [0,atomIndex) uninitialised
    }
    const float px = point[0], py = point[1], pz = point[2];
    Basis B;
    if (PBC) load_basis_dev(basis, B);
    const int64_t i0 = (int64_t)blockIdx.x * 256 * per + threadIdx.x, i1 = min((int64_t)n, i0 + 256 * (int64_t)per);
#pragma unroll 4
    for (int64_t i = i0; i < i1; i += 256) {
        if (i < from) continue;
        // pairs_distances.pyx:373-375 / 461-463: diff = point - coords[i]
        const float dx = px - coords[3 * i], dy = py - coords[3 * i + 1], dz = pz - coords[3 * i + 2];
        float rx = dx, ry = dy, rz = dz;
        if (PBC) pbc_real(dx, dy, dz, B, rx, ry, rz);
        if (DIFF) {
            out[3 * i] = rx;
            out[3 * i + 1] = ry;
            out[3 * i + 2] = rz;
        } else {
            out[i] = cr_sqrt(norm2(rx, ry, rz));
        }
    }
}

// Row-wise pairs: from_to_points_differences (diff = to[i]-from[i]),
// pair_difference_to_point (n=1, diff = p2-p1), point_to_point_distance
// (n=1, diff = p1-p2, distance).
template <bool PBC, bool DIFF>
__global__ void __launch_bounds__(256) k_rowwise(const float *__restrict__ a, const float *__restrict__ b,
                                                 int32_t n, const float *__restrict__ basis,
                                                 float *__restrict__ out) {
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float dx = a[3 * (int64_t)i] - b[3 * (int64_t)i];
    float dy = a[3 * (int64_t)i + 1] - b[3 * (int64_t)i + 1];
    float dz = a[3 * (int64_t)i + 2] - b[3 * (int64_t)i + 2];
    float rx, ry, rz;
    if (PBC) {
        Basis B;
        load_basis_dev(basis, B);
        pbc_real(dx, dy, dz, B, rx, ry, rz);
    } else {
        rx = dx;
        ry = dy;
        rz = dz;
    }
    if (DIFF) {
        out[3 * (int64_t)i] = rx;
        out[3 * (int64_t)i + 1] = ry;
        out[3 * (int64_t)i + 2] = rz;
    } else {
        out[i] = cr_sqrt(norm2(rx, ry, rz));
    }
}

static int launch_vs_all(bool diff, const float *coords, int32_t n, const float *basis, int isPBC, int mode,
                         const int32_t *indexes, int32_t atomIndex, const float *points, int32_t k, int allAtoms,
                         float *out, void *stream) {
    FRMC_REQUIRE(n >= 0 && k >= 0, "negative size (n=%d, k=%d)", n, k);
    FRMC_REQUIRE(coords != nullptr || n == 0, "coords is NULL");
    FRMC_REQUIRE(out != nullptr || n == 0 || k == 0, "out is NULL");
    FRMC_REQUIRE(!isPBC || basis != nullptr, "basis is NULL");
    if (n == 0 || k == 0) return FRMC_OK;
    FRMC_REQUIRE(k <= 65535, "too many points (k=%d > 65535)", k);
    hipStream_t st = as_stream(stream);
    if (k == 1) {
        const int32_t per = n > kPointRows ? 4 : 1;
        const unsigned blocks = blocks_for(n, 256 * per);
        if (isPBC && diff)
            k_point_vs_all<true, true><<<blocks, 256, 0, st>>>(coords, n, basis, mode, indexes, atomIndex, points, k,
                                                               allAtoms, per, out);
        else if (isPBC)
            k_point_vs_all<true, false><<<blocks, 256, 0, st>>>(coords, n, basis, mode, indexes, atomIndex, points, k,
                                                                allAtoms, per, out);
        else if (diff)
            k_point_vs_all<false, true><<<blocks, 256, 0, st>>>(coords, n, basis, mode, indexes, atomIndex, points, k,
                                                                allAtoms, per, out);
        else
            k_point_vs_all<false, false><<<blocks, 256, 0, st>>>(coords, n, basis, mode, indexes, atomIndex, points, k,
                                                                 allAtoms, per, out);
        FRMC_CHECK_LAUNCH();
        return FRMC_OK;
    }
    // about 4,096 elements per workgroup
    const int32_t nc = k < kVsCols ? k : kVsCols;
    const int32_t rows = 4096 / nc < kVsRows ? (4096 / nc < 1 ? 1 : 4096 / nc) : kVsRows;
    dim3 grid(blocks_for(n, rows), (unsigned)((k + kVsCols - 1) / kVsCols));
    if (isPBC) {
        if (diff)
            k_vs_all<true, true><<<grid, 256, 0, st>>>(coords, n, basis, mode, indexes, atomIndex, points, k,
                                                       allAtoms, rows, out);
        else
            k_vs_all<true, false><<<grid, 256, 0, st>>>(coords, n, basis, mode, indexes, atomIndex, points, k,
                                                        allAtoms, rows, out);
    } else {
        if (diff)
            k_vs_all<false, true><<<grid, 256, 0, st>>>(coords, n, basis, mode, indexes, atomIndex, points, k,
                                                        allAtoms, rows, out);
        else
            k_vs_all<false, false><<<grid, 256, 0, st>>>(coords, n, basis, mode, indexes, atomIndex, points,
                                                         k, allAtoms, rows, out);
    }
    FRMC_CHECK_LAUNCH();
    return FRMC_OK;
}

static int launch_rowwise(bool diff, const float *a, const float *b, int32_t n, const float *basis, int isPBC,
                          float *out, void *stream) {
    FRMC_REQUIRE(n >= 0, "negative size");
    FRMC_REQUIRE(!isPBC || basis != nullptr, "basis is NULL");
    if (n == 0) return FRMC_OK;
    FRMC_REQUIRE(a && b && out, "NULL pointer argument");
    hipStream_t st = as_stream(stream);
    unsigned g = blocks_for(n, 256);
    if (isPBC) {
        if (diff) k_rowwise<true, true><<<g, 256, 0, st>>>(a, b, n, basis, out);
        else      k_rowwise<true, false><<<g, 256, 0, st>>>(a, b, n, basis, out);
    } else {
        if (diff) k_rowwise<false, true><<<g, 256, 0, st>>>(a, b, n, basis, out);
        else      k_rowwise<false, false><<<g, 256, 0, st>>>(a, b, n, basis, out);
    }
    FRMC_CHECK_LAUNCH();
    return FRMC_OK;
}

}  // namespace frmc

using namespace frmc;

extern "C" {

int frmc_pairs_distances_to_indexcoords(int32_t atomIndex, const float *coords, int32_t n, const float *basis,
                                        int isPBC, int allAtoms, float *out, void *stream) {
    FRMC_REQUIRE(atomIndex >= 0 && atomIndex < n, "atomIndex %d out of range [0,%d)", atomIndex, n);
    return launch_vs_all(false, coords, n, basis, isPBC, PM_INDEX, nullptr, atomIndex, nullptr, 1, allAtoms, out,
                         stream);
}

int frmc_pairs_distances_to_multi_indexcoords(const int32_t *indexes, int32_t k, const float *coords, int32_t n,
                                              const float *basis, int isPBC, int allAtoms, float *out,
                                              void *stream) {
    FRMC_REQUIRE(indexes != nullptr || k == 0, "indexes is NULL");
    return launch_vs_all(false, coords, n, basis, isPBC, PM_INDEX, indexes, 0, nullptr, k, allAtoms, out, stream);
}

int frmc_pairs_distances_to_point(const float *point, const float *coords, int32_t n, const float *basis,
                                  int isPBC, float *out, void *stream) {
    FRMC_REQUIRE(point != nullptr, "point is NULL");
    return launch_vs_all(false, coords, n, basis, isPBC, PM_POINTS, nullptr, 0, point, 1, 1, out, stream);
}

int frmc_pairs_distances_to_multi_points(const float *points, int32_t k, const float *coords, int32_t n,
                                         const float *basis, int isPBC, float *out, void *stream) {
    FRMC_REQUIRE(points != nullptr || k == 0, "points is NULL");
    return launch_vs_all(false, coords, n, basis, isPBC, PM_POINTS, nullptr, 0, points, k, 1, out, stream);
}

int frmc_point_to_point_distance(const float *point1, const float *point2, const float *basis, int isPBC,
                                 float *out, void *stream) {
    // pairs_distances.pyx:256-282: diff = point1 - point2
    return launch_rowwise(false, point1, point2, 1, basis, isPBC, out, stream);
}

int frmc_pairs_differences_to_indexcoords(int32_t atomIndex, const float *coords, int32_t n, const float *basis,
                                          int isPBC, int allAtoms, float *out, void *stream) {
    FRMC_REQUIRE(atomIndex >= 0 && atomIndex < n, "atomIndex %d out of range [0,%d)", atomIndex, n);
    return launch_vs_all(true, coords, n, basis, isPBC, PM_INDEX, nullptr, atomIndex, nullptr, 1, allAtoms, out,
                         stream);
}

int frmc_pairs_differences_to_multi_indexcoords(const int32_t *indexes, int32_t k, const float *coords,
                                                int32_t n, const float *basis, int isPBC, int allAtoms,
                                                float *out, void *stream) {
    FRMC_REQUIRE(indexes != nullptr || k == 0, "indexes is NULL");
    return launch_vs_all(true, coords, n, basis, isPBC, PM_INDEX, indexes, 0, nullptr, k, allAtoms, out, stream);
}

int frmc_pairs_differences_to_point(const float *point, const float *coords, int32_t n, const float *basis,
                                    int isPBC, float *out, void *stream) {
    FRMC_REQUIRE(point != nullptr, "point is NULL");
    return launch_vs_all(true, coords, n, basis, isPBC, PM_POINTS, nullptr, 0, point, 1, 1, out, stream);
}

int frmc_pairs_differences_to_multi_points(const float *points, int32_t k, const float *coords, int32_t n,
                                           const float *basis, int isPBC, float *out, void *stream) {
    FRMC_REQUIRE(points != nullptr || k == 0, "points is NULL");
    return launch_vs_all(true, coords, n, basis, isPBC, PM_POINTS, nullptr, 0, points, k, 1, out, stream);
}

int frmc_from_to_points_differences(const float *pointsFrom, const float *pointsTo, int32_t n,
                                    const float *basis, int isPBC, float *out, void *stream) {
    // pairs_distances.pyx:84-93 / 127-132: diff = to[i] - from[i]
    return launch_rowwise(true, pointsTo, pointsFrom, n, basis, isPBC, out, stream);
}

int frmc_pair_difference_to_point(const float *point1, const float *point2, const float *basis, int isPBC,
                                  float *out, void *stream) {
    // pairs_distances.pyx:54-59 / 108-114: diff = point2 - point1
    return launch_rowwise(true, point2, point1, 1, basis, isPBC, out, stream);
}

}  // extern "C"
