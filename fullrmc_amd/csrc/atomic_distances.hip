// atomic_distances.hip -- the atomic_distances extension
// (Extensions/atomic_distances.pyx) on gfx950: per element pair, the number
// and the float32 sum of the (reduced) distances of atom pairs that pass the
// molecule and distance-limit filters, as InterMolecularDistanceConstraint
// and IntraMolecularDistanceConstraint use them.
//
// The reference adds each selected distance to its slot in a fixed order
// (atoms in `indexes` order, then other atoms by index), and float32
// addition is not associative, so the sums are rebuilt in that order:
//   k_ad_pass    every (atom, other atom) pair in parallel, or k_ad_chunks the
//                pairs near enough to be inside the limits (chunks.h): filters,
//                per-slot counts (LDS, then global atomics), each selected pair
//                as a 64-bit key (slot, atom position, other index) and its value
//   k_ad_few     up to kFew selected pairs: sorted and summed in one workgroup
//   radix sort   more of them: rocPRIM, by key: each slot's terms become
//                contiguous and in the reference's order
//   k_ad_sum     one workgroup per slot adds its terms sequentially onto the
//                slot's existing float32 value and adds the count
// Counts are integers and need no order.  The host waits once, for the number
// of selected pairs.
//
// Measured (MI355X, whole calls): all close pairs (2.6 A) of 13,500 atoms 155 us
// against 1,600 (two passes of a workgroup per 256 pairs, sums with one memory
// access per add); 13 atoms against 13,500 63 against 139.  What is left: the
// sort of the keys, the sequential sums (34 us for 9,100 terms per slot, 9
// cycles per dependent add) and the launches.
#include <rocprim/device/device_radix_sort.hpp>
#include <algorithm>

#include "chunks.h"

namespace frmc {

namespace {

enum AdSource { AD_PBC = 0, AD_IBC = 1, AD_DISTS = 2 };

struct AdArgs {
    const float *coords;     // (n,3) box (PBC) or real (IBC) coordinates, or NULL
    const float *dists;      // (n,k) distances, or NULL
    int32_t n, k;            // atoms (rows), atoms in the index list (columns of dists)
    const float *basis;      // (3,3) or NULL
    const int32_t *indexes;  // [k] atom of each column, or NULL: atomIndex
    int32_t atomIndex;
    const int32_t *mol, *elem;
    int32_t nel;
    const float *lower, *upper;  // [nel][nel], read as [other][atom]
    int32_t flags, allAtoms;
};

// Where the selected pairs go: the slots' counts, the pairs' number, and as many
// keys and values as the buffers hold.
struct AdOut {
    uint32_t *cnt;              // [2*nel*nel], or NULL: counted before
    unsigned long long *total;
    unsigned long long cap;
    int32_t shift;              // bits of (list position, other atom) below the slot
    uint64_t *keys;
    float *vals;
};

// the basis through one lane-varying load and broadcasts (see load_dev)
__device__ __forceinline__ Basis basis_of(const float *basis) {
    Basis B;
    const int v = __float_as_int(basis[min((int)(threadIdx.x & 63), 8)]);
#pragma unroll
    for (int k = 0; k < 9; k++) B.b[k] = __int_as_float(__builtin_amdgcn_readlane(v, k));
    return B;
}

// distance as pairs_distances computes it (pairs_distances.pyx:343-386 / :438-471: diff = coords[a] - coords[i])
template <bool PBC>
__device__ __forceinline__ float ad_distance(const Basis &B, float px, float py, float pz, float x, float y, float z) {
    const float dx = px - x, dy = py - y, dz = pz - z;
    float rx = dx, ry = dy, rz = dz;
    if (PBC) pbc_real(dx, dy, dz, B, rx, ry, rz);
    return cr_sqrt(norm2(rx, ry, rz));
}

// _single_atomic_distances_dists (atomic_distances.pyx:42-118) for one pair:
// true if counted, with the counted value and the slot
// ws = (0 intra | 1 inter)*nel*nel + e_atom*nel + e_other.
__device__ __forceinline__ bool ad_select(const AdArgs &A, float d, bool same, int32_t ei, int32_t ea, float &v,
                                          int32_t &ws) {
    if (!(A.flags & FRMC_AD_INTRA) && same) return false;
    if (!(A.flags & FRMC_AD_INTER) && !same) return false;
    const float lower = A.lower[ei * A.nel + ea], upper = A.upper[ei * A.nel + ea];
    if (A.flags & FRMC_AD_WITHIN) {
        if (d < lower) return false;
        if (d >= upper) return false;
    } else if (d >= lower && d < upper) {
        return false;
    }
    if (A.flags & FRMC_AD_RED_UPPER) {
        d = fabsf(upper - d);
    } else if (A.flags & FRMC_AD_RED_LOWER) {
        d = fabsf(lower - d);
    } else if (A.flags & FRMC_AD_RED) {
        const float mid = (lower + upper) / 2.0f;
        d = d > mid ? fabsf(upper - d) : fabsf(lower - d);
    }
    v = d;
    ws = (same ? 0 : A.nel * A.nel) + ea * A.nel + ei;
    return true;
}

// One key and value per lane with sel: a single atomic per wave takes their places.
__device__ __forceinline__ void ad_emit(const AdOut &O, bool sel, int32_t ws, uint64_t order, float v) {
    const uint64_t m = __ballot(sel);
    if (!m) return;
    unsigned long long at = 0;
    const int lane = threadIdx.x & 63, lead = __builtin_ctzll(m);
    if (lane == lead) at = atomicAdd(O.total, (unsigned long long)__popcll(m));
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)at, lead),
                   hi = __builtin_amdgcn_readlane((uint32_t)(at >> 32), lead);
    at = ((unsigned long long)hi << 32 | lo) +
         __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
    if (sel && at < O.cap) {
        O.keys[at] = ((uint64_t)ws << O.shift) | order;
        O.vals[at] = v;
    }
}

__device__ __forceinline__ void ad_flush(const AdOut &O, const uint32_t *lcnt, int32_t nws) {
    __syncthreads();
    for (int32_t s = threadIdx.x; s < nws; s += blockDim.x)
        if (lcnt[s]) atomicAdd(&O.cnt[s], lcnt[s]);
}

// grid (ceil(n/256), ceil(k/per)): one other atom per thread against `per`
// (at most kAdCols) columns c, column c = atom indexes[c].
constexpr int kAdCols = 32;

template <int SRC>
__global__ void __launch_bounds__(256) k_ad_pass(AdArgs A, AdOut O, int32_t per) {
    extern __shared__ uint32_t lcnt[];  // [2*nel*nel] when counting
    __shared__ int32_t sa[kAdCols], sm[kAdCols], se[kAdCols];
    __shared__ float sp[kAdCols][3];
    const int32_t nws = 2 * A.nel * A.nel, c0 = blockIdx.y * per, nc = min(per, A.k - c0);
    if (O.cnt)
        for (int32_t s = threadIdx.x; s < nws; s += blockDim.x) lcnt[s] = 0;
    if ((int32_t)threadIdx.x < nc) {
        const int32_t a = A.indexes ? A.indexes[c0 + threadIdx.x] : A.atomIndex;
        const bool ok = a >= 0 && a < A.n;  // the host shims reject other indexes; nothing is counted for them
        sa[threadIdx.x] = ok ? a : -1;
        if (ok) {
            sm[threadIdx.x] = A.mol[a];
            se[threadIdx.x] = A.elem[a];
            if (SRC != AD_DISTS)
                for (int d = 0; d < 3; d++) sp[threadIdx.x][d] = A.coords[3 * (int64_t)a + d];
        }
    }
    Basis B;
    if (SRC == AD_PBC) B = basis_of(A.basis);
    __syncthreads();
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x, ii = min(i, A.n - 1);
    const int32_t mi = A.mol[ii], ei = A.elem[ii];
    float x = 0.f, y = 0.f, z = 0.f;
    if (SRC != AD_DISTS) {
        x = A.coords[3 * (int64_t)ii];
        y = A.coords[3 * (int64_t)ii + 1];
        z = A.coords[3 * (int64_t)ii + 2];
    }
    const int32_t last = min(A.n, (int32_t)(blockIdx.x + 1) * 256) - 1;
    for (int32_t q = 0; q < nc; q++) {
        const int32_t a = sa[q];
        if (a < 0 || (!A.allAtoms && last < a)) continue;
        float v = 0.f;
        int32_t ws = 0;
        bool sel = i < A.n && i != a && (A.allAtoms || i > a);
        if (sel) {
            const float d = SRC == AD_DISTS ? A.dists[(int64_t)i * A.k + c0 + q]
                                            : ad_distance<SRC == AD_PBC>(B, sp[q][0], sp[q][1], sp[q][2], x, y, z);
            sel = ad_select(A, d, mi == sm[q], ei, se[q], v, ws);
        }
        if (O.cnt && sel) atomicAdd(&lcnt[ws], 1u);
        ad_emit(O, sel, ws, (uint64_t)(c0 + q) * (uint64_t)A.n + (uint64_t)i, v);
    }
    if (O.cnt) ad_flush(O, lcnt, nws);
}

// The list's positions of every atom, as chains: head[atom], then next[position].
__global__ void __launch_bounds__(256) k_ad_chains(const int32_t *__restrict__ indexes, int32_t k, int32_t n,
                                                   int32_t *__restrict__ head, int32_t *__restrict__ next) {
    const int32_t c = blockIdx.x * 256 + threadIdx.x;
    if (c >= k) return;
    const int32_t a = indexes[c];
    if (a >= 0 && a < n) next[c] = atomicExch(&head[a], c);
}

// Pairs inside the limits over sorted chunks (chunks.h).  A wave takes a row
// chunk and kAdOffsets of the chunks after it around the ring, tests boxes,
// then atoms against the row chunk's box, and queues the pairs within the
// largest limit; full waves evaluate the queue exactly, in both directions
// where both atoms are listed.
// The items grow as the square of the atoms, so the launch is bounded and its
// waves stride over them: 64 listed atoms of 200,000 take 472 us with at most 16,384
// workgroups, 497 with 4,096, 513 with 65,536, 1,066 with an item per wave, and from
// 889,632 atoms on that is more than a launch holds.
constexpr int64_t kAdBlocks = 1 << 14;
constexpr int kAdOffsets = 4;  // 13,500 atoms: 155 us a call; 2: 181, 8: 177, 16: 180

template <bool PBC>
__global__ void __launch_bounds__(256) k_ad_chunks(AdArgs A, AdOut O, ChunkSort S, const int32_t *__restrict__ head,
                                                   const int32_t *__restrict__ next) {
    extern __shared__ uint32_t lcnt[];
    __shared__ float4 list_of[4][64];
    __shared__ int32_t pos_of[4][64];
    __shared__ uint32_t queue_of[4][128];
    const int32_t nws = 2 * A.nel * A.nel;
    if (O.cnt)
        for (int32_t s = threadIdx.x; s < nws; s += blockDim.x) lcnt[s] = 0;
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    float4 *list = list_of[wave];
    int32_t *pos = pos_of[wave];
    uint32_t *queue = queue_of[wave];
    const ChunkPlan P = plan_of(S.meta);
    // the largest upper limit; one that is not a number excludes nothing
    float range = 0.0f;
    for (int32_t s = lane; s < A.nel * A.nel; s += 64) range = fmaxf(range, abs_or_inf(fmaxf(A.upper[s], 0.0f) + 0.0f * A.upper[s]));
    for (int o = 32; o > 0; o >>= 1) range = fmaxf(range, __shfl_xor(range, o));
    const float cut2 = cut_squared(P.C, range, coord_max<PBC>(S.meta));
    const int32_t N = (int32_t)load_dev(S.meta + M_NCHUNK), ndist = N / 2 + 1;
    const int32_t nsub = (ndist + kAdOffsets - 1) / kAdOffsets;
    // item sub * N + i of nsub * N, which may not fit 32 bits: both parts advance
    const uint32_t first = blockIdx.x * 4 + wave, stride = gridDim.x * 4;
    const int32_t dsub = (int32_t)(stride / N), di = (int32_t)(stride % N);
    int32_t sub = (int32_t)(first / N), i = (int32_t)(first % N);
    for (; sub < nsub; sub += dsub + (i + di >= N), i = i + di >= N ? i + di - N : i + di) {
        const int32_t e0 = sub * kAdOffsets, e1 = min(ndist, e0 + kAdOffsets);
        const float4 r = S.sx[(int64_t)i * 64 + lane];
        const int bx = __float_as_int(reinterpret_cast<const float *>(S.cbox + kBox * (int64_t)i)[lane & 7]);
        auto of = [&](int k) { return __int_as_float(__builtin_amdgcn_readlane(bx, k)); };
        const float3 bm = make_float3(of(0), of(1), of(2)), bh = make_float3(of(4), of(5), of(6));
        int32_t qn = 0;
        auto drain = [&](int32_t len) {
            bool on = lane < len;
            float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b = a;
            bool same = false;
            int32_t ca = -1, cb = -1;
            if (on) {
                const uint32_t q = queue[lane];
                const int64_t pa = (int64_t)i * 64 + (q >> 26), pb = q & 0x3ffffffu;
                a = S.sx[pa];
                b = S.sx[pb];
                same = S.smol[pa] == S.smol[pb];
                if (__float_as_int(b.w) < __float_as_int(a.w)) {
                    const float4 t = a;
                    a = b;
                    b = t;
                }
                ca = head[__float_as_int(a.w) >> 6];
                cb = A.allAtoms ? head[__float_as_int(b.w) >> 6] : -1;
            }
            const int32_t ia = __float_as_int(a.w) >> 6, ib = __float_as_int(b.w) >> 6, ea = __float_as_int(a.w) & 63,
                          eb = __float_as_int(b.w) & 63;
            const float d = ad_distance<PBC>(P.B, a.x, a.y, a.z, b.x, b.y, b.z);
            auto along = [&](int32_t c, int32_t other, int32_t ei, int32_t el) {
                float v = 0.f;
                int32_t ws = 0;
                const bool sel = on && c >= 0 && ad_select(A, d, same, ei, el, v, ws);
                while (__ballot(sel && c >= 0)) {
                    const bool now = sel && c >= 0;
                    if (O.cnt && now) atomicAdd(&lcnt[ws], 1u);
                    ad_emit(O, now, ws, (uint64_t)(uint32_t)c * (uint64_t)A.n + (uint64_t)other, v);
                    if (now) c = next[c];
                }
            };
            along(ca, ib, eb, ea);  // the earlier atom listed
            along(cb, ia, ea, eb);  // the later one
        };
        const int32_t el = e0 + lane;
        int32_t j = i + el;
        j = j >= N ? j - N : j;
        bool near = false;
        if (el < e1 && (2 * el != N || i < el || el == 0)) {
            const float4 m = S.cbox[kBox * (int64_t)j], h = S.cbox[kBox * (int64_t)j + 1];
            near = !(lower_bound2<PBC, false>(m.x - bm.x, m.y - bm.y, m.z - bm.z, h.x + bh.x, h.y + bh.y, h.z + bh.z,
                                              P.C) > cut2);
        }
        uint64_t todo = __ballot(near);
        while (todo) {
            int32_t jc = i + e0 + __builtin_ctzll(todo);
            todo &= todo - 1;
            jc = jc >= N ? jc - N : jc;
            const float4 c = S.sx[(int64_t)jc * 64 + lane];
            const float fx = PBC ? c.x - floorf(c.x) : c.x, fy = PBC ? c.y - floorf(c.y) : c.y,
                        fz = PBC ? c.z - floorf(c.z) : c.z;
            const bool keep = __float_as_int(c.w) >= 0 &&
                              !(lower_bound2<PBC, false>(fx - bm.x, fy - bm.y, fz - bm.z, bh.x, bh.y, bh.z, P.C) > cut2);
            const uint64_t km = __ballot(keep);
            __builtin_amdgcn_wave_barrier();
            if (keep) {
                const int at = __builtin_amdgcn_mbcnt_hi((uint32_t)(km >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)km, 0));
                list[at] = c;
                pos[at] = jc * 64 + lane;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            const int cnt = __popcll(km);
            for (int t = 0; t < cnt; t++) {
                const float4 q = list[t];
                const int32_t p = pos[t];
                const float s = pair_s<PBC, false>(r.x, r.y, r.z, q.x, q.y, q.z, P.B);
                // within a chunk each pair once; padding rows are not in range (NaN) unless nothing is cut
                const bool in = __float_as_int(r.w) >= 0 && !(s > cut2) && (jc != i || p > i * 64 + lane);
                const uint64_t m = __ballot(in);
                if (!m) continue;
                if (in)
                    queue[qn + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0))] =
                        ((uint32_t)lane << 26) | (uint32_t)p;
                qn += __popcll(m);
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
                if (qn >= 64) {
                    drain(64);
                    __builtin_amdgcn_wave_barrier();
                    qn -= 64;
                    const uint32_t rest = queue[64 + lane];
                    __builtin_amdgcn_wave_barrier();
                    if (lane < qn) queue[lane] = rest;
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                }
            }
        }
        drain(qn);
        __builtin_amdgcn_wave_barrier();
    }
    if (O.cnt) ad_flush(O, lcnt, nws);
}

// The number of selected pairs to a host word, and, when at most kFew, their
// sort (bitonic, by key: each slot's terms in the reference's order) and sums.
constexpr int kFew = 2048;

__global__ void __launch_bounds__(1024) k_ad_few(AdOut O, const uint32_t *__restrict__ cnt, int32_t nws,
                                                 float *__restrict__ dintra, float *__restrict__ dinter,
                                                 int32_t *__restrict__ nintra, int32_t *__restrict__ ninter,
                                                 int64_t *total) {
    __shared__ uint64_t key[kFew];
    __shared__ float val[kFew];
    const int tid = threadIdx.x;
    const unsigned long long all = load_dev(O.total);
    if (tid == 0) *total = (int64_t)all;
    if (all > (unsigned)kFew || all > O.cap) return;
    const int len = (int)all;
    int size = 2;
    while (size < len) size *= 2;
    for (int i = tid; i < size; i += 1024) {
        key[i] = i < len ? O.keys[i] : ~(uint64_t)0;
        val[i] = i < len ? O.vals[i] : 0.0f;
    }
    __syncthreads();
    for (int k = 2; k <= size; k *= 2)
        for (int j = k / 2; j > 0; j /= 2) {
            for (int i = tid; i < size; i += 1024) {
                const int l = i ^ j;
                if (l > i && ((key[i] > key[l]) == ((i & k) == 0))) {
                    const uint64_t tk = key[i];
                    key[i] = key[l];
                    key[l] = tk;
                    const float tv = val[i];
                    val[i] = val[l];
                    val[l] = tv;
                }
            }
            __syncthreads();
        }
    for (int32_t s = tid; s < nws; s += 1024) {
        const int32_t n = (int32_t)cnt[s];
        if (!n) continue;
        int lo = 0, hi = len;  // first key of slot s
        while (lo < hi) {
            const int mid = (lo + hi) / 2;
            if ((int32_t)(key[mid] >> O.shift) < s) lo = mid + 1;
            else hi = mid;
        }
        const int32_t half = nws / 2;
        float *d = s < half ? dintra + s : dinter + (s - half);
        int32_t *nn = s < half ? nintra + s : ninter + (s - half);
        float acc = *d;
        int j = 0;
        for (; j + 8 <= n; j += 8) {  // the loads together, then the dependent adds
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = val[lo + j + u];
#pragma unroll
            for (int u = 0; u < 8; u++) acc = acc + v[u];
        }
        for (; j < n; j++) acc = acc + val[lo + j];
        *d = acc;
        *nn = *nn + n;
    }
}

// One workgroup per slot: dsum[slot] += terms in order (float32), nsum[slot] +=
// count.  The four waves stage the next kSumChunk terms while the first adds
// the present ones, a dependent add at a time (one lane with a memory access per
// add: 569 us for 9,100 terms per slot).
constexpr int kSumChunk = 2048;

__global__ void __launch_bounds__(256) k_ad_sum(const uint32_t *__restrict__ cnt, int32_t nws,
                                                const float *__restrict__ vals, float *__restrict__ dintra,
                                                float *__restrict__ dinter, int32_t *__restrict__ nintra,
                                                int32_t *__restrict__ ninter) {
    __shared__ __align__(16) float buf[2][kSumChunk];
    __shared__ unsigned long long before;
    const int32_t s = blockIdx.x;
    const int tid = threadIdx.x;
    if (tid == 0) before = 0;
    __syncthreads();
    unsigned long long mine = 0;
    for (int32_t t = tid; t < s; t += 256) mine += cnt[t];
    if (mine) atomicAdd(&before, mine);
    const uint32_t len = load_dev(cnt + s);
    __syncthreads();
    if (!len) return;
    const float *v = vals + before;
    const int32_t half = nws / 2;
    float *d = s < half ? dintra + s : dinter + (s - half);
    int32_t *nn = s < half ? nintra + s : ninter + (s - half);
    float acc = load_dev(d);
    auto stage = [&](uint32_t c0, float *to) {
#pragma unroll
        for (int u = 0; u < kSumChunk / 256; u++) {
            const uint32_t at = c0 + tid + 256 * u;
            to[tid + 256 * u] = at < len ? v[at] : 0.0f;
        }
    };
    stage(0, buf[0]);
    for (uint32_t c0 = 0, which = 0; c0 < len; c0 += kSumChunk, which ^= 1) {
        __syncthreads();
        if (c0 + kSumChunk < len) stage(c0 + kSumChunk, buf[which ^ 1]);
        if (tid < 64) {
            const float *b = buf[which];
            const int n = (int)min((uint32_t)kSumChunk, len - c0);
            int j = 0;
            for (; j + 32 <= n; j += 32) {
                float4 q[8];
#pragma unroll
                for (int u = 0; u < 8; u++) q[u] = reinterpret_cast<const float4 *>(b + j)[u];
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    acc = acc + q[u].x;
                    acc = acc + q[u].y;
                    acc = acc + q[u].z;
                    acc = acc + q[u].w;
                }
            }
            for (; j < n; j++) acc = acc + b[j];
        }
    }
    if (tid == 0) {
        *d = acc;
        *nn = *nn + (int32_t)len;
    }
}

__global__ void __launch_bounds__(256) k_ad_clear(uint32_t *__restrict__ p, int64_t n, int32_t *__restrict__ head,
                                                  int64_t nhead) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x, stride = (int64_t)gridDim.x * 256;
    for (int64_t i = t; i < n; i += stride) p[i] = 0;
    for (int64_t i = t; i < nhead; i += stride) head[i] = -1;
}

// pair_elements_stats (atomic_distances.pyx:632-656): every pair i<j once,
// nintra/ninter[e_i][e_j] += 1 by molecule.  Grid (row tiles of 256,
// column chunks of kPeChunk); LDS-private counters.
constexpr int kPeChunk = 2048;

__global__ void __launch_bounds__(256) k_pair_elements_stats(const int32_t *__restrict__ elem,
                                                             const int32_t *__restrict__ mol, int32_t n, int32_t nel,
                                                             int32_t *__restrict__ nintra,
                                                             int32_t *__restrict__ ninter) {
    extern __shared__ int32_t sm[];
    const int32_t nn = nel * nel;
    int32_t *lc = sm;                  // [2*nn]
    int32_t *ce = sm + 2 * nn;         // [kPeChunk] chunk elements
    int32_t *cm = ce + kPeChunk;       // [kPeChunk] chunk molecules
    const int32_t r0 = blockIdx.x * 256, j0 = blockIdx.y * kPeChunk;
    if (j0 + kPeChunk <= r0 + 1) return;  // chunk entirely at or below the row tile's diagonal (uniform)
    for (int32_t s = threadIdx.x; s < 2 * nn; s += blockDim.x) lc[s] = 0;
    const int32_t len = min(kPeChunk, n - j0);
    for (int32_t t = threadIdx.x; t < len; t += blockDim.x) {
        ce[t] = elem[j0 + t];
        cm[t] = mol[j0 + t];
    }
    __syncthreads();
    const int32_t i = r0 + threadIdx.x;
    if (i < n) {
        const int32_t ei = elem[i], mi = mol[i];
        for (int32_t t = max(0, i + 1 - j0); t < len; t++) {
            const int32_t slot = (cm[t] == mi ? 0 : nn) + ei * nel + ce[t];
            atomicAdd(&lc[slot], 1);
        }
    }
    __syncthreads();
    for (int32_t s = threadIdx.x; s < 2 * nn; s += blockDim.x)
        if (lc[s]) atomicAdd(s < nn ? &nintra[s] : &ninter[s - nn], lc[s]);
}

// Scratch of one call, returned to the stream-ordered pool at scope exit.
struct AdScratch {
    hipStream_t st = nullptr;
    void *p[3] = {nullptr, nullptr, nullptr};
    ~AdScratch() {
        for (void *q : p)
            if (q) (void)hipFreeAsync(q, st);
    }
};

// Whether k listed atoms of n take the chunks.  They pay for their sort (five
// launches and a chain pass, about 25 us) from all pairs of 2,048 atoms on (3,000
// atoms: 138 us against 166; 1,000: 127 without).  Their pass tests all pairs of chunks
// whatever the list: about 55 us + 9e-9 n^2 more than a call's launches, where the
// direct pass takes k (0.08 + 1.1e-6 n), with limits of 2.6 A, and up to k (0.8 +
// 1.1e-6 n) at 6 A, where each listed atom has ten times the pairs to sort.  The line
// is at 0.15: 200,000 atoms, us direct and by chunks at 2.6 A: 84 and 472 for 64
// listed atoms, 387 and 516 for 1,024, 678 and 524 for 2,048; at 6 A: 136 and 544, 1,191
// and 759, 2,323 and 1,056; 1,000,000 atoms, 2,048 listed: 2,926 and 8,967.
constexpr int64_t kChunkPairs = (int64_t)1 << 22;

bool chunks_pay(int64_t k, int64_t n) {
    return k * n >= kChunkPairs && (double)k * (16e6 + 120.0 * n) >= 6e9 + (double)n * n;
}

template <int SRC>
int ad_run(AdArgs A, float *dintra, float *dinter, int32_t *nintra, int32_t *ninter, hipStream_t st) {
    const int32_t nws = 2 * A.nel * A.nel;
    const size_t lds = sizeof(uint32_t) * nws;
    FRMC_REQUIRE(lds <= 64 * 1024, "atomic_distances: %d element types is too many", A.nel);
    FRMC_REQUIRE((uint64_t)A.k * (uint64_t)A.n < ((uint64_t)1 << 40), "atomic_distances: too many pairs");
    FRMC_REQUIRE(A.k <= 65535, "atomic_distances: at most 65535 atoms per call");
    if (A.k == 0 || A.n == 0) return FRMC_OK;
    const int64_t pairs = (int64_t)A.k * A.n;
    // only pairs inside the limits can be skipped by their distance
    const bool chunks = SRC != AD_DISTS && (A.flags & FRMC_AD_WITHIN) && A.indexes && A.nel <= 64 &&
                        A.n < (1 << 25) && chunks_pay(A.k, A.n);
    ChunkSort S;
    memset(&S, 0, sizeof(S));
    if (chunks) S = chunk_layout(A.n);
    // scratch: [chunks | counts, total | chains | keys | values]; room for 64
    // selected pairs per listed atom at first
    AdOut O;
    O.shift = 1;
    while (((int64_t)1 << O.shift) < pairs) O.shift++;
    O.cap = (unsigned long long)std::min<int64_t>(pairs, std::max<int64_t>(1 << 16, 64 * (int64_t)A.k));
    const int64_t ncnt = (nws + 3) & ~1;  // the total after them, 8-byte aligned
    const size_t o_cnt = S.bytes, o_head = o_cnt + 4 * (size_t)ncnt + 8, nchain = chunks ? (size_t)A.n + A.k : 0,
                 o_keys = (o_head + 4 * nchain + 255) & ~(size_t)255, o_vals = o_keys + 8 * (size_t)O.cap;
    AdScratch R;
    R.st = st;
    FRMC_CHECK_HIP(pool_malloc(&R.p[0], o_vals + 4 * (size_t)O.cap, st));
    char *scr = (char *)R.p[0];
    uint32_t *cnt = O.cnt = (uint32_t *)(scr + o_cnt);
    O.total = (unsigned long long *)(scr + o_cnt + 4 * (size_t)ncnt);
    O.keys = (uint64_t *)(scr + o_keys);
    O.vals = (float *)(scr + o_vals);
    int32_t *head = (int32_t *)(scr + o_head), *next = head + A.n;
    const int64_t nclear = ncnt + 2;
    k_ad_clear<<<std::min(256u, blocks_for(nclear + (chunks ? A.n : 0), 256)), 256, 0, st>>>(cnt, nclear, head,
                                                                                            chunks ? A.n : 0);
    FRMC_CHECK_LAUNCH();
    const unsigned nb = blocks_for(A.n, 256);
    // columns per workgroup: about 1,024 workgroups, none of more than kAdCols
    const int32_t per = (int32_t)std::max<int64_t>(
        std::max<int64_t>(1, (A.k + 65534) / 65535),
        std::min<int64_t>(kAdCols, ((int64_t)A.k * nb + 1023) / 1024));
    if (chunks) {
        Basis none;
        memset(&none, 0, sizeof(none));
        launch_chunk_sort(S, scr, A.coords, A.n, SRC == AD_PBC ? A.basis : nullptr, none, SRC == AD_PBC, A.mol, A.elem,
                          A.nel, nullptr, 0, st);
        k_ad_chains<<<blocks_for(A.k, 256), 256, 0, st>>>(A.indexes, A.k, A.n, head, next);
        FRMC_CHECK_LAUNCH();
    }
    const int64_t items = chunks ? S.maxchunks * ((S.maxchunks / 2 + kAdOffsets) / kAdOffsets) : 0;
    const unsigned cblocks = (unsigned)std::min<int64_t>((items + 3) / 4, kAdBlocks);
    auto pass = [&]() {
        if (chunks)
            k_ad_chunks<SRC == AD_PBC><<<cblocks, 256, lds, st>>>(A, O, S, head, next);
        else
            k_ad_pass<SRC><<<dim3(nb, (unsigned)((A.k + per - 1) / per)), 256, lds, st>>>(A, O, per);
    };
    pass();
    FRMC_CHECK_LAUNCH();
    HostWords found(st);
    if (!found.p) {
        set_error("allocation of pinned host words failed");
        return FRMC_ENOMEM;
    }
    k_ad_few<<<1, 1024, 0, st>>>(O, cnt, nws, dintra, dinter, nintra, ninter, found.p);
    FRMC_CHECK_LAUNCH();
    FRMC_CHECK_HIP(found.wait());
    const uint64_t L = (uint64_t)found.p[0];
    FRMC_REQUIRE(L < ((uint64_t)1 << 28), "atomic_distances: %llu counted pairs exceed the 2^28 limit",
                 (unsigned long long)L);
    if (L <= (uint64_t)kFew && L <= O.cap) return FRMC_OK;
    if (L > O.cap) {  // more than the first room: again, into buffers of their size
        FRMC_CHECK_HIP(pool_malloc(&R.p[1], (8 + 4) * (size_t)L, st));
        O.cap = L;
        O.keys = (uint64_t *)R.p[1];
        O.vals = (float *)(O.keys + L);
        O.cnt = nullptr;
        k_ad_clear<<<1, 256, 0, st>>>((uint32_t *)O.total, 2, head, 0);
        pass();
        FRMC_CHECK_LAUNCH();
    }
    unsigned end_bit = O.shift;
    while ((1u << (end_bit - O.shift)) < (unsigned)nws) end_bit++;
    size_t tmp_bytes = 0;
    uint64_t *none = nullptr;
    FRMC_CHECK_HIP(rocprim::radix_sort_pairs(nullptr, tmp_bytes, O.keys, none, O.vals, (float *)nullptr, (size_t)L, 0,
                                             end_bit, st));
    const size_t o_tmp = ((8 + 4) * (size_t)L + 255) & ~(size_t)255;
    FRMC_CHECK_HIP(pool_malloc(&R.p[2], o_tmp + std::max<size_t>(tmp_bytes, 1), st));
    uint64_t *keys_s = (uint64_t *)R.p[2];
    float *vals_s = (float *)(keys_s + L);
    FRMC_CHECK_HIP(rocprim::radix_sort_pairs((char *)R.p[2] + o_tmp, tmp_bytes, O.keys, keys_s, O.vals, vals_s,
                                             (size_t)L, 0, end_bit, st));
    k_ad_sum<<<nws, 256, 0, st>>>(cnt, nws, vals_s, dintra, dinter, nintra, ninter);
    FRMC_CHECK_LAUNCH();
    return FRMC_OK;
}

}  // namespace

}  // namespace frmc

using namespace frmc;

extern "C" int frmc_single_atomic_distances_dists(int32_t atomIndex, const float *distances, int32_t n,
                                                  const int32_t *moleculeIndex, const int32_t *elementIndex,
                                                  float *dintra, float *dinter, int32_t *nintra, int32_t *ninter,
                                                  int32_t numberOfElements, const float *lowerLimit,
                                                  const float *upperLimit, int flags, int allAtoms, void *stream) {
    FRMC_REQUIRE(numberOfElements >= 1 && n >= 0, "atomic_distances: bad sizes");
    FRMC_REQUIRE(atomIndex >= 0 && atomIndex < n, "atomIndex %d outside [0,%d)", atomIndex, n);
    AdArgs A{};
    A.dists = distances;
    A.n = n;
    A.k = 1;
    A.indexes = nullptr;
    A.atomIndex = atomIndex;
    A.mol = moleculeIndex;
    A.elem = elementIndex;
    A.nel = numberOfElements;
    A.lower = lowerLimit;
    A.upper = upperLimit;
    A.flags = flags;
    A.allAtoms = allAtoms;
    return ad_run<AD_DISTS>(A, dintra, dinter, nintra, ninter, as_stream(stream));
}

extern "C" int frmc_multiple_atomic_distances_coords(const int32_t *indexes, int32_t nidx, const float *boxCoords,
                                                     int32_t n, const float *basis, int isPBC,
                                                     const int32_t *moleculeIndex, const int32_t *elementIndex,
                                                     int32_t numberOfElements, const float *lowerLimit,
                                                     const float *upperLimit, int flags, int allAtoms,
                                                     int32_t *nintra, float *dintra, int32_t *ninter, float *dinter,
                                                     void *stream) {
    FRMC_REQUIRE(numberOfElements >= 1 && n >= 0 && nidx >= 0, "atomic_distances: bad sizes");
    FRMC_REQUIRE(!isPBC || basis, "basis is NULL");
    hipStream_t st = as_stream(stream);
    AdArgs A{};
    A.coords = boxCoords;
    A.n = n;
    A.k = nidx;
    A.indexes = indexes;
    A.mol = moleculeIndex;
    A.elem = elementIndex;
    A.nel = numberOfElements;
    A.lower = lowerLimit;
    A.upper = upperLimit;
    A.flags = flags;
    A.allAtoms = allAtoms;
    A.basis = basis;
    return isPBC ? ad_run<AD_PBC>(A, dintra, dinter, nintra, ninter, st)
                 : ad_run<AD_IBC>(A, dintra, dinter, nintra, ninter, st);
}

extern "C" int frmc_multiple_atomic_distances_dists(const int32_t *indexes, int32_t nidx, const float *distances,
                                                    int32_t n, int32_t k, const int32_t *moleculeIndex,
                                                    const int32_t *elementIndex, int32_t numberOfElements,
                                                    const float *lowerLimit, const float *upperLimit, int flags,
                                                    int allAtoms, int32_t *nintra, float *dintra, int32_t *ninter,
                                                    float *dinter, void *stream) {
    FRMC_REQUIRE(numberOfElements >= 1 && n >= 0 && nidx >= 0 && nidx <= k, "atomic_distances: bad sizes");
    AdArgs A{};
    A.dists = distances;
    A.n = n;
    A.k = nidx;
    A.indexes = indexes;
    A.mol = moleculeIndex;
    A.elem = elementIndex;
    A.nel = numberOfElements;
    A.lower = lowerLimit;
    A.upper = upperLimit;
    A.flags = flags;
    A.allAtoms = allAtoms;
    // column c of the (n,k) array belongs to indexes[c]; the kernel indexes it with stride k
    (void)k;
    return ad_run<AD_DISTS>(A, dintra, dinter, nintra, ninter, as_stream(stream));
}

extern "C" int frmc_pair_elements_stats(const int32_t *elementIndex, const int32_t *moleculeIndex, int32_t n,
                                        int32_t numberOfElements, int32_t *nintra, int32_t *ninter, void *stream) {
    FRMC_REQUIRE(numberOfElements >= 1 && n >= 0, "pair_elements_stats: bad sizes");
    const size_t lds = sizeof(int32_t) * (2 * (size_t)numberOfElements * numberOfElements + 2 * kPeChunk);
    FRMC_REQUIRE(lds <= 64 * 1024, "pair_elements_stats: %d element types is too many", numberOfElements);
    hipStream_t st = as_stream(stream);
    const size_t nn = (size_t)numberOfElements * numberOfElements;
    FRMC_CHECK_HIP(hipMemsetAsync(nintra, 0, sizeof(int32_t) * nn, st));
    FRMC_CHECK_HIP(hipMemsetAsync(ninter, 0, sizeof(int32_t) * nn, st));
    if (n < 2) return FRMC_OK;
    const dim3 grid(blocks_for(n, 256), (n + kPeChunk - 1) / kPeChunk);
    hipLaunchKernelGGL(k_pair_elements_stats, grid, dim3(256), lds, st, elementIndex, moleculeIndex, n,
                       numberOfElements, nintra, ninter);
    FRMC_CHECK_LAUNCH();
    return FRMC_OK;
}
