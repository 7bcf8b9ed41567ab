// abd_cull.hip — candidate culling (culling.py / culling2.py) and the sparse
// structure of the Newton matrix (orthogonal_energy.py:138-165).
//
// Culling replaces the reference's per-body Warp BVHs with an exact two-level
// scheme that needs no tree build or refit:
//   1. body pairs: every (i < j) pair tested against the FP32 body boxes;
//   2. per body pair and side, the primitives whose box overlaps the hull of the
//      OTHER side's primitive boxes are kept (a primitive box that misses that
//      hull cannot overlap any box of the other side, so nothing is lost);
//   3. the filtered lists are tested exhaustively in chunks of `chunk` tests (a tunable
//      launch shape: the emitted list is the same for every chunk size).
// Every list is produced by a count -> exclusive scan -> write sequence with
// wave-ballot ranks, so outputs are emitted in sorted order (ii, order, a, b)
// and are identical from run to run.
#include <hip/hip_runtime.h>

#include <math.h>

#include <algorithm>

#include "abd_block.h"
#include "abd_device.h"
#include "abd_internal.h"
#include "abd_profile.h"

namespace abd {

__device__ __forceinline__ bool overlap(const float* __restrict__ alo, const float* __restrict__ ahi,
                                        const float* __restrict__ blo, const float* __restrict__ bhi) {
    // every bound is loaded before any is compared: as one condition after the other the six
    // loads waited for each other
    const float a0 = alo[0], a1 = alo[1], a2 = alo[2], A0 = ahi[0], A1 = ahi[1], A2 = ahi[2];
    const float b0 = blo[0], b1 = blo[1], b2 = blo[2], B0 = bhi[0], B1 = bhi[1], B2 = bhi[2];
    return !((a0 > B0) | (A0 < b0) | (a1 > B1) | (A1 < b1) | (a2 > B2) | (A2 < b2));
}

// ---------------------------------------------------------------- bodies
constexpr int kItems = 8;      // entries per thread in the vertex-ground compaction
constexpr int kPairItems = 1;  // pairs per thread in the body-pair compaction: enough workgroups to fill the device

// k -> (i, j), i < j.  Order 0: row-major (i, j); order 1: sorted by (j, i).
__device__ __forceinline__ void pair_of(int64_t k, int nb, int order, int& i, int& j) {
    if (order == 0) {
        double n2 = 2.0 * nb - 1.0;
        int64_t r = (int64_t)floor((n2 - sqrt(n2 * n2 - 8.0 * (double)k)) * 0.5);
        if (r < 0) r = 0;
        auto off = [nb](int64_t q) { return q * nb - q * (q + 1) / 2; };
        while (r > 0 && off(r) > k) --r;
        while (off(r + 1) <= k) ++r;
        i = (int)r;
        j = (int)(k - off(r) + r + 1);
    } else {
        int64_t c = (int64_t)floor((1.0 + sqrt(1.0 + 8.0 * (double)k)) * 0.5);
        if (c < 1) c = 1;
        while (c > 1 && c * (c - 1) / 2 > k) --c;
        while ((c + 1) * c / 2 <= k) ++c;
        j = (int)c;
        i = (int)(k - c * (c - 1) / 2);
    }
}

__device__ __forceinline__ bool body_pred(int i, int j, const int32_t* __restrict__ scene,
                                          const float* __restrict__ lo, const float* __restrict__ hi) {
    if (scene && scene[i] != scene[j]) return false;
    return overlap(lo + 3 * i, hi + 3 * i, lo + 3 * j, hi + 3 * j);
}

// Scene segmentation: pairs enumerated scene by scene (bodies of a scene are
// contiguous), so the concatenation stays sorted in both orders.
struct SceneSeg {
    int n;                 // scenes (<= 1: no segmentation)
    const int32_t* boff;   // [n+1] body offsets
    const int64_t* poff;   // [n+1] pair offsets
};

__device__ __forceinline__ void seg_pair_of(int64_t k, int nb, int order, const SceneSeg& sg, int& i, int& j) {
    if (sg.n <= 1) {
        pair_of(k, nb, order, i, j);
        return;
    }
    int lo = 0, hi = sg.n;  // last s with poff[s] <= k
    while (hi - lo > 1) {
        int mid = (lo + hi) >> 1;
        if (sg.poff[mid] <= k)
            lo = mid;
        else
            hi = mid;
    }
    const int b0 = sg.boff[lo];
    pair_of(k - sg.poff[lo], sg.boff[lo + 1] - b0, order, i, j);
    i += b0;
    j += b0;
}

// blockIdx.y: the order of the enumeration, its counts and offsets nblk + 1 apart.
template <bool WRITE>
__global__ __launch_bounds__(kBlock) void body_pairs_kernel(int nb, int64_t npairs, SceneSeg sg,
                                                             const int32_t* __restrict__ scene,
                                                             const float* __restrict__ lo,
                                                             const float* __restrict__ hi, int64_t* __restrict__ bcnt,
                                                             const int64_t* __restrict__ boff, int32_t* out_ij,
                                                             int32_t* out_ji, int64_t cap) {
    __shared__ int shw[kBlock / kWave];
    const int order = blockIdx.y;
    int32_t* out = order ? out_ji : out_ij;
    bcnt += order * ((int64_t)gridDim.x + 1);
    if (WRITE) boff += order * ((int64_t)gridDim.x + 1);
    int64_t base = (int64_t)blockIdx.x * kBlock * kPairItems;
    int64_t run = WRITE ? boff[blockIdx.x] : 0;
    for (int it = 0; it < kPairItems; ++it) {
        int64_t k = base + (int64_t)it * kBlock + threadIdx.x;
        bool pred = false;
        int i = 0, j = 0;
        if (k < npairs) {
            seg_pair_of(k, nb, order, sg, i, j);
            pred = body_pred(i, j, scene, lo, hi);
        }
        int tot;
        int r = block_rank(pred, shw, &tot);
        if (WRITE && pred) {
            int64_t o = run + r;
            if (o < cap) {
                out[2 * o] = i;
                out[2 * o + 1] = j;
            }
        }
        run += tot;
    }
    if (!WRITE && threadIdx.x == 0) bcnt[blockIdx.x] = run;
}

// ------------------------------------------------------------- primitives

// unit -> (ii, I (set-1 body), J (set-2 body))
__device__ __forceinline__ void unit_bodies(int pt, int64_t u, const int32_t* __restrict__ ij, int64_t& ii, int& I,
                                            int& J) {
    if (pt) {
        ii = u >> 1;
        int a = ij[2 * ii], b = ij[2 * ii + 1];
        I = (u & 1) ? b : a;  // intersection_prims: odd threads take (ij1, ij0), culling.py:88-91
        J = a + b - I;
    } else {
        ii = u;
        I = ij[2 * ii];
        J = ij[2 * ii + 1];
    }
}

constexpr int kXcds = 8;
// Which of n blocks the workgroup `loc` of a list takes (-1: none): the workgroups of one XCD
// (they are dealt to the XCDs in turn) take a contiguous run of blocks, whose entries share
// vertices in its L2.  n: the blocks in use, of a launch over at least as many rounded up.
__device__ __forceinline__ int64_t xcd_block(int64_t loc, int64_t n) {
    const int64_t run = (n + kXcds - 1) / kXcds, y = loc / kXcds, b = loc % kXcds * run + y;
    return y < run && b < n ? b : -1;
}

// The hull of the boxes of primitives [p0, p1) over the workgroup (four loads in flight a
// thread, past the end the last primitive again; sh: 6 floats a wave).
__device__ __forceinline__ void prims_hull(const float* __restrict__ lo, const float* __restrict__ hi, int p0, int p1,
                                           float* sh, float (&mn)[3], float (&mx)[3]) {
    constexpr int kAtOnce = 4;
    for (int k = 0; k < 3; ++k) {
        mn[k] = INFINITY;
        mx[k] = -INFINITY;
    }
    for (int p = p0 + threadIdx.x; p < p1; p += kAtOnce * kBlock) {
        float l[kAtOnce][3], h[kAtOnce][3];
#pragma unroll
        for (int j = 0; j < kAtOnce; ++j) {
            const int64_t q = 3 * (int64_t)min(p + j * kBlock, p1 - 1);
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                l[j][k] = lo[q + k];
                h[j][k] = hi[q + k];
            }
        }
#pragma unroll
        for (int j = 0; j < kAtOnce; ++j)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                mn[k] = fminf(mn[k], l[j][k]);
                mx[k] = fmaxf(mx[k], h[j][k]);
            }
    }
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            mn[k] = fminf(mn[k], __shfl_xor(mn[k], off, kWave));
            mx[k] = fmaxf(mx[k], __shfl_xor(mx[k], off, kWave));
        }
    if (lane_id() == 0)
        for (int k = 0; k < 3; ++k) {
            sh[6 * wave_id() + k] = mn[k];
            sh[6 * wave_id() + 3 + k] = mx[k];
        }
    __syncthreads();
    for (int w = 0; w < kBlock / kWave; ++w)
        for (int k = 0; k < 3; ++k) {
            mn[k] = fminf(mn[k], sh[6 * w + k]);
            mx[k] = fmaxf(mx[k], sh[6 * w + 3 + k]);
        }
}

// One workgroup per (unit, side): side 0 keeps the set-1 prims of I whose box overlaps the hull
// of J's set-2 prims, side 1 the set-2 prims of J against the hull of I's set-1 prims; local
// ids in ascending order.  Four primitives a thread and one barrier a pass.  (With the hulls
// of all bodies in a kernel before it, one wave a body, and one primitive a thread here, 634
// pairs of bodies of 3200 edges took 43 + 46 us; 33 here: the XCD order gives about 8 of that
// and overlap() loading all its bounds at once 30.)
__global__ __launch_bounds__(kBlock) void filter_kernel(int pt, const int32_t* __restrict__ ij, int64_t ntasks,
                                                         PrimSets S, int64_t maxs, int32_t* __restrict__ flist,
                                                         int64_t* __restrict__ fcnt) {
    constexpr int kWaves = kBlock / kWave, kPer = 4;
    __shared__ float sh[6 * kWaves];
    __shared__ int cnt[2][kWaves];
    // neighbouring units share bodies: the workgroups of one XCD take them in runs
    const int64_t task = xcd_block(blockIdx.x, ntasks);
    if (task < 0) return;  // uniform
    const int64_t u = task >> 1;
    const bool side = task & 1;
    int64_t ii;
    int I, J;
    unit_bodies(pt, u, ij, ii, I, J);
    const int32_t *offs = side ? S.off2 : S.off1, *offs_h = side ? S.off1 : S.off2;
    const float *lo = side ? S.lo2 : S.lo1, *hi = side ? S.hi2 : S.hi1;
    const int body = side ? J : I, other = side ? I : J;
    float mn[3], mx[3];
    prims_hull(side ? S.lo1 : S.lo2, side ? S.hi1 : S.hi2, offs_h[other], offs_h[other + 1], sh, mn, mx);
    const int p0 = offs[body], p1 = offs[body + 1];
    int32_t* dst = flist + task * maxs;
    int64_t run = 0;
    int turn = 0;
    for (int base = p0; base < p1; base += kPer * kBlock, turn ^= 1) {
        const int p = base + kPer * threadIdx.x;
        bool pred[kPer];
        int before = 0, mine = 0;
        const unsigned long long below = (1ull << lane_id()) - 1ull;
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const int64_t q = 3 * (int64_t)min(p + j, p1 - 1);
            pred[j] = overlap(lo + q, hi + q, mn, mx) && p + j < p1;
        }
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const unsigned long long m = __ballot(pred[j]);
            before += __popcll(m & below);
            mine += __popcll(m);
        }
        if (lane_id() == 0) cnt[turn][wave_id()] = mine;  // (buffers in turn: one barrier a pass)
        __syncthreads();
        int tot = 0;
        for (int w = 0; w < kWaves; ++w) {
            if (w < wave_id()) before += cnt[turn][w];
            tot += cnt[turn][w];
        }
        int64_t o = run + before;
#pragma unroll
        for (int j = 0; j < kPer; ++j)
            if (pred[j]) dst[o++] = p + j - p0;
        run += tot;
    }
    if (threadIdx.x == 0) fcnt[task] = run;
}

// The units' chunks of `chunk` primitive tests, scanned into their first chunks choff.
__global__ __launch_bounds__(kScanThreads) void unit_chunks_kernel(int64_t nunits, int chunk,
                                                                   const int64_t* __restrict__ fcnt,
                                                                   int64_t* __restrict__ choff,
                                                                   int64_t* __restrict__ total,
                                                                   int64_t* __restrict__ total2) {
    scan_block_exclusive_by(
        [=](int64_t u) { return (fcnt[2 * u] * fcnt[2 * u + 1] + chunk - 1) / chunk; }, choff, nunits, total, total2);
}

// last u with choff[u] <= c (choff non-decreasing, choff[0] = 0)
__device__ __forceinline__ int64_t find_unit(const int64_t* __restrict__ choff, int64_t nunits, int64_t c) {
    int64_t lo = 0, hi = nunits;  // invariant: choff[lo] <= c, answer in [lo, hi)
    while (hi - lo > 1) {
        int64_t mid = (lo + hi) >> 1;
        if (choff[mid] <= c)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

template <bool WRITE>
__global__ __launch_bounds__(kBlock) void prim_pairs_kernel(int pt, int chunk, const int32_t* __restrict__ ij,
                                                             PrimSets S, int64_t maxs, const int32_t* __restrict__ flist,
                                                             const int64_t* __restrict__ fcnt,
                                                             const int64_t* __restrict__ choff, int64_t nunits,
                                                             const int64_t* __restrict__ total_chunks,
                                                             int64_t* __restrict__ ccnt,
                                                             const int64_t* __restrict__ ccoff,
                                                             int32_t* __restrict__ out, int64_t cap) {
    __shared__ int shw[kBlock / kWave];
    const int64_t T = *total_chunks;
    for (int64_t c = blockIdx.x; c < T; c += gridDim.x) {
        int64_t u = find_unit(choff, nunits, c);
        int64_t ii;
        int I, J;
        unit_bodies(pt, u, ij, ii, I, J);
        const uint32_t nA = (uint32_t)fcnt[2 * u], nB = (uint32_t)fcnt[2 * u + 1];
        const uint32_t nt = nA * nB;
        const int32_t* LA = flist + (2 * u) * maxs;
        const int32_t* LB = flist + (2 * u + 1) * maxs;
        const int oA = S.off1[I], oB = S.off2[J];
        const uint32_t f0 = (uint32_t)(c - choff[u]) * (uint32_t)chunk;
        const uint32_t f1 = f0 + (uint32_t)chunk < nt ? f0 + (uint32_t)chunk : nt;
        int64_t run = WRITE ? ccoff[c] : 0;
        for (uint32_t base = f0; base < f1; base += kBlock) {
            uint32_t f = base + threadIdx.x;
            bool pred = false;
            int32_t a = 0, b = 0;
            if (f < f1) {
                uint32_t i = f / nB, j = f - i * nB;
                a = LA[i];
                b = LB[j];
                int64_t ga = oA + a, gb = oB + b;
                pred = overlap(S.lo1 + 3 * ga, S.hi1 + 3 * ga, S.lo2 + 3 * gb, S.hi2 + 3 * gb);
            }
            int tot;
            int r = block_rank(pred, shw, &tot);
            if (WRITE && pred) {
                int64_t o = run + r;
                if (o < cap) {
                    int32_t* t5 = out + 5 * o;
                    t5[0] = I;
                    t5[1] = J;
                    t5[2] = (int32_t)ii;
                    t5[3] = a;
                    t5[4] = b;
                }
            }
            run += tot;
        }
        if (!WRITE && threadIdx.x == 0) ccnt[c] = run;
    }
}

// ------------------------------------------------------------------- VG
template <bool WRITE>
__global__ __launch_bounds__(kBlock) void vg_kernel(int64_t nv, const int32_t* __restrict__ vert_body,
                                                     const int32_t* __restrict__ voff, const float* __restrict__ blo,
                                                     const float* __restrict__ plo, const float* __restrict__ phi,
                                                     double ythresh, float fground, int64_t* __restrict__ bcnt,
                                                     const int64_t* __restrict__ boff, int32_t* __restrict__ out,
                                                     int64_t cap) {
    constexpr int kWaves = kBlock / kWave;
    __shared__ int cnt[kItems * kWaves];
    const float qlo[3] = {-1e3f, -1e3f, -1e3f};
    const float qhi[3] = {1e3f, fground, 1e3f};
    const int64_t base = (int64_t)blockIdx.x * kBlock * kItems;
    // all of a thread's items first (their loads in flight together), then one ranking
    bool pred[kItems];
    int32_t body[kItems];
#pragma unroll
    for (int it = 0; it < kItems; ++it) {
        const int64_t v = base + (int64_t)it * kBlock + threadIdx.x, u = v < nv ? v : nv - 1;
        body[it] = vert_body[u];
        // culling.py:67: lowers[i][1] < 0.5 * dhat + ground (FP64)
        pred[it] = overlap(plo + 3 * u, phi + 3 * u, qlo, qhi) && v < nv;
    }
#pragma unroll
    for (int it = 0; it < kItems; ++it) pred[it] = pred[it] && (double)blo[3 * body[it] + 1] < ythresh;
    int rank[kItems];
#pragma unroll
    for (int it = 0; it < kItems; ++it) {
        const unsigned long long m = __ballot(pred[it]);
        rank[it] = __popcll(m & ((1ull << lane_id()) - 1ull));
        if (lane_id() == 0) cnt[it * kWaves + wave_id()] = __popcll(m);
    }
    __syncthreads();
    int64_t run = WRITE ? boff[blockIdx.x] : 0;
#pragma unroll
    for (int it = 0; it < kItems; ++it)
        for (int w = 0; w < kWaves; ++w) {
            if (WRITE && pred[it] && w == wave_id()) {
                const int64_t o = run + rank[it];
                if (o < cap) {
                    const int64_t v = base + (int64_t)it * kBlock + threadIdx.x;
                    out[2 * o] = body[it];
                    out[2 * o + 1] = (int32_t)(v - voff[body[it]]);
                }
            }
            run += cnt[it * kWaves + w];
        }
    if (!WRITE && threadIdx.x == 0) bcnt[blockIdx.x] = run;
}

// ------------------------------------------------------------ structure
__global__ void triplets_kernel(int nb, int64_t nij, const int32_t* __restrict__ ij, int32_t* __restrict__ rows,
                                int32_t* __restrict__ cols) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t nslot = nb + 2 * nij;
    if (t >= 16 * nslot) return;
    int64_t i = t / 16;
    int e = (int)(t % 16), ii = e % 4, jj = e / 4;
    int64_t I, J;
    if (i < nb) {
        I = J = i;
    } else if (i < nb + nij) {
        I = ij[2 * (i - nb)];
        J = ij[2 * (i - nb) + 1];
    } else {
        I = ij[2 * (i - nb - nij) + 1];
        J = ij[2 * (i - nb - nij)];
    }
    rows[16 * i + ii + jj * 4] = (int32_t)(ii + 4 * I);
    cols[16 * i + ii + jj * 4] = (int32_t)(jj + 4 * J);
}

// first k in [lo, hi) with key(k) >= v; keys non-decreasing, key(k) = a[2k + comp]
__device__ __forceinline__ int64_t lower_bound2(const int32_t* __restrict__ a, int comp, int64_t lo, int64_t hi,
                                                int v) {
    while (lo < hi) {
        int64_t mid = (lo + hi) >> 1;
        if (a[2 * mid + comp] < v)
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

// The block structure from the sorted pairs, one thread per body row: before row b lie one
// diagonal entry a body, the pairs whose first body is below b and those whose second is
// (found in the sorted lists, so no scan of row lengths).  dnij (nullable): the pair count on
// the device (nij is then unused).
__global__ void structure_kernel(int nb, int64_t nij, const int64_t* __restrict__ dnij,
                                 const int32_t* __restrict__ ij, const int32_t* __restrict__ ji,
                                 int32_t* __restrict__ row_ptr, int32_t* __restrict__ cols,
                                 int32_t* __restrict__ slots) {
    int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nb) return;
    if (dnij) nij = *dnij;
    const int64_t l0 = lower_bound2(ji, 1, 0, nij, b), u0 = lower_bound2(ij, 0, 0, nij, b);
    int64_t o = b + l0 + u0;
    row_ptr[b] = (int32_t)o;
    if (b == nb - 1) row_ptr[nb] = (int32_t)(nb + 2 * nij);
    for (int64_t k = l0; k < nij && ji[2 * k + 1] == b; ++k) {
        const int i = ji[2 * k];
        const int64_t v0 = lower_bound2(ij, 0, 0, nij, i), v1 = lower_bound2(ij, 0, v0, nij, i + 1);
        cols[o] = i;
        slots[o] = (int32_t)(nb + nij + lower_bound2(ij, 1, v0, v1, b));
        ++o;
    }
    cols[o] = b;
    slots[o] = b;
    ++o;
    for (int64_t k = u0; k < nij && ij[2 * k] == b; ++k) {
        cols[o] = ij[2 * k + 1];
        slots[o] = (int32_t)(nb + k);
        ++o;
    }
}

// ------------------------------------------------------- staged culling
// The primitive-pair culling in three stages that leave their counts on the device,
// so that a caller can run several cullings side by side and read all their counts in
// one host synchronization.  `set` selects one of two independent workspaces.
namespace {
const int kCullSlots[2][5] = {
    {kSlotFilter, kSlotFilterCount, kSlotScanB, kSlotChunkCount, kSlotChunk},
    {kSlotFilterB, kSlotFilterCountB, kSlotScanBB, kSlotChunkCountB, kSlotChunkB}};
}  // namespace

int prim_cull_begin(hipStream_t s, const AbdScene* sc, int mode, const int32_t* ij, int64_t nij, const float* lo1,
                    const float* hi1, const float* lo2, const float* hi2, int set, PrimCull& C,
                    int64_t* total_copy) {
    const int* slot = kCullSlots[set];
    C.set = set;
    C.pt = mode == ABD_CULL_PT;
    C.ij = ij;
    PrimSets& S = C.S;
    S.off1 = C.pt ? sc->voff : sc->eoff;
    S.off2 = C.pt ? sc->foff : sc->eoff;
    S.lo1 = lo1;
    S.hi1 = hi1;
    S.lo2 = lo2;
    S.hi2 = hi2;
    const int64_t max1 = C.pt ? sc->max_verts : sc->max_edges;
    const int64_t max2 = C.pt ? sc->max_tris : sc->max_edges;
    C.maxs = max1 > max2 ? max1 : max2;
    if (C.maxs > 65535) return ABD_ERR_ARG;  // n1 * n2 tests per body pair must fit in 32 bits
    C.nunits = C.pt ? 2 * nij : nij;
    if (2 * C.nunits > INT32_MAX) return ABD_ERR_ARG;
    int rc;
    if ((rc = arena_get(slot[0], sizeof(int32_t) * (size_t)(2 * C.nunits * C.maxs), (void**)&C.flist))) return rc;
    if ((rc = arena_get(slot[1], sizeof(int64_t) * (size_t)(2 * C.nunits), (void**)&C.fcnt))) return rc;
    if ((rc = arena_get(slot[2], sizeof(int64_t) * (size_t)(C.nunits + 1), (void**)&C.choff))) return rc;
    int ph = prof_start(kProfFilter, s, 0.0);
    launch_kernel(filter_kernel, dim3((unsigned)(ceil_div(2 * C.nunits, (int64_t)kXcds) * kXcds)), dim3(kBlock), 0, s,
                  C.pt, ij, 2 * C.nunits, S, C.maxs,
                       C.flist, C.fcnt);
    ABD_CHECK_LAUNCH();
    prof_stop(ph, s);
    C.tune = tuning();
    launch_kernel(unit_chunks_kernel, dim3(1), dim3(kScanThreads), 0, s, C.nunits, C.tune.cull_chunk,
                       (const int64_t*)C.fcnt, C.choff, C.choff + C.nunits, total_copy);
    ABD_CHECK_LAUNCH();
    C.total_chunks = C.choff + C.nunits;
    C.total_pairs = nullptr;
    return ABD_OK;
}

int prim_cull_count(hipStream_t s, PrimCull& C, int64_t T, int64_t* total_copy) {
    const int* slot = kCullSlots[C.set];
    C.T = T;
    if (T == 0) return ABD_OK;
    int rc;
    if ((rc = arena_get(slot[3], sizeof(int64_t) * (size_t)(T + 1), (void**)&C.ccnt))) return rc;
    if ((rc = arena_get(slot[4], sizeof(int64_t) * (size_t)(T + 1), (void**)&C.ccoff))) return rc;
    C.grid = (unsigned)(T < C.tune.cull_grid ? T : C.tune.cull_grid);
    int ph = prof_start(kProfPrimCount, s, 0.0);
    launch_kernel(prim_pairs_kernel<false>, dim3(C.grid), dim3(kBlock), 0, s, C.pt, C.tune.cull_chunk, C.ij, C.S,
                       C.maxs, (const int32_t*)C.flist, (const int64_t*)C.fcnt, (const int64_t*)C.choff, C.nunits,
                       (const int64_t*)C.total_chunks, C.ccnt, (const int64_t*)nullptr, (int32_t*)nullptr, (int64_t)0);
    ABD_CHECK_LAUNCH();
    prof_stop(ph, s);
    if ((rc = scan_exclusive_i64(s, C.ccnt, C.ccoff, T, C.ccoff + T, total_copy))) return rc;
    C.total_pairs = C.ccoff + T;
    return ABD_OK;
}

int prim_cull_fill(hipStream_t s, PrimCull& C, int32_t* out, int64_t cap, int64_t n) {
    if (C.T == 0 || n == 0) return ABD_OK;
    int ph = prof_start(kProfPrimFill, s, 20.0 * n);
    launch_kernel(prim_pairs_kernel<true>, dim3(C.grid), dim3(kBlock), 0, s, C.pt, C.tune.cull_chunk, C.ij, C.S,
                       C.maxs, (const int32_t*)C.flist, (const int64_t*)C.fcnt, (const int64_t*)C.choff, C.nunits,
                       (const int64_t*)C.total_chunks, C.ccnt, (const int64_t*)C.ccoff, out, cap);
    ABD_CHECK_LAUNCH();
    prof_stop(ph, s);
    return ABD_OK;
}

int vg_cull_begin(hipStream_t s, const AbdScene* sc, const float* blo, const float* plo, const float* phi, double dhat,
                  double ground, VgCull& C,
                  int64_t* total_copy) {
    C.sc = sc;
    C.blo = blo;
    C.plo = plo;
    C.phi = phi;
    C.yth = 0.5 * dhat + ground;
    C.fg = (float)ground;
    const int64_t nv = sc->n_verts;
    C.nblk = ceil_div(nv, (int64_t)kBlock * kItems);
    C.total = nullptr;
    if (nv == 0) return ABD_OK;
    int rc;
    if ((rc = arena_get(kSlotVgA, sizeof(int64_t) * (C.nblk + 1), (void**)&C.bcnt))) return rc;
    if ((rc = arena_get(kSlotVgB, sizeof(int64_t) * (C.nblk + 1), (void**)&C.boff))) return rc;
    int ph = prof_start(kProfVg, s, 28.0 * nv);
    launch_kernel(vg_kernel<false>, dim3((unsigned)C.nblk), dim3(kBlock), 0, s, nv, sc->vert_body, sc->voff, blo,
                       plo, phi, C.yth, C.fg, C.bcnt, (const int64_t*)nullptr, (int32_t*)nullptr, (int64_t)0);
    ABD_CHECK_LAUNCH();
    prof_stop(ph, s);
    if ((rc = scan_exclusive_i64(s, C.bcnt, C.boff, C.nblk, C.boff + C.nblk, total_copy))) return rc;
    C.total = C.boff + C.nblk;
    return ABD_OK;
}

int vg_cull_fill(hipStream_t s, VgCull& C, int32_t* out, int64_t cap, int64_t n) {
    if (n == 0 || !C.total) return ABD_OK;
    const AbdScene* sc = C.sc;
    launch_kernel(vg_kernel<true>, dim3((unsigned)C.nblk), dim3(kBlock), 0, s, (int64_t)sc->n_verts,
                       sc->vert_body, sc->voff, C.blo, C.plo, C.phi, C.yth, C.fg, C.bcnt, (const int64_t*)C.boff, out,
                       cap);
    ABD_CHECK_LAUNCH();
    return ABD_OK;
}

// abd_cull_bodies; ji == nullptr skips the (j, i) order.
int cull_bodies(hipStream_t s, const AbdScene* sc, const float* lo, const float* hi, int32_t* ij, int32_t* ji,
                int64_t cap, int64_t* count) {
    const int nb = sc->n_bodies;
    SceneSeg sg{0, nullptr, nullptr};
    int64_t npairs = (int64_t)nb * (nb - 1) / 2;
    if (sc->n_scenes > 1 && sc->scene_boff && sc->scene_poff) {
        sg = SceneSeg{sc->n_scenes, sc->scene_boff, sc->scene_poff};
        npairs = sc->n_scene_pairs;
    }
    *count = 0;
    if (npairs <= 0) return ABD_OK;
    const int64_t nblk = ceil_div(npairs, (int64_t)kBlock * kPairItems);
    if (nblk > INT32_MAX) return ABD_ERR_ARG;
    // both orders at once: counts, scans (the totals are equal), then the lists
    const int orders = ji ? 2 : 1;
    int64_t *bcnt, *boff;
    int rc = arena_get(kSlotScanA, sizeof(int64_t) * orders * (nblk + 1), (void**)&bcnt);
    if (rc) return rc;
    rc = arena_get(kSlotScanB, sizeof(int64_t) * orders * (nblk + 1), (void**)&boff);
    if (rc) return rc;
    int ph = prof_start(kProfBodyPairs, s, 24.0 * nb);
    launch_kernel(body_pairs_kernel<false>, dim3((unsigned)nblk, orders), dim3(kBlock), 0, s, nb, npairs, sg,
                       sc->body_scene, lo, hi, bcnt, (const int64_t*)nullptr, (int32_t*)nullptr, (int32_t*)nullptr,
                       (int64_t)0);
    ABD_CHECK_LAUNCH();
    prof_stop(ph, s);
    ScanSeg sg2[2];
    for (int k = 0; k < orders; ++k) {
        const int64_t o = k * (nblk + 1);
        sg2[k] = ScanSeg{bcnt + o, boff + o, nblk, boff + o + nblk, nullptr};
    }
    if ((rc = scan_exclusive_i64_multi(s, sg2, orders))) return rc;
    int64_t n;
    if ((rc = read_i64(s, boff + nblk, &n))) return rc;
    *count = n;
    if (n > cap) return ABD_ERR_OVERFLOW;
    if (n == 0) return ABD_OK;
    launch_kernel(body_pairs_kernel<true>, dim3((unsigned)nblk, orders), dim3(kBlock), 0, s, nb, npairs, sg,
                       sc->body_scene, lo, hi, bcnt, (const int64_t*)boff, ij, ji, cap);
    ABD_CHECK_LAUNCH();
    return ABD_OK;
}


}  // namespace abd

using namespace abd;

extern "C" {

int abd_cull_bodies(abd_stream_t stream, const AbdScene* sc, const float* lo, const float* hi, int32_t* ij,
                    int32_t* ji, int64_t cap, int64_t* count) {
    if (!sc || !lo || !hi || !count || cap < 0 || (cap > 0 && (!ij || !ji))) return ABD_ERR_ARG;
    return cull_bodies(to_stream(stream), sc, lo, hi, ij, ji, cap, count);
}

int abd_cull_prims(abd_stream_t stream, const AbdScene* sc, int32_t mode, const int32_t* ij, int64_t nij,
                   const float* lo1, const float* hi1, const float* lo2, const float* hi2, int32_t* out, int64_t cap,
                   int64_t* count) {
    if (!sc || !count || nij < 0 || cap < 0 || (nij > 0 && !ij) || !lo1 || !hi1 || !lo2 || !hi2 ||
        (cap > 0 && !out))
        return ABD_ERR_ARG;
    if (mode != ABD_CULL_PT && mode != ABD_CULL_EE) return ABD_ERR_ARG;
    *count = 0;
    if (nij == 0) return ABD_OK;
    hipStream_t s = to_stream(stream);
    PrimCull C;
    int rc = prim_cull_begin(s, sc, mode, ij, nij, lo1, hi1, lo2, hi2, 0, C);
    if (rc) return rc;
    int64_t T;
    if ((rc = read_i64(s, C.total_chunks, &T))) return rc;
    if ((rc = prim_cull_count(s, C, T))) return rc;
    if (T == 0) return ABD_OK;
    int64_t n;
    if ((rc = read_i64(s, C.total_pairs, &n))) return rc;
    *count = n;
    if (n > cap) return ABD_ERR_OVERFLOW;
    if (n == 0) return ABD_OK;
    return prim_cull_fill(s, C, out, cap, n);
}

int abd_cull_vg(abd_stream_t stream, const AbdScene* sc, const float* blo, const float* plo, const float* phi,
                double dhat, double ground, int32_t* out, int64_t cap, int64_t* count) {
    if (!sc || !blo || !plo || !phi || !count || cap < 0 || (cap > 0 && !out)) return ABD_ERR_ARG;
    hipStream_t s = to_stream(stream);
    *count = 0;
    if (sc->n_verts == 0) return ABD_OK;
    VgCull C;
    int rc = vg_cull_begin(s, sc, blo, plo, phi, dhat, ground, C);
    if (rc) return rc;
    int64_t n;
    if ((rc = read_i64(s, C.total, &n))) return rc;
    *count = n;
    if (n > cap) return ABD_ERR_OVERFLOW;
    return vg_cull_fill(s, C, out, cap, n);
}

int abd_set_triplets(abd_stream_t stream, int32_t nb, const int32_t* ij, int64_t nij, int32_t* rows,
                     int32_t* cols) {
    if (nb < 0 || nij < 0 || (nij > 0 && !ij) || !rows || !cols) return ABD_ERR_ARG;
    int64_t n = 16 * ((int64_t)nb + 2 * nij);
    if (n == 0) return ABD_OK;
    launch_kernel(triplets_kernel, dim3(grid_for(n, kBlock, INT32_MAX)), dim3(kBlock), 0, to_stream(stream), nb,
                       nij, ij, rows, cols);
    ABD_CHECK_LAUNCH();
    return ABD_OK;
}

int abd_bsr_structure(abd_stream_t stream, int32_t nb, const int32_t* ij, const int32_t* ji, int64_t nij,
                      int32_t* row_ptr, int32_t* cols, int32_t* slots) {
    if (nb <= 0 || nij < 0 || (nij > 0 && (!ij || !ji)) || !row_ptr || !cols || !slots) return ABD_ERR_ARG;
    return bsr_structure(to_stream(stream), nb, ij, ji, nij, nullptr, row_ptr, cols, slots);
}

}  // extern "C"

namespace abd {

int bsr_structure(hipStream_t s, int nb, const int32_t* ij, const int32_t* ji, int64_t nij, const int64_t* dnij,
                  int32_t* row_ptr, int32_t* cols, int32_t* slots) {
    launch_kernel(structure_kernel, dim3(grid_for(nb, kWave, INT32_MAX)), dim3(kWave), 0, s, nb, nij, dnij, ij, ji,
                       row_ptr, cols, slots);
    ABD_CHECK_LAUNCH();
    return ABD_OK;
}

// ------------------------------------------------- collision set from a superset
// The pairs and candidates of a candidate set made from larger boxes (the swept set of
// the last step: boxes over x - alpha dq, alpha in [0, 1], dilated as the collision set's)
// that pass the culling predicates on the current boxes.  When the current boxes lie
// inside those the superset was made from, this is the culling's own output: the same
// predicates on the same boxes, and the superset's sorted order restricted to the kept
// entries (pair indices renumbered through `remap`).
namespace {

// The five lists of a keep pass: 0 ij, 1 ji, 2 PT, 3 EE, 4 VG.
constexpr int kKeepLists = 5;
// blocks of a super-block: a block's offset is the sum of the super-blocks' counts before its
// own (added to by the count pass: integers, any order) and of the blocks' before it inside
constexpr int kSuper = 64;
// words between super-block counts: adds to one cache line wait for each other (about 10 ns
// each: packed, a count pass of 18 k blocks took 108 us instead of 87)
constexpr int kSuperStride = 8;
constexpr int kFlagAlign = 16;
// blocks of PT / EE entries a workgroup of the sweep's write pass takes
constexpr int kSweepBlocks = 4;  // (a thread's flags are one word)
struct KeepArgs {
    KeepInput in;
    KeepBoxes bx;
    KeepOutput out;
    const int32_t *voff, *foff, *eoff;
    int32_t* remap;
    double yth;
    float fg;
    int64_t n[kKeepLists];
    int64_t blk0[kKeepLists + 1];  // first workgroup of each list (one per block of kBlock
                                   // entries, rounded up to a multiple of kXcds)
    uint32_t* bcnt[kKeepLists];    // kept entries of each block
    uint32_t* scnt[kKeepLists];    // and of each super-block
    const int64_t* pair_off;       // the pair blocks' offsets when a scan made them
    int64_t* dcount;               // the five totals
    uint8_t* flag;                 // each entry's predicate (count pass), read by the write pass
    int64_t flag0[kKeepLists];     // first flag of each list (a multiple of kFlagAlign)
    int64_t grp0[kKeepLists + 1];  // first workgroup of each list in the sweep's write pass
    // primitive boxes from the vertices when x is set (KeepAtX)
    const double *x, *x1;
    const int32_t *tris, *edges;
    float pdil;
    double edil, tdil;
    const float4* ebox;   // KeepAtX
    const double* alpha;  // KeepAtX: entries apart at their scene's step length are dropped
    const int32_t* body_scene;
    KeepSweep W;
};

// point_boxes_kernel's box of vertex v at x, or with x1 set swept_point_boxes_kernel's
// (the union with the box at x1)
__device__ __forceinline__ void point_box_at(const double* __restrict__ x, const double* __restrict__ x1,
                                             int64_t v, float dil, float* lo, float* hi) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float c = (float)x[3 * v + k];
        if (x1) {
            const float c1 = (float)x1[3 * v + k];
            lo[k] = fminf(c - dil, c1 - dil);
            hi[k] = fmaxf(c + dil, c1 + dil);
        } else {
            lo[k] = c - dil;
            hi[k] = c + dil;
        }
    }
}

// prim_boxes_kernel's box of the primitive with scene vertices vi[0..NV) (its topology's
// order) at x, or with x1 set swept_prim_boxes_kernel's
template <int NV>
__device__ __forceinline__ void prim_box_of(const double* __restrict__ x, const double* __restrict__ x1,
                                            const int64_t (&vi)[NV], double dil, float* lo, float* hi) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        double mn = x[3 * vi[0] + k], mx = mn;
#pragma unroll
        for (int j = 1; j < NV; ++j) {
            const double c = x[3 * vi[j] + k];
            mn = c < mn ? c : mn;
            mx = c > mx ? c : mx;
        }
        float l = (float)(mn - dil), h = (float)(mx + dil);
        if (x1) {
            double mn1 = x1[3 * vi[0] + k], mx1 = mn1;
#pragma unroll
            for (int j = 1; j < NV; ++j) {
                const double c = x1[3 * vi[j] + k];
                mn1 = c < mn1 ? c : mn1;
                mx1 = c > mx1 ? c : mx1;
            }
            l = fminf(l, (float)(mn1 - dil));
            h = fmaxf(h, (float)(mx1 + dil));
        }
        lo[k] = l;
        hi[k] = h;
    }
}
// the same for primitive i (NV vertices from topo, numbered from vb)
template <int NV>
__device__ __forceinline__ void prim_box_at(const double* __restrict__ x, const double* __restrict__ x1,
                                            const int32_t* __restrict__ topo, int64_t i, int vb, double dil,
                                            float* lo, float* hi) {
    int64_t vi[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) vi[j] = vb + topo[NV * i + j];
    prim_box_of<NV>(x, x1, vi, dil, lo, hi);
}

// an entry of body b apart at the step length its scene has taken: the boxes there do not
// overlap, and neither they nor the vertices need to be read
__device__ __forceinline__ bool keep_apart(const KeepArgs& A, int b, float apart) {
    return A.alpha[A.body_scene ? A.body_scene[b] : 0] < (double)apart;
}

__device__ __forceinline__ bool keep_pred(const KeepArgs& A, int k, int64_t i) {
    const KeepBoxes& B = A.bx;
    if (k <= 1) {
        const int32_t* pr = (k == 0 ? A.in.ij : A.in.ji) + 2 * i;
        const int a = pr[0], b = pr[1];
        return overlap(B.blo + 3 * a, B.bhi + 3 * a, B.blo + 3 * b, B.bhi + 3 * b);
    }
    if (k <= 3) {  // (I, J, ii, a, b): both bodies' boxes and the two primitives' boxes
        const int32_t* t5 = (k == 2 ? A.in.pt : A.in.ee) + 5 * i;
        const int I = t5[0], J = t5[1];
        if (A.alpha && keep_apart(A, I, (k == 2 ? A.in.vids.apart_pt : A.in.vids.apart_ee)[i])) return false;
        const int32_t* vid = k == 2 ? A.in.vids.pt : A.in.vids.ee;
        if (A.x && vid) {  // the candidate's vertex ids stored beside the list
            vid += 4 * i;
            const int64_t v0 = vid[0], v1 = vid[1], v2 = vid[2], v3 = vid[3];
            if (!overlap(B.blo + 3 * I, B.bhi + 3 * I, B.blo + 3 * J, B.bhi + 3 * J)) return false;
            if (k == 3 && A.ebox) {
                // an edge's swept box is the union of its vertices': rounding and the dilation
                // are monotone, so the bounds are prim_box_of's.  Half the gathers, which bound
                // this pass (4.5 M entries 90 -> 70 us, for 11 us more in body_end, 1.06 M vertices)
                float4 a[4], b[4];
                const int64_t v[4] = {v0, v1, v2, v3};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    a[j] = A.ebox[2 * v[j]];
                    b[j] = A.ebox[2 * v[j] + 1];
                }
                const float l1[3] = {fminf(a[0].x, a[1].x), fminf(a[0].y, a[1].y), fminf(a[0].z, a[1].z)};
                const float l2[3] = {fminf(a[2].x, a[3].x), fminf(a[2].y, a[3].y), fminf(a[2].z, a[3].z)};
                const float h1[3] = {fmaxf(a[0].w, a[1].w), fmaxf(b[0].x, b[1].x), fmaxf(b[0].y, b[1].y)};
                const float h2[3] = {fmaxf(a[2].w, a[3].w), fmaxf(b[2].x, b[3].x), fmaxf(b[2].y, b[3].y)};
                return overlap(l1, h1, l2, h2);
            }
            float l1[3], h1[3], l2[3], h2[3];
            if (k == 2) {
                point_box_at(A.x, A.x1, v0, A.pdil, l1, h1);
                const int64_t tv[3] = {v1, v2, v3};
                prim_box_of<3>(A.x, A.x1, tv, A.tdil, l2, h2);
            } else {
                const int64_t ea[2] = {v0, v1}, eb[2] = {v2, v3};
                prim_box_of<2>(A.x, A.x1, ea, A.edil, l1, h1);
                prim_box_of<2>(A.x, A.x1, eb, A.edil, l2, h2);
            }
            return overlap(l1, h1, l2, h2);
        }
        if (!overlap(B.blo + 3 * I, B.bhi + 3 * I, B.blo + 3 * J, B.bhi + 3 * J)) return false;
        const int64_t a = (k == 2 ? A.voff : A.eoff)[I] + (int64_t)t5[3];
        const int64_t b = (k == 2 ? A.foff : A.eoff)[J] + (int64_t)t5[4];
        if (A.x) {
            // a: a point of I (PT) or an edge of I; b: a triangle or an edge of J
            float l1[3], h1[3], l2[3], h2[3];
            if (k == 2) {
                point_box_at(A.x, A.x1, a, A.pdil, l1, h1);
                prim_box_at<3>(A.x, A.x1, A.tris, b, A.voff[J], A.tdil, l2, h2);
            } else {
                prim_box_at<2>(A.x, A.x1, A.edges, a, A.voff[I], A.edil, l1, h1);
                prim_box_at<2>(A.x, A.x1, A.edges, b, A.voff[J], A.edil, l2, h2);
            }
            return overlap(l1, h1, l2, h2);
        }
        const float *lo1 = k == 2 ? B.plo : B.elo, *hi1 = k == 2 ? B.phi : B.ehi;
        const float *lo2 = k == 2 ? B.tlo : B.elo, *hi2 = k == 2 ? B.thi : B.ehi;
        return overlap(lo1 + 3 * a, hi1 + 3 * a, lo2 + 3 * b, hi2 + 3 * b);
    }
    // VG (b, v): the predicate of vg_kernel
    const float qlo[3] = {-1e3f, -1e3f, -1e3f};
    const float qhi[3] = {1e3f, A.fg, 1e3f};
    const int b = A.in.vg[2 * i];
    if (A.alpha && keep_apart(A, b, A.in.vids.apart_vg[i])) return false;
    const int64_t v = A.voff[b] + (int64_t)A.in.vg[2 * i + 1];
    if (!((double)B.blo[3 * b + 1] < A.yth)) return false;
    if (A.x) {
        float l[3], h[3];
        point_box_at(A.x, A.x1, v, A.pdil, l, h);
        return overlap(l, h, qlo, qhi);
    }
    return overlap(B.plo + 3 * v, B.phi + 3 * v, qlo, qhi);
}

template <class Off>
__device__ __forceinline__ void keep_write(const KeepArgs& A, const Off& pair_off, int k, int64_t i, int64_t o) {
    if (k <= 1) {
        const int32_t* pr = (k == 0 ? A.in.ij : A.in.ji) + 2 * i;
        int32_t* q = (k == 0 ? A.out.ij : A.out.ji) + 2 * o;
        q[0] = pr[0];
        q[1] = pr[1];
    } else if (k <= 3) {
        const int32_t* t5 = (k == 2 ? A.in.pt : A.in.ee) + 5 * i;
        int32_t* q = (k == 2 ? A.out.pt : A.out.ee) + 5 * o;
        q[0] = t5[0];
        q[1] = t5[1];
        // the pair's index in the kept ij: its block's offset + its rank in the block (the
        // tuple is kept only if its pair's body boxes overlap, so the pair is kept)
        q[2] = (int32_t)(pair_off[t5[2] / kBlock] + A.remap[t5[2]]);
        q[3] = t5[3];
        q[4] = t5[4];
        const int32_t* vin = k == 2 ? A.in.vids.pt : A.in.vids.ee;
        int32_t* vout = k == 2 ? A.out.ptv : A.out.eev;
        if (vin && vout) {
#pragma unroll
            for (int j = 0; j < 4; ++j) vout[4 * o + j] = vin[4 * i + j];
        }
    } else {
        A.out.vg[2 * o] = A.in.vg[2 * i];
        A.out.vg[2 * o + 1] = A.in.vg[2 * i + 1];
    }
}

// The count: one entry per thread (its predicate's gathers need many waves in flight to
// hide their latency), the kept entries of each workgroup's kBlock entries to bcnt; each
// entry's predicate is stored for the write pass, and each kept pair's rank in its
// workgroup's kept pairs (ij) to remap, so that the write pass places pairs and tuples in one
// launch.
// entries of input list k: A.n[k], or with the input sizes on the device (A.in.dn, the
// keep output layout) that count (A.n[k] then bounds it)
__device__ __forceinline__ int64_t keep_n(const KeepArgs& A, int k) {
    return A.in.dn ? (k == 1 && !A.in.ji ? 0 : A.in.dn[k]) : A.n[k];
}

__device__ __forceinline__ int64_t blocks_of(int64_t n) { return (n + kBlock - 1) / kBlock; }

__global__ __launch_bounds__(kBlock) void keep_count_kernel(KeepArgs A) {
    __shared__ int shw[kBlock / kWave];
    const int64_t g = blockIdx.x;
    int k = 0;
    while (k + 1 < kKeepLists && g >= A.blk0[k + 1]) ++k;
    const int64_t nk = keep_n(A, k), blk = xcd_block(g - A.blk0[k], blocks_of(nk));
    if (blk < 0) return;  // uniform
    const int64_t i = blk * kBlock + threadIdx.x;
    const bool in_list = i < nk;
    const bool pred = in_list && keep_pred(A, k, i);
    if (in_list) A.flag[A.flag0[k] + i] = pred ? 1 : 0;
    int tot;
    const int r = block_rank(pred, shw, &tot);
    if (k == 0 && in_list) A.remap[i] = pred ? r : -1;
    if (threadIdx.x == 0) {
        A.bcnt[k][blk] = (uint32_t)tot;
        if (tot) atomicAdd(A.scnt[k] + kSuperStride * (blk / kSuper), (uint32_t)tot);
    }
}

// The kept entries before block blk of list k: whole super-blocks, then the blocks of its own.
__device__ __forceinline__ int64_t block_offset(const KeepArgs& A, int k, int64_t blk, int64_t* sh) {
    const int64_t sb = blk / kSuper;
    int64_t v = 0;
    for (int64_t q = threadIdx.x; q < sb; q += kBlock) v += A.scnt[k][kSuperStride * q];
    const int64_t b = sb * kSuper + threadIdx.x;
    if (b < blk) v += A.bcnt[k][b];
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) v += __shfl_xor(v, off);
    if (lane_id() == 0) sh[wave_id()] = v;
    __syncthreads();
    v = 0;
    for (int w = 0; w < kBlock / kWave; ++w) v += sh[w];
    __syncthreads();
    return v;
}

// The pair blocks' offsets, which place the tuples' pair indices: summed in LDS where there
// are at most kBlock of them (65536 pairs), else scanned before.
__device__ __forceinline__ void pair_offsets(const KeepArgs& A, int64_t* poff, int64_t* sh) {
    if (A.pair_off) return;
    const int t = threadIdx.x;
    poff[t] = block_exclusive_scan_i64(t < blocks_of(keep_n(A, 0)) ? (int64_t)A.bcnt[0][t] : 0, sh);
    __syncthreads();
}
__device__ __forceinline__ void write_entry(const KeepArgs& A, const int64_t* poff, int k, int64_t i, int64_t o) {
    if (A.pair_off)
        keep_write(A, A.pair_off, k, i, o);
    else
        keep_write(A, poff, k, i, o);
}

// The write pass, one entry per thread: the kept entries at their ordered ranks (the block's
// offset + the rank in the block), the totals by each list's last block.
__global__ __launch_bounds__(kBlock) void keep_write_kernel(KeepArgs A) {
    __shared__ int shw[kBlock / kWave];
    __shared__ int64_t sh[kBlock / kWave];
    __shared__ int64_t poff[kBlock];
    const int64_t g = blockIdx.x;
    const int t = threadIdx.x;
    if (g == 0 && t < kKeepLists && A.blk0[t] == A.blk0[t + 1]) A.dcount[t] = 0;  // an empty list
    if (g >= A.blk0[kKeepLists]) return;
    int k = 0;
    while (k + 1 < kKeepLists && g >= A.blk0[k + 1]) ++k;
    const int64_t nk = keep_n(A, k), nblk = blocks_of(nk), blk = xcd_block(g - A.blk0[k], nblk);
    if (nk == 0 && g == A.blk0[k] && t == 0) A.dcount[k] = 0;
    if (blk < 0) return;  // uniform
    const bool last = blk + 1 == nblk;
    const uint32_t mine = A.bcnt[k][blk];
    if (mine == 0 && !last) return;  // uniform: nothing kept
    const int64_t off = block_offset(A, k, blk, sh);
    if (last && t == 0) A.dcount[k] = off + mine;
    if (mine == 0) return;
    if (k == 2 || k == 3) pair_offsets(A, poff, sh);
    const int64_t i = blk * kBlock + t;
    const bool pred = i < nk && A.flag[A.flag0[k] + i] != 0;
    int tot;
    const int64_t r = off + block_rank(pred, shw, &tot);
    if (pred) write_entry(A, poff, k, i, r);
}

// The scenes of the lanes with `kept` counted in list l (EE, PT, VG): one add a wave, or one a
// lane where a wave holds entries of several scenes.
__device__ __forceinline__ void count_scene(const KeepSweep& W, int l, bool kept, int s) {
    const unsigned long long m = __ballot(kept);
    if (W.S == 1 || !m) return;
    const int leader = __ffsll((long long)m) - 1;
    const int s0 = __shfl(s, leader);
    uint32_t* c = W.scnt + (int64_t)l * W.S;
    if (__ballot(kept && s != s0) == 0) {
        if (lane_id() == leader) atomicAdd(c + s0, (uint32_t)__popcll(m));
    } else if (kept) {
        atomicAdd(c + s, 1u);
    }
}

// The write pass of a swept set with its CCD (KeepSweep).  PT / EE entries: kSweepBlocks
// blocks a workgroup, whose kept entries are listed in LDS, so that the lanes are full where a
// third of the superset is kept; each then has its tuple written and, from one gather of its
// eight vertices, its apart_until and cubic taken.  The gathers' latency bounds it (3/4 of the
// wave cycles wait, the address units are busy a third of the time).  1.3 M kept of 4.5 M:
// 119 us, against 46 (write) + 121 (scan of the written lists) + 19 (plan) as passes of their
// own.  What it cost on the way: one counter for the queue and every wave adding to it 40 us
// more (hence one add a workgroup); blocks dealt to the XCDs in turn 11-24 us more (hence
// xcd_block); four waves a SIMD, with 25 registers spilled, 20 us more than three; all in the
// count pass, whose waves then hold the CCD's registers, 55 us more.
__global__ __launch_bounds__(kBlock, 3) void sweep_write_kernel(KeepArgs A) {
    constexpr int kWaves = kBlock / kWave;
    __shared__ int64_t woff[kWaves];
    __shared__ int wcnt[kWaves], wpair[kWaves], qn, qbase;
    __shared__ int64_t poff[kBlock];
    __shared__ uint16_t list[kSweepBlocks * kBlock], qlist[kSweepBlocks * kBlock];
    const int64_t g = blockIdx.x;
    const int t = threadIdx.x;
    const KeepSweep& W = A.W;
    if (g == 0 && t < kKeepLists && A.blk0[t] == A.blk0[t + 1]) A.dcount[t] = 0;  // an empty list
    if (g >= A.grp0[kKeepLists]) return;
    int k = 0;
    while (k + 1 < kKeepLists && g >= A.grp0[k + 1]) ++k;
    const bool tuples = k == 2 || k == 3;
    const int64_t nk = keep_n(A, k), nblk = blocks_of(nk);
    const int64_t ngrp = tuples ? (nblk + kSweepBlocks - 1) / kSweepBlocks : nblk;
    const int64_t grp = xcd_block(g - A.grp0[k], ngrp);
    if (nk == 0 && g == A.grp0[k] && t == 0) A.dcount[k] = 0;
    if (grp < 0) return;  // uniform
    const int64_t blk = tuples ? grp * kSweepBlocks : grp;
    const bool last = grp + 1 == ngrp;
    const int64_t i0 = blk * kBlock;
    // the kept entries before the workgroup's (block_offset's), its own, and the pair
    // blocks' offsets (pair_offsets'), their loads in flight together and one scan for all
    uint32_t word = 0;
    if (tuples) {
        const int64_t i = i0 + kSweepBlocks * t;
        if (i < nk) word = *reinterpret_cast<const uint32_t*>(A.flag + A.flag0[k] + i);
        for (int j = 0; j < kSweepBlocks; ++j)
            if (i + j >= nk || (word >> (8 * j) & 0xff) == 0) word &= ~(0xffu << (8 * j));
    } else if (i0 + t < nk) {
        word = A.flag[A.flag0[k] + i0 + t];
    }
    const int64_t sb = blk / kSuper;
    int64_t before = 0;
    for (int64_t q = t; q < sb; q += kBlock) before += A.scnt[k][kSuperStride * q];
    if (sb * kSuper + t < blk) before += A.bcnt[k][sb * kSuper + t];
    const int pairs = tuples && !A.pair_off && t < blocks_of(keep_n(A, 0)) ? (int)A.bcnt[0][t] : 0;
    int c = 0;
#pragma unroll
    for (int j = 0; j < kSweepBlocks; ++j) c += (word >> (8 * j) & 0xff) != 0;
    int ci = c, pi = pairs;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const int u = __shfl_up(ci, o), v = __shfl_up(pi, o);
        if (lane_id() >= o) {
            ci += u;
            pi += v;
        }
        before += __shfl_xor(before, o);
    }
    if (lane_id() == kWave - 1) {
        woff[wave_id()] = before;
        wcnt[wave_id()] = ci;
        wpair[wave_id()] = pi;
    }
    if (t == 0) qn = 0;
    __syncthreads();
    int64_t off = 0;
    int mine = 0;
    for (int w = 0; w < kWaves; ++w) {
        if (w < wave_id()) {
            ci += wcnt[w];
            pi += wpair[w];
        }
        off += woff[w];
        mine += wcnt[w];
    }
    if (last && t == 0) A.dcount[k] = off + mine;
    if (mine == 0) return;  // uniform: nothing kept
    if (!tuples) {
        const bool pred = c != 0;
        const int64_t i = i0 + t, r = off + ci - c;
        if (pred) write_entry(A, poff, k, i, r);
        if (k < 4) return;  // uniform
        int s = 0;
        if (pred) {
            const int32_t* tu = A.in.vg + 2 * i;
            s = W.S > 1 ? W.body_scene[tu[0]] : 0;
            float apart = 0.0f;
            if (W.body_on[tu[0]]) {
                const int64_t v = A.voff[tu[0]] + (int64_t)tu[1];
                apart = apart_until_vg(A.x[3 * v + 1], A.x1[3 * v + 1], W.ground, W.dhat);
                const double tv = cand_toi_vg(A.voff, A.x, A.x1, tu, W.ground);
                // a TOI below 0 gives the first length that 0 gives
                if (tv < 1.0 && W.use_vg)
                    atomicMin(W.slots + s, (unsigned long long)__double_as_longlong(tv > 0.0 ? tv : 0.0));
            }
            W.avg[r] = apart;
        }
        count_scene(W, 2, pred, s);
        return;
    }
    poff[t] = pi - pairs;
    {
        int r = ci - c;
#pragma unroll
        for (int j = 0; j < kSweepBlocks; ++j)
            if (word >> (8 * j) & 0xff) list[r++] = (uint16_t)(kSweepBlocks * t + j);
    }
    __syncthreads();
    const SceneView V{A.voff, A.foff, A.eoff, A.tris, A.edges, nullptr};
    const int32_t* tuple = k == 2 ? A.in.pt : A.in.ee;
    const int32_t* vids = k == 2 ? A.in.vids.pt : A.in.vids.ee;
    float* out = k == 2 ? W.apt : W.aee;
    const bool use = k == 2 ? W.use_pt : W.use_ee;
    for (int j0 = wave_id() * kWave; j0 < mine; j0 += kBlock) {
        const int j = j0 + lane_id();
        const bool in = j < mine;
        bool queued = false;
        int s = 0;
        if (in) {
            const int64_t i = i0 + list[j], o = off + j;
            const int32_t* tu = tuple + 5 * i;
            s = W.S > 1 ? W.body_scene[tu[0]] : 0;
            write_entry(A, poff, k, i, o);
            float apart = 0.0f;
            if (W.body_on[tu[0]]) {
                d3 a[4], b[4];
                cand_verts(k == 2 ? 0 : 1, V, A.x, A.x1, tu, a, b, vids ? vids + 4 * i : nullptr);
                apart = apart_until(k == 2 ? 0 : 1, a, b, W.dhat);
                queued = use && toi_bracketed(a, b);
            }
            out[o] = apart;
        }
        count_scene(W, k == 3 ? 0 : 1, in, s);
        const unsigned long long mq = __ballot(queued);
        if (mq) {
            const int leader = __ffsll((long long)mq) - 1;
            int32_t base = 0;
            if (lane_id() == leader) base = atomicAdd(&qn, (int)__popcll(mq));
            base = __shfl(base, leader);
            if (queued) qlist[base + __popcll(mq & ((1ull << lane_id()) - 1ull))] = (uint16_t)j;
        }
    }
    __syncthreads();
    if (qn == 0) return;  // uniform
    if (t == 0) qbase = atomicAdd(W.qcount, qn);
    __syncthreads();
    for (int q = t; q < qn; q += kBlock)
        W.queue[qbase + q] = (int32_t)(((off + qlist[q]) << 1) | (k == 3 ? 1 : 0));
}

// The pair blocks' offsets of more than kBlock blocks.
__global__ __launch_bounds__(kScanThreads) void keep_pair_scan_kernel(const uint32_t* __restrict__ cnt, int64_t n,
                                                                      int64_t* __restrict__ off) {
    scan_block_exclusive_by([cnt](int64_t i) { return (int64_t)cnt[i]; }, off, n, nullptr, nullptr);
}

}  // namespace

size_t keep_counters(int64_t nij, int64_t npt, int64_t nee, int64_t nvg) {
    size_t n = 0;
    for (int64_t m : {nij, nij, npt, nee, nvg}) n += (size_t)ceil_div(ceil_div(m, (int64_t)kBlock), kSuper);
    return kSuperStride * n;
}

namespace {
__global__ __launch_bounds__(kBlock) void cand_vid_kernel(SceneView V, int kind, const int32_t* __restrict__ tuples,
                                                          int64_t n, int32_t* __restrict__ vid) {
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        int64_t v[4];
        cand_idx(kind, V, tuples + 5 * i, nullptr, v);
#pragma unroll
        for (int j = 0; j < 4; ++j) vid[4 * i + j] = (int32_t)v[j];
    }
}
}  // namespace

int cand_vertex_ids(hipStream_t s, const AbdScene* sc, int kind, const int32_t* tuples, int64_t n, int32_t* vid) {
    if (n <= 0) return ABD_OK;
    const SceneView V{sc->voff, sc->foff, sc->eoff, sc->tris, sc->edges, sc->x0};
    launch_kernel(cand_vid_kernel, dim3(grid_for(n, kBlock, 1 << 16)), dim3(kBlock), 0, s, V, kind, tuples, n, vid);
    ABD_CHECK_LAUNCH();
    return ABD_OK;
}

int keep_from_superset(hipStream_t s, const AbdScene* sc, const KeepInput& in, const KeepBoxes& bx, double dhat,
                       double ground, const KeepOutput& out, int64_t* dcount, int64_t* hcount, bool sync,
                       const KeepAtX* at, uint32_t* counters, const KeepSweep* sweep) {
    KeepArgs A{};
    A.in = in;
    A.bx = bx;
    A.out = out;
    A.voff = sc->voff;
    A.foff = sc->foff;
    A.eoff = sc->eoff;
    A.x = at ? at->x : nullptr;
    A.x1 = at ? at->x1 : nullptr;
    A.tris = sc->tris;
    A.edges = sc->edges;
    A.pdil = at ? (float)at->pdil : 0.0f;
    A.edil = at ? at->edil : 0.0;
    A.tdil = at ? at->tdil : 0.0;
    A.ebox = at && at->x1 ? at->ebox : nullptr;
    A.alpha = at && in.vids.apart_pt ? at->alpha : nullptr;
    A.body_scene = at ? at->body_scene : nullptr;
    A.yth = 0.5 * dhat + ground;
    A.fg = (float)ground;
    A.dcount = dcount;
    if (sweep) A.W = *sweep;
    const int64_t n[kKeepLists] = {in.nij, in.ji ? in.nij : 0, in.npt, in.nee, in.nvg};
    int64_t nblk[kKeepLists], total = 0, nflag = 0, nsup = 0;
    A.blk0[0] = 0;
    for (int k = 0; k < kKeepLists; ++k) {
        A.flag0[k] = nflag;
        nflag += ceil_div(n[k], (int64_t)kFlagAlign) * kFlagAlign;
        A.n[k] = n[k];
        nblk[k] = ceil_div(n[k], (int64_t)kBlock);
        A.blk0[k + 1] = A.blk0[k] + ceil_div(nblk[k], (int64_t)kXcds) * kXcds;
        total += nblk[k];
        nsup += ceil_div(nblk[k], kSuper);
    }
    if (A.blk0[kKeepLists] >= INT32_MAX) return ABD_ERR_ARG;
    if (sweep && in.npt + in.nee > (int64_t)INT32_MAX / 2) return ABD_ERR_ARG;  // the queue's indices
    // more pair blocks than the write pass sums in LDS: scanned, their offsets beside the counts
    const bool scan = nblk[0] > kBlock;
    uint32_t* buf;
    int rc;
    const size_t own = counters ? 0 : keep_counters(in.nij, in.npt, in.nee, in.nvg);
    const size_t even = ((size_t)total + own + 1) & ~(size_t)1;
    if ((rc = arena_get(kSlotKeep, sizeof(uint32_t) * even + (scan ? sizeof(int64_t) * (size_t)nblk[0] : 0),
                        (void**)&buf)))
        return rc;
    if ((rc = arena_get(kSlotKeepMap, sizeof(int32_t) * ((size_t)in.nij + 1), (void**)&A.remap))) return rc;
    int64_t* pair_off = scan ? reinterpret_cast<int64_t*>(buf + even) : nullptr;
    A.pair_off = pair_off;
    if (!counters) {
        counters = buf;
        buf += own;
        if ((rc = zero_fill(s, counters, sizeof(uint32_t) * own))) return rc;
    }
    for (int k = 0; k < kKeepLists; ++k) {
        A.bcnt[k] = buf;
        buf += nblk[k];
        A.scnt[k] = counters;
        counters += kSuperStride * ceil_div(nblk[k], kSuper);
    }
    // counts of all five lists in one launch (with the kept pairs' ranks in their
    // workgroups), then every list written in one launch, with the totals to dcount
    const int64_t nall = A.blk0[kKeepLists];
    if ((rc = arena_get(kSlotKeepFlags, (size_t)nflag + 1, (void**)&A.flag))) return rc;
    const int ph = prof_start(kProfKeep, s, 0.0);
    if (nall > 0) {
        launch_kernel(keep_count_kernel, dim3((unsigned)nall), dim3(kBlock), 0, s, A);
        ABD_CHECK_LAUNCH();
    }
    if (scan) {
        launch_kernel(keep_pair_scan_kernel, dim3(1), dim3(kScanThreads), 0, s, (const uint32_t*)A.bcnt[0],
                           nblk[0], pair_off);
        ABD_CHECK_LAUNCH();
    }
    prof_stop(ph, s);
    if (sweep) {
        A.grp0[0] = 0;
        for (int k = 0; k < kKeepLists; ++k)
            A.grp0[k + 1] = A.grp0[k] +
                            ceil_div(nblk[k], (int64_t)kXcds * (k == 2 || k == 3 ? kSweepBlocks : 1)) * kXcds;
        // bytes: the CCD's tuple, ids and vertices at both ends of each kept entry, counted on the
        // device (the host knows only the superset's bounds, many times the kept entries)
        const int phw = prof_start(kProfToi, s, 1.0);
        launch_kernel(sweep_write_kernel, dim3((unsigned)std::max<int64_t>(A.grp0[kKeepLists], 1)),
                           dim3(kBlock), 0, s, A);
        ABD_CHECK_LAUNCH();
        prof_stop(phw, s);
        if ((rc = prof_count_bytes(phw, s, dcount, 224.0, 228.0, 56.0, 0.0))) return rc;
    } else {
        const int phw = prof_start(kProfKeep, s, 0.0);
        launch_kernel(keep_write_kernel, dim3((unsigned)std::max<int64_t>(nall, 1)), dim3(kBlock), 0, s, A);
        ABD_CHECK_LAUNCH();
        prof_stop(phw, s);
    }
    if (hcount) {
        ABD_CHECK(hipMemcpyAsync(hcount, dcount, kKeepLists * sizeof(int64_t), hipMemcpyDeviceToHost, s));
        if (sync) ABD_CHECK(hipStreamSynchronize(s));
    }
    return ABD_OK;
}

}  // namespace abd

using namespace abd;

extern "C" int abd_cull_keep(abd_stream_t stream, const AbdScene* sc, const int32_t* ij, const int32_t* ji,
                             int64_t nij, const int32_t* pt, int64_t npt, const int32_t* ee, int64_t nee,
                             const int32_t* vg, int64_t nvg, const float* blo, const float* bhi, const float* plo,
                             const float* phi, const float* elo, const float* ehi, const float* tlo,
                             const float* thi, double dhat, double ground, int32_t* ij_out, int32_t* ji_out,
                             int32_t* pt_out, int32_t* ee_out, int32_t* vg_out, int64_t* counts) {
    if (!sc || !counts || nij < 0 || npt < 0 || nee < 0 || nvg < 0) return ABD_ERR_ARG;
    if ((nij && (!ij || !ij_out || (ji && !ji_out))) || (npt && (!pt || !pt_out)) || (nee && (!ee || !ee_out)) ||
        (nvg && (!vg || !vg_out)))
        return ABD_ERR_ARG;
    if (!blo || !bhi || !plo || !phi || !elo || !ehi || !tlo || !thi) return ABD_ERR_ARG;
    hipStream_t s = to_stream(stream);
    int64_t *dcount, *hcount;
    int rc = arena_get(kSlotKeepCount, 8 * sizeof(int64_t), (void**)&dcount);
    if (!rc) rc = arena_host(8 * sizeof(int64_t), (void**)&hcount);
    if (rc) return rc;
    const KeepInput in{ij, ji, pt, ee, vg, nij, npt, nee, nvg};
    const KeepBoxes bx{blo, bhi, plo, phi, elo, ehi, tlo, thi};
    const KeepOutput out{ij_out, ji_out, pt_out, ee_out, vg_out};
    if ((rc = keep_from_superset(s, sc, in, bx, dhat, ground, out, dcount, hcount))) return rc;
    for (int k = 0; k < 5; ++k) counts[k] = hcount[k];
    return ABD_OK;
}

