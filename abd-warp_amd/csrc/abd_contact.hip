// abd_contact.hip — barrier energy, gradient and PSD-projected Hessian of the
// point-triangle (PT), edge-edge (EE) and vertex-ground (VG) contacts, and the
// inertia / orthogonality terms (ipc.py, ipcsk/, psd/, orthogonal_energy.py).
//
// Hessian structure.  For one contact the reference forms (ipcsk/pt_ipc.py:111-185)
//   Hl  = sum_k L_k q_k q_k^T / |q_k|^2          (9x9, psd/hl.py:156-195; L_4 = 2)
//   H12 = D~^T Hl D~,  g12 = D~^T q_4           (D~ = dcdx (x) I3, 9x12)
//   Hipc = b' H12 + b'' g12 g12^T,   Hi/Hj/Hij = J^T Hipc J   (J = [1, x0^T] (x) I3)
// which is a sum of five rank-one terms in body space: with V_k = J^T D~^T q_k
// (24 entries: 12 per body),
//   H24 = sum_{k<4} (b' L_k/|q_k|^2) V_k V_k^T + (b' L_4/|q_4|^2 + b'') V_4 V_4^T,
//   g24 = b' V_4.
// A contact is therefore stored as 5 coefficients + 5 x 24 vectors, and the
// body-pair blocks are reduced from those in a fixed order (no atomics):
//   stage A  classify every candidate (active = s < d2hat and valid)      [HBM stream]
//   stage B  ordered compaction of the active candidates
//   stage C  per active contact: coefficients and V_k (one thread each)
//   stage D  per body pair: sum of its contacts' 24x24 terms; the off-diagonal
//            12x12 goes straight into the pair's two slots
//   stage E  per body: diagonal slot and gradient += its pairs' diagonal parts
//            + its vertex-ground terms.
#include <hip/hip_runtime.h>

#include <cstring>

#include "abd_block.h"
#include "abd_dense.h"
#include "abd_device.h"
#include "abd_inertia.h"
#include "abd_internal.h"
#include "abd_profile.h"

namespace abd {

constexpr int kSuperBlocks = 64;   // blocks (kBlock candidates) per super-block of active counts
constexpr int kSuperStride = 8;    // words between those: adds to one cache line wait for each other
constexpr int kGhBoundMib = 8192;  // stored contacts sized by a list bound, at most (default)
constexpr int kContactStride = 128;  // doubles per stored contact: c[0..4], b', pad, then V[5][24]
constexpr int kCoefOff = 0;
constexpr int kB1Off = 5;
constexpr int kVOff = 8;

__device__ __forceinline__ SceneView view_of(const AbdScene& sc) {
    SceneView v;
    v.voff = sc.voff;
    v.foff = sc.foff;
    v.eoff = sc.eoff;
    v.tris = sc.tris;
    v.edges = sc.edges;
    v.x0 = sc.x0;
    return v;
}

__device__ __forceinline__ void load4(const double* __restrict__ x, const int64_t v[4], d3 out[4]) {
#pragma unroll
    for (int k = 0; k < 4; ++k) out[k] = ld3(x + 3 * v[k]);
}


// ------------------------------------------------------------ contact terms
// One contact: writes coefficients and V_k into out[kContactStride]; returns
// active.  kind 0 PT (x0 point; x1..x3 triangle), 1 EE (x0x1, x2x3).
__device__ bool contact_terms(int kind, const d3 v[4], const d3 r[4], double d2hat, double kappa, int psd,
                              double* __restrict__ out) {
    CMap c = kind == 0 ? cmap_pt(v[0], v[1], v[2], v[3]) : cmap_ee(v[0], v[1], v[2], v[3]);
    bool valid = kind == 0 ? valid_pt(c.beta, c.gamma) : valid_ee(c.beta, c.gamma);
    double l = signed_distance(c.e0, c.e1p, c.e2p);
    // _mask_valid: PT gh uses l^2 (pt_ipc.py:20-22), EE gh |e2p|^2 (ee_ipc.py:23)
    double s = kind == 0 ? l * l : dot(c.e2p, c.e2p);
    if (!(s < d2hat && valid)) return false;
    double b1 = barrier_d1(s, d2hat, kappa);
    double b2 = barrier_d2(s, d2hat, kappa);
    // psd/hl.py:156-195 eigensystem of d2(l^2)/dc2
    double e0pn = dot(c.e0, c.e0), e1pn = dot(c.e1p, c.e1p), e2pn = dot(c.e2p, c.e2p);
    double f12 = sqrt(1.0 + 4.0 * (e1pn / e2pn));
    double f02 = sqrt(1.0 + 4.0 * (e0pn / e2pn));
    double lam[4];
    lam[0] = -l / (2.0 * e1pn) * (1.0 + f12);
    lam[1] = -l / (2.0 * e1pn) * (1.0 - f12);
    lam[2] = -l / (2.0 * e0pn) * (1.0 + f02);
    lam[3] = -l / (2.0 * e0pn) * (1.0 - f02);
    const double lt = l / e2pn;
    // dcdx (psd/vf.py:44-72, psd/ee.py:135-163), row-major 3x4
    double D[12];
    if (kind == 0) {
        D[0] = 0.0; D[1] = 1.0; D[2] = -1.0; D[3] = 0.0;
        D[4] = 0.0; D[5] = -c.alpha; D[6] = c.alpha - 1.0; D[7] = 1.0;
        D[8] = 1.0; D[9] = -c.beta; D[10] = c.beta + c.gamma - 1.0; D[11] = -c.gamma;
    } else {
        D[0] = -1.0; D[1] = 1.0; D[2] = 0.0; D[3] = 0.0;
        D[4] = c.alpha; D[5] = -c.alpha; D[6] = -1.0; D[7] = 1.0;
        D[8] = c.beta - 1.0; D[9] = -c.beta; D[10] = c.gamma + 1.0; D[11] = -c.gamma;
    }
    const int nI = kind == 0 ? 1 : 2;  // contact vertices on body I
    const d3 gl2 = (c.e2p * l) / e2pn;  // psd/hl.py:37-39
    const d3 q4 = (gl2 * 2.0) * l;
    for (int k = 0; k < 5; ++k) {
        d3 qb[3];
        double L;
        if (k < 4) {
            double om = lam[k] / (lam[k] - lt);
            L = lam[k] * 2.0 * l;
            // pt_ipc.py:266-269 (EE unclamped, ee_ipc.py:33-36); the psd mode projects the
            // whole contact-space Hessian below and starts from the unclamped eigenvalue
            if (kind == 0 && !psd) L = L > 0.0 ? L : 0.0;
            if (k < 2) {
                qb[0] = mk(0.0, 0.0, 0.0);
                qb[1] = c.e2p;
                qb[2] = c.e1p * om;
            } else {
                qb[0] = c.e2p;
                qb[1] = mk(0.0, 0.0, 0.0);
                qb[2] = c.e0 * om;
            }
        } else {
            L = 2.0;
            qb[0] = mk(0.0, 0.0, 0.0);
            qb[1] = mk(0.0, 0.0, 0.0);
            qb[2] = q4;
        }
        double qn = dot(qb[0], qb[0]) + dot(qb[1], qb[1]) + dot(qb[2], qb[2]);
        if (psd) {
            // contact-space eigenvalue of b' Hl + b'' q4 q4^T, clamped at zero
            double mu = k < 4 ? b1 * L : b1 * L + b2 * qn;
            out[kCoefOff + k] = (mu > 0.0 ? mu : 0.0) * (1.0 / qn);
        } else {
            double w = L * (1.0 / qn);
            out[kCoefOff + k] = k < 4 ? b1 * w : b1 * w + b2;
        }
        // u = D~^T q (12, per contact vertex), then V = J^T u per body
        double V[24];
#pragma unroll
        for (int i = 0; i < 24; ++i) V[i] = 0.0;
#pragma unroll
        for (int vtx = 0; vtx < 4; ++vtx) {
            d3 u = (qb[0] * D[0 * 4 + vtx] + qb[1] * D[1 * 4 + vtx]) + qb[2] * D[2 * 4 + vtx];
            const double Jr[4] = {1.0, r[vtx].x, r[vtx].y, r[vtx].z};
            const int base = vtx < nI ? 0 : 12;
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                V[base + 3 * a + 0] += Jr[a] * u.x;
                V[base + 3 * a + 1] += Jr[a] * u.y;
                V[base + 3 * a + 2] += Jr[a] * u.z;
            }
        }
#pragma unroll
        for (int i = 0; i < 24; ++i) out[kVOff + 24 * k + i] = V[i];
    }
    out[kB1Off] = b1;
    return true;
}

// stage A: active flags over [PT | EE] and their counts per block of kBlock candidates (bcnt)
// and per super-block (scnt, 0 before), plus ordering checks.
// dn (nullable): the list sizes on the device, [nij, nij, npt, nee, nvg] (the arguments are
// then upper bounds that only size the launch)
__global__ __launch_bounds__(kBlock) void classify_kernel(AbdScene sc, AbdParams P, const double* __restrict__ x,
                                                           const int32_t* __restrict__ pt, int64_t npt,
                                                           const int32_t* __restrict__ ee, int64_t nee,
                                                           const int32_t* __restrict__ vg, int64_t nvg,
                                                           const int64_t* __restrict__ dn,
                                                           uint8_t* __restrict__ flag, int* __restrict__ err,
                                                           uint32_t* __restrict__ bcnt,
                                                           uint32_t* __restrict__ scnt) {
    const SceneView S = view_of(sc);
    if (dn) {
        npt = dn[2];
        nee = dn[3];
        nvg = dn[4];
    }
    const int64_t n = npt + nee, nblk = (n + kBlock - 1) / kBlock, nvblk = (nvg + kBlock - 1) / kBlock;
    for (int64_t blk = blockIdx.x; blk < nblk + nvblk; blk += gridDim.x) {  // uniform over the workgroup
        if (blk >= nblk) {
            const int64_t k = (blk - nblk) * kBlock + threadIdx.x;
            if (k > 0 && k < nvg && vg[2 * k] < vg[2 * (k - 1)]) *err = 1;
            continue;
        }
        bool act = false;
        const int64_t i = blk * kBlock + threadIdx.x;
        if (i < n) {
        const bool is_ee = i >= npt;
        const int64_t k = is_ee ? i - npt : i;
        const int32_t* t5 = (is_ee ? ee : pt) + 5 * k;
        if (k > 0 && t5[2] < t5[2 - 5]) *err = 1;
        int64_t vi[4];
        d3 v[4];
        if (is_ee)
            fetch_ee_idx(S, t5, vi);
        else
            fetch_pt_idx(S, t5, vi);
        load4(x, vi, v);
        if (P.psd == 3) {  // full IPC: the closest feature pair, no validity gate
            const Feat f = is_ee ? ee_feature(v) : pt_feature(v);
            act = (is_ee ? P.ee : P.pt) && feature_dist2_value(is_ee ? 1 : 0, f, v) < P.d2hat;
        } else if (is_ee) {
            CMap c = cmap_ee(v[0], v[1], v[2], v[3]);
            act = P.ee && dot(c.e2p, c.e2p) < P.d2hat && valid_ee(c.beta, c.gamma);
        } else {
            CMap c = cmap_pt(v[0], v[1], v[2], v[3]);
            double l = signed_distance(c.e0, c.e1p, c.e2p);
            act = P.pt && l * l < P.d2hat && valid_pt(c.beta, c.gamma);
        }
        flag[i] = act ? 1 : 0;
        }
        const int c = __syncthreads_count(act);
        if (threadIdx.x == 0) {
            bcnt[blk] = (uint32_t)c;
            if (c) atomicAdd(scnt + kSuperStride * (blk / kSuperBlocks), (uint32_t)c);
        }
    }
}

// The active candidates before block blk (its workgroup's threads together; sh: one per wave).
__device__ __forceinline__ int64_t active_before(const uint32_t* __restrict__ bcnt, const uint32_t* __restrict__ scnt,
                                                 int64_t blk, int64_t* sh) {
    const int64_t sb = blk / kSuperBlocks, b = sb * kSuperBlocks + threadIdx.x;
    int64_t v = b < blk ? (int64_t)bcnt[b] : 0;
    for (int64_t q = threadIdx.x; q < sb; q += kBlock) v += scnt[kSuperStride * q];
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if (lane_id() == 0) sh[wave_id()] = v;
    __syncthreads();
    v = 0;
    for (int w = 0; w < kBlock / kWave; ++w) v += sh[w];
    return v;
}

// The active count (one workgroup), where it is wanted before stage C's sizes.
__global__ __launch_bounds__(kBlock) void active_total_kernel(const uint32_t* __restrict__ scnt, int64_t nsup,
                                                              int64_t* __restrict__ total) {
    __shared__ int64_t sh[kBlock / kWave];
    const int64_t v = active_before(nullptr, scnt, nsup * kSuperBlocks, sh);
    if (threadIdx.x == 0) *total = v;
}

// A block's share of stages B and C: its active candidates in order (their places in the block
// listed in LDS) and the index of the first among all; the last block writes the total.
// Returns their number; uniform over the workgroup, whose threads meet before the next block.
struct ActiveArgs {
    const uint8_t* flag;
    int64_t n;            // PT + EE candidates (dn, nullable: counted on the device)
    const int64_t* dn;
    const uint32_t *bcnt, *scnt;
    int64_t *total, *total2;  // total2 nullable
};
__device__ __forceinline__ int64_t active_blocks(const ActiveArgs& A, int64_t& n) {
    n = A.dn ? A.dn[2] + A.dn[3] : A.n;
    if (n == 0 && blockIdx.x == 0 && threadIdx.x == 0) {
        *A.total = 0;
        if (A.total2) *A.total2 = 0;
    }
    return (n + kBlock - 1) / kBlock;
}
__device__ __forceinline__ int active_block(const ActiveArgs& A, int64_t n, int64_t blk, int64_t nblk, uint8_t* list,
                                            int64_t& first) {
    __shared__ int64_t sh[kBlock / kWave];
    __shared__ int shw[kBlock / kWave];
    const int c = (int)A.bcnt[blk];
    if (c == 0 && blk + 1 < nblk) return 0;
    __syncthreads();  // the last block's list is read
    first = active_before(A.bcnt, A.scnt, blk, sh);
    if (blk + 1 == nblk && threadIdx.x == 0) {
        *A.total = first + c;
        if (A.total2) *A.total2 = first + c;
    }
    const int64_t i = blk * kBlock + threadIdx.x;
    const bool pred = i < n && A.flag[i];
    int tot;
    const int r = block_rank(pred, shw, &tot);
    if (pred) list[r] = (uint8_t)threadIdx.x;
    __syncthreads();
    return c;
}
// workgroups of the kernels over those blocks, at most
constexpr int64_t kActiveGrid = 4096;

// stage B on its own (the dense modes): the active candidates in order.
__global__ __launch_bounds__(kBlock) void compact_flags_kernel(ActiveArgs A, int32_t* __restrict__ out) {
    __shared__ uint8_t list[kBlock];
    int64_t n;
    const int64_t nblk = active_blocks(A, n);
    for (int64_t blk = blockIdx.x; blk < nblk; blk += gridDim.x) {
        int64_t first;
        const int c = active_block(A, n, blk, nblk, list, first);
        if (threadIdx.x < c) out[first + threadIdx.x] = (int32_t)(blk * kBlock + list[threadIdx.x]);
    }
}

// sort key of candidate i of [PT | EE]: (type << 32) | body pair
__device__ __forceinline__ int64_t active_key(const int32_t* __restrict__ pt, int64_t npt,
                                              const int32_t* __restrict__ ee, int64_t i) {
    const bool is_ee = i >= npt;
    const int32_t* t5 = is_ee ? ee + 5 * (i - npt) : pt + 5 * i;
    return ((int64_t)(is_ee ? 1 : 0) << 32) | (int64_t)t5[2];
}

// A run of contacts [begin, end) as stored in pseg: (kRunBase - begin, end), each the largest of
// its writers' (0, 0: empty), so the contacts of a run need not meet in one workgroup.
constexpr unsigned long long kRunBase = 1ull << 40;
__device__ __forceinline__ void read_run(const unsigned long long* __restrict__ ps, int64_t& begin, int64_t& end) {
    begin = ps[0] ? (int64_t)(kRunBase - ps[0]) : 0;
    end = (int64_t)ps[1];
}

// Where stage C leaves what stage D needs of the active contacts, beside their terms.
struct ContactOut {
    double* __restrict__ cbuf;
    uint8_t* __restrict__ swap;
    uint8_t* __restrict__ hl_pt;
    uint8_t* __restrict__ hl_ee;
    uint8_t* __restrict__ pflag;
    int64_t nij;
    unsigned long long* __restrict__ pseg;
};

// The pair's flags and run of active contact e, tuple t5, key; kprev, knext: the keys of its
// neighbours in the sorted active list (-1: none known; the contact then also offers its ends).
__device__ __forceinline__ void contact_bookkeeping(const ContactOut& O, int64_t e, int64_t key, int64_t kprev,
                                                    int64_t knext, const int32_t* __restrict__ t5) {
    const bool is_ee = (key >> 32) != 0;
    O.pflag[t5[2]] = 1;  // the body pair has an active contact (every writer stores 1)
    unsigned long long* ps = O.pseg + 2 * ((is_ee ? O.nij : 0) + t5[2]);
    if (kprev != key) atomicMax(ps, kRunBase - (unsigned long long)e);
    if (knext != key) atomicMax(ps + 1, (unsigned long long)(e + 1));
    O.swap[e] = t5[0] > t5[1] ? 1 : 0;  // body I is ij1 (PT second order)
    if (is_ee)
        O.hl_ee[t5[1]] = 1;
    else
        O.hl_pt[t5[1]] = 1;
}

// stages B and C: the active contacts of a block of kBlock candidates, one thread each (the
// contact-space terms, psd 0 and 1).  As a compaction and a kernel over its list these were
// two launches, with the scan between them three (4.6 + 8.1 + 16.4 us at 87 k candidates, 2 k
// active; 12.7 us here).
__global__ __launch_bounds__(kBlock) void contact_kernel(AbdScene sc, AbdParams P, const double* __restrict__ x,
                                                          const int32_t* __restrict__ pt, int64_t npt,
                                                          const int32_t* __restrict__ ee, ActiveArgs A,
                                                          ContactOut O) {
    __shared__ uint8_t list[kBlock];
    __shared__ int64_t keys[kBlock];
    const SceneView S = view_of(sc);
    int64_t n;
    const int64_t nblk = active_blocks(A, n);
    if (A.dn) npt = A.dn[2];
    const int t = threadIdx.x;
    for (int64_t blk = blockIdx.x; blk < nblk; blk += gridDim.x) {
        int64_t first;
        const int c = active_block(A, n, blk, nblk, list, first);
        if (c == 0) continue;  // uniform
        const int64_t i = blk * kBlock + (t < c ? list[t] : 0);
        if (t < c) keys[t] = active_key(pt, npt, ee, i);
        __syncthreads();
        if (t < c) {
            const int64_t e = first + t;
            const bool is_ee = i >= npt;
            const int32_t* t5 = is_ee ? ee + 5 * (i - npt) : pt + 5 * i;
            int64_t vi[4];
            if (is_ee)
                fetch_ee_idx(S, t5, vi);
            else
                fetch_pt_idx(S, t5, vi);
            d3 v[4], r[4];
            load4(x, vi, v);
            load4(sc.x0, vi, r);
            contact_terms(is_ee ? 1 : 0, v, r, P.d2hat, P.kappa, P.psd, O.cbuf + e * kContactStride);
            contact_bookkeeping(O, e, keys[t], t > 0 ? keys[t - 1] : -1, t + 1 < c ? keys[t + 1] : -1, t5);
        }
    }
}

// stage C of the dense modes (MODE 2 the exact Hessian, 3 full IPC): one wave per active
// contact (grid-stride), see abd_dense.h.
template <int MODE>
__global__ __launch_bounds__(kWave) void contact_dense_kernel(AbdScene sc, AbdParams P, const double* __restrict__ x,
                                                              const int32_t* __restrict__ pt, int64_t npt,
                                                              const int32_t* __restrict__ ee,
                                                              const int32_t* __restrict__ act, int64_t nact,
                                                              const int64_t* __restrict__ dnact,
                                                              const int64_t* __restrict__ dn, ContactOut O) {
    __shared__ DenseLds D;
    const SceneView S = view_of(sc);
    if (dnact) nact = *dnact;
    if (dn) npt = dn[2];
    const int lane = threadIdx.x;
    for (int64_t e = blockIdx.x; e < nact; e += gridDim.x) {  // uniform over the wave
        const int64_t i = act[e];
        const bool is_ee = i >= npt;
        const int32_t* t5 = is_ee ? ee + 5 * (i - npt) : pt + 5 * i;
        int64_t vi[4];
        if (is_ee)
            fetch_ee_idx(S, t5, vi);
        else
            fetch_pt_idx(S, t5, vi);
        d3 v[4], r[4];
        load4(x, vi, v);
        load4(sc.x0, vi, r);
        if (MODE == 3)
            wave_contact_full(lane, is_ee ? 1 : 0, v, r, P.d2hat, P.kappa, D, O.cbuf + e * kDenseStride);
        else
            wave_contact_exact(lane, is_ee ? 1 : 0, v, r, P.d2hat, P.kappa, D, O.cbuf + e * kDenseStride);
        if (lane == 0)
            contact_bookkeeping(O, e, active_key(pt, npt, ee, i), e > 0 ? active_key(pt, npt, ee, act[e - 1]) : -1,
                                e + 1 < nact ? active_key(pt, npt, ee, act[e + 1]) : -1, t5);
    }
}

// workgroups of the dense modes' stage C, at most: one wave each, 16 a CU, as many as the exact
// mode's registers let a CU hold (127 of them: four waves a SIMD; full IPC's 162: three).  Each
// takes 4 KB of the CU's LDS.
constexpr int64_t kDenseGrid = 4096;

constexpr int kPairThreads = 576;  // one thread per entry of the 24x24 body-pair block
constexpr int64_t kPairGrid = 2048;           // workgroups of stage D (grid-stride over pairs)

constexpr int kPairChunk = 64;  // contacts of one stage-D work item
constexpr int kPartStride = 600;  // one chunk's partial sums: the 24x24 block, then g (24)

// stage D1: the work items of each body pair: its PT run and its EE run cut into chunks of
// kPairChunk contacts (runs from stage C).  Pair ii owns the items [pitem[ii].x, + pitem[ii].y),
// taken from a counter in any order (where a pair's items lie changes no result), its PT run's
// chunks then its EE run's; item i's descriptor idesc is its first contact | its contact count
// << 56.  The order the rank-one partial sums run them in takes the full chunks first (odesc /
// oitem from the front, counters[0] of them) and the others after them (from cap on,
// counters[1]): the longest sums start first.  counters[2]: all items.  A workgroup takes kBlock
// pairs and one add per counter (adds to one cache line wait for each other: with three a pair
// this took 28 us for 700 pairs with contacts; 5 us here), then its threads stride over the items.
constexpr int kItemShift = 56;
struct PairItems {
    int2* pitem;
    int64_t *idesc, *odesc, *oitem;
    int64_t cap;
    int* counters;
};
__global__ __launch_bounds__(kBlock) void pair_items_kernel(int64_t nij, const int64_t* __restrict__ dn,
                                                            const uint8_t* __restrict__ pflag,
                                                            const unsigned long long* __restrict__ pseg,
                                                            int64_t nij_cap, PairItems I) {
    if (dn) nij = dn[0];
    __shared__ int64_t sh[kBlock / kWave];
    __shared__ int64_t run[kBlock][4];   // PT and EE runs of the workgroup's pairs
    __shared__ int ifirst[kBlock], ffirst[kBlock], pfirst[kBlock];  // first item, full and other chunk
    __shared__ int base[3], nitems;
    const int t = threadIdx.x;
    constexpr int kPartialShift = 40;
    for (int64_t ii0 = (int64_t)blockIdx.x * kBlock; ii0 < nij; ii0 += (int64_t)gridDim.x * kBlock) {
        const int64_t ii = ii0 + t;
        int64_t p0 = 0, p1 = 0, e0 = 0, e1 = 0;
        if (ii < nij && pflag[ii]) {
            read_run(pseg + 2 * ii, p0, p1);
            read_run(pseg + 2 * (nij_cap + ii), e0, e1);
        }
        const int64_t full = (p1 - p0) / kPairChunk + (e1 - e0) / kPairChunk;
        const int64_t partial = ((p1 - p0) % kPairChunk != 0) + ((e1 - e0) % kPairChunk != 0);
        const int64_t mine = full | partial << kPartialShift;
        const int64_t before = block_exclusive_scan_i64(mine, sh);
        const int nf = (int)(before & ((int64_t(1) << kPartialShift) - 1)), np = (int)(before >> kPartialShift);
        run[t][0] = p0;
        run[t][1] = p1;
        run[t][2] = e0;
        run[t][3] = e1;
        ifirst[t] = nf + np;
        ffirst[t] = nf;
        pfirst[t] = np;
        if (t == kBlock - 1) {
            const int tf = nf + (int)full, tp = np + (int)partial;
            nitems = tf + tp;
            if (tf) base[0] = atomicAdd(I.counters, tf);
            if (tp) base[1] = atomicAdd(I.counters + 1, tp);
            if (tf + tp) base[2] = atomicAdd(I.counters + 2, tf + tp);
        }
        __syncthreads();
        if (full + partial) I.pitem[ii] = make_int2(base[2] + ifirst[t], (int)(full + partial));
        for (int q = t; q < nitems; q += kBlock) {
            int lo = 0, hi = kBlock - 1;  // the pair: the last whose first item is <= q
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (ifirst[mid] <= q)
                    lo = mid;
                else
                    hi = mid - 1;
            }
            const int64_t a0 = run[lo][0], a1 = run[lo][1], b0 = run[lo][2], b1 = run[lo][3];
            const int64_t npc = (a1 - a0 + kPairChunk - 1) / kPairChunk, c = q - ifirst[lo];
            const bool pt = c < npc;
            const int64_t c0 = pt ? a0 + c * kPairChunk : b0 + (c - npc) * kPairChunk;
            const int64_t end = pt ? a1 : b1;
            const int64_t nc = end - c0 < kPairChunk ? end - c0 : kPairChunk;
            const int64_t d = c0 | (nc << kItemShift);
            I.idesc[base[2] + q] = d;
            // PT's full chunks come first among the pair's, its partial one (if any) too
            const bool whole = nc == kPairChunk, pt_rest = (a1 - a0) % kPairChunk != 0;
            const int64_t slot = whole ? base[0] + ffirst[lo] + c - (!pt && pt_rest ? 1 : 0)
                                       : I.cap + base[1] + pfirst[lo] + (!pt && pt_rest ? 1 : 0);
            I.odesc[slot] = d;
            I.oitem[slot] = base[2] + q;
        }
        __syncthreads();  // the tables are free for the next pairs
    }
}

// stage D2: one work item per workgroup (grid-stride over the *total items): the sums, in
// contact order, of one chunk's contacts into part[item] (24x24 block in the pair's body
// order [ij0 | ij1], then g), for contacts stored whole by contact_dense_kernel.
__global__ __launch_bounds__(kPairThreads) void pair_partial_dense_kernel(const double* __restrict__ cbuf,
                                                                           const uint8_t* __restrict__ swap,
                                                                           PairItems I, double* __restrict__ part) {
    constexpr int kStride = kDenseStride;
    constexpr int kBatch = 4;
    __shared__ double sc[kBatch][kStride];
    __shared__ uint8_t ssw[kBatch];
    const int t = threadIdx.x;
    const int R = t / 24, C = t % 24;
    const int64_t nitem = I.counters[2];
    for (int64_t gc = blockIdx.x; gc < nitem; gc += gridDim.x) {
        const int64_t d = I.idesc[gc];
        const int64_t c0 = d & ((int64_t(1) << kItemShift) - 1);
        const int64_t c1 = c0 + (d >> kItemShift);
        double h = 0.0, gacc = 0.0;
        for (int64_t e0 = c0; e0 < c1; e0 += kBatch) {
            const int nbat = (int)((c1 - e0) < kBatch ? (c1 - e0) : kBatch);
            for (int q = t; q < nbat * kStride; q += kPairThreads)
                sc[q / kStride][q % kStride] = cbuf[(e0 + q / kStride) * kStride + q % kStride];
            if (t < nbat) ssw[t] = swap[e0 + t];
            __syncthreads();
            for (int bq = 0; bq < nbat; ++bq) {
                // body order [ij0 | ij1]: swap halves when body I is ij1
                const int sw = ssw[bq] ? 12 : 0;
                const int r = (R + sw) % 24, cc = (C + sw) % 24;
                h += sc[bq][24 * r + cc];
                if (t < 24) gacc += sc[bq][kDenseGOff + (t + sw) % 24];
            }
            __syncthreads();
        }
        double* pp = part + gc * kPartStride;
        pp[t] = h;
        if (t < 24) pp[576 + t] = gacc;
    }
}

// stage D2 for rank-one contacts (the stored form of contact_terms): the items of a
// workgroup (grid-stride) cut into batches of kRankBatch contacts, each staged into LDS
// (without the pad) from registers loaded while the previous batch was summed; one thread
// per entry of the upper triangle of the 24x24 block sums c_k (V_k[r] V_k[c]) over the
// item's contacts in order, and threads 0..23 the gradient; an entry of the lower triangle
// is the same sum (V_k[r] V_k[c] == V_k[c] V_k[r]), written from its mirror.
constexpr int kRankThreads = 320;                   // 300 upper-triangle entries, 5 waves
constexpr int kRankBatch = 32;                      // contacts staged at a time
constexpr int kStaged = 126;                        // doubles per staged contact: c[5], b', V[5][24]
constexpr int kRankPieces = (kRankBatch * 63 + kRankThreads - 1) / kRankThreads;  // 16-byte loads a thread
static_assert(kContactStride == 128 && kCoefOff == 0 && kB1Off == 5 && kVOff == 8, "staged layout");
static_assert(kPairChunk <= kWave, "one swap bit a lane");
typedef double dbl2 __attribute__((ext_vector_type(2)));  // a 16-byte piece (kept in registers)
// read-only data reached through the constant address space: uniform loads become scalar ones
typedef __attribute__((address_space(4))) const double kconst_double;

// A thread's pieces of the batch of n contacts from src (63 pieces of 16 bytes a contact:
// c[0..5] in pieces 0-2, V from piece 4 of the stored row), piece U onwards.  A thread past
// the batch reloads its last piece (stored to a spare slot), so the loads are unconditional
// and issue together; the recursion keeps every index a constant (the pieces in registers).
template <int U>
__device__ __forceinline__ void rank_batch_load(const dbl2* __restrict__ src, int np, int t,
                                                dbl2 (&piece)[kRankPieces]) {
    if constexpr (U < kRankPieces) {
        const int q = min(t + U * kRankThreads, np - 1), e = q / 63, pc = q - 63 * e;
        piece[U] = src[e * (kContactStride / 2) + pc + (pc >= 3 ? 1 : 0)];
        rank_batch_load<U + 1>(src, np, t, piece);
    }
}
// The pieces into the staged batch (the pieces past it into the spare slot).
template <int U>
__device__ __forceinline__ void rank_batch_store(dbl2* dst, int np, int t, const dbl2 (&piece)[kRankPieces]) {
    if constexpr (U < kRankPieces) {
        const int q = t + U * kRankThreads, e = q / 63, pc = q - 63 * e;
        dst[q < np ? e * (kStaged / 2) + pc : kRankBatch * kStaged / 2] = piece[U];
        rank_batch_store<U + 1>(dst, np, t, piece);
    }
}

__global__ __launch_bounds__(kRankThreads, 5) void pair_partial_rank_kernel(const double* __restrict__ cbuf,
                                                                         const uint8_t* __restrict__ swap,
                                                                         PairItems I, double* __restrict__ part) {
    // the staged batch, then a 16-byte slot the pieces past the batch are stored to
    __shared__ __align__(16) double st[kRankBatch * kStaged + 2];
    const int t = threadIdx.x, lane = t % kWave;
    // this thread's entry (r, c), r <= c, of the upper triangle (rows of 24 - r entries)
    int r = 0, j = t;
    while (r < 24 && j >= 24 - r) {
        j -= 24 - r;
        ++r;
    }
    const bool ent = r < 24;
    const int c = ent ? r + j : 0;
    if (!ent) r = 0;
    // V indices in the stored order, without and with the halves swapped (body I is ij1)
    const int tg = t % 24;
    const int rA = r, rB = (r + 12) % 24, cA = c, cB = (c + 12) % 24, gA = tg, gB = (tg + 12) % 24;
    const int64_t nfull = I.counters[0], nitem = nfull + I.counters[1];
    const int64_t gap = I.cap - nfull;  // execution slots past the full chunks are stored from cap on
    int64_t gc = blockIdx.x;  // the execution slot
    if (gc >= nitem) return;  // uniform
    const int64_t kMask = (int64_t(1) << kItemShift) - 1;
    const int64_t d0 = I.odesc[gc < nfull ? gc : gc + gap];
    int64_t c0 = d0 & kMask;
    int nc = (int)(d0 >> kItemShift), b0 = 0;
    dbl2 piece[kRankPieces];
    rank_batch_load<0>(reinterpret_cast<const dbl2*>(cbuf + c0 * kContactStride), 63 * min(nc, kRankBatch), t,
                       piece);
    // the item's swap flags, one bit a contact, in every wave
    uint64_t swm = __ballot(lane < nc && swap[c0 + lane] != 0);
    double h = 0.0, gacc = 0.0;
    for (;;) {
        const int nbat = min(kRankBatch, nc - b0);
        __syncthreads();  // the previous batch is summed: its LDS is free
        rank_batch_store<0>(reinterpret_cast<dbl2*>(st), 63 * nbat, t, piece);
        __syncthreads();
        // the next batch: the rest of this item, else the workgroup's next item; its loads
        // are in flight while this batch is summed
        int64_t gn = gc, cn = c0;
        int nn = nc, bn = b0 + kRankBatch;
        if (bn >= nc) {
            gn = gc + gridDim.x;
            bn = 0;
            if (gn < nitem) {
                const int64_t dn_ = I.odesc[gn < nfull ? gn : gn + gap];
                cn = dn_ & kMask;
                nn = (int)(dn_ >> kItemShift);
            }
        }
        // (past the workgroup's last item this batch is loaded again, unused: the loads stay
        // unconditional and the pieces in registers)
        const bool more = gn < nitem;
        rank_batch_load<0>(reinterpret_cast<const dbl2*>(cbuf + (more ? cn + bn : c0 + b0) * kContactStride),
                           63 * (more ? min(nn - bn, kRankBatch) : nbat), t, piece);
        const uint8_t swn = more && gn != gc && lane < nn ? swap[cn + lane] : 0;
        // every thread also runs the gradient chain of entry t % 24 (kept by threads 0..23),
        // so the loop has no branch and the loads of unrolled contacts issue together
#pragma unroll 4
        for (int e = 0; e < nbat; ++e) {
            const double* S = st + e * kStaged;
            // the coefficients are the same for every lane: scalar loads from the stored row
            const kconst_double* K = (const kconst_double*)cbuf + (c0 + b0 + e) * kContactStride;
            // body order [ij0 | ij1]: halves swapped when body I is ij1
            const bool sw = (swm >> (b0 + e)) & 1;
            const double* Vr = S + 6 + (sw ? rB : rA);
            const double* Vc = S + 6 + (sw ? cB : cA);
#pragma unroll
            for (int k = 0; k < 5; ++k) h += K[k] * (Vr[24 * k] * Vc[24 * k]);
            gacc += K[5] * S[6 + 96 + (sw ? gB : gA)];
        }
        if (gn != gc) {  // uniform: the item is summed
            double* pp = part + I.oitem[gc < nfull ? gc : gc + gap] * kPartStride;
            if (ent) {
                pp[24 * r + c] = h;
                pp[24 * c + r] = h;
            }
            if (t < 24) pp[576 + t] = gacc;
            h = gacc = 0.0;
            if (gn >= nitem) break;
            swm = __ballot(swn != 0);
        }
        gc = gn;
        c0 = cn;
        nc = nn;
        b0 = bn;
    }
}

// The first vertex-ground candidate of body b and of body b + 1 in a list grouped by body
// ascending, found by the whole workgroup at once: each half probes 128 evenly spaced
// entries for its key and the count of entries below the key narrows the range 128-fold,
// so a list of n entries takes about log_128(n) + 1 dependent loads instead of log_2(n).
// Every thread runs the same trip count (the ranges are computed from block-wide counts).
__device__ __forceinline__ void body_vg_range(const int32_t* __restrict__ vg, int64_t n, int b, int64_t& k0,
                                              int64_t& k1) {
    static_assert(kBlock == 256, "two halves of 128 probes");
    __shared__ int s_cnt[2][kBlock / kWave];
    const int t = threadIdx.x, h = t >> 7, j = t & 127, w = t / kWave;
    const int key = b + h;
    int64_t lo[2] = {0, 0}, len[2] = {n, n};
    for (int it = 0; len[0] > 0 || len[1] > 0; ++it) {
        const int64_t L = len[h];
        bool below = false;
        if (L > 128)
            below = vg[2 * (lo[h] + (int64_t)j * L / 128)] < key;
        else if (j < L)
            below = vg[2 * (lo[h] + j)] < key;
        const uint64_t m = __ballot(below);
        if ((t & (kWave - 1)) == 0) s_cnt[it & 1][w] = __popcll(m);
        __syncthreads();
        for (int q = 0; q < 2; ++q) {
            const int c = s_cnt[it & 1][2 * q] + s_cnt[it & 1][2 * q + 1];
            const int64_t Lq = len[q];
            if (Lq <= 128) {
                lo[q] += c;
                len[q] = 0;
            } else {
                // entries before probe c-1 (inclusive) are below the key, probe c is not
                const int64_t a = c > 0 ? lo[q] + (int64_t)(c - 1) * Lq / 128 + 1 : lo[q];
                const int64_t e = c < 128 ? lo[q] + (int64_t)c * Lq / 128 : lo[q] + Lq;
                lo[q] = a;
                len[q] = e - a;
            }
        }
    }
    k0 = lo[0];
    k1 = lo[1];
}

// stage E: one workgroup per body: its 144 Hessian and 12 gradient entries; and the off-diagonal
// block of every pair.  A pair's chunks' partial sums (part, in the pair's body order [ij0 |
// ij1]) are added in order (PT chunks, then EE), the pairs in row order; nij: the pairs, or with
// dn a bound of dn[0] that only sizes the launch.  nact (nullable): an active count no stage
// wrote, zeroed.
// Without LONG a row's pairs are taken one after the other, each with its off-diagonal block where
// the row's body is its first: a few load latencies, hidden by the other bodies' workgroups (59
// VGPRs, eight waves a SIMD).  A long row makes that a chain with nothing beside it: with LONG
// its pairs with active contacts are listed, kPairsAtOnce of them have their loads in flight, and
// the workgroups past the bodies add the off-diagonal blocks.  A plate under 400 cubes takes 93 us
// with it and 392 without, 8217 bodies in 256 scenes 23.8 and 19.0.  Hence the line at kLongRow
// bodies to a scene, which bound a row.
constexpr int kLongRow = 64;
constexpr int kPairsAtOnce = 8;
constexpr int64_t kOffGrid = 4096;  // workgroups of the off-diagonal blocks, at most

// the off-diagonal block of pair ii (threads 0..143, one an entry): the upper slot holds rows ij0
// x cols ij1, the lower one its transpose
__device__ __forceinline__ void add_off_diagonal(int R, int C, int64_t up, int64_t lo, double h,
                                                 double* __restrict__ blocks) {
    const int bi = R / 3, rr = R % 3, bj = C / 3, cc = C % 3;
    blocks[9 * (16 * up + bi + 4 * bj) + 3 * rr + cc] += h;
    blocks[9 * (16 * lo + bj + 4 * bi) + 3 * cc + rr] += h;
}
template <bool LONG>
__global__ __launch_bounds__(kBlock) void body_finalize_kernel(AbdScene sc, AbdParams P,
                                                                const double* __restrict__ x, int64_t nij,
                                                                const int64_t* __restrict__ dn,
                                                                const int32_t* __restrict__ row_ptr,
                                                                const int32_t* __restrict__ slots,
                                                                const uint8_t* __restrict__ pflag,
                                                                const int2* __restrict__ pitem,
                                                                const double* __restrict__ part,
                                                                const int32_t* __restrict__ vg, int64_t nvg,
                                                                double* __restrict__ g, double* __restrict__ blocks,
                                                                const uint8_t* __restrict__ hl_pt,
                                                                const uint8_t* __restrict__ hl_ee,
                                                                uint8_t* __restrict__ highlight,
                                                                int64_t* __restrict__ nact) {
    __shared__ int s_item[kBlock], s_n[kBlock], s_slot[kBlock];
    const int b = blockIdx.x;
    const int t = threadIdx.x;
    const int nb = sc.n_bodies;
    if (dn) {
        nij = dn[0];
        nvg = dn[4];
    }
    if (LONG && b >= nb) {  // off-diagonal blocks (part is not null), grid-stride over the pairs
        if (t >= 144) return;
        const double* off = part + 24 * (t / 12) + 12 + t % 12;
        for (int64_t ii = b - nb; ii < nij; ii += gridDim.x - nb) {
            if (!pflag[ii]) continue;  // uniform
            const int2 it = pitem[ii];
            double h = 0.0;
            for (int c = 0; c < it.y; ++c) h += off[(int64_t)(it.x + c) * kPartStride];
            add_off_diagonal(t / 12, t % 12, nb + ii, nb + nij + ii, h, blocks);
        }
        return;
    }
    if (nact && b == 0 && t == 0) *nact = 0;
    // threads 0..143: the entries of the diagonal block; 144..155: the gradient; the rest
    // only help to evaluate the vertex-ground terms
    const bool act = t < 156;
    const bool isg = t >= 144;
    const int R = isg ? t - 144 : t / 12, C = isg ? 0 : t % 12;
    double acc = 0.0;
    if (part && nij > 0) {  // uniform
        const int e1 = row_ptr[b + 1];
        for (int eb = row_ptr[b]; eb < e1; eb += kBlock) {
            int ne = e1 - eb < kBlock ? e1 - eb : kBlock, s = 0;
            int2 it = make_int2(0, 0);
            if (t < ne) {  // the row's pairs with active contacts: their items, side
                s = slots[eb + t];
                if (s >= nb) {
                    const int64_t ii = s < nb + nij ? s - nb : s - nb - nij;
                    if (pflag[ii]) it = pitem[ii];
                }
            }
            if constexpr (!LONG) {
                if (t < ne) {
                    s_item[t] = it.x;
                    s_n[t] = it.y;
                    s_slot[t] = s;
                }
                __syncthreads();
                if (act)
                    for (int q = 0; q < ne; ++q) {
                        const int n = s_n[q];
                        if (n == 0) continue;  // the diagonal, or a pair without active contacts
                        const int s = s_slot[q];
                        const int side = s < nb + nij ? 0 : 1;  // upper slot in row b: b is ij0
                        const double* pp = part + (int64_t)s_item[q] * kPartStride;
                        const int at = isg ? 576 + 12 * side + R : 24 * (12 * side + R) + 12 * side + C;
                        double h = 0.0, ho = 0.0;
                        for (int c = 0; c < n; ++c) {
                            h += pp[(int64_t)c * kPartStride + at];
                            if (!isg && side == 0) ho += pp[(int64_t)c * kPartStride + 24 * R + 12 + C];
                        }
                        acc += h;
                        if (!isg && side == 0) add_off_diagonal(R, C, s, s + nij, ho, blocks);
                    }
            } else {
                __shared__ int shw[kBlock / kWave];
                const int r = block_rank(it.y > 0, shw, &ne);
                if (it.y > 0) {
                    s_item[r] = it.x;
                    s_n[r] = it.y;
                    s_slot[r] = s;
                }
                __syncthreads();
                if (act)
                    for (int q = 0; q < ne; q += kPairsAtOnce) {
                        const double* src[kPairsAtOnce];
                        int n[kPairsAtOnce], most = 0;
                        double h[kPairsAtOnce];
#pragma unroll
                        for (int j = 0; j < kPairsAtOnce; ++j) {
                            const int u = q + j < ne ? q + j : q;  // past the end: read, not added
                            const int side = s_slot[u] < nb + nij ? 0 : 1;
                            src[j] = part + (int64_t)s_item[u] * kPartStride +
                                     (isg ? 576 + 12 * side + R : 24 * (12 * side + R) + 12 * side + C);
                            n[j] = q + j < ne ? s_n[u] : 0;
                            most = n[j] > most ? n[j] : most;
                            h[j] = 0.0;
                        }
                        for (int c = 0; c < most; ++c) {  // uniform
                            double v[kPairsAtOnce];
#pragma unroll
                            for (int j = 0; j < kPairsAtOnce; ++j)
                                v[j] = src[j][c < n[j] ? (int64_t)c * kPartStride : 0];
#pragma unroll
                            for (int j = 0; j < kPairsAtOnce; ++j)
                                if (c < n[j]) h[j] += v[j];
                        }
#pragma unroll
                        for (int j = 0; j < kPairsAtOnce; ++j)
                            if (n[j] > 0) acc += h[j];
                    }
            }
            __syncthreads();
        }
    }
    if (P.vg && nvg > 0) {
        // ipcsk/vg_ipc.py:5-34 (no 2 b' grad d grad d^T term, D11).  The barrier derivatives
        // of each contact are evaluated once per tile into LDS, then every entry adds the
        // tile's terms in contact order.
        __shared__ double s_d[kBlock], s_db[kBlock], s_d2b[kBlock], s_vt[kBlock][3];
        int64_t k0, k1;
        body_vg_range(vg, nvg, b, k0, k1);
        const int ia = R / 3, ra = R % 3, ja = C / 3, ca = C % 3;
        for (int64_t base = k0; base < k1; base += kBlock) {
            const int nt = (int)(k1 - base < kBlock ? k1 - base : kBlock);
            if (t < nt) {
                const int64_t vid = sc.voff[b] + vg[2 * (base + t) + 1];
                const double d = x[3 * vid + 1] - P.ground;
                s_d[t] = d;
                s_d2b[t] = barrier_d2(d * d, P.d2hat, P.kappa);
                s_db[t] = barrier_d1(d * d, P.d2hat, P.kappa);
                s_vt[t][0] = sc.x0[3 * vid];
                s_vt[t][1] = sc.x0[3 * vid + 1];
                s_vt[t][2] = sc.x0[3 * vid + 2];
            }
            __syncthreads();
            if (act)
                for (int q = 0; q < nt; ++q) {
                    const double d = s_d[q], d2b = s_d2b[q], db = s_db[q];
                    const double th_i = ia == 0 ? 1.0 : s_vt[q][ia - 1];
                    if (isg) {
                        const double nr = ra == 1 ? 1.0 : 0.0;
                        acc += (((d * 2.0) * nr) * th_i) * db;
                    } else {
                        const double th_j = ja == 0 ? 1.0 : s_vt[q][ja - 1];
                        double scl = th_i * th_j * d2b * 4.0 * d * d;
                        if (P.psd == 2) scl += th_i * th_j * 2.0 * db;  // exact mode: the b' term
                        if (P.psd == 3) {  // full IPC: d2b/dy2 = 4 d^2 b'' + 2 b' clamped at 0
                            const double cy = d2b * 4.0 * d * d + 2.0 * db;
                            scl = th_i * th_j * (cy > 0.0 ? cy : 0.0);
                        }
                        const double nn = (ra == 1 ? 1.0 : 0.0) * (ca == 1 ? 1.0 : 0.0);
                        acc += nn * scl;
                    }
                }
            __syncthreads();
        }
    }
    if (!act) return;
    if (isg) {
        g[3 * (4 * (int64_t)b + R / 3) + R % 3] += acc;
    } else {
        const int ia = R / 3, ra = R % 3, ja = C / 3, ca = C % 3;
        blocks[9 * (16 * (int64_t)b + ia + 4 * ja) + 3 * ra + ca] += acc;
    }
    if (t == 0 && highlight) highlight[b] = (uint8_t)((hl_pt[b] ? 1 : 0) | (hl_ee[b] ? 2 : 0));
}

// The gh stage's flags and counters, 0 before it: the ordering flag, stage D's counters and the
// active count (16 words), the active counts of the super-blocks, the pairs' runs, then the
// bodies' highlight bytes (PT, EE) and the pairs' active flags.
struct GhScratch {
    int* err;
    int* counters;
    int64_t* total;
    uint32_t* scnt;
    unsigned long long* pseg;  // [2][nij][2]
    uint8_t *hl_pt, *hl_ee, *pflag;
    int64_t nsup, words;       // 8-byte words in all
};
int gh_scratch(int nb, int64_t nij, int64_t n, GhScratch& G) {
    G.nsup = ceil_div(ceil_div(n, (int64_t)kBlock), (int64_t)kSuperBlocks);
    const size_t bytes = 2 * (size_t)nb + (size_t)nij;
    G.words = 8 + kSuperStride * G.nsup / 2 + 4 * nij + (int64_t)((bytes + 7) / 8);
    uint64_t* p;
    const int rc = arena_get(kSlotMisc, sizeof(uint64_t) * (size_t)G.words, (void**)&p);
    if (rc) return rc;
    G.err = reinterpret_cast<int*>(p);
    G.counters = G.err + 1;
    G.total = reinterpret_cast<int64_t*>(p + 4);
    G.scnt = reinterpret_cast<uint32_t*>(p + 8);
    G.pseg = reinterpret_cast<unsigned long long*>(p + 8 + kSuperStride * G.nsup / 2);
    G.hl_pt = reinterpret_cast<uint8_t*>(G.pseg + 4 * nij);
    G.hl_ee = G.hl_pt + nb;
    G.pflag = G.hl_ee + nb;
    return ABD_OK;
}

// Per-contact entry (tests, microbenchmarks): dense 24x24 and gradient per contact.
__global__ __launch_bounds__(kBlock) void pair_gh_kernel(int kind, AbdParams P, const double* __restrict__ x4,
                                                          const double* __restrict__ r4, int64_t n,
                                                          uint8_t* __restrict__ active, double* __restrict__ g24,
                                                          double* __restrict__ H24, double* __restrict__ scratch) {
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        d3 v[4], r[4];
        for (int k = 0; k < 4; ++k) {
            v[k] = ld3(x4 + 12 * i + 3 * k);
            r[k] = ld3(r4 + 12 * i + 3 * k);
        }
        double* buf = scratch + i * kContactStride;
        bool act = contact_terms(kind, v, r, P.d2hat, P.kappa, P.psd, buf);
        active[i] = act ? 1 : 0;
        for (int a = 0; a < 24; ++a) {
            g24[24 * i + a] = act ? buf[kB1Off] * buf[kVOff + 24 * 4 + a] : 0.0;
            for (int c = 0; c < 24; ++c) {
                double h = 0.0;
                if (act)
                    for (int k = 0; k < 5; ++k) {
                        const double* V = buf + kVOff + 24 * k;
                        h += buf[kCoefOff + k] * (V[a] * V[c]);
                    }
                H24[576 * i + 24 * a + c] = h;
            }
        }
    }
}

// The same in the dense modes, one wave per contact.
__global__ __launch_bounds__(kWave) void pair_gh_dense_kernel(int kind, AbdParams P, const double* __restrict__ x4,
                                                              const double* __restrict__ r4, int64_t n,
                                                              uint8_t* __restrict__ active, double* __restrict__ g24,
                                                              double* __restrict__ H24,
                                                              double* __restrict__ scratch) {
    __shared__ DenseLds D;
    const int lane = threadIdx.x;
    for (int64_t i = blockIdx.x; i < n; i += gridDim.x) {
        d3 v[4], r[4];
        for (int k = 0; k < 4; ++k) {
            v[k] = ld3(x4 + 12 * i + 3 * k);
            r[k] = ld3(r4 + 12 * i + 3 * k);
        }
        double* buf = scratch + i * kDenseStride;
        const bool act = P.psd == 3 ? wave_contact_full(lane, kind, v, r, P.d2hat, P.kappa, D, buf)
                                    : wave_contact_exact(lane, kind, v, r, P.d2hat, P.kappa, D, buf);
        dense_sync();
        if (lane == 0) active[i] = act ? 1 : 0;
        // every lane reads back what it wrote (entry q of the block and gradient is lane q % 64's)
        for (int q = lane; q < kDenseStride; q += kWave) {
            const double h = act ? buf[q] : 0.0;
            if (q < kDenseGOff)
                H24[576 * i + q] = h;
            else
                g24[24 * i + q - kDenseGOff] = h;
        }
    }
}

// -------------------------------------------------------------- inertia
// orthogonal_energy.py:99-112 (overwrites g)
__global__ void inertia_gradient_kernel(int nb, AbdParams P, const double* __restrict__ mass,
                                        const double* __restrict__ I0v, const double* __restrict__ A,
                                        const double* __restrict__ p, const double* __restrict__ A0,
                                        const double* __restrict__ p0, const double* __restrict__ Adot,
                                        const double* __restrict__ pdot, double* __restrict__ g) {
    int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nb) return;
    const double m = mass ? mass[b] : P.mass, i0 = I0v ? I0v[b] : P.I0;
    for (int e = 0; e < 4; ++e) {
        double r[3];
        inertia_gradient_row(P, e, A + 9 * b, p + 3 * b, A0 + 9 * b, p0 + 3 * b, Adot + 9 * b, pdot + 3 * b, m, i0, r);
        for (int k = 0; k < 3; ++k) g[3 * (4 * b + e) + k] = r[k];
    }
}

// orthogonal_energy.py:63-96 (+= into the diagonal slots); one thread per (body, sub-block).
__global__ void inertia_hessian_kernel(int nb, AbdParams P, const double* __restrict__ mass,
                                       const double* __restrict__ I0v, const double* __restrict__ A,
                                       double* __restrict__ blocks) {
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 16 * nb) return;
    const int b = t / 16, e = t % 16;
    double dh[9];
    inertia_hessian_block(P, e % 4, e / 4, A + 9 * b, mass ? mass[b] : P.mass, I0v ? I0v[b] : P.I0, dh);
    double* B = blocks + 9 * (16 * (int64_t)b + e);
    for (int k = 0; k < 9; ++k) B[k] += dh[k];
}

// The gh stage (stages A-E).  With L.dn the list sizes are on the device (L's counts bound
// them and size the launches and buffers), nothing is read back and the lists are taken
// as grouped (the drivers' own culling output); n_active_dev (nullable) then receives the
// active count on the device.  Without it the call reads the active count and the
// ordering flag back (n_active, host, nullable) and returns ABD_ERR_UNSORTED for lists
// that are not grouped.
int contact_gh(hipStream_t s, const AbdScene* sc, const AbdParams* P, const double* x, const GhLists& L,
               const int32_t* row_ptr, const int32_t* slots, double* g, double* blocks, uint8_t* highlight,
               int64_t* n_active, int64_t* n_active_dev, bool zeroed, int row_bodies) {
    const int nb = sc->n_bodies;
    if (nb == 0) return ABD_OK;
    if (row_bodies <= 0) row_bodies = nb;
    const int32_t *pt = L.pt, *ee = L.ee, *vg = L.vg;
    const int64_t npt = L.npt, nee = L.nee, nij = L.nij;
    const int64_t nvg = P->vg ? L.nvg : 0;
    const int64_t* dn = L.dn;
    const int64_t n = npt + nee;
    int rc;
    GhScratch G;
    if ((rc = gh_scratch(nb, nij, n, G))) return rc;
    if (!zeroed && (rc = zero_fill(s, G.err, sizeof(uint64_t) * (size_t)G.words))) return rc;
    int64_t nact = 0;
    const int64_t nblk = ceil_div(n, (int64_t)kBlock);
    uint8_t* flag = nullptr;
    uint32_t* bcnt = nullptr;
    if (n + nvg > 0) {
        if ((rc = arena_get(kSlotFlags, (size_t)n + 1, (void**)&flag))) return rc;
        if ((rc = arena_get(kSlotScanA, sizeof(uint32_t) * ((size_t)nblk + 1), (void**)&bcnt))) return rc;
        int ph = prof_start(kProfClassify, s, dn ? 1.0 : 129.0 * npt + 133.0 * nee + 8.0 * nvg);
        const int64_t blocks_all = nblk + ceil_div(nvg, (int64_t)kBlock);
        launch_kernel(classify_kernel, dim3((unsigned)std::min<int64_t>(blocks_all, 8192)), dim3(kBlock), 0, s, *sc,
                      *P, x, pt, npt, ee, nee, vg, nvg, dn, flag, G.err, bcnt, G.scnt);
        ABD_CHECK_LAUNCH();
        prof_stop(ph, s);
        if ((rc = prof_count_bytes(ph, s, dn, 129.0, 133.0, 8.0, 0.0))) return rc;
    }
    const auto total_now = [&]() -> int {  // the active count for the host
        launch_kernel(active_total_kernel, dim3(1), dim3(kBlock), 0, s, (const uint32_t*)G.scnt, G.nsup,
                           G.total);
        ABD_CHECK_LAUNCH();
        return ABD_OK;
    };
    const bool dense = P->psd >= 2;
    const int stride = dense ? kDenseStride : kContactStride;
    if (dn) {
        nact = n;  // an upper bound: the stages below read the count on the device
        // The bound is the capacity of the candidate lists, which a superset swept by a very
        // long step can make many times the contacts: past the tuning's contact_bound_mib of
        // stored contacts the active count is read back and sizes the buffers instead (never
        // while a graph is recorded: that iteration then runs eagerly)
        const int mib = tuning().contact_bound_mib;
        if ((double)nact * (8.0 * stride + 9.0) > (mib > 0 ? mib : kGhBoundMib) * 1048576.0) {
            if (capturing()) return ABD_ERR_CAPACITY;
            int64_t* hv;
            if ((rc = arena_host(sizeof(int64_t), (void**)&hv))) return rc;
            if ((rc = total_now())) return rc;
            ABD_CHECK(hipMemcpyAsync(hv, G.total, sizeof(int64_t), hipMemcpyDeviceToHost, s));
            ABD_CHECK(hipStreamSynchronize(s));
            nact = hv[0];
        }
    } else {
        // the active count and the ordering flag in one read-back
        int64_t* hv;
        if ((rc = arena_host(2 * sizeof(int64_t), (void**)&hv))) return rc;
        hv[0] = 0;
        if (n > 0) {
            if ((rc = total_now())) return rc;
            ABD_CHECK(hipMemcpyAsync(hv, G.total, sizeof(int64_t), hipMemcpyDeviceToHost, s));
        }
        ABD_CHECK(hipMemcpyAsync(hv + 1, G.err, sizeof(int), hipMemcpyDeviceToHost, s));
        ABD_CHECK(hipStreamSynchronize(s));
        nact = hv[0];
        int herr = 0;
        memcpy(&herr, hv + 1, sizeof(int));
        if (herr) return ABD_ERR_UNSORTED;
        if (n_active) *n_active = nact;
    }
    double* part = nullptr;
    int2* pitem = nullptr;
    // a count read back is 0: no stage below writes the device's
    int64_t* const nact_unwritten = nact > 0 ? nullptr : n_active_dev;
    if (nact > 0) {
        double* cbuf;
        uint8_t* swp;
        if ((rc = arena_get(kSlotContact, (sizeof(double) * stride + 1) * (size_t)nact, (void**)&cbuf))) return rc;
        swp = reinterpret_cast<uint8_t*>(cbuf + stride * nact);
        const double cbytes = 4.0 + 20 + 16 + 192 + 8.0 * stride + 9;
        int ph = prof_start(kProfContact, s, dn ? 1.0 : cbytes * nact);
        const int64_t* dnact = dn ? G.total : nullptr;
        const ContactOut O{cbuf, swp, G.hl_pt, G.hl_ee, G.pflag, nij, G.pseg};
        const ActiveArgs A{flag, n, dn, bcnt, G.scnt, G.total, n_active_dev};
        if (dense) {
            int32_t* act;
            if ((rc = arena_get(kSlotList, sizeof(int32_t) * (size_t)n, (void**)&act))) return rc;
            launch_kernel(compact_flags_kernel, dim3((unsigned)std::min(nblk, kActiveGrid)), dim3(kBlock), 0, s, A,
                               act);
            ABD_CHECK_LAUNCH();
            const dim3 dgrid((unsigned)std::min<int64_t>(nact, kDenseGrid));
            if (P->psd == 3)
                launch_kernel(contact_dense_kernel<3>, dgrid, dim3(kWave), 0, s, *sc, *P, x, pt, npt, ee,
                                   (const int32_t*)act, nact, dnact, dn, O);
            else
                launch_kernel(contact_dense_kernel<2>, dgrid, dim3(kWave), 0, s, *sc, *P, x, pt, npt, ee,
                                   (const int32_t*)act, nact, dnact, dn, O);
        } else {
            launch_kernel(contact_kernel, dim3((unsigned)std::min(nblk, kActiveGrid)), dim3(kBlock), 0, s, *sc, *P, x,
                               pt, npt, ee, A, O);
        }
        ABD_CHECK_LAUNCH();
        prof_stop(ph, s);
        if ((rc = prof_count_bytes(ph, s, dnact, cbytes, 0.0, 0.0, 0.0, true))) return rc;
        // stage D: chunks of each pair's runs (count, scan), their partial sums, the per-pair sums
        // items: at most one per kPairChunk contacts plus one per run (a run per pair and type)
        const int64_t pgrid = tuning().pair_grid > 0 ? tuning().pair_grid : kPairGrid;
        const int64_t runs = 2 * nij < nact ? 2 * nij : nact;
        const int64_t cap_items = nact / kPairChunk + runs + 1;
        PairItems I{};
        if ((rc = arena_get(kSlotPairChunk, sizeof(int64_t) * ((size_t)nij + 5 * (size_t)cap_items),
                            (void**)&I.pitem)))
            return rc;
        I.idesc = reinterpret_cast<int64_t*>(I.pitem + nij);
        I.odesc = I.idesc + cap_items;
        I.oitem = I.odesc + 2 * cap_items;
        I.cap = cap_items;
        I.counters = G.counters;
        pitem = I.pitem;
        if ((rc = arena_get(kSlotPairPart, sizeof(double) * kPartStride * (size_t)cap_items, (void**)&part)))
            return rc;
        launch_kernel(pair_items_kernel, dim3(grid_for(nij, kBlock)), dim3(kBlock), 0, s, nij, dn,
                           (const uint8_t*)G.pflag, (const unsigned long long*)G.pseg, nij, I);
        ABD_CHECK_LAUNCH();
        // timed: the partial sums (each stored contact read once, its body-order flag once)
        ph = prof_start_ext(kProfPairReduce, dn ? 1.0 : (8.0 * stride + 1) * nact);
        if (dense)
            prof_launch(ph, pair_partial_dense_kernel, dim3((unsigned)pgrid), dim3(kPairThreads), 0, s,
                        (const double*)cbuf, (const uint8_t*)swp, I, part);
        else
            prof_launch(ph, pair_partial_rank_kernel, dim3((unsigned)pgrid), dim3(kRankThreads), 0, s,
                        (const double*)cbuf, (const uint8_t*)swp, I, part);
        ABD_CHECK_LAUNCH();
        if ((rc = prof_count_bytes(ph, s, dnact, 8.0 * stride + 1, 0.0, 0.0, 0.0, true))) return rc;
    }
    const double fbytes = 2.0 * 8 * 156 * nb;
    const double pbytes = 8.0 * 2 * 312;  // a pair's partial sums, read by both bodies (one chunk)
    int phf = prof_start(kProfBodyFinalize, s, dn ? 1.0 : fbytes + pbytes * nij + 40.0 * nvg);
    const bool rows = row_bodies > kLongRow;  // that can be long
    const int64_t off = rows && part ? std::min(nij, kOffGrid) : 0;
    launch_kernel(rows ? body_finalize_kernel<true> : body_finalize_kernel<false>, dim3((unsigned)(nb + off)),
                       dim3(kBlock), 0, s, *sc, *P, x, nij, dn, row_ptr, slots,
                       (const uint8_t*)G.pflag, (const int2*)pitem, (const double*)part, vg, nvg, g, blocks,
                       (const uint8_t*)G.hl_pt, (const uint8_t*)G.hl_ee, highlight, nact_unwritten);
    ABD_CHECK_LAUNCH();
    prof_stop(phf, s);
    if ((rc = prof_count_bytes(phf, s, dn, 0.0, 0.0, 40.0, pbytes, false, fbytes))) return rc;
    return ABD_OK;
}

int gh_zero_region(int nb, int64_t nij, int64_t n, void** p, int64_t* words) {
    GhScratch G;
    const int rc = gh_scratch(nb, nij, n, G);
    *p = G.err;
    *words = G.words;
    return rc;
}

}  // namespace abd

using namespace abd;

extern "C" {

int abd_contact_gh(abd_stream_t stream, const AbdScene* sc, const AbdParams* P, const double* x, const int32_t* pt,
                   int64_t npt, const int32_t* ee, int64_t nee, const int32_t* vg, int64_t nvg, int64_t nij,
                   const int32_t* row_ptr, const int32_t* slots, double* g, double* blocks, uint8_t* highlight,
                   int64_t* n_active) {
    if (!sc || !P || !x || !g || !blocks || npt < 0 || nee < 0 || nvg < 0 || nij < 0) return ABD_ERR_ARG;
    if (P->psd < 0 || P->psd > 3) return ABD_ERR_ARG;
    if ((npt && !pt) || (nee && !ee) || (nvg && !vg) || (nij && (!row_ptr || !slots))) return ABD_ERR_ARG;
    if (nij == 0 && (npt || nee)) return ABD_ERR_ARG;
    if (n_active) *n_active = 0;
    GhLists L{pt, npt, ee, nee, vg, nvg, nij, nullptr};
    return contact_gh(to_stream(stream), sc, P, x, L, row_ptr, slots, g, blocks, highlight, n_active, nullptr);
}

int abd_pair_gh(abd_stream_t stream, int32_t kind, const AbdParams* P, const double* x4, const double* r4, int64_t n,
                uint8_t* active, double* g24, double* H24) {
    if (!P || n < 0 || (n && (!x4 || !r4 || !active || !g24 || !H24)) || (kind != 0 && kind != 1)) return ABD_ERR_ARG;
    if (P->psd < 0 || P->psd > 3) return ABD_ERR_ARG;
    if (n == 0) return ABD_OK;
    double* scratch;
    const int stride = P->psd >= 2 ? kDenseStride : kContactStride;
    int rc = arena_get(kSlotContact, sizeof(double) * stride * (size_t)n, (void**)&scratch);
    if (rc) return rc;
    if (P->psd >= 2)
        launch_kernel(pair_gh_dense_kernel, dim3((unsigned)std::min<int64_t>(n, kDenseGrid)), dim3(kWave), 0,
                           to_stream(stream), kind, *P, x4, r4, n, active, g24, H24, scratch);
    else
        launch_kernel(pair_gh_kernel, dim3(grid_for(n)), dim3(kBlock), 0, to_stream(stream), kind, *P, x4, r4, n,
                           active, g24, H24, scratch);
    ABD_CHECK_LAUNCH();
    return ABD_OK;
}

int abd_inertia_gradient(abd_stream_t stream, const AbdScene* sc, const AbdParams* P, const double* A, const double* p,
                         const double* A0, const double* p0, const double* Adot, const double* pdot, double* g) {
    if (!sc || !P || !A || !p || !A0 || !p0 || !Adot || !pdot || !g) return ABD_ERR_ARG;
    const int nb = sc->n_bodies;
    if (!nb) return ABD_OK;
    launch_kernel(inertia_gradient_kernel, dim3(grid_for(nb)), dim3(kBlock), 0, to_stream(stream), nb, *P,
                       sc->mass, sc->I0, A, p, A0, p0, Adot, pdot, g);
    ABD_CHECK_LAUNCH();
    return ABD_OK;
}

int abd_inertia_hessian(abd_stream_t stream, const AbdScene* sc, const AbdParams* P, const double* A,
                        double* blocks) {
    if (!sc || !P || !A || !blocks) return ABD_ERR_ARG;
    const int nb = sc->n_bodies;
    if (!nb) return ABD_OK;
    launch_kernel(inertia_hessian_kernel, dim3(grid_for(16 * (int64_t)nb)), dim3(kBlock), 0, to_stream(stream),
                       nb, *P, sc->mass, sc->I0, A, blocks);
    ABD_CHECK_LAUNCH();
    return ABD_OK;
}

}  // extern "C"
