// abd_reduce.hip — the scalar reductions of the Newton loop (barrier energy,
// inertia energy, CCD time of impact, dot products), per independent scene.
//
// Every reduction is evaluated in an order fixed by the scene's own data: a
// scene's candidate lists are cut into chunks of kChunkItems counted from the
// scene's first candidate, each chunk is summed (or min-reduced) by one
// workgroup in a fixed pattern, and the chunk results are reduced per scene in
// chunk order.  The same scene therefore gives bit-identical results whether it
// is evaluated alone (n_scenes = 1: the plain entry points) or inside a batch of
// any other scenes, and the plain and batched drivers follow the same Newton
// path to the last bit.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>

#include "abd_block.h"
#include "abd_device.h"
#include "abd_inertia.h"
#include "abd_internal.h"
#include "abd_profile.h"

namespace abd {

constexpr int kRedThreads = 256;
constexpr int kChunkItems = 2048;
constexpr int kLists = 3;

enum { kListPT = 0, kListEE = 1, kListVG = 2 };

struct ListRef {
    const int32_t* p;
    int64_t n;
    int kind;                   // kListPT / kListEE / kListVG
    const int32_t* v = nullptr;  // PT / EE: the candidates' scene vertex ids, 4 per tuple (nullable)
    float* apart = nullptr;      // the candidates' apart_until (nullable)
};
__device__ __forceinline__ const int32_t* vids_of(const ListRef& r, int64_t i) { return r.v ? r.v + 4 * i : nullptr; }
// dn (nullable): the lists' sizes on the device, [nij, nij, npt, nee, nvg] (the keep
// filter's layout); the n of each ListRef then bounds its size (a list with n = 0 is empty).
struct Lists {
    ListRef l[kLists];
    const int64_t* dn = nullptr;
};

__device__ __forceinline__ int64_t list_n(const Lists& L, int l) {
    const ListRef& r = L.l[l];
    if (!L.dn || r.n == 0) return r.n;
    return L.dn[r.kind == kListPT ? 2 : r.kind == kListEE ? 3 : 4];
}

__device__ __forceinline__ int width_of(int kind) { return kind == kListVG ? 2 : 5; }

// first k in [0, n) whose tuple's first body belongs to a scene >= s
__device__ __forceinline__ int64_t scene_lower_bound(const ListRef& L, int64_t n,
                                                     const int32_t* __restrict__ body_scene, int s) {
    const int w = width_of(L.kind);
    int64_t lo = 0, hi = n;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (body_scene[L.p[w * mid]] < s)
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

__device__ __forceinline__ int64_t n_chunks(int64_t len) { return (len + kChunkItems - 1) / kChunkItems; }

// Per scene: the segment [a, b) of each list and the offset of its first chunk.  One
// workgroup: first the S + 1 scene boundaries of every list, one binary search per
// thread (scene s ends where scene s + 1 begins), then the chunk counts of the scenes in
// tiles of blockDim with a running offset.
constexpr int kPlanThreads = 1024;
constexpr unsigned long long kBitsOne = 0x3FF0000000000000ull;  // 1.0
// What the plan's kernel also sets for the CCD that follows it (nullable): the scene slots to
// 1, the queue count to 0.
struct ToiInit {
    unsigned long long* slots = nullptr;
    int32_t* qcount = nullptr;
};
__global__ __launch_bounds__(kPlanThreads) void plan_kernel(int S, const int32_t* __restrict__ body_scene, Lists L,
                                                            int64_t* __restrict__ seg, int64_t* __restrict__ choff,
                                                            ToiInit I) {
    __shared__ int64_t sh[kPlanThreads];
    if (I.slots) {
        for (int s = threadIdx.x; s < S; s += blockDim.x) I.slots[s] = kBitsOne;
        if (threadIdx.x == 0) *I.qcount = 0;
    }
    __shared__ int64_t tile_total;
    for (int idx = threadIdx.x; idx < kLists * (S + 1); idx += blockDim.x) {
        const int l = idx / (S + 1), s = idx % (S + 1);
        const int64_t n = list_n(L, l);
        int64_t v;
        if (S == 1)
            v = s == 0 ? 0 : n;
        else
            v = n > 0 ? scene_lower_bound(L.l[l], n, body_scene, s) : 0;
        if (s < S) seg[2 * (kLists * (int64_t)s + l)] = v;
        if (s > 0) seg[2 * (kLists * (int64_t)(s - 1) + l) + 1] = v;
    }
    __syncthreads();  // the boundaries written above are read by other threads below
    int64_t carry = 0;
    for (int base = 0; base < S; base += blockDim.x) {
        const int s = base + threadIdx.x;
        int64_t cnt = 0;
        if (s < S)
            for (int l = 0; l < kLists; ++l)
                cnt += n_chunks(seg[2 * (kLists * (int64_t)s + l) + 1] - seg[2 * (kLists * (int64_t)s + l)]);
        const int64_t excl = block_exclusive_scan_i64(cnt, sh);
        if (s < S) choff[s] = carry + excl;
        if (threadIdx.x == blockDim.x - 1) tile_total = excl + cnt;
        __syncthreads();
        carry += tile_total;
        __syncthreads();
    }
    if (threadIdx.x == 0) choff[S] = carry;
}

// the scene whose chunks contain chunk c: the largest s with choff[s] <= c
__device__ __forceinline__ int scene_of_chunk(const int64_t* __restrict__ choff, int S, int64_t c) {
    int lo = 0, hi = S - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (choff[mid] <= c)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// Vertex positions at a line-search trial state, placed on the fly from the bodies' trial
// states st ([nb][12], A then p: trial_states_kernel) with the arithmetic of
// abd_update_q + abd_project_vertices (abd.py:305-353), so that they equal the projected
// vertices of the updated state bit for bit.
struct VertsTrial {
    const double *xr, *st;  // rest positions, trial states (16-byte aligned)
    __device__ __forceinline__ void state(int b, double (&q)[12]) const {
        typedef double v2 __attribute__((ext_vector_type(2)));
        const v2* p = reinterpret_cast<const v2*>(st + 12 * (int64_t)b);
#pragma unroll
        for (int i = 0; i < 6; ++i) {
            const v2 v = p[i];
            q[2 * i] = v.x;
            q[2 * i + 1] = v.y;
        }
    }
    __device__ __forceinline__ static d3 place(const double (&q)[12], const double* __restrict__ r) {
        double x[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            double v = q[9 + c] + r[0] * q[c];
            v = v + r[1] * q[3 + c];
            v = v + r[2] * q[6 + c];
            x[c] = v;
        }
        return mk(x[0], x[1], x[2]);
    }
    __device__ __forceinline__ void load4(int I, int J, const int64_t vi[4], int nI, d3 v[4]) const {
        double qI[12], qJ[12];
        state(I, qI);
        state(J, qJ);
        for (int k = 0; k < 4; ++k) v[k] = k < nI ? place(qI, xr + 3 * vi[k]) : place(qJ, xr + 3 * vi[k]);
    }
    __device__ __forceinline__ double y(int b, int64_t vid) const {
        double q[12];
        state(b, q);
        return place(q, xr + 3 * vid).y;
    }
};

// Trial i = k nb + b of the bodies' states q - alpha dq and inertia energies: its state st[i]
// (12) and energy e[i] at length al; a negative length leaves it unwritten.
struct StateArgs {
    const double *A, *p, *dq, *A0, *p0, *Adot, *pdot;
    double *st, *e;
};
__device__ __forceinline__ void trial_state_of(const AbdScene& sc, const AbdParams& P, const StateArgs& Q, int64_t i,
                                               int b, double al) {
    if (al < 0.0) return;
    double Ab[9], pb[3];
    trial_state(b, al, Q.A, Q.p, Q.dq, Ab, pb);
    double* o = Q.st + 12 * i;
#pragma unroll
    for (int q = 0; q < 9; ++q) o[q] = Ab[q];
#pragma unroll
    for (int q = 0; q < 3; ++q) o[9 + q] = pb[q];
    Q.e[i] = inertia_energy_q(P, sc.mass, sc.I0, b, Ab, pb, Q.A0, Q.p0, Q.Adot, Q.pdot);
}
// The states of K trials of lengths alpha [K][S].  One thread per (body, trial): the energies'
// kernels and every candidate evaluated then read 96 bytes of a body instead of forming its
// state.
__global__ __launch_bounds__(kRedThreads) void trial_states_kernel(AbdScene sc, AbdParams P, int S, int K,
                                                                   const double* __restrict__ alpha, StateArgs Q) {
    const int64_t i = (int64_t)blockIdx.x * kRedThreads + threadIdx.x;
    const int nb = sc.n_bodies;
    if (i >= (int64_t)nb * K) return;
    const int b = (int)(i % nb), k = (int)(i / nb);
    trial_state_of(sc, P, Q, i, b, alpha[(int64_t)k * S + (S > 1 ? sc.body_scene[b] : 0)]);
}

// The line search's start: workgroup s < S takes scene s's TOI from its slot to out and the
// first step length to alpha (first_step_length; -1 for a scene not in `active`) with the
// scene's dots (seg_dot_kernel's sums); the others form the states of K trials, the first
// lengths and their halvings (known with the TOI).
__global__ __launch_bounds__(kRedThreads) void search_start_kernel(AbdScene sc, AbdParams P, int S, int K,
                                                                   const unsigned long long* __restrict__ slots,
                                                                   const uint8_t* __restrict__ active,
                                                                   double* __restrict__ out,
                                                                   double* __restrict__ alpha, SceneDots D,
                                                                   StateArgs Q) {
    __shared__ double sh[34];
    if ((int)blockIdx.x >= S) {
        const int64_t i = (int64_t)(blockIdx.x - S) * kRedThreads + threadIdx.x;
        const int nb = sc.n_bodies;
        if (i >= (int64_t)nb * K) return;
        const int b = (int)(i % nb), s = S > 1 ? sc.body_scene[b] : 0;
        double al = active[s] ? first_step_length(__longlong_as_double((long long)slots[s])) : -1.0;
        for (int q = (int)(i / nb); q > 0; --q) al *= 0.5;
        trial_state_of(sc, P, Q, i, b, al);
        return;
    }
    const int s = blockIdx.x;
    if (threadIdx.x == 0) {
        const double r = __longlong_as_double((long long)slots[s]);
        out[s] = r;
        alpha[s] = active[s] ? first_step_length(r) : -1.0;
    }
    const int64_t i0 = D.sboff ? 12 * (int64_t)D.sboff[s] : 0, i1 = D.sboff ? 12 * (int64_t)D.sboff[s + 1] : D.n;
    double acc1 = 0.0, acc2 = 0.0;
    constexpr int kAtOnce = 4;  // terms whose loads are in flight together
    for (int64_t i = i0 + threadIdx.x; i < i1; i += kAtOnce * kRedThreads) {
        double v1[kAtOnce], v2[kAtOnce];
#pragma unroll
        for (int j = 0; j < kAtOnce; ++j) {
            const int64_t q = i + j * kRedThreads < i1 ? i + j * kRedThreads : i;
            v1[j] = D.a[q] * D.b[q];
            v2[j] = D.c[q] * D.d[q];
        }
#pragma unroll
        for (int j = 0; j < kAtOnce; ++j)
            if (i + j * kRedThreads < i1) {
                acc1 += v1[j];
                acc2 += v2[j];
            }
    }
    block_sum2_fast(acc1, acc2, sh);
    if (threadIdx.x == 0) {
        D.out1[s] = acc1;
        D.out2[s] = acc2;
    }
}

// ipcsk/energy.py:10-48 per candidate
template <class Src>
__device__ __forceinline__ double energy_term(int kind, const AbdScene& sc, const SceneView& V, const AbdParams& P,
                                              const Src& X, const int32_t* t, const int32_t* vid) {
    if (P.psd == 3 && kind != kListVG)  // full IPC (beyond the reference)
        return cand_energy_full(kind == kListPT ? 0 : 1, V, X, t, P.d2hat, P.kappa);
    if (kind == kListEE) return cand_energy_ee(V, X, t, P.d2hat, P.kappa, vid);
    if (kind == kListPT) return cand_energy_pt(V, X, t, P.d2hat, P.kappa, vid);
    return cand_energy_vg(sc.voff, X, t, P.ground, P.d2hat, P.kappa);
}

// Chunk c of the plan: its scene s, list l (kLists: none) and candidates [start, end).
struct ChunkRange {
    int s, l;
    int64_t start, end;
};
__device__ __forceinline__ ChunkRange chunk_range(int S, const int64_t* __restrict__ seg,
                                                  const int64_t* __restrict__ choff, int64_t c) {
    ChunkRange r{scene_of_chunk(choff, S, c), 0, 0, 0};
    int64_t k = c - choff[r.s];
    for (; r.l < kLists; ++r.l) {
        const int64_t a = seg[2 * (kLists * (int64_t)r.s + r.l)], b = seg[2 * (kLists * (int64_t)r.s + r.l) + 1];
        const int64_t nch = n_chunks(b - a);
        if (k < nch) {
            r.start = a + k * kChunkItems;
            r.end = r.start + kChunkItems < b ? r.start + kChunkItems : b;
            break;
        }
        k -= nch;
    }
    return r;
}

// Energies at positions x0, one chunk per workgroup.
__global__ __launch_bounds__(kRedThreads) void chunk_kernel(AbdScene sc, AbdParams P, const double* __restrict__ x0,
                                                            Lists L, int S, const int64_t* __restrict__ seg,
                                                            const int64_t* __restrict__ choff,
                                                            double* __restrict__ part) {
    __shared__ double sh[17];
    const int64_t c = blockIdx.x;
    if (c >= choff[S]) return;
    const ChunkRange r = chunk_range(S, seg, choff, c);
    double acc = 0.0;
    if (r.l < kLists) {
        const SceneView V{sc.voff, sc.foff, sc.eoff, sc.tris, sc.edges, sc.x0};
        const int kind = L.l[r.l].kind, w = width_of(kind);
        const Verts X{x0};
        for (int64_t i = r.start + threadIdx.x; i < r.end; i += kRedThreads)
            acc += energy_term(kind, sc, V, P, X, L.l[r.l].p + w * i, vids_of(L.l[r.l], i));
    }
    acc = block_sum_fast(acc, sh);
    if (threadIdx.x == 0) part[c] = acc;
}

// The line-search trials: step lengths alpha [trial][S] (a negative length skips that
// scene's trial: its sums are 0) and the bodies' states at each ([trial][nb][12]).
struct TrialArgs {
    const double *alpha, *st;
};

// The energies of up to kMaxTrials trials, one chunk per workgroup, the trials dealt over blockIdx.y
// (partials part + part_stride trial).  Nearly every candidate of a step's set is inactive at
// a trial (its boxes meet only further along the step, or not at all), so the (trial,
// candidate) pairs that may be active (apart_until at most the trial's length: 4 bytes read
// a candidate) are listed in LDS, all trials together, and evaluated side by side; each
// thread then adds its own candidates' terms in order: the sum of every candidate in turn,
// whose other terms are zeros.  A pair's place in the list is its trial's and wave's first
// place plus its rank among the wave's ballots, so that the owner finds it again.  Bound by
// the latency of a workgroup's few dependent gathers: evaluating every candidate at every
// trial took 60 us for a pass of one trial and 130 us for one of twelve over 1.3M
// candidates (256 scenes), this 32 and 73 us (0.35M and 1.1M pairs evaluated).  Where most
// candidates are near and listed all the same (256 scenes of 2 to 64 bodies, 0.8 of the bytes),
// the listing is not repaid: 30 and 58 us against 19 and 44.
constexpr int kTrialItems = kChunkItems / kRedThreads;
constexpr int kTrialBatch = 1024;  // pairs listed at a time
__global__ __launch_bounds__(kRedThreads, 4) void trial_chunk_kernel(AbdScene sc, AbdParams P, TrialArgs T, Lists L,
                                                                     int S, int K, const int64_t* __restrict__ seg,
                                                                     const int64_t* __restrict__ choff,
                                                                     double* __restrict__ part, int64_t part_stride) {
    constexpr int kWaves = kRedThreads / kWave;
    __shared__ double term[kTrialBatch];
    __shared__ uint16_t pair[kTrialBatch];  // trial << 11 | candidate of the chunk
    __shared__ int first[kMaxTrials * kWaves + 1];
    __shared__ double wsum[kMaxTrials][kWaves];
    __shared__ double sal[kMaxTrials];
    static_assert(kChunkItems == 2048 && kMaxTrials <= 32, "a pair fits 16 bits");
    static_assert(kMaxTrials * kWaves <= kWave, "one lane a (trial, wave)");
    const int64_t c = blockIdx.x;
    if (c >= choff[S]) return;
    const ChunkRange r = chunk_range(S, seg, choff, c);
    const int t = threadIdx.x, lane = lane_id(), w = wave_id();
    const int nk = (K - (int)blockIdx.y + (int)gridDim.y - 1) / (int)gridDim.y;  // this workgroup's trials
    if (t < nk) sal[t] = T.alpha[(int64_t)S * (blockIdx.y + t * gridDim.y) + r.s];
    __syncthreads();
    bool any = false;
    for (int k = 0; k < nk; ++k) any |= !(sal[k] < 0.0);
    double* const out = part + part_stride * blockIdx.y + c;
    if (!any) {  // uniform: no trial of the scene is wanted, the neutral element of the sum
        if (t < nk) out[part_stride * t * gridDim.y] = 0.0;
        return;
    }
    const ListRef& Lr = L.l[r.l < kLists ? r.l : 0];
    float apart[kTrialItems];
#pragma unroll
    for (int u = 0; u < kTrialItems; ++u) {
        const int64_t i = r.start + u * kRedThreads + t;
        apart[u] = i < r.end ? (Lr.apart ? Lr.apart[i] : 0.0f) : 4.0f;
    }
    // (trial, candidate) pairs of each wave, then their exclusive prefix sum over (trial, wave)
    for (int k = 0; k < nk; ++k) {
        const double al = sal[k];
        int n = 0;
        if (!(al < 0.0))
#pragma unroll
            for (int u = 0; u < kTrialItems; ++u) n += __popcll(__ballot(!(al < (double)apart[u])));
        if (lane == 0) first[k * kWaves + w] = n;
    }
    __syncthreads();
    if (w == 0) {
        const int n = lane < nk * kWaves ? first[lane] : 0;
        int incl = n;
#pragma unroll
        for (int off = 1; off < kWave; off <<= 1) {
            const int y = __shfl_up(incl, off);
            if (lane >= off) incl += y;
        }
        if (lane < nk * kWaves) first[lane] = incl - n;
        if (lane == kWave - 1) first[nk * kWaves] = incl;
    }
    __syncthreads();
    const SceneView V{sc.voff, sc.foff, sc.eoff, sc.tris, sc.edges, sc.x0};
    const int width = width_of(Lr.kind);
    const unsigned long long below = (1ull << lane) - 1ull;
    // batches of whole trials, or of a part of one trial's pairs (its sums then carried on)
    double acc = 0.0;
    for (int k0 = 0, b0 = 0; k0 < nk;) {  // uniform
        int k1 = k0 + 1;
        while (k1 < nk && first[(k1 + 1) * kWaves] - b0 <= kTrialBatch) ++k1;
        const int b1 = min(first[k1 * kWaves], b0 + kTrialBatch);
        for (int k = k0; k < k1; ++k) {
            const double al = sal[k];
            if (al < 0.0) continue;
            int at = first[k * kWaves + w] - b0;
#pragma unroll
            for (int u = 0; u < kTrialItems; ++u) {
                const bool on = !(al < (double)apart[u]);
                const unsigned long long m = __ballot(on);
                const int q = at + __popcll(m & below);
                if (on && q >= 0 && q < b1 - b0) pair[q] = (uint16_t)((k << 11) | (u * kRedThreads + t));
                at += __popcll(m);
            }
        }
        __syncthreads();
        for (int q = t; q < b1 - b0; q += kRedThreads) {
            const int64_t i = r.start + (pair[q] & 2047);
            const int64_t k = blockIdx.y + (pair[q] >> 11) * gridDim.y;
            const VertsTrial X{sc.x0, T.st + 12 * k * sc.n_bodies};
            term[q] = energy_term(Lr.kind, sc, V, P, X, Lr.p + width * i, vids_of(Lr, i));
        }
        __syncthreads();
        const bool whole = b1 == first[k1 * kWaves];  // the last trial of the batch ends in it
        for (int k = k0; k < k1; ++k) {
            const double al = sal[k];
            if (!(al < 0.0)) {
                int at = first[k * kWaves + w] - b0;
#pragma unroll
                for (int u = 0; u < kTrialItems; ++u) {
                    const bool on = !(al < (double)apart[u]);
                    const unsigned long long m = __ballot(on);
                    const int q = at + __popcll(m & below);
                    if (on && q >= 0 && q < b1 - b0) acc += term[q];
                    at += __popcll(m);
                }
            }
            if (whole || k + 1 < k1) {
                const double v = wave_sum(acc);
                if (lane == 0) wsum[k][w] = v;
                acc = 0.0;
            }
        }
        __syncthreads();
        b0 = b1;
        k0 = whole ? k1 : k1 - 1;
    }
    // the trials' sums with block_sum_fast's pairing (four waves of its sixteen: the shuffles
    // by 8 and 4 add the empty waves' zeros, those by 2 and 1 give (w0 + w2) + (w1 + w3))
    if (t < nk) out[part_stride * t * gridDim.y] = (wsum[t][0] + wsum[t][2]) + (wsum[t][1] + wsum[t][3]);
}

__global__ __launch_bounds__(kRedThreads) void scene_final_kernel(const int64_t* __restrict__ choff,
                                                                  const double* __restrict__ part,
                                                                  double* __restrict__ out) {
    __shared__ double sh[17];
    const int s = blockIdx.x;
    double acc = 0.0;
    for (int64_t i = choff[s] + threadIdx.x; i < choff[s + 1]; i += blockDim.x) acc += part[i];
    const double r = block_sum_fast(acc, sh);
    if (threadIdx.x == 0) out[s] = r;
}

// ---------------------------------------------------------------- CCD TOI
// The scene minimum of the TOIs below 1 (ccd.py:9-40, abd.py:284-299) in two passes.
// toi_scan_kernel: one candidate per thread (kToiSplit workgroups of kRedThreads per chunk
// of the plan): the vertex-ground TOI directly, and for a PT / EE candidate its
// coplanarity cubic and bracket test; the few candidates with a bracketed root in [0, 1] go
// to a queue (one atomic per wave).  (The native driver's filter of the swept set does this
// per entry: KeepSweep.)  toi_solve_kernel: the full collision_time of each
// queued candidate (root searches and validity), its TOI below 1 min-ed into its scene's
// slot (non-negative doubles order like their bit patterns, so an integer atomic min is
// exact).  toi_final_kernel: per scene the minimum of its chunks' partials and its slot.
// A minimum does not depend on the order, so the result is the one of evaluating every
// candidate in turn.
constexpr int kToiSplit = kChunkItems / kRedThreads;  // one candidate per thread
constexpr int kToiSolveThreads = 64;
constexpr int kToiSolveGrid = 2048;

__device__ __forceinline__ double wave_min(double v) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
        const double u = __shfl_xor(v, o);
        v = u < v ? u : v;
    }
    return v;
}

__global__ __launch_bounds__(kRedThreads, 4) void toi_scan_kernel(AbdScene sc, AbdParams P, const double* __restrict__ x0,
                                                               const double* __restrict__ x1, Lists L, int S,
                                                               const int64_t* __restrict__ seg,
                                                               const int64_t* __restrict__ choff,
                                                               double* __restrict__ part, int32_t* __restrict__ queue,
                                                               int32_t* __restrict__ qcount) {
    __shared__ double sh[kRedThreads / kWave];
    const int64_t c = blockIdx.x;
    if (c >= choff[S]) return;  // uniform over the workgroup
    const ChunkRange r = chunk_range(S, seg, choff, c);
    const SceneView V{sc.voff, sc.foff, sc.eoff, sc.tris, sc.edges, sc.x0};
    const ListRef& Lr = L.l[r.l < kLists ? r.l : 0];
    const int kind = Lr.kind, ck = kind == kListPT ? 0 : 1;
    const int64_t i = r.start + (int64_t)blockIdx.y * kRedThreads + threadIdx.x;
    double acc = 1.0;
    bool queued = false;
    int32_t entry = 0;
    if (r.l < kLists && i < r.end) {
        const int32_t* t = Lr.p + (int64_t)width_of(kind) * i;
        if (kind == kListVG) {
            const double tv = cand_toi_vg(sc.voff, x0, x1, t, P.ground);
            if (tv < 1.0) acc = tv;  // `if t < 1: atomic_min`
        } else {
            d3 a[4], b[4];
            cand_verts(ck, V, x0, x1, t, a, b, vids_of(Lr, i));
            queued = toi_bracketed(a, b);
            entry = (int32_t)((i << 1) | (kind == kListEE ? 1 : 0));
        }
    }
    // wave-aggregated push of the queued candidates
    const unsigned long long mask = __ballot(queued);
    if (mask) {
        const int lane = lane_id();
        const int leader = __ffsll((long long)mask) - 1;
        int32_t base = 0;
        if (lane == leader) base = atomicAdd(qcount, (int32_t)__popcll(mask));
        base = __shfl(base, leader);
        if (queued) queue[base + __popcll(mask & ((1ull << lane) - 1ull))] = entry;
    }
    const double wm = wave_min(acc);
    if (lane_id() == 0) sh[wave_id()] = wm;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = sh[0];
        for (int w = 1; w < kRedThreads / kWave; ++w) m = sh[w] < m ? sh[w] : m;
        part[c * kToiSplit + blockIdx.y] = m;
    }
}

// The reduction plan of the EE, PT and VG lists a sweep wrote (plan_kernel's) from its
// per-scene counts (S = 1: the lists' sizes dn), by one wave.
struct SweepPlan {
    const uint32_t* scnt = nullptr;
    const int64_t* dn = nullptr;
    int use[kLists] = {};
    int64_t* plan = nullptr;  // nullptr: no plan
};
__device__ __forceinline__ void sweep_plan(int S, const SweepPlan& Q) {
    int64_t *seg = Q.plan, *choff = seg + 2 * kLists * (int64_t)S;
    int64_t carry[kLists + 1] = {};
    for (int base = 0; base < S; base += kWave) {
        const int s = base + lane_id();
        int64_t v[kLists + 1] = {};
#pragma unroll
        for (int l = 0; l < kLists; ++l) {
            if (s < S && Q.use[l])
                v[l] = S > 1 ? (int64_t)Q.scnt[(int64_t)l * S + s] : Q.dn[l == 0 ? 3 : l == 1 ? 2 : 4];
            v[kLists] += n_chunks(v[l]);
        }
#pragma unroll
        for (int l = 0; l <= kLists; ++l) {
            int64_t incl = v[l];
            for (int o = 1; o < kWave; o <<= 1) {
                const int64_t u = __shfl_up(incl, o);
                if (lane_id() >= o) incl += u;
            }
            const int64_t e = carry[l] + incl;
            if (s < S) {
                if (l < kLists) {
                    seg[2 * (kLists * (int64_t)s + l)] = e - v[l];
                    seg[2 * (kLists * (int64_t)s + l) + 1] = e;
                } else {
                    choff[s] = e - v[l];
                }
            }
            carry[l] = __shfl(e, kWave - 1);
        }
    }
    if (lane_id() == 0) choff[S] = carry[kLists];
}

__global__ __launch_bounds__(kToiSolveThreads) void toi_solve_kernel(AbdScene sc, Lists L, int S,
                                                                     const double* __restrict__ x0,
                                                                     const double* __restrict__ x1,
                                                                     const int32_t* __restrict__ queue,
                                                                     const int32_t* __restrict__ qcount,
                                                                     unsigned long long* __restrict__ slots,
                                                                     SweepPlan Q) {
    int block = blockIdx.x, blocks = gridDim.x;
    if (Q.plan) {  // block 0 makes the plan, the others solve
        if (block == 0) {
            sweep_plan(S, Q);
            return;
        }
        --block;
        --blocks;
    }
    const int32_t n = *qcount;
    const SceneView V{sc.voff, sc.foff, sc.eoff, sc.tris, sc.edges, sc.x0};
    for (int32_t q = block * kToiSolveThreads + threadIdx.x; q < n; q += blocks * kToiSolveThreads) {
        const int32_t e = queue[q];
        const int ee = e & 1;
        const ListRef& Lr = L.l[ee ? 0 : 1];  // the lists' order: EE, PT, VG
        const int32_t* t = Lr.p + 5 * (int64_t)(e >> 1);
        const double tt = cand_toi(ee, V, x0, x1, t, vids_of(Lr, e >> 1));
        if (tt < 1.0) {
            const int s = S > 1 ? sc.body_scene[t[0]] : 0;
            atomicMin(slots + s, (unsigned long long)__double_as_longlong(tt));
        }
    }
}

__global__ __launch_bounds__(kRedThreads) void toi_final_kernel(const int64_t* __restrict__ choff,
                                                                const double* __restrict__ part,
                                                                const unsigned long long* __restrict__ slots,
                                                                double* __restrict__ out) {
    __shared__ double sh[kRedThreads / kWave];
    const int s = blockIdx.x;
    double acc = __longlong_as_double((long long)slots[s]);
    for (int64_t i = choff[s] * kToiSplit + threadIdx.x; i < choff[s + 1] * kToiSplit; i += blockDim.x) {
        const double v = part[i];
        acc = v < acc ? v : acc;
    }
    const double r = block_min(acc, sh);
    if (threadIdx.x == 0) out[s] = r;
}

// out[s] = sum over the rows [12 sboff[s], 12 sboff[s + 1]) of a * b (one workgroup per scene;
// sboff == nullptr: one segment [0, n))
__global__ __launch_bounds__(kRedThreads) void seg_dot_kernel(const int32_t* __restrict__ sboff, int64_t n,
                                                              const double* __restrict__ a,
                                                              const double* __restrict__ b, double* __restrict__ out) {
    __shared__ double sh[17];
    const int s = blockIdx.x;
    const int64_t i0 = sboff ? 12 * (int64_t)sboff[s] : 0, i1 = sboff ? 12 * (int64_t)sboff[s + 1] : n;
    double acc = 0.0;
    for (int64_t i = i0 + threadIdx.x; i < i1; i += blockDim.x) acc += a[i] * b[i];
    const double r = block_sum_fast(acc, sh);
    if (threadIdx.x == 0) out[s] = r;
}

// orthogonal_energy.py:25-51 summed over the bodies of each scene (one workgroup per scene)
__global__ __launch_bounds__(kRedThreads) void seg_inertia_kernel(const int32_t* __restrict__ sboff, int nb,
                                                                  AbdParams P, const double* __restrict__ mass,
                                                                  const double* __restrict__ I0v,
                                                                  const double* __restrict__ Ak,
                                                                  const double* __restrict__ pk,
                                                                  const double* __restrict__ A0,
                                                                  const double* __restrict__ p0,
                                                                  const double* __restrict__ Adot,
                                                                  const double* __restrict__ pdot,
                                                                  double* __restrict__ E) {
    __shared__ double sh[17];
    const int s = blockIdx.x;
    const int b0 = sboff ? sboff[s] : 0, b1 = sboff ? sboff[s + 1] : nb;
    double acc = 0.0;
    for (int b = b0 + threadIdx.x; b < b1; b += blockDim.x)
        acc += inertia_energy_body(P, mass, I0v, b, Ak, pk, A0, p0, Adot, pdot);
    const double r = block_sum_fast(acc, sh);
    if (threadIdx.x == 0) E[s] = r;
}

// Upper bound on the chunks of the lists over S scenes (each scene's lists may end in a
// partial chunk).
int64_t chunk_bound(const Lists& L, int S) {
    int64_t bound = 3 * (int64_t)S;
    for (int l = 0; l < kLists; ++l) bound += (L.l[l].n + kChunkItems - 1) / kChunkItems;
    return bound;
}

// Caller-provided scratch of the TOI (the allocation-free entry point's): the plan, the
// scene slots and queue count, room for part_cap chunk partials (kToiSplit per chunk) and
// queue_cap queued candidates.  Null: the arena's.
struct ReduceScratch {
    int64_t* plan = nullptr;
    unsigned long long* slots = nullptr;
    int32_t* qcount = nullptr;
    double* part = nullptr;
    int64_t part_cap = 0;
    int32_t* queue = nullptr;
    int64_t queue_cap = 0;
};

// The per-scene segments and chunk offsets of the lists: plan_in when given (made by
// reduce_plan for these lists), else computed into plan_buf (nullable: the arena).
int get_plan(hipStream_t s, const AbdScene& sc, int S, const Lists& L, const int64_t* plan_in,
             const int64_t** seg, const int64_t** choff, int64_t* plan_buf = nullptr, ToiInit init = {}) {
    if (plan_in) {
        *seg = plan_in;
        *choff = plan_in + 2 * kLists * (size_t)S;
        return ABD_OK;
    }
    int64_t* plan = plan_buf;
    int rc = plan ? ABD_OK : arena_get(kSlotPlan, sizeof(int64_t) * reduce_plan_elems(S), (void**)&plan);
    if (rc) return rc;
    launch_kernel(plan_kernel, dim3(1), dim3(kPlanThreads), 0, s, S, sc.body_scene, L, plan,
                       plan + 2 * kLists * (size_t)S, init);
    ABD_CHECK_LAUNCH();
    *seg = plan;
    *choff = plan + 2 * kLists * (size_t)S;
    return ABD_OK;
}

int toi_scratch(int S, int64_t nq, unsigned long long** slots, int32_t** qcount, int32_t** queue) {
    int rc = arena_get(kSlotToiQueue, sizeof(int32_t) * (size_t)(nq + 1), (void**)queue);
    if (!rc) rc = arena_get(kSlotToiSlots, sizeof(unsigned long long) * (size_t)(S + 1), (void**)slots);
    if (!rc) *qcount = reinterpret_cast<int32_t*>(*slots + S);
    return rc;
}

// Plan + chunks + per-scene energies over the lists at x; S = 1 treats the lists as one scene.
// Algorithmic bytes: 128 per PT, 132 per EE and 32 per VG candidate.
int seg_reduce(hipStream_t s, const AbdScene& sc, const AbdParams& P, int S, const double* x, const Lists& L,
               double* out, int prof_id) {
    const int64_t bound = chunk_bound(L, S);
    if (bound > INT32_MAX) return ABD_ERR_ARG;
    const int64_t *seg, *choff;
    double* part = nullptr;
    int rc = get_plan(s, sc, S, L, nullptr, &seg, &choff);
    if (!rc) rc = arena_get(kSlotReduce, sizeof(double) * (size_t)bound, (void**)&part);
    if (rc) return rc;
    int ph = prof_start_ext(prof_id, L.dn ? 1.0 : 128.0 * L.l[1].n + 132.0 * L.l[0].n + 32.0 * L.l[2].n);
    prof_launch(ph, chunk_kernel, dim3((unsigned)bound), dim3(kRedThreads), 0, s, sc, P, x, L, S, seg, choff, part);
    ABD_CHECK_LAUNCH();
    if ((rc = prof_count_bytes(ph, s, L.dn, 128.0, 132.0, 32.0, 0.0))) return rc;
    launch_kernel(scene_final_kernel, dim3(S), dim3(kRedThreads), 0, s, choff, (const double*)part, out);
    ABD_CHECK_LAUNCH();
    return ABD_OK;
}

// Algorithmic bytes of a launch over the plan's scenes: c_ee, c_pt, c_vg per EE, PT and VG
// candidate of the plan's per-scene segments.
__global__ __launch_bounds__(kRedThreads) void seg_bytes_kernel(int S, const int64_t* __restrict__ seg, double c_ee,
                                                                double c_pt, double c_vg, double* __restrict__ out) {
    __shared__ double sh[kRedThreads];
    double acc = 0.0;
    for (int64_t i = threadIdx.x; i < S; i += blockDim.x) {
        const int64_t* q = seg + 2 * (int64_t)kLists * i;
        acc += c_ee * (double)(q[1] - q[0]) + c_pt * (double)(q[3] - q[2]) + c_vg * (double)(q[5] - q[4]);
    }
    acc = block_sum(acc, sh);
    if (threadIdx.x == 0) *out = acc;
}

// Attaches to `handle` the bytes of seg_bytes_kernel (nothing when the handle is -1).
int attach_seg_bytes(int handle, hipStream_t s, int S, const int64_t* seg, double c_ee, double c_pt, double c_vg) {
    double* out;
    int rc = prof_byte_slot(handle, &out);
    if (rc || !out) return rc;
    launch_kernel(seg_bytes_kernel, dim3(1), dim3(kRedThreads), 0, s, S, seg, c_ee, c_pt, c_vg, out);
    ABD_CHECK_LAUNCH();
    prof_stop(handle, s, nullptr, out);
    return ABD_OK;
}

// Algorithmic bytes of trial_chunk_kernel, one workgroup per chunk.  Per candidate, once a launch
// however many of its trials take it: its apart_until where a trial of its scene is wanted, and
// 132, 128 or 32 bytes (EE, PT, VG: tuple, indices and rest vertices) where one lists it; per
// wanted trial of a scene, the states of the scene's bodies (96 bytes each; workgroup 0).  Sums
// of whole numbers: their order is free.
__global__ __launch_bounds__(kRedThreads) void trial_bytes_kernel(Lists L, int S, int K, int nb,
                                                                  const int32_t* __restrict__ scene_boff,
                                                                  const double* __restrict__ alpha,
                                                                  const int64_t* __restrict__ seg,
                                                                  const int64_t* __restrict__ choff,
                                                                  double* __restrict__ out) {
    __shared__ double sh[kRedThreads];
    const int64_t c = blockIdx.x;
    double acc = 0.0;
    if (c == 0)
        for (int i = threadIdx.x; i < S * K; i += blockDim.x)
            if (!(alpha[i] < 0.0)) acc += 96.0 * (S > 1 ? scene_boff[i % S + 1] - scene_boff[i % S] : nb);
    if (c < choff[S]) {
        const ChunkRange r = chunk_range(S, seg, choff, c);
        const ListRef& Lr = L.l[r.l < kLists ? r.l : 0];
        const double each = Lr.kind == kListEE ? 132.0 : Lr.kind == kListPT ? 128.0 : 32.0;
        for (int64_t i = r.start + threadIdx.x; i < r.end; i += blockDim.x) {
            const double apart = Lr.apart ? (double)Lr.apart[i] : 0.0;
            bool wanted = false, listed = false;
            for (int k = 0; k < K; ++k) {
                const double al = alpha[(int64_t)S * k + r.s];
                if (al < 0.0) continue;
                wanted = true;
                if (!(al < apart)) listed = true;
            }
            if (wanted && Lr.apart) acc += 4.0;
            if (listed) acc += each;
        }
    }
    acc = block_sum(acc, sh);
    if (threadIdx.x == 0) atomicAdd(out, acc);
}

// Attaches to `handle` the bytes of trial_bytes_kernel (nothing when the handle is -1).
int attach_trial_bytes(int handle, hipStream_t s, const AbdScene& sc, const Lists& L, int S, int K,
                       const double* alpha, const int64_t* seg, const int64_t* choff, int64_t chunks) {
    double* out;
    int rc = prof_byte_slot(handle, &out);
    if (rc || !out) return rc;
    if ((rc = zero_fill(s, out, sizeof(double)))) return rc;
    launch_kernel(trial_bytes_kernel, dim3((unsigned)chunks), dim3(kRedThreads), 0, s, L, S, K, sc.n_bodies,
                  sc.scene_boff, alpha, seg, choff, out);
    ABD_CHECK_LAUNCH();
    prof_stop(handle, s, nullptr, out);
    return ABD_OK;
}

// The queued candidates of the EE and PT lists (L.l[0], L.l[1]) solved into the slots.
int toi_solve(hipStream_t s, const AbdScene& sc, int S, const double* x0, const double* x1, const Lists& L,
              const int32_t* queue, const int32_t* qcount, unsigned long long* slots, bool prof,
              const SweepPlan& Q = {}) {
    const int64_t nq = L.l[0].n + L.l[1].n;
    const int64_t gmax = tuning().toi_grid > 0 ? tuning().toi_grid : kToiSolveGrid;
    const unsigned grid = (unsigned)std::min<int64_t>(gmax, std::max<int64_t>(1, ceil_div(nq, 4 * kToiSolveThreads)));
    const int ph = prof ? prof_start_ext(kProfToiSolve, 0.0) : -1;
    prof_launch(ph, toi_solve_kernel, dim3(grid + (Q.plan ? 1 : 0)), dim3(kToiSolveThreads), 0, s, sc, L, S, x0, x1,
                queue, qcount, slots, Q);
    ABD_CHECK_LAUNCH();
    return ABD_OK;
}

// Per-scene TOI (toi_scan_kernel, toi_solve_kernel, toi_final_kernel) with scratch from
// scr (nullable: the arena; then the scan and the solve are timed when profiling).
int toi_reduce(hipStream_t s, const AbdScene& sc, const AbdParams& P, int S, const double* x0, const double* x1,
               const Lists& L, double* out, const ReduceScratch* scr) {
    const int64_t bound = chunk_bound(L, S);
    if (bound * kToiSplit > INT32_MAX) return ABD_ERR_ARG;
    const int64_t nq = L.l[0].n + L.l[1].n;  // every PT and EE candidate may queue
    if (nq > (int64_t)INT32_MAX / 2) return ABD_ERR_ARG;
    if (scr && (bound * kToiSplit > scr->part_cap || nq > scr->queue_cap)) return ABD_ERR_CAPACITY;
    ReduceScratch w;
    if (scr) {
        w = *scr;
    } else {
        int rc;
        if ((rc = arena_get(kSlotReduce, sizeof(double) * (size_t)(bound * kToiSplit), (void**)&w.part))) return rc;
        if ((rc = toi_scratch(S, nq, &w.slots, &w.qcount, &w.queue))) return rc;
    }
    const int64_t *seg, *choff;
    int rc = get_plan(s, sc, S, L, nullptr, &seg, &choff, w.plan, ToiInit{w.slots, w.qcount});
    if (rc) return rc;
    // algorithmic bytes of the scan: tuple, indices and four vertices at both ends per PT / EE
    // candidate (224 / 228 B), tuple, offset and a vertex at both ends per VG candidate (56 B),
    // over the scenes it evaluates (counted on the device)
    const int ph = scr ? -1 : prof_start_ext(kProfToi, 1.0);
    prof_launch(ph, toi_scan_kernel, dim3((unsigned)bound, kToiSplit), dim3(kRedThreads), 0, s, sc, P, x0, x1, L, S,
                seg, choff, w.part, w.queue, w.qcount);
    ABD_CHECK_LAUNCH();
    if ((rc = attach_seg_bytes(ph, s, S, seg, 228.0, 224.0, 56.0))) return rc;
    if ((rc = toi_solve(s, sc, S, x0, x1, L, w.queue, w.qcount, w.slots, !scr))) return rc;
    launch_kernel(toi_final_kernel, dim3(S), dim3(kRedThreads), 0, s, choff, (const double*)w.part,
                       (const unsigned long long*)w.slots, out);
    ABD_CHECK_LAUNCH();
    return ABD_OK;
}

// The candidate lists of energies and TOIs, in the one order every reduction uses (the
// sum order of the energy; a minimum does not depend on it).  The switches of
// const_params.py:42-44 drop a whole list.
Lists contact_lists(const AbdParams& P, const int32_t* pt, int64_t npt, const int32_t* ee, int64_t nee,
                    const int32_t* vg, int64_t nvg, const int64_t* dn = nullptr, CandSide vids = {}) {
    if (!P.pt) npt = 0;
    if (!P.ee) nee = 0;
    if (!P.vg) nvg = 0;
    return Lists{{{ee, nee, kListEE, vids.ee, vids.apart_ee},
                  {pt, npt, kListPT, vids.pt, vids.apart_pt},
                  {vg, nvg, kListVG, nullptr, vids.apart_vg}},
                 dn};
}

size_t reduce_plan_elems(int S) { return 2 * kLists * (size_t)S + (size_t)S + 1; }

// ---------------------------------------------------------- line-search trials
// K trial states q - alpha dq evaluated together (alpha: [K][S] on the device; S = 1
// treats the scene as one): per scene the chunks' contact energies of every trial, each
// bit-identical to the chunk sums at that state.

int trial_states(hipStream_t s, const AbdScene* sc, const AbdParams* P, int S, int K, const double* alpha,
                 const double* A, const double* p, const double* dq, const double* A0, const double* p0,
                 const double* Adot, const double* pdot, double* st, double* e) {
    const int64_t n = (int64_t)sc->n_bodies * K;
    if (n <= 0) return ABD_OK;
    launch_kernel(trial_states_kernel, dim3(grid_for(n, kRedThreads, INT32_MAX)), dim3(kRedThreads), 0, s, *sc, *P, S,
                  K, alpha, StateArgs{A, p, dq, A0, p0, Adot, pdot, st, e});
    ABD_CHECK_LAUNCH();
    return ABD_OK;
}

// workgroups of a line-search pass: twice what the device holds at once (four a CU)
constexpr int64_t kTrialGrid = 2048;
int line_chunks(hipStream_t s, const AbdScene* sc, const AbdParams* P, int S, int K, const double* alpha,
                const double* st, const int32_t* pt, int64_t npt, const int32_t* ee, int64_t nee, const int32_t* vg,
                int64_t nvg, const int64_t* plan, const int64_t* dn, CandSide vids, TrialSums* out) {
    int rc;
    const Lists L = contact_lists(*P, pt, npt, ee, nee, vg, nvg, dn, vids);
    const int64_t bound = chunk_bound(L, S);
    if (bound > INT32_MAX || K < 1 || K > kMaxTrials || !plan) return ABD_ERR_ARG;
    const int64_t *seg, *choff;
    double* part;
    if ((rc = get_plan(s, *sc, S, L, plan, &seg, &choff))) return rc;
    if ((rc = arena_get(kSlotReduce, sizeof(double) * (size_t)bound * K, (void**)&part))) return rc;
    // bytes: those of the candidates that some trial lists, counted on the device
    int ph = prof_start_ext(kProfEnergy, 1.0);
    // a workgroup's trials share its listing and fill its batches, but its threads evaluate
    // them in turn: two trials each, or one where the chunks leave the device fewer than
    // kTrialGrid workgroups.  The pass of twelve trials in 3, 4, 6 and 12 groups: 78, 67, 58
    // and 58 us for 256 scenes with most candidates near; three frames of 256 scenes with few
    // near 18.6, 18.6, 18.65 and 19.2 ms (the listing repeated); a 1024-body pile's 7.87,
    // 7.85, 7.80 and 7.82 ms
    const int64_t most = std::max<int64_t>(6, kTrialGrid / bound);
    const unsigned groups = (unsigned)std::min<int64_t>(K, most);
    prof_launch(ph, trial_chunk_kernel, dim3((unsigned)bound, groups), dim3(kRedThreads), 0, s, *sc, *P,
                TrialArgs{alpha, st}, L, S, K, seg, choff, part, bound);
    ABD_CHECK_LAUNCH();
    if ((rc = attach_trial_bytes(ph, s, *sc, L, S, K, alpha, seg, choff, bound))) return rc;
    *out = TrialSums{choff, part, bound};
    return ABD_OK;
}

namespace {

bool scenes_ok(const AbdScene* sc) { return sc && sc->n_scenes > 0 && sc->scene_boff && sc->body_scene; }

int energy_impl(abd_stream_t stream, const AbdScene* sc, const AbdParams* P, int S, const double* xk,
                const int32_t* pt, int64_t npt, const int32_t* ee, int64_t nee, const int32_t* vg, int64_t nvg,
                double* E) {
    if (!P || !xk || !E || npt < 0 || nee < 0 || nvg < 0 || P->psd < 0 || P->psd > 3) return ABD_ERR_ARG;
    if ((npt && !pt) || (nee && !ee) || (nvg && !vg)) return ABD_ERR_ARG;
    return contact_energy(to_stream(stream), sc, P, S, xk, pt, npt, ee, nee, vg, nvg, nullptr, E);
}

}  // namespace

int contact_energy(hipStream_t s, const AbdScene* sc, const AbdParams* P, int S, const double* xk, const int32_t* pt,
                   int64_t npt, const int32_t* ee, int64_t nee, const int32_t* vg, int64_t nvg, const int64_t* dn,
                   double* E) {
    const Lists L = contact_lists(*P, pt, npt, ee, nee, vg, nvg, dn);
    return seg_reduce(s, *sc, *P, S, xk, L, E, kProfEnergy);
}

int sweep_toi(hipStream_t s, const AbdScene* sc, const AbdParams* P, int S, const double* x_t0, const double* x_t1,
              const int32_t* pt, int64_t npt, const int32_t* ee, int64_t nee, const int64_t* dn, CandSide side,
              const KeepSweep& W, int64_t* plan, double* toi, double* first_alpha, const SceneDots& dots, int K,
              const double* A, const double* p, const double* dq, const double* A0, const double* p0,
              const double* Adot, const double* pdot, double* st, double* e) {
    const Lists L = contact_lists(*P, pt, npt, ee, nee, nullptr, 0, nullptr, side);
    SweepPlan Q;
    Q.scnt = W.scnt;
    Q.dn = dn;
    Q.use[0] = W.use_ee;
    Q.use[1] = W.use_pt;
    Q.use[2] = W.use_vg;
    Q.plan = plan;
    int rc;
    if ((rc = toi_solve(s, *sc, S, x_t0, x_t1, L, W.queue, W.qcount, W.slots, true, Q))) return rc;
    const int64_t blocks = S + ceil_div((int64_t)sc->n_bodies * K, (int64_t)kRedThreads);
    if (blocks > INT32_MAX) return ABD_ERR_ARG;
    launch_kernel(search_start_kernel, dim3((unsigned)blocks), dim3(kRedThreads), 0, s, *sc, *P, S, K,
                  (const unsigned long long*)W.slots, W.active, toi, first_alpha, dots,
                  StateArgs{A, p, dq, A0, p0, Adot, pdot, st, e});
    ABD_CHECK_LAUNCH();
    return ABD_OK;
}

namespace {
int scene_toi(hipStream_t s, const AbdScene* sc, const AbdParams* P, int S, const double* x_t0, const double* x_t1,
              const int32_t* pt, int64_t npt, const int32_t* ee, int64_t nee, const int32_t* vg, int64_t nvg,
              double* toi) {
    if (!P || !x_t0 || !x_t1 || !toi || npt < 0 || nee < 0 || nvg < 0) return ABD_ERR_ARG;
    if ((npt && !pt) || (nee && !ee) || (nvg && !vg)) return ABD_ERR_ARG;
    const Lists L = contact_lists(*P, pt, npt, ee, nee, vg, nvg);  // abd.py:288-299
    return toi_reduce(s, *sc, *P, S, x_t0, x_t1, L, toi, nullptr);
}
}  // namespace

// ------------------------------------------------- allocation-free TOI scratch
// The fixed scratch of abd_toi_noalloc: the chunk plan (kNoAllocPlanElems int64), the scene
// slot and queue count, kNoAllocPartElems chunk partials and a queue of
// ABD_TOI_NOALLOC_MAX_CANDIDATES int32 (in doubles: 2 entries each).  In host code `scratch`
// names a host-side stand-in, not device memory: its device address is looked up once per
// device (noalloc_scratch) and only that address reaches kernels.
constexpr int64_t kNoAllocPlanElems = 64;
constexpr int64_t kNoAllocSlotElems = 64;
// chunks of every list at most: 3 + (all candidates in one list) / 2048, kToiSplit partials each
constexpr int64_t kNoAllocPartElems = kToiSplit * (8 + ABD_TOI_NOALLOC_MAX_CANDIDATES / kChunkItems);
constexpr int64_t kNoAllocQueueElems = ABD_TOI_NOALLOC_MAX_CANDIDATES / 2;
static __device__ __align__(256) double scratch[kNoAllocPlanElems + kNoAllocSlotElems + kNoAllocPartElems +
                                                kNoAllocQueueElems];

namespace {
constexpr int kNoAllocDevices = 64;
std::mutex g_noalloc_mu;
void* g_noalloc_ptr[kNoAllocDevices] = {};

// The device address of `scratch` on the current device (looked up on its first use there).
int noalloc_scratch(ReduceScratch* out) {
    int dev = -1;
    ABD_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kNoAllocDevices) return ABD_ERR_NODEVICE;
    std::lock_guard<std::mutex> lock(g_noalloc_mu);
    if (!g_noalloc_ptr[dev]) {
        void* p = nullptr;
        ABD_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        g_noalloc_ptr[dev] = p;
    }
    double* base = static_cast<double*>(g_noalloc_ptr[dev]);
    out->plan = reinterpret_cast<int64_t*>(base);
    out->slots = reinterpret_cast<unsigned long long*>(base + kNoAllocPlanElems);
    out->qcount = reinterpret_cast<int32_t*>(base + kNoAllocPlanElems + 1);
    out->part = base + kNoAllocPlanElems + kNoAllocSlotElems;
    out->part_cap = kNoAllocPartElems;
    out->queue = reinterpret_cast<int32_t*>(base + kNoAllocPlanElems + kNoAllocSlotElems + kNoAllocPartElems);
    out->queue_cap = ABD_TOI_NOALLOC_MAX_CANDIDATES;
    return ABD_OK;
}
static_assert(2 * kLists + 2 <= kNoAllocPlanElems, "one scene's plan fits the front of the scratch");
}  // namespace

}  // namespace abd

using namespace abd;

extern "C" {

int abd_contact_energy(abd_stream_t stream, const AbdScene* sc, const AbdParams* P, const double* xk,
                       const int32_t* pt, int64_t npt, const int32_t* ee, int64_t nee, const int32_t* vg, int64_t nvg,
                       double* E) {
    if (!sc) return ABD_ERR_ARG;
    return energy_impl(stream, sc, P, 1, xk, pt, npt, ee, nee, vg, nvg, E);
}

int abd_scene_contact_energy(abd_stream_t stream, const AbdScene* sc, const AbdParams* P, const double* xk,
                             const int32_t* pt, int64_t npt, const int32_t* ee, int64_t nee, const int32_t* vg,
                             int64_t nvg, double* E) {
    if (!scenes_ok(sc)) return ABD_ERR_ARG;
    return energy_impl(stream, sc, P, sc->n_scenes, xk, pt, npt, ee, nee, vg, nvg, E);
}

int abd_toi(abd_stream_t stream, const AbdScene* sc, const AbdParams* P, const double* x_t0, const double* x_t1,
            const int32_t* pt, int64_t npt, const int32_t* ee, int64_t nee, const int32_t* vg, int64_t nvg,
            double* toi) {
    if (!sc) return ABD_ERR_ARG;
    return scene_toi(to_stream(stream), sc, P, 1, x_t0, x_t1, pt, npt, ee, nee, vg, nvg, toi);
}

int abd_toi_noalloc(abd_stream_t stream, const AbdScene* sc, const AbdParams* P, const double* x_t0,
                    const double* x_t1, const int32_t* pt, int64_t npt, const int32_t* ee, int64_t nee,
                    const int32_t* vg, int64_t nvg, double* toi) {
    if (!sc || !P || !x_t0 || !x_t1 || !toi || npt < 0 || nee < 0 || nvg < 0) return ABD_ERR_ARG;
    if ((npt && !pt) || (nee && !ee) || (nvg && !vg)) return ABD_ERR_ARG;
    const Lists L = contact_lists(*P, pt, npt, ee, nee, vg, nvg);
    // before any device call
    if (L.l[0].n + L.l[1].n + L.l[2].n > ABD_TOI_NOALLOC_MAX_CANDIDATES) return ABD_ERR_CAPACITY;
    ReduceScratch scr;
    int rc = noalloc_scratch(&scr);
    if (rc) return rc;
    return toi_reduce(to_stream(stream), *sc, *P, 1, x_t0, x_t1, L, toi, &scr);
}

int abd_scene_toi(abd_stream_t stream, const AbdScene* sc, const AbdParams* P, const double* x_t0,
                  const double* x_t1, const int32_t* pt, int64_t npt, const int32_t* ee, int64_t nee,
                  const int32_t* vg, int64_t nvg, double* toi) {
    if (!scenes_ok(sc)) return ABD_ERR_ARG;
    return scene_toi(to_stream(stream), sc, P, sc->n_scenes, x_t0, x_t1, pt, npt, ee, nee, vg, nvg, toi);
}

int abd_dot(abd_stream_t stream, const double* a, const double* b, int64_t n, double* out) {
    if (n < 0 || (!a && n) || (!b && n) || !out) return ABD_ERR_ARG;
    launch_kernel(seg_dot_kernel, dim3(1), dim3(kRedThreads), 0, to_stream(stream), nullptr, n, a, b, out);
    ABD_CHECK_LAUNCH();
    return ABD_OK;
}

int abd_scene_dot(abd_stream_t stream, const AbdScene* sc, const double* a, const double* b, double* out) {
    if (!scenes_ok(sc) || !a || !b || !out) return ABD_ERR_ARG;
    launch_kernel(seg_dot_kernel, dim3(sc->n_scenes), dim3(kRedThreads), 0, to_stream(stream), sc->scene_boff,
                       (int64_t)0, a, b, out);
    ABD_CHECK_LAUNCH();
    return ABD_OK;
}

int abd_inertia_energy(abd_stream_t stream, const AbdScene* sc, const AbdParams* P, const double* Ak, const double* pk,
                       const double* A0, const double* p0, const double* Adot, const double* pdot, double* E) {
    if (!sc || !P || !Ak || !pk || !A0 || !p0 || !Adot || !pdot || !E) return ABD_ERR_ARG;
    launch_kernel(seg_inertia_kernel, dim3(1), dim3(kRedThreads), 0, to_stream(stream), nullptr, sc->n_bodies,
                       *P, sc->mass, sc->I0, Ak, pk, A0, p0, Adot, pdot, E);
    ABD_CHECK_LAUNCH();
    return ABD_OK;
}

int abd_scene_inertia_energy(abd_stream_t stream, const AbdScene* sc, const AbdParams* P, const double* Ak,
                             const double* pk, const double* A0, const double* p0, const double* Adot,
                             const double* pdot, double* E) {
    if (!scenes_ok(sc) || !P || !Ak || !pk || !A0 || !p0 || !Adot || !pdot || !E) return ABD_ERR_ARG;
    launch_kernel(seg_inertia_kernel, dim3(sc->n_scenes), dim3(kRedThreads), 0, to_stream(stream),
                       sc->scene_boff, sc->n_bodies, *P, sc->mass, sc->I0, Ak, pk, A0, p0, Adot, pdot, E);
    ABD_CHECK_LAUNCH();
    return ABD_OK;
}

}  // extern "C"
