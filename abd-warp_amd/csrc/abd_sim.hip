// abd_sim.hip — native frame driver: AffineBodySimulator.step (abd.py:212-276)
// run from C++ over the stage entry points of this library.  The candidate lists a
// Newton iteration filters from the candidate superset keep their sizes on the device
// (every launch sized by the superset's, which bound them), and line searches and
// convergence tests run on the device, so an iteration is one recorded graph (or its
// launches) and one wait, for the lists' sizes and the number of scenes still iterating.
// One scene is a batch of one: the same iteration.  The arithmetic is the same sequence
// of kernels as the Python mirror, so both give identical states.
#include <hip/hip_runtime.h>

#include <math.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "abd_block.h"
#include "abd_internal.h"
#include "abd_profile.h"

namespace abd {

namespace {

template <class T>
struct DevBuf {
    T* p = nullptr;
    size_t cap = 0;  // elements
    int reserve(size_t n) {
        if (n <= cap && p) return ABD_OK;
        if (capturing()) return ABD_ERR_CAPACITY;  // no allocation inside a recorded graph
        note_reallocation();
        size_t want = std::max<size_t>(n + n / 2, 64);
        if (p) {
            ABD_CHECK(hipDeviceSynchronize());
            ABD_CHECK(hipFree(p));
            p = nullptr;
        }
        const hipError_t e = hipMalloc((void**)&p, want * sizeof(T));
        if (e != hipSuccess) {
            p = nullptr;
            if (std::getenv("ABD_DEBUG_ERRORS"))
                std::fprintf(stderr, "abd: simulator buffer of %zu bytes not allocated\n", want * sizeof(T));
            return hip_failure(e, __FILE__, __LINE__, "hipMalloc");
        }
        cap = want;
        return ABD_OK;
    }
    void release() {  // teardown: a failure leaves nothing to recover
        if (p) (void)hipFree(p);
        p = nullptr;
        cap = 0;
    }
};

struct BoxBuf {
    DevBuf<float> lo, hi;
    int reserve(size_t n) {
        int rc = lo.reserve(3 * n);
        return rc ? rc : hi.reserve(3 * n);
    }
};

// Body pairs (ij sorted by (i, j), ji the same pairs sorted by (j, i)) and the PT / EE / VG
// candidate tuples of one set of boxes.  The counts are exact when the set was culled
// (exact: consumers take them from here); a set filtered on the device has its sizes at dn
// ([nij, nij, npt, nee, nvg], device) and the counts here bound them.
// With `vids`, the PT and EE tuples' scene vertex ids (4 each, CandSide) are kept beside them.
struct CandSet {
    DevBuf<int32_t> ij, ji, ptl, eel, vgl;
    DevBuf<int32_t> ptv, eev;
    DevBuf<float> apt, aee, avg;  // the candidates' apart_until (the swept set's)
    int64_t nij = 0, npt = 0, nee = 0, nvg = 0;
    bool exact = true;
    bool vids = false;
    const int64_t* dn = nullptr;
    const int64_t* counts() const { return exact ? nullptr : dn; }
    CandSide side() const {
        return CandSide{vids ? ptv.p : nullptr, vids ? eev.p : nullptr, apt.p, aee.p, avg.p};
    }
    int reserve_like(const CandSet& o, bool with_vids = false) {
        int rc = ij.reserve(2 * (size_t)o.nij + 2);
        if (!rc) rc = ji.reserve(2 * (size_t)o.nij + 2);
        if (!rc) rc = ptl.reserve(5 * (size_t)o.npt + 5);
        if (!rc) rc = eel.reserve(5 * (size_t)o.nee + 5);
        if (!rc) rc = vgl.reserve(2 * (size_t)o.nvg + 2);
        if (!rc && with_vids) rc = ptv.reserve(4 * (size_t)o.npt + 4);
        if (!rc && with_vids) rc = eev.reserve(4 * (size_t)o.nee + 4);
        return rc;
    }
    void release() {
        ij.release();
        ji.release();
        ptl.release();
        eel.release();
        vgl.release();
        ptv.release();
        eev.release();
        apt.release();
        aee.release();
        avg.release();
    }
};

// words of a recorded iteration's key (graph_key)
constexpr int kKeyWords = 5;

struct Sim {
    Arena arena;  // the stages' scratch during this simulator's calls
    AbdScene sc;
    AbdParams P;
    AbdSimState st;
    int nb, nv, ne, nf;
    BoxBuf body, tri, edge, pt;         // boxes of the last collision_set
    BoxBuf tbody;                       // swept body boxes (the primitives' are evaluated per entry)
    // the collision set at xk (gh, BSR structure) and the swept set of the last CCD step
    // (CCD, line search; the next iteration's collision set is filtered from it)
    CandSet col, sw;
    bool sw_valid = false;  // sw covers the current state (set by the CCD, cleared per frame)
    // candidate superset: the culling of the swept boxes of vertex ranges (a CCD step's two
    // ends widened by a skin); every later step whose two ends stay inside the ranges
    // takes its swept set from it by filtering instead of culling
    CandSet sup;
    BoxBuf sbody, stri, sedge, spt;  // the superset's boxes
    DevBuf<double> vlo, vhi;         // its vertex ranges
    DevBuf<uint8_t> body_on;         // body_end's
    DevBuf<float> ebox;              // body_end's, 8 per vertex
    bool ebox_ready = false;         // written by this iteration's step end (writes_ebox)
    DevBuf<uint32_t> kcnt;           // the filters' counters (sweep_words)
    unsigned long long* toi_slots = nullptr;  // the CCD's scratch (arena)
    int32_t *toi_qcount = nullptr, *toi_queue = nullptr;
    DevBuf<double> qref;             // the states they were made around
    DevBuf<double> rest_max, rest_ref;  // the bodies' rest extents and the rest positions then
    bool sup_valid = false;
    bool col_fresh = false;  // col (with its structure) is the collision set at the current x
    DevBuf<int32_t> row_ptr, cols, slots;
    DevBuf<double> blocks;
    DevBuf<double> scal;        // the residual of hessian_solve
    DevBuf<int32_t> iters;
    DevBuf<int64_t> dcount;     // culling totals gathered for one read-back
    DevBuf<int64_t> cnt;        // device sizes of the filtered sets (kCnt*), read back per iteration
    int64_t* hcnt = nullptr;    // pinned copy of cnt
    int64_t* hcount = nullptr;  // pinned list counts
    int64_t stats[10] = {};
    // per-scene device values (one scene: a batch of one)
    int ns = 1, max_scene_bodies = 0;
    DevBuf<double> sv;          // [kSv][ns]
    // the Newton / line-search state of every scene on the device (ls_pass_kernel): rows
    // of the current iteration (lcur) and of the next, so that a step redone from a
    // recomputed swept set repeats the same decisions
    DevBuf<uint8_t> lsflag;     // [kLfRows][ns]
    DevBuf<double> lsval;       // [kLvRows][ns]
    DevBuf<int32_t> lsit;       // [2][ns] Newton iterations of each scene in this frame
    // the Newton iteration recorded as a HIP graph and replayed while the launches it
    // holds stay valid (GraphKey); a key met for the first time runs eagerly, the second
    // time it is recorded
    bool graphs = true;
    bool solve_waits = false;  // the solver reads back between its launches: never recorded
    int64_t gcount[3] = {};  // iterations replayed, recorded (then replayed), launched eagerly
    hipGraphExec_t gexec = nullptr;
    uint64_t gkey[kKeyWords] = {}, gseen[kKeyWords] = {}, gfailed[kKeyWords] = {};
    int32_t* hiters = nullptr;  // pinned [ns]: the iteration counts read back at a frame's end
    std::vector<int32_t> scene_it;  // Newton iterations of each scene in the last frame
    // line-search candidates evaluated together: states, vertices and per-candidate scalars
    DevBuf<double> cand_alpha;      // [kLsSpec][ns]
    DevBuf<double> trial_st;        // [1 + kLsSpec][nb][12] the bodies' trial states
    DevBuf<double> trial_e;         // [1 + kLsSpec][nb] and inertia energies
    DevBuf<int64_t> plan;           // reduction plan of the swept candidate set (CCD + line search)
};

// Step lengths evaluated per line-search pass after the first: the trials alpha,
// alpha/2, ..., alpha/2^(kLsSpec-1) of the backtracking loop (abd.py:146-160), whose
// accept test depends only on each trial's own energy, so taking the first accepted
// trial of a pass gives exactly the sequential loop's step.
constexpr int kLsSpec = kMaxTrials;

// Trials a pass needs from step length a on: a, a/2, ... up to the first one below
// alpha_min, which the loop accepts whatever its energy (at most kLsSpec; a pass that
// ends above alpha_min is followed by another).  With alpha <= 1 and alpha_min = 1e-3
// one pass after the first always decides.
__host__ __device__ inline int trials_to_floor(double a, double alpha_min) {
    int k = 1;
    while (k < kLsSpec && !(a < alpha_min)) {
        a *= 0.5;
        ++k;
    }
    return k;
}

// per-scene value rows of Sim::sv
enum { kSvEc = 0, kSvEi, kSvToi, kSvQtg, kSvGtg, kSvAlpha, kSv };
// Sim::cnt: the collision set's sizes, the swept set's, the active contacts of the gh
// stage, the flag of a step leaving the superset's ranges, the batched line search's
// outputs (scenes iterating after this iteration, scenes still searching, trials of the
// second pass and of the next, the solver's iterations summed over the iterating scenes);
// the host's copy holds staging rows for the exact sizes of a culled collision set and of
// the superset after it
enum {
    kCntCol = 0,
    kCntSw = 8,
    kCntNact = 16,
    kCntRange = 17,
    kCntNewton = 18,
    kCntSearch = 19,
    kCntK1 = 20,
    kCntK2 = 21,
    kCntSolver = 22,
    kCntSup = 24,  // the candidate superset's sizes
    kCntLen = 32
};
// rows of Sim::lsflag (iterating: the current and the next iteration's; searching) and of
// Sim::lsval (E0: the current and the next); the next
// iteration's rows are copied over the current ones at the start of every iteration
// (body_start)
enum { kLfNewton = 0, kLfSearch = 2, kLfRows };
enum { kLvE0 = 0, kLvRows = 2 };

// The EE, PT and VG candidate lists of one set of boxes (culling.py:32-76), culled side
// by side so that their counts come back in two host synchronizations instead of five;
// the stages copy their totals into S.dcount, one read-back each.
int cull_lists(hipStream_t s, Sim& S, CandSet& C, const BoxBuf& body, const BoxBuf& pts, const BoxBuf& tris,
               const BoxBuf& edges) {
    PrimCull ce, cp;
    VgCull cv;
    const bool pairs = C.nij > 0;
    int64_t* dc = S.dcount.p;
    int rc;
    if (pairs) {
        if ((rc = prim_cull_begin(s, &S.sc, ABD_CULL_EE, C.ij.p, C.nij, edges.lo.p, edges.hi.p, edges.lo.p,
                                  edges.hi.p, 0, ce, dc + 0)))
            return rc;
        if ((rc = prim_cull_begin(s, &S.sc, ABD_CULL_PT, C.ij.p, C.nij, pts.lo.p, pts.hi.p, tris.lo.p, tris.hi.p, 1,
                                  cp, dc + 1)))
            return rc;
    }
    if ((rc = vg_cull_begin(s, &S.sc, body.lo.p, pts.lo.p, pts.hi.p, S.P.dhat, S.P.ground, cv, dc + 2))) return rc;
    int64_t* hv = S.hcount;
    if (pairs || cv.total) {
        ABD_CHECK(hipMemcpyAsync(hv, dc, 3 * sizeof(int64_t), hipMemcpyDeviceToHost, s));
        ABD_CHECK(hipStreamSynchronize(s));
    }
    const int64_t T_ee = pairs ? hv[0] : 0, T_pt = pairs ? hv[1] : 0;
    C.nvg = cv.total ? hv[2] : 0;
    if ((rc = C.vgl.reserve(2 * (size_t)C.nvg + 2))) return rc;
    if ((rc = vg_cull_fill(s, cv, C.vgl.p, (int64_t)(C.vgl.cap / 2), C.nvg))) return rc;
    C.nee = C.npt = 0;
    if (!pairs) return ABD_OK;
    if ((rc = prim_cull_count(s, ce, T_ee, dc + 3))) return rc;
    if ((rc = prim_cull_count(s, cp, T_pt, dc + 4))) return rc;
    if (T_ee || T_pt) {
        ABD_CHECK(hipMemcpyAsync(hv + 3, dc + 3, 2 * sizeof(int64_t), hipMemcpyDeviceToHost, s));
        ABD_CHECK(hipStreamSynchronize(s));
    }
    C.nee = T_ee ? hv[3] : 0;
    C.npt = T_pt ? hv[4] : 0;
    if ((rc = C.eel.reserve(5 * (size_t)C.nee + 5))) return rc;
    if ((rc = C.ptl.reserve(5 * (size_t)C.npt + 5))) return rc;
    if ((rc = prim_cull_fill(s, ce, C.eel.p, (int64_t)(C.eel.cap / 5), C.nee))) return rc;
    return prim_cull_fill(s, cp, C.ptl.p, (int64_t)(C.ptl.cap / 5), C.npt);
}

// Body pairs of C (with the (j, i) order when with_ji), then the BSR structure of the
// collision set when `structure`.
int body_pairs(hipStream_t s, Sim& S, CandSet& C, const BoxBuf& body, bool with_ji) {
    for (;;) {
        int64_t cnt = 0;
        int rc = cull_bodies(s, &S.sc, body.lo.p, body.hi.p, C.ij.p, with_ji ? C.ji.p : nullptr,
                             (int64_t)(C.ij.cap / 2), &cnt);
        if (rc == ABD_ERR_OVERFLOW) {
            if ((rc = C.ij.reserve(2 * (size_t)cnt))) return rc;
            if ((rc = C.ji.reserve(2 * (size_t)cnt))) return rc;
            continue;
        }
        if (rc) return rc;
        C.nij = cnt;
        break;
    }
    return ABD_OK;
}

// abd.py:240-243: the slot layout of the collision set's body pairs (its pair count on the
// device when the set was filtered)
int structure_of(hipStream_t s, Sim& S) {
    int rc;
    if ((rc = S.cols.reserve(S.nb + 2 * (size_t)S.col.nij))) return rc;
    if ((rc = S.slots.reserve(S.nb + 2 * (size_t)S.col.nij))) return rc;
    return bsr_structure(s, S.nb, S.col.ij.p, S.col.ji.p, S.col.nij, S.col.counts(), S.row_ptr.p, S.cols.p,
                         S.slots.p);
}

// abd.py:187-207 on the vertices xv (xk of the reference's compute_energy, or x = xk at the
// start of a Newton iteration).  The culled counts are exact; with `structure` they are also
// staged to the device row the filtered sets use, so that every consumer of the collision
// set reads its sizes there.
int collision_set(hipStream_t s, Sim& S, bool structure, const double* xv) {
    const double dh = S.P.dhat * 0.5;
    int rc;
    if ((rc = abd_body_boxes(s, &S.sc, xv, dh, S.body.lo.p, S.body.hi.p))) return rc;
    if ((rc = body_pairs(s, S, S.col, S.body, structure))) return rc;
    S.col.exact = true;
    if (structure && (rc = structure_of(s, S))) return rc;
    if ((rc = abd_prim_boxes(s, &S.sc, ABD_KIND_TRI, xv, 0.0, S.tri.lo.p, S.tri.hi.p))) return rc;
    if ((rc = abd_prim_boxes(s, &S.sc, ABD_KIND_EDGE, xv, dh, S.edge.lo.p, S.edge.hi.p))) return rc;
    if ((rc = abd_prim_boxes(s, &S.sc, ABD_KIND_POINT, xv, S.P.dhat, S.pt.lo.p, S.pt.hi.p))) return rc;
    if ((rc = cull_lists(s, S, S.col, S.body, S.pt, S.tri, S.edge))) return rc;
    if (structure) {
        // the pinned staging row is rewritten only after the next read-back of the iteration
        int64_t* h = S.hcnt + kCntLen;
        h[0] = h[1] = S.col.nij;
        h[2] = S.col.npt;
        h[3] = S.col.nee;
        h[4] = S.col.nvg;
        ABD_CHECK(hipMemcpyAsync(S.cnt.p + kCntCol, h, 5 * sizeof(int64_t), hipMemcpyHostToDevice, s));
        S.col.dn = S.cnt.p + kCntCol;
        S.col.exact = false;  // consumers read the staged sizes (equal to the counts here)
    }
    return ABD_OK;
}

// The collision set at the vertices xv = x(q) of the accepted step (with its structure)
// filtered from a set that holds every pair and candidate of it (the swept set of the last
// CCD step: q = q_prev - alpha dq lies on that step and the swept boxes contain the boxes at
// every point of it; or the candidate superset while xv lies inside its ranges).  The result
// is the culling's own (keep_from_superset); its sizes stay on the device.
int collision_from(hipStream_t s, Sim& S, const CandSet& W, const double* xv) {
    const double dh = S.P.dhat * 0.5;
    int rc;
    // S.body: the body boxes at xv; the primitive boxes of collision_set's dilations are
    // evaluated per entry of W by the filter: W holds far fewer entries than the scene has
    // primitives
    if ((rc = S.col.reserve_like(W))) return rc;
    const KeepInput in{W.ij.p, W.ji.p, W.ptl.p, W.eel.p, W.vgl.p, W.nij, W.npt, W.nee, W.nvg, W.counts(),
                       W.side()};
    const KeepBoxes bx{S.body.lo.p, S.body.hi.p, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
    const KeepOutput out{S.col.ij.p, S.col.ji.p, S.col.ptl.p, S.col.eel.p, S.col.vgl.p};
    // (the swept set's entries apart at the accepted step length are dropped first)
    const KeepAtX at{xv,   nullptr, S.P.dhat,
                     dh,   0.0,     &W == &S.sw ? S.sv.p + kSvAlpha * S.ns : nullptr,
                     S.ns > 1 ? S.sc.body_scene : nullptr};
    if ((rc = keep_from_superset(s, &S.sc, in, bx, S.P.dhat, S.P.ground, out, S.cnt.p + kCntCol, nullptr, false,
                                 &at, &W == &S.sw ? S.kcnt.p : nullptr)))
        return rc;
    S.col.nij = W.nij;
    S.col.npt = W.npt;
    S.col.nee = W.nee;
    S.col.nvg = W.nvg;
    S.col.dn = S.cnt.p + kCntCol;
    S.col.exact = false;
    return structure_of(s, S);
}
int collision_from_swept(hipStream_t s, Sim& S, const double* xv) { return collision_from(s, S, S.sw, xv); }

// Skin of the candidate superset's vertex ranges, in units of dhat: wide enough that the
// later Newton steps of a frame (and of the next frames while the scenes rest) stay inside,
// so that a batch of scenes, which reuses the superset only when all of them do, skips
// most cullings; 30 measured best among 2, 10, 30 and 100 on the 256-scene workload.
constexpr double kSkinOverDhat = 30.0;
double skin_of(const Sim& S) { return kSkinOverDhat * S.P.dhat; }
// What the range tests leave of it, far above the rounding of positions: a point of a step
// whose ends pass them is inside the ranges too.
double range_margin(const Sim& S) { return 1e-6 * skin_of(S); }

// A frame's first collision set: filtered from the candidate superset when the state lies
// inside its vertex ranges (boxes at any positions inside them lie inside its boxes, so the
// culling output is a subset of it), else culled.
int collision_at_frame_start(hipStream_t s, Sim& S, const double* xv) {
    if (S.sup_valid) {
        int rc;
        ABD_CHECK(hipMemsetAsync(S.dcount.p + 7, 0, sizeof(int64_t), s));
        if ((rc = within_ranges(s, 3 * (int64_t)S.nv, xv, S.vlo.p, S.vhi.p, range_margin(S), S.sc.x0, S.rest_ref.p,
                                S.dcount.p + 7))) return rc;
        ABD_CHECK(hipMemcpyAsync(S.hcount + 7, S.dcount.p + 7, sizeof(int64_t), hipMemcpyDeviceToHost, s));
        ABD_CHECK(hipStreamSynchronize(s));
        if (S.hcount[7] == 0) {
            if ((rc = abd_body_boxes(s, &S.sc, xv, 0.5 * S.P.dhat, S.body.lo.p, S.body.hi.p))) return rc;
            return collision_from(s, S, S.sup, xv);
        }
        S.sup_valid = false;  // the frame starts outside it (or with another rest shape)
    }
    return collision_set(s, S, true, xv);
}


// abd.py:170-185, with both ends of every box dilated as in collision_set: one candidate
// set per Newton iteration that holds both the CCD candidates of the step (a pair that
// collides at some t has overlapping boxes at t, inside these) and every candidate of a
// collision set at any point of the step (x - alpha dq, alpha in [0, 1]).  The CCD then
// finds the same time of impact as the reference's trajectory lists (extra pairs have no
// verified root), and the line search's energies need no re-culling: a pair missing from
// the collision set at x - alpha dq has boxes apart, hence distance >= dhat and a zero
// barrier, so only the order of the nonzero terms' partial sums changes.
// The set is the culling output of the step's swept boxes, taken by filtering the
// candidate superset (keep_from_superset: the same predicates), valid while both ends of
// the step lie inside the superset's vertex ranges (every vertex of every scene).  Launched
// only: the range test's flag (cnt[kCntRange]) comes back with the iteration's scalars, and
// a step that left the ranges is redone after swept_set_recull.  Without a superset the
// superset is culled first (swept_set_recull's path).  The range test itself runs with
// the step's end (step_end).
int swept_set_launch(hipStream_t s, Sim& S);

// n rounded up to a multiple of an eighth of its power of two (at least 64; 0 stays 0: an
// empty list is launched over nothing).
int64_t size_bound(int64_t n) {
    if (n <= 64) return n > 0 ? 64 : 0;
    int64_t step = 8;
    while (step * 16 <= n) step *= 2;
    return (n + step - 1) / step * step;
}

// The counters of the filters of an iteration, 0 before it: the collision set's, the swept
// set's, then its kept entries per list and scene; with the CCD's scratch for the superset.
int64_t filter_words(const Sim& S) { return (int64_t)keep_counters(S.sup.nij, S.sup.npt, S.sup.nee, S.sup.nvg); }
int64_t sweep_words(const Sim& S) { return 2 * filter_words(S) + kSweepLists * (int64_t)S.ns; }
int sweep_buffers(Sim& S) {
    int rc;
    if ((rc = S.kcnt.reserve((size_t)sweep_words(S)))) return rc;
    return toi_scratch(S.ns, S.sup.npt + S.sup.nee, &S.toi_slots, &S.toi_qcount, &S.toi_queue);
}
__global__ __launch_bounds__(kBlock) void sweep_reset_kernel(uint32_t* __restrict__ words, int64_t nwords,
                                                                 unsigned long long* __restrict__ slots, int ns,
                                                                 int32_t* __restrict__ qcount,
                                                                 int64_t* __restrict__ counters, int ncounters) {
    const int64_t i0 = blockIdx.x * (int64_t)kBlock + threadIdx.x, step = gridDim.x * (int64_t)kBlock;
    for (int64_t i = i0; i < nwords; i += step) words[i] = 0;
    for (int64_t i = i0; i < ns; i += step) slots[i] = 0x3FF0000000000000ull;  // 1.0
    if (i0 < ncounters) counters[i0] = 0;
    if (i0 == 0) *qcount = 0;
}
KeepSweep sweep_of(Sim& S) {
    KeepSweep W{};
    W.S = S.ns;
    W.active = S.lsflag.p + (size_t)kLfNewton * S.ns;
    W.body_on = S.body_on.p;
    W.body_scene = S.sc.body_scene;
    W.ground = S.P.ground;
    W.dhat = std::max(S.P.dhat, sqrt(S.P.d2hat));  // the boxes' dilation, the barrier's range
    W.queue = S.toi_queue;
    W.qcount = S.toi_qcount;
    W.slots = S.toi_slots;
    W.apt = S.sw.apt.p;
    W.aee = S.sw.aee.p;
    W.avg = S.sw.avg.p;
    W.scnt = S.kcnt.p + 2 * filter_words(S);
    W.use_pt = S.P.pt != 0;
    W.use_ee = S.P.ee != 0;
    W.use_vg = S.P.vg != 0;
    return W;
}

// The superset culled anew around the current step (its ends widened by the skin; host
// synchronizations for the culling counts), then the swept set filtered from it.
int swept_set_recull(hipStream_t s, Sim& S) {
    const double dh = S.P.dhat * 0.5;
    const AbdSimState& st = S.st;
    const int64_t n3 = 3 * (int64_t)S.nv;
    int rc;
    S.sup_valid = false;
    if ((rc = vertex_ranges(s, n3, st.x, st.xk, skin_of(S), S.vlo.p, S.vhi.p))) return rc;
    if ((rc = step_states(s, &S.sc, st.A, st.p, st.dq, S.lsflag.p + (size_t)kLfNewton * S.ns, S.qref.p))) return rc;
    if ((rc = rest_max(s, &S.sc, S.rest_max.p, S.rest_ref.p))) return rc;
    if ((rc = swept_boxes(s, &S.sc, -1, S.vlo.p, S.vhi.p, dh, S.sbody.lo.p, S.sbody.hi.p))) return rc;
    // with the (j, i) order: the swept set (and the collision sets after it) keep it
    if ((rc = body_pairs(s, S, S.sup, S.sbody, true))) return rc;
    if ((rc = swept_boxes(s, &S.sc, ABD_KIND_TRI, S.vlo.p, S.vhi.p, 0.0, S.stri.lo.p, S.stri.hi.p))) return rc;
    if ((rc = swept_boxes(s, &S.sc, ABD_KIND_EDGE, S.vlo.p, S.vhi.p, dh, S.sedge.lo.p, S.sedge.hi.p))) return rc;
    if ((rc = swept_boxes(s, &S.sc, ABD_KIND_POINT, S.vlo.p, S.vhi.p, S.P.dhat, S.spt.lo.p, S.spt.hi.p))) return rc;
    if ((rc = cull_lists(s, S, S.sup, S.sbody, S.spt, S.stri, S.sedge))) return rc;
    // the tuples' vertex ids, read by the filters and, carried into the swept set, by the CCD
    // and the line search (the superset serves many steps)
    if ((rc = S.sup.ptv.reserve(4 * (size_t)S.sup.npt + 4))) return rc;
    if ((rc = S.sup.eev.reserve(4 * (size_t)S.sup.nee + 4))) return rc;
    if ((rc = cand_vertex_ids(s, &S.sc, 0, S.sup.ptl.p, S.sup.npt, S.sup.ptv.p))) return rc;
    if ((rc = cand_vertex_ids(s, &S.sc, 1, S.sup.eel.p, S.sup.nee, S.sup.eev.p))) return rc;
    S.sup.vids = true;
    // its exact sizes to the device; from here the counts are bounds in steps of an eighth,
    // which size the launches and buffers of the sets filtered from it, so that an iteration
    // recorded for one superset replays for the next of about its size
    int64_t* h = S.hcnt + kCntLen + 8;  // rewritten only after the next recull's synchronizations
    h[0] = h[1] = S.sup.nij;
    h[2] = S.sup.npt;
    h[3] = S.sup.nee;
    h[4] = S.sup.nvg;
    ABD_CHECK(hipMemcpyAsync(S.cnt.p + kCntSup, h, 5 * sizeof(int64_t), hipMemcpyHostToDevice, s));
    S.sup.nij = size_bound(S.sup.nij);
    S.sup.npt = size_bound(S.sup.npt);
    S.sup.nee = size_bound(S.sup.nee);
    S.sup.nvg = size_bound(S.sup.nvg);
    S.sup.dn = S.cnt.p + kCntSup;
    S.sup.exact = false;
    S.sup_valid = true;
    // the filters' counters of the new sizes and the CCD's start values (an iteration that
    // starts with this superset has them from body_start)
    if ((rc = sweep_buffers(S))) return rc;
    const int64_t n = std::max<int64_t>(sweep_words(S), S.ns);
    launch_kernel(sweep_reset_kernel, dim3(grid_for(n, kBlock, 1024)), dim3(kBlock), 0, s, S.kcnt.p,
                       sweep_words(S), S.toi_slots, S.ns, S.toi_qcount, S.cnt.p + kCntNewton,
                       kCntSolver - kCntNewton + 1);
    ABD_CHECK_LAUNCH();
    return swept_set_launch(s, S);
}

int swept_set_launch(hipStream_t s, Sim& S) {
    const double dh = S.P.dhat * 0.5;
    const AbdSimState& st = S.st;
    int rc;
    if (!S.sup_valid) return swept_set_recull(s, S);
    // the swept body boxes come from the step's end (body_end); the primitives' are evaluated
    // by the filter per entry of the superset from both ends (far fewer entries than
    // primitives)
    if ((rc = S.sw.reserve_like(S.sup, S.sup.vids))) return rc;
    if ((rc = S.sw.apt.reserve((size_t)S.sup.npt + 1))) return rc;
    if ((rc = S.sw.aee.reserve((size_t)S.sup.nee + 1))) return rc;
    if ((rc = S.sw.avg.reserve((size_t)S.sup.nvg + 1))) return rc;
    const CandSet& W = S.sup;
    const KeepInput in{W.ij.p, W.ji.p, W.ptl.p, W.eel.p, W.vgl.p, W.nij, W.npt, W.nee, W.nvg, W.counts(),
                       W.side()};
    const KeepBoxes bx{S.tbody.lo.p, S.tbody.hi.p, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
    KeepOutput o{S.sw.ij.p, S.sw.ji.p, S.sw.ptl.p, S.sw.eel.p, S.sw.vgl.p};
    if (W.vids) {
        o.ptv = S.sw.ptv.p;
        o.eev = S.sw.eev.p;
    }
    KeepAtX at{st.x, st.xk, S.P.dhat, dh, 0.0};
    at.ebox = S.ebox_ready ? reinterpret_cast<const float4*>(S.ebox.p) : nullptr;
    const KeepSweep sweep = sweep_of(S);
    if ((rc = keep_from_superset(s, &S.sc, in, bx, S.P.dhat, S.P.ground, o, S.cnt.p + kCntSw, nullptr, false, &at,
                                 S.kcnt.p + filter_words(S), &sweep)))
        return rc;
    S.sw.nij = W.nij;
    S.sw.npt = W.npt;
    S.sw.nee = W.nee;
    S.sw.nvg = W.nvg;
    S.sw.dn = S.cnt.p + kCntSw;
    S.sw.exact = false;
    S.sw.vids = W.vids;
    S.sw_valid = true;
    return ABD_OK;
}

// The lists' sizes for the statistics (after the iteration's synchronization).
void count_stats(Sim& S) {
    const int64_t* h = S.hcnt;
    S.stats[1] += h[kCntCol + 2];
    S.stats[2] += h[kCntCol + 3];
    S.stats[3] += h[kCntCol + 4];
    S.stats[4] += h[kCntNact];
    S.stats[8] += h[kCntSw + 2];
    S.stats[9] += h[kCntSw + 3];
}

// ---------------------------------------------------------------- batched
// The independent scenes of a batch (or the one scene) advanced together: one launch per
// stage covers every scene, and each scene keeps its own Newton loop, step length and
// stopping test (abd.py:212-276).  A scene that has converged is masked out of the solve
// and takes zero-length steps.  The line searches and the stopping tests run on the
// device (ls_pass_kernel), so an iteration waits for the device once.

// The device rows of the Newton / line-search state for the current iteration.
struct LsDev {
    int ns;
    const uint8_t* newton;  // scenes iterating (the solver's mask of this iteration)
    uint8_t* newton_nxt;
    uint8_t* search;        // scenes whose line search has not accepted a trial
    const double* E0;       // energy at the iteration's start (abd.py:225)
    double* E0_nxt;
    double* dalpha;         // the accepted step length (0: a scene not iterating)
    const int32_t* it;      // Newton iterations of the frame so far
    int32_t* it_nxt;
    const double* qtg;      // q.g and g.g of the iteration (abd.py:148, 265)
    const double* gtg;
    const int32_t* iters;   // the solver's iterations
    int64_t* cnt;           // Sim::cnt
};

LsDev ls_dev(Sim& S) {
    const int ns = S.ns, c = 0, n = 1;
    LsDev L;
    L.ns = ns;
    L.newton = S.lsflag.p + (size_t)(kLfNewton + c) * ns;
    L.newton_nxt = S.lsflag.p + (size_t)(kLfNewton + n) * ns;
    L.search = S.lsflag.p + (size_t)kLfSearch * ns;
    L.E0 = S.lsval.p + (size_t)(kLvE0 + c) * ns;
    L.E0_nxt = S.lsval.p + (size_t)(kLvE0 + n) * ns;
    L.dalpha = S.sv.p + (size_t)kSvAlpha * ns;
    L.it = S.lsit.p + (size_t)c * ns;
    L.it_nxt = S.lsit.p + (size_t)n * ns;
    L.qtg = S.sv.p + (size_t)kSvQtg * ns;
    L.gtg = S.sv.p + (size_t)kSvGtg * ns;
    L.iters = S.iters.p;
    L.cnt = S.cnt.p;
    return L;
}

constexpr int kLsThreads = 256;

// One pass of a scene's line search (abd.py:146-160; the Armijo test as written, a trial
// below alpha_min accepted whatever its energy): the energies of this pass's trials alpha
// [K][ns] (negative: no further trial), one after the other up to the first that passes: the
// contact energy from the chunks' sums C, the inertia energy from the bodies' e [K][nb],
// each added as a reduction of its own would.  first: the pass of the first trial, over the
// iterating scenes (the others get step length 0).  A scene that takes a trial has its
// stopping test (abd.py:265-268: g.g < tol or the iteration cap) written to the next
// iteration's rows; one that does not has its next pass's trials written to alpha
// [kLsSpec][ns]: a, a/2, ... from half the last rejected trial down to the first below
// alpha_min (trials_to_floor), -1 past them and for the scenes not searching.  One workgroup
// per scene; the totals over the scenes are integers, added by atomics (zeroed before the
// first pass).
// M: trials of the pass at most (1 for the first).
template <int M>
__global__ __launch_bounds__(kLsThreads) void ls_pass_kernel(LsDev L, double c1, double alpha_min, double tol,
                                                              int max_iter, int first, int K,
                                                              double* __restrict__ alpha, TrialSums C,
                                                              const double* __restrict__ e,
                                                              const int32_t* __restrict__ sboff, int nb) {
    __shared__ double sh[M][2][kLsThreads / kWave];
    const int s = blockIdx.x, ns = L.ns, t = threadIdx.x;
    const bool searching = first ? L.newton[s] != 0 : L.search[s] != 0;  // uniform
    if (!searching) {
        if (first) {
            if (t < kLsSpec) alpha[(int64_t)t * ns + s] = -1.0;
            if (t == 0) {
                L.dalpha[s] = 0.0;
                L.search[s] = 0;
                L.E0_nxt[s] = L.E0[s];
                L.it_nxt[s] = L.it[s];
                L.newton_nxt[s] = 0;
            }
        }
        return;
    }
    const int b0 = sboff ? sboff[s] : 0, b1 = sboff ? sboff[s + 1] : nb;
    const int64_t c0 = C.choff[s], c1_ = C.choff[s + 1];
    const double e0 = L.E0[s], qtg = L.qtg[s];
    // the trials' sums side by side, then one barrier for all (one trial after the other, with
    // its loads' latency and two barriers each, the second pass of 1024 bodies took 20 us; 10.5
    // here)
    double al[M], ec[M], ei[M];
#pragma unroll
    for (int k = 0; k < M; ++k) {
        al[k] = k < K ? alpha[(int64_t)k * ns + s] : -1.0;
        ec[k] = ei[k] = 0.0;
    }
    int nk = 0;  // this scene's trials
#pragma unroll
    for (int k = 0; k < M; ++k)
        if (nk == k && al[k] >= 0.0) nk = k + 1;
    // (a trial past nk reads the first one's: the loads have no branch and issue together)
    for (int64_t i = c0 + t; i < c1_; i += kLsThreads) {
        double v[M];
#pragma unroll
        for (int k = 0; k < M; ++k) v[k] = C.part[k < nk ? C.stride * k + i : i];
#pragma unroll
        for (int k = 0; k < M; ++k) ec[k] += v[k];
    }
    for (int b = b0 + t; b < b1; b += kLsThreads) {
        double v[M];
#pragma unroll
        for (int k = 0; k < M; ++k) v[k] = e[k < nk ? (int64_t)nb * k + b : b];
#pragma unroll
        for (int k = 0; k < M; ++k) ei[k] += v[k];
    }
#pragma unroll
    for (int k = 0; k < M; ++k)
        if (k < nk) {  // uniform
            const double wc = wave_sum(ec[k]), wi = wave_sum(ei[k]);
            if (lane_id() == 0) {
                sh[k][0][wave_id()] = wc;
                sh[k][1][wave_id()] = wi;
            }
        }
    __syncthreads();  // (and every thread has read this pass's trials)
    double last = 0.0, e1 = 0.0;
    bool acc = false;
#pragma unroll
    for (int k = 0; k < M; ++k)
        if (k < nk && !acc) {
            last = al[k];
            e1 = waves_sum(sh[k][0], kLsThreads / kWave) + waves_sum(sh[k][1], kLsThreads / kWave);
            const bool wolfe = e1 < e0 + c1 * last * qtg;
            acc = wolfe || last < alpha_min;
        }
    const double a0 = last * 0.5;  // the next pass's first trial
    const int need = acc ? 0 : trials_to_floor(a0, alpha_min);
    if (t < kLsSpec) {
        double ak = a0;
        for (int k = 0; k < t; ++k) ak *= 0.5;
        alpha[(int64_t)t * ns + s] = t >= need ? -1.0 : ak;
    }
    if (t != 0) return;
    L.search[s] = acc ? 0 : 1;
    unsigned long long* cnt = reinterpret_cast<unsigned long long*>(L.cnt);
    if (!acc) {
        if (first) atomicAdd(cnt + kCntSearch, 1ull);
        atomicMax(cnt + (first ? kCntK1 : kCntK2), (unsigned long long)need);
        return;
    }
    if (!first) atomicAdd(cnt + kCntSearch, ~0ull);  // one less
    const int32_t itn = L.it[s] + 1, si = L.iters[s];
    const uint8_t nn = (L.gtg[s] < tol || itn >= max_iter) ? 0 : 1;
    L.dalpha[s] = last;
    L.E0_nxt[s] = e1;
    L.it_nxt[s] = itn;
    L.newton_nxt[s] = nn;
    if (nn) atomicAdd(cnt + kCntNewton, 1ull);
    if (si > 0) atomicAdd(cnt + kCntSolver, (unsigned long long)si);
}

// A frame's start: E0 = the energy at q0 (abd.py:224-225), every scene iterating, no
// iterations yet.
__global__ __launch_bounds__(kLsThreads) void ls_frame_start_kernel(int ns, const double* __restrict__ Ec,
                                                                     const double* __restrict__ Ei,
                                                                     double* __restrict__ E0,
                                                                     uint8_t* __restrict__ newton,
                                                                     int32_t* __restrict__ it) {
    for (int s = blockIdx.x * kLsThreads + threadIdx.x; s < ns; s += gridDim.x * kLsThreads) {
        E0[s] = Ec[s] + Ei[s];
        newton[s] = 1;
        it[s] = 0;
    }
}

// q_gets_q0 (abd.py:124-128): q = (Ak, pk) = q0, and the accepted step lengths 0.
__global__ __launch_bounds__(kLsThreads) void frame_state_kernel(int nb, int ns, const double* __restrict__ A0,
                                                                  const double* __restrict__ p0,
                                                                  double* __restrict__ A, double* __restrict__ p,
                                                                  double* __restrict__ Ak, double* __restrict__ pk,
                                                                  double* __restrict__ dalpha) {
    const int i = blockIdx.x * kLsThreads + threadIdx.x;
    if (i < 9 * nb) A[i] = Ak[i] = A0[i];
    if (i < 3 * nb) p[i] = pk[i] = p0[i];
    if (i < ns) dalpha[i] = 0.0;
}

// A frame's start: q = q0 and the energies there (abd.py:224-225), sv rows Ec, Ei
int frame_start_scenes(hipStream_t s, Sim& S) {
    int rc;
    const AbdSimState& st = S.st;
    const int ns = S.ns;
    launch_kernel(frame_state_kernel, dim3(grid_for(std::max(9 * (int64_t)S.nb, (int64_t)ns), kLsThreads, INT32_MAX)),
                       dim3(kLsThreads), 0, s, S.nb, ns, st.A0, st.p0, st.A, st.p, st.Ak, st.pk,
                       S.sv.p + kSvAlpha * ns);
    ABD_CHECK_LAUNCH();
    if ((rc = abd_project_vertices(s, &S.sc, st.Ak, st.pk, st.xk))) return rc;
    // xk = x: the first Newton iteration's collision set too, with its structure
    if ((rc = collision_at_frame_start(s, S, st.xk))) return rc;
    S.col_fresh = true;
    const CandSet& C = S.col;
    if ((rc = contact_energy(s, &S.sc, &S.P, ns, st.xk, C.ptl.p, C.npt, C.eel.p, C.nee, C.vgl.p, C.nvg, C.counts(),
                             S.sv.p + kSvEc * ns)))
        return rc;
    if (ns > 1)
        rc = abd_scene_inertia_energy(s, &S.sc, &S.P, st.Ak, st.pk, st.A0, st.p0, st.Adot, st.pdot,
                                      S.sv.p + kSvEi * ns);
    else
        rc = abd_inertia_energy(s, &S.sc, &S.P, st.Ak, st.pk, st.A0, st.p0, st.Adot, st.pdot, S.sv.p + kSvEi);
    if (rc) return rc;
    S.stats[5] += 1;
    return ABD_OK;
}

// One line-search pass over every scene: the energies at q - alpha dq of the K trials (their
// states from trial k0 of trial_st on) over the swept candidate set of this iteration, and
// the scenes' decisions
int line_pass(hipStream_t s, Sim& S, const LsDev& L, bool first, int K, int k0) {
    int rc;
    const int64_t nb = S.nb;
    TrialSums C;
    if ((rc = line_chunks(s, &S.sc, &S.P, S.ns, K, S.cand_alpha.p, S.trial_st.p + 12 * nb * k0, S.sw.ptl.p, S.sw.npt,
                          S.sw.eel.p, S.sw.nee, S.sw.vgl.p, S.sw.nvg, S.plan.p, S.sw.counts(), S.sw.side(), &C)))
        return rc;
    launch_kernel(K == 1 ? ls_pass_kernel<1> : ls_pass_kernel<kLsSpec>, dim3(S.ns), dim3(kLsThreads), 0, s, L, S.P.c1,
                  S.P.alpha_min, S.P.tol, (int)S.P.max_iter, first ? 1 : 0, K, S.cand_alpha.p, C,
                       (const double*)(S.trial_e.p + nb * k0), S.ns > 1 ? S.sc.scene_boff : nullptr, S.nb);
    ABD_CHECK_LAUNCH();
    return ABD_OK;
}

// The trial states of K trials into trial_st from trial k0 on
int pass_states(hipStream_t s, Sim& S, int K, int k0) {
    const AbdSimState& st = S.st;
    const int64_t nb = S.nb;
    return trial_states(s, &S.sc, &S.P, S.ns, K, S.cand_alpha.p, st.A, st.p, st.dq, st.A0, st.p0, st.Adot,
                        st.pdot, S.trial_st.p + 12 * nb * k0, S.trial_e.p + nb * k0);
}

int read_counts(hipStream_t s, Sim& S) {
    ABD_CHECK(hipMemcpyAsync(S.hcnt, S.cnt.p, kCntLen * sizeof(int64_t), hipMemcpyDeviceToHost, s));
    ABD_CHECK(hipStreamSynchronize(s));
    return ABD_OK;
}

// Whether an iteration's step end writes the vertices' boxes: they cost 10 ns per 1000 vertices
// there and save the swept filter 6 ns per 1000 EE entries of the superset.  A function of the
// size bounds that a recorded iteration is replayed for, so the same for its replays; a step
// that leaves the ranges is filtered again from what its own iteration wrote.
bool writes_ebox(const Sim& S) { return S.sup_valid && S.sup.nee >= 2 * (int64_t)S.nv; }

// The end of the step (xk = x(q - dq) for the scenes in `active`), the swept body boxes and
// the range test against the superset's ranges when there is a superset (a vertex outside
// writes 1 over the 0 of body_start).
int step_end_scenes(hipStream_t s, Sim& S, const uint8_t* active) {
    const AbdSimState& st = S.st;
    BodyEnd U{};
    U.A = st.A;
    U.p = st.p;
    U.dq = st.dq;
    U.active = active;
    U.ns = S.ns;
    U.x = st.xk;
    U.dil = 0.5 * S.P.dhat;
    U.blo = S.body.lo.p;
    U.bhi = S.body.hi.p;
    U.slo = S.tbody.lo.p;
    U.shi = S.tbody.hi.p;
    if (S.sup_valid) {
        U.lo = S.vlo.p;
        U.hi = S.vhi.p;
        U.qref = S.qref.p;
        U.rest_max = S.rest_max.p;
    }
    U.skin = skin_of(S);
    U.margin = range_margin(S);
    U.flag = S.cnt.p + kCntRange;
    U.on = S.body_on.p;
    U.ebox = S.ebox_ready ? reinterpret_cast<float4*>(S.ebox.p) : nullptr;
    return body_end(s, &S.sc, U);
}

// The swept set's TOI (from its filter's slots and queue), q.g and g.g, and both line-search
// passes with their decisions, then the counts' read-back (launched; the caller waits).
int ccd_and_search_scenes(hipStream_t s, Sim& S, const LsDev& L) {
    const AbdSimState& st = S.st;
    const AbdParams& P = S.P;
    const int ns = S.ns;
    const CandSet& W = S.sw;
    int rc;
    // the TOI of the scenes still iterating and from it the first trial's step lengths; in the
    // same final pass q.g and g.g of the Armijo and stopping tests (abd.py:148,265: g and dq
    // are final here)
    SceneDots qg;
    qg.sboff = ns > 1 ? S.sc.scene_boff : nullptr;
    qg.n = 12 * (int64_t)S.sc.n_bodies;
    qg.a = st.dq;
    qg.b = st.g;
    qg.c = st.g;
    qg.d = st.g;
    qg.out1 = S.sv.p + kSvQtg * ns;
    qg.out2 = S.sv.p + kSvGtg * ns;
    if ((rc = sweep_toi(s, &S.sc, &P, ns, st.x, st.xk, W.ptl.p, W.npt, W.eel.p, W.nee, W.counts(), W.side(),
                        sweep_of(S), S.plan.p, S.sv.p + kSvToi * ns, S.cand_alpha.p, qg,
                        1 + kLsSpec, st.A, st.p, st.dq, st.A0, st.p0, st.Adot, st.pdot, S.trial_st.p, S.trial_e.p)))
        return rc;
    // the line search: the first trial, then every remaining halving of the scenes that
    // rejected it, each decided on the device
    if ((rc = line_pass(s, S, L, true, 1, 0))) return rc;
    if ((rc = line_pass(s, S, L, false, kLsSpec, 1))) return rc;
    return copy_to_host(s, S.hcnt, S.cnt.p, kCntLen * sizeof(int64_t));
}

// One Newton iteration of every scene up to the read-back of its counts (abd.py:224-271): the last
// iteration's accepted steps applied, then collision set, gradient and Hessian, solve, step
// end with the range test, swept set, TOI and line search.  With no host branch on device
// values, the same launches every time for the same sizes: the form a HIP graph records.
int iteration_scenes(hipStream_t s, Sim& S) {
    const AbdSimState& st = S.st;
    const AbdParams& P = S.P;
    const int nb = S.nb, ns = S.ns;
    const LsDev L = ls_dev(S);
    int rc;
    // q and (Ak, pk) = the accepted trial of every scene (step length 0: an exact copy), the
    // rows committed, x and its body boxes, the inertia terms, the off-diagonal slots zeroed
    const int64_t nij = S.col_fresh ? S.col.nij : S.sw.nij;
    if ((rc = S.blocks.reserve((nb + 2 * (size_t)nij) * 144))) return rc;
    BodyStart U{};
    U.alpha = L.dalpha;
    U.A = st.A;
    U.p = st.p;
    U.Ak = st.Ak;
    U.pk = st.pk;
    U.dq = st.dq;
    U.x = st.x;
    U.dil = 0.5 * P.dhat;
    U.lo = S.body.lo.p;
    U.hi = S.body.hi.p;
    U.A0 = st.A0;
    U.p0 = st.p0;
    U.Adot = st.Adot;
    U.pdot = st.pdot;
    U.g = st.g;
    U.blocks = S.blocks.p;
    U.zero = S.blocks.p + 144 * (int64_t)nb;
    U.nzero = 2 * 144 * nij;
    // contact_gh's flags and counters, over the collision set it will take
    const CandSet& Wn = S.col_fresh ? S.col : S.sw;
    void* ghz;
    if ((rc = gh_zero_region(nb, nij, Wn.npt + Wn.nee, &ghz, &U.nzero2))) return rc;
    U.zero2 = static_cast<double*>(ghz);
    if (S.sup_valid) {  // (else the superset's culling sets them)
        if ((rc = sweep_buffers(S))) return rc;
        U.zero32 = S.kcnt.p;
        U.nzero32 = sweep_words(S);
        U.slots = S.toi_slots;
        U.qcount = S.toi_qcount;
    }
    U.counters = S.cnt.p + kCntNewton;
    U.ncounters = kCntSolver - kCntNewton + 1;
    U.ns = ns;
    U.newton = S.lsflag.p + (size_t)kLfNewton * ns;
    U.E0 = S.lsval.p + (size_t)kLvE0 * ns;
    U.it = S.lsit.p;
    U.range_flag = S.cnt.p + kCntRange;
    if ((rc = body_start(s, &S.sc, &P, U))) return rc;
    // the collision set at x: the frame start's (the same positions), else from the last
    // iteration's swept set
    if (S.col_fresh)
        S.col_fresh = false;
    else if ((rc = collision_from_swept(s, S, st.x)))
        return rc;
    const CandSet& C = S.col;
    const GhLists GL{C.ptl.p, C.npt, C.eel.p, C.nee, C.vgl.p, C.nvg, C.nij, C.counts()};
    if ((rc = contact_gh(s, &S.sc, &P, st.x, GL, S.row_ptr.p, S.slots.p, st.g, S.blocks.p, nullptr, nullptr,
                         S.cnt.p + kCntNact, true, ns > 1 ? S.max_scene_bodies : 0)))
        return rc;
    if (ns > 1)
        rc = abd_bsr_solve_scenes(s, P.solver, &S.sc, S.max_scene_bodies, S.row_ptr.p, S.cols.p, S.slots.p,
                                  S.blocks.p, st.g, st.dq, P.solver_tol, P.solver_maxiter, 10, L.newton, S.iters.p,
                                  nullptr);
    else
        rc = abd_bsr_solve(s, P.solver, nb, S.row_ptr.p, S.cols.p, S.slots.p, S.blocks.p, st.g, st.dq, P.solver_tol,
                           P.solver_maxiter, 10, S.iters.p, nullptr);
    if (rc) return rc;
    // CCD over the full steps of the scenes still iterating (abd.py:278-303)
    if ((rc = step_end_scenes(s, S, L.newton))) return rc;
    if ((rc = swept_set_launch(s, S))) return rc;
    return ccd_and_search_scenes(s, S, L);
}

// What a recorded iteration depends on besides device values: the candidate superset's
// size bounds (they size every launch), the scratch pointers and the culling tiles.
void graph_key(const Sim& S, uint64_t key[kKeyWords]) {
    const AbdTuning t = tuning();
    key[0] = (uint64_t)S.sup.nij << 32 | (uint64_t)S.sup.nvg;
    key[1] = (uint64_t)S.sup.npt;
    key[2] = (uint64_t)S.sup.nee;
    key[3] = alloc_generation();
    key[4] = ((uint64_t)(uint32_t)t.cull_chunk << 32) | (uint32_t)t.cull_grid;
}
bool same_key(const uint64_t a[kKeyWords], const uint64_t b[kKeyWords]) {
    return !memcmp(a, b, kKeyWords * sizeof(uint64_t));
}

// Records iteration_scenes into S.gexec (updated in place when the topology allows); nothing
// runs.  A failure leaves no error state behind, and the caller launches the iteration instead.
int record_iteration(hipStream_t s, Sim& S) {
    hipGraph_t g = nullptr;
    const hipError_t ce = hipGraphCreate(&g, 0);
    if (ce != hipSuccess) {
        (void)hipGetLastError();
        return -static_cast<int>(ce);
    }
    graph_record(g);
    int rc = iteration_scenes(s, S);
    const int node_rc = graph_record_end();
    if (!rc) rc = node_rc;
    if (rc) {
        (void)hipGraphDestroy(g);
        (void)hipGetLastError();
        return rc;
    }
    if (S.gexec) {
        hipGraphNode_t err_node = nullptr;
        hipGraphExecUpdateResult res;
        if (hipGraphExecUpdate(S.gexec, g, &err_node, &res) != hipSuccess || res != hipGraphExecUpdateSuccess) {
            (void)hipGetLastError();
            (void)hipGraphExecDestroy(S.gexec);
            S.gexec = nullptr;
        }
    }
    hipError_t ie = hipSuccess;
    if (!S.gexec) ie = hipGraphInstantiate(&S.gexec, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (ie != hipSuccess) {
        S.gexec = nullptr;
        (void)hipGetLastError();
        return -static_cast<int>(ie);
    }
    return ABD_OK;
}

int step_scenes(hipStream_t s, Sim& S) {
    const AbdSimState& st = S.st;
    const AbdParams& P = S.P;
    const int nb = S.nb, ns = S.ns;
    int rc;
    double* dalpha = S.sv.p + kSvAlpha * ns;
    S.sw_valid = false;  // a frame starts from the state the caller holds
    if ((rc = frame_start_scenes(s, S))) return rc;
    {
        // the first iteration's rows, taken over by its body_start_kernel
        const LsDev L = ls_dev(S);
        launch_kernel(ls_frame_start_kernel, dim3((unsigned)ceil_div(ns, kLsThreads)), dim3(kLsThreads), 0, s,
                           ns, (const double*)(S.sv.p + kSvEc * ns), (const double*)(S.sv.p + kSvEi * ns), L.E0_nxt,
                           L.newton_nxt, L.it_nxt);
        ABD_CHECK_LAUNCH();
    }
    int64_t n_active = ns;
    while (n_active > 0) {
        const LsDev L = ls_dev(S);
        S.ebox_ready = writes_ebox(S);  // launched or replayed
        // a steady iteration (collision set from the last swept set, superset kept) replays
        // its recorded graph; the first time a key is met the iteration runs eagerly, the
        // second time it is recorded (every buffer then holds its size for these launches)
        const bool steady =
            S.graphs && !S.solve_waits && S.sw_valid && !S.col_fresh && S.sup_valid && !prof_enabled();
        uint64_t key[kKeyWords];
        graph_key(S, key);
        bool ran = false;
        if (steady && S.gexec && same_key(key, S.gkey)) {
            ABD_CHECK(hipGraphLaunch(S.gexec, s));
            ran = true;
            ++S.gcount[0];
        } else if (steady && same_key(key, S.gseen) && !same_key(key, S.gfailed)) {
            if (record_iteration(s, S) == ABD_OK) {
                ABD_CHECK(hipGraphLaunch(S.gexec, s));
                memcpy(S.gkey, key, sizeof(key));
                ran = true;
                ++S.gcount[1];
            } else {
                memcpy(S.gfailed, key, sizeof(key));  // this key runs eagerly
            }
        }
        if (!ran) {
            ++S.gcount[2];
            if ((rc = iteration_scenes(s, S))) return rc;
            if (steady) {
                graph_key(S, key);  // the eager run may have grown buffers
                memcpy(S.gseen, key, sizeof(key));
            }
        }
        ABD_CHECK(hipStreamSynchronize(s));
        if (S.hcnt[kCntRange] != 0) {
            // the step left the superset's ranges: the swept set (and all after it) again from
            // a superset culled around this very step, which holds it
            if ((rc = swept_set_recull(s, S))) return rc;
            if ((rc = ccd_and_search_scenes(s, S, L))) return rc;
            ABD_CHECK(hipStreamSynchronize(s));
        }
        count_stats(S);
        S.stats[5] += 1 + S.hcnt[kCntK1];
        // further passes: only when alpha_min lies more than kLsSpec halvings below a first trial
        while (S.hcnt[kCntSearch] > 0) {
            const int64_t K = S.hcnt[kCntK2];
            if ((rc = zero_fill(s, S.cnt.p + kCntK2, sizeof(int64_t)))) return rc;
            if ((rc = pass_states(s, S, kLsSpec, 1))) return rc;
            if ((rc = line_pass(s, S, L, false, kLsSpec, 1))) return rc;
            if ((rc = read_counts(s, S))) return rc;
            S.stats[5] += K;
        }
        S.stats[0] += n_active;
        S.stats[6] += S.hcnt[kCntSolver];
        n_active = S.hcnt[kCntNewton];
    }
    if ((rc = update_q_scenes_dual(s, &S.sc, st.A, st.p, st.dq, dalpha, st.A, st.p, st.Ak, st.pk))) return rc;
    if ((rc = abd_update_q0qdot(s, nb, P.dt, st.A, st.p, st.A0, st.p0, st.Adot, st.pdot))) return rc;
    if ((rc = abd_project_vertices(s, &S.sc, st.A0, st.p0, st.x_view))) return rc;
    ABD_CHECK(hipMemcpyAsync(S.hiters, S.lsit.p + ns, sizeof(int32_t) * ns, hipMemcpyDeviceToHost, s));
    ABD_CHECK(hipStreamSynchronize(s));
    S.scene_it.assign(S.hiters, S.hiters + ns);
    S.stats[7] += 1;
    return ABD_OK;
}

}  // namespace

}  // namespace abd

using namespace abd;

extern "C" {

int abd_sim_create(const AbdScene* scene, const AbdParams* params, const AbdSimState* state, void** out) {
    if (!scene || !params || !state || !out || scene->n_bodies <= 0) return ABD_ERR_ARG;
    if (params->psd < 0 || params->psd > 3) return ABD_ERR_ARG;
    Sim* S = new (std::nothrow) Sim();
    if (!S) return ABD_ERR_ARG;
    S->sc = *scene;
    S->P = *params;
    S->st = *state;
    S->nb = scene->n_bodies;
    S->nv = scene->n_verts;
    S->ne = scene->n_edges;
    S->nf = scene->n_tris;
    int rc = 0;
    const size_t nb = S->nb;
    BoxBuf* b4[] = {&S->body, &S->tbody};
    for (BoxBuf* b : b4)
        if (!rc) rc = b->reserve(nb);
    if (!rc) rc = S->tri.reserve(S->nf + 1);
    if (!rc) rc = S->edge.reserve(S->ne + 1);
    if (!rc) rc = S->pt.reserve(S->nv);
    if (!rc) rc = S->sbody.reserve(nb);
    if (!rc) rc = S->stri.reserve(S->nf + 1);
    if (!rc) rc = S->sedge.reserve(S->ne + 1);
    if (!rc) rc = S->spt.reserve(S->nv);
    if (!rc) rc = S->vlo.reserve(3 * (size_t)S->nv + 3);
    if (!rc) rc = S->vhi.reserve(3 * (size_t)S->nv + 3);
    if (!rc) rc = S->qref.reserve(24 * nb);
    if (!rc) rc = S->rest_max.reserve(3 * nb);
    if (!rc) rc = S->rest_ref.reserve(3 * (size_t)S->nv + 3);
    if (!rc) rc = S->body_on.reserve(nb);
    if (!rc) rc = S->ebox.reserve(8 * (size_t)S->nv + 8);
    for (CandSet* C : {&S->col, &S->sw, &S->sup}) {
        if (!rc) rc = C->ij.reserve(2 * 256);
        if (!rc) rc = C->ji.reserve(2 * 256);
        if (!rc) rc = C->ptl.reserve(5 * 4096);
        if (!rc) rc = C->eel.reserve(5 * 4096);
        if (!rc) rc = C->vgl.reserve(2 * 1024);
    }
    if (!rc) rc = S->row_ptr.reserve(nb + 1);
    if (!rc) rc = S->cols.reserve(nb + 512);
    if (!rc) rc = S->slots.reserve(nb + 512);
    if (!rc) rc = S->blocks.reserve((nb + 512) * 144);
    if (!rc) rc = S->scal.reserve(1);
    if (!rc && hipHostMalloc((void**)&S->hcount, 8 * sizeof(int64_t), hipHostMallocDefault) != hipSuccess)
        rc = ABD_ERR_ARG;
    {
        const int nsc = scene->n_scenes > 1 ? scene->n_scenes : 1;
        if (!rc) rc = S->cand_alpha.reserve((size_t)nsc * kLsSpec);
        if (!rc) rc = S->trial_st.reserve(12 * nb * (1 + kLsSpec));
        if (!rc) rc = S->trial_e.reserve(nb * (1 + kLsSpec));
        if (!rc) rc = S->plan.reserve(reduce_plan_elems(nsc));
        if (!rc) rc = S->dcount.reserve(8);
        if (!rc) rc = S->cnt.reserve(kCntLen);
        if (!rc && hipMemset(S->cnt.p, 0, sizeof(int64_t) * S->cnt.cap) != hipSuccess) rc = ABD_ERR_ARG;
        if (!rc && hipHostMalloc((void**)&S->hcnt, 2 * kCntLen * sizeof(int64_t), hipHostMallocDefault) != hipSuccess)
            rc = ABD_ERR_ARG;
        if (!rc) rc = S->sv.reserve((size_t)kSv * nsc);
        if (!rc) rc = S->lsflag.reserve((size_t)kLfRows * nsc);
        if (!rc) rc = S->lsval.reserve((size_t)kLvRows * nsc);
        if (!rc) rc = S->lsit.reserve(2 * (size_t)nsc);
        if (!rc) rc = S->iters.reserve(nsc);
        if (!rc && hipHostMalloc((void**)&S->hiters, sizeof(int32_t) * nsc, hipHostMallocDefault) != hipSuccess)
            rc = ABD_ERR_ARG;
    }
    if (!rc && scene->n_scenes > 1) {
        // scene ranges from the host copy of scene_boff
        const int ns = scene->n_scenes;
        std::vector<int32_t> sb(ns + 1);
        if (!scene->scene_boff || !scene->body_scene ||
            hipMemcpy(sb.data(), scene->scene_boff, sizeof(int32_t) * (ns + 1), hipMemcpyDeviceToHost) != hipSuccess)
            rc = ABD_ERR_ARG;
        for (int k = 0; !rc && k < ns; ++k) {
            if (sb[k + 1] < sb[k]) rc = ABD_ERR_ARG;
            S->max_scene_bodies = std::max(S->max_scene_bodies, sb[k + 1] - sb[k]);
        }
        if (!rc && (sb[0] != 0 || sb[ns] != scene->n_bodies)) rc = ABD_ERR_ARG;
        S->ns = ns;
    }
    S->solve_waits = S->ns == 1 && solve_waits(params->solver, scene->n_bodies);
    if (rc) {
        abd_sim_destroy(S);
        return rc;
    }
    *out = S;
    return ABD_OK;
}

int abd_sim_step(void* sim, abd_stream_t stream, int64_t* stats) {
    if (!sim) return ABD_ERR_ARG;
    Sim& S = *static_cast<Sim*>(sim);
    ArenaScope scope(&S.arena);
    const int rc = step_scenes(to_stream(stream), S);
    if (stats)
        for (int k = 0; k < 10; ++k) stats[k] = S.stats[k];
    return rc;
}

int abd_sim_hessian_solve(void* sim, abd_stream_t stream, int32_t method, double tol, int32_t maxiter,
                          const double* rhs, double* y, int32_t* iters, double* resid) {
    if (!sim || !rhs || !y) return ABD_ERR_ARG;
    if (method != ABD_SOLVER_BICGSTAB && method != ABD_SOLVER_CG_JACOBI && method != ABD_SOLVER_CG_BLOCK)
        return ABD_ERR_ARG;
    Sim& S = *static_cast<Sim*>(sim);
    if (S.ns > 1) return ABD_ERR_ARG;
    ArenaScope scope(&S.arena);
    hipStream_t s = to_stream(stream);
    const AbdSimState& st = S.st;
    int rc;
    // the Newton matrix of abd.py:230-243 at q = (A, p), contacts from x(q)
    if ((rc = abd_project_vertices(s, &S.sc, st.A, st.p, st.x))) return rc;
    if ((rc = collision_set(s, S, true, st.x))) return rc;
    const size_t nslot = S.nb + 2 * (size_t)S.col.nij;
    if ((rc = S.blocks.reserve(nslot * 16 * 9))) return rc;
    ABD_CHECK(hipMemsetAsync(S.blocks.p, 0, sizeof(double) * nslot * 16 * 9, s));
    ABD_CHECK(hipMemsetAsync(st.g, 0, sizeof(double) * 12 * S.nb, s));
    if ((rc = abd_inertia_hessian(s, &S.sc, &S.P, st.A, S.blocks.p))) return rc;
    int64_t nact = 0;
    if ((rc = abd_contact_gh(s, &S.sc, &S.P, st.x, S.col.ptl.p, S.col.npt, S.col.eel.p, S.col.nee, S.col.vgl.p, S.col.nvg, S.col.nij,
                             S.row_ptr.p, S.slots.p, st.g, S.blocks.p, nullptr, &nact)))
        return rc;
    ABD_CHECK(hipMemsetAsync(y, 0, sizeof(double) * 12 * S.nb, s));
    if ((rc = abd_bsr_solve(s, method, S.nb, S.row_ptr.p, S.cols.p, S.slots.p, S.blocks.p, rhs, y, tol, maxiter, 10,
                            S.iters.p, S.scal.p)))
        return rc;
    if (iters) ABD_CHECK(hipMemcpyAsync(iters, S.iters.p, sizeof(int32_t), hipMemcpyDeviceToHost, s));
    if (resid) ABD_CHECK(hipMemcpyAsync(resid, S.scal.p, sizeof(double), hipMemcpyDeviceToHost, s));
    ABD_CHECK(hipStreamSynchronize(s));
    return ABD_OK;
}

int abd_sim_autotune(void* sim, abd_stream_t stream, AbdTuning* chosen) {
    if (!sim) return ABD_ERR_ARG;
    Sim& S = *static_cast<Sim*>(sim);
    ArenaScope scope(&S.arena);
    hipStream_t s = to_stream(stream);
    const AbdTuning saved = tuning();
    int rc;
    // the candidate lists at the current state (xk) are what every collision_set of a frame culls
    if ((rc = abd_project_vertices(s, &S.sc, S.st.Ak, S.st.pk, S.st.xk))) return rc;
    hipEvent_t e0, e1;
    ABD_CHECK(hipEventCreate(&e0));
    ABD_CHECK(hipEventCreate(&e1));
    AbdTuning best = saved;
    float best_ms = 1e30f;
    const int chunks[] = {1024, 2048, 4096, 8192, 16384};
    const int grids[] = {4096, 16384, 65536};
    for (int c : chunks)
        for (int g : grids) {
            AbdTuning t{c, g, saved.contact_bound_mib, saved.pair_grid, saved.toi_grid};
            if ((rc = abd_set_tuning(&t))) break;
            float ms_min = 1e30f;
            for (int rep = 0; rep < 3 && !rc; ++rep) {
                hipError_t he = hipEventRecord(e0, s);
                if (he != hipSuccess) {
                    rc = -static_cast<int>(he);
                    break;
                }
                rc = collision_set(s, S, false, S.st.xk);
                if (!rc && (he = hipEventRecord(e1, s)) != hipSuccess) rc = -static_cast<int>(he);
                float ms = 0.f;
                if (!rc && hipEventSynchronize(e1) == hipSuccess && hipEventElapsedTime(&ms, e0, e1) == hipSuccess)
                    ms_min = ms < ms_min ? ms : ms_min;
            }
            if (rc) break;
            if (ms_min < best_ms) {
                best_ms = ms_min;
                best = t;
            }
        }
    // stage D's grid, with the chosen tiles: the contact Hessian of the collision set at this
    // state (its structure built once), best of three per grid; g and the Hessian slots are
    // scratch that the next iteration rewrites
    if (!rc && (rc = abd_set_tuning(&best)) == ABD_OK && (rc = collision_set(s, S, true, S.st.xk)) == ABD_OK) {
        const size_t nslot = S.sc.n_bodies + 2 * (size_t)S.col.nij;
        rc = S.blocks.reserve(nslot * 16 * 9);
        const CandSet& C = S.col;
        const GhLists L{C.ptl.p, C.npt, C.eel.p, C.nee, C.vgl.p, C.nvg, C.nij, C.counts()};
        // one or two rounds of the workgroups the device holds at once (four a CU): larger
        // grids, and smaller ones, measured faster on an early frame's few contacts and slower
        // on the later frames' many
        const int pgrids[] = {1024, 2048};
        float bestp = 1e30f;
        int32_t pbest = best.pair_grid;
        for (int pg : pgrids) {
            if (rc) break;
            AbdTuning t = best;
            t.pair_grid = pg;
            if ((rc = abd_set_tuning(&t))) break;
            float ms_min = 1e30f;
            for (int rep = 0; rep < 3 && !rc; ++rep) {
                hipError_t he = hipEventRecord(e0, s);
                if (he != hipSuccess) {
                    rc = -static_cast<int>(he);
                    break;
                }
                rc = contact_gh(s, &S.sc, &S.P, S.st.xk, L, S.row_ptr.p, S.slots.p, S.st.g, S.blocks.p, nullptr,
                                nullptr, S.cnt.p + kCntNact);
                if (!rc && (he = hipEventRecord(e1, s)) != hipSuccess) rc = -static_cast<int>(he);
                float ms = 0.f;
                if (!rc && hipEventSynchronize(e1) == hipSuccess && hipEventElapsedTime(&ms, e0, e1) == hipSuccess)
                    ms_min = ms < ms_min ? ms : ms_min;
            }
            if (!rc && ms_min < bestp) {
                bestp = ms_min;
                pbest = pg;
            }
        }
        best.pair_grid = pbest;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    abd_set_tuning(rc ? &saved : &best);
    if (rc) return rc;
    if (chosen) *chosen = best;
    return ABD_OK;
}

int abd_sim_set_graphs(void* sim, int32_t on) {
    if (!sim) return ABD_ERR_ARG;
    static_cast<Sim*>(sim)->graphs = on != 0;
    return ABD_OK;
}

int abd_sim_graph_counts(void* sim, int64_t* counts) {
    if (!sim || !counts) return ABD_ERR_ARG;
    const Sim& S = *static_cast<Sim*>(sim);
    for (int k = 0; k < 3; ++k) counts[k] = S.gcount[k];
    return ABD_OK;
}

int abd_sim_scene_iters(void* sim, int32_t* iters) {
    if (!sim || !iters) return ABD_ERR_ARG;
    const Sim& S = *static_cast<Sim*>(sim);
    for (int k = 0; k < S.ns; ++k) iters[k] = k < (int)S.scene_it.size() ? S.scene_it[k] : 0;
    return ABD_OK;
}

int abd_sim_destroy(void* sim) {
    if (!sim) return ABD_OK;
    Sim* S = static_cast<Sim*>(sim);
    (void)hipDeviceSynchronize();  // queued work may still use the buffers released below
    if (S->gexec) (void)hipGraphExecDestroy(S->gexec);
    (void)arena_free(S->arena);
    for (BoxBuf* b : {&S->body, &S->tri, &S->edge, &S->pt, &S->tbody, &S->sbody,
                      &S->stri, &S->sedge, &S->spt}) {
        b->lo.release();
        b->hi.release();
    }
    S->col.release();
    S->sw.release();
    S->sup.release();
    S->vlo.release();
    S->vhi.release();
    S->qref.release();
    S->kcnt.release();
    S->body_on.release();
    S->ebox.release();
    S->rest_max.release();
    S->rest_ref.release();
    S->row_ptr.release();
    S->cols.release();
    S->slots.release();
    S->blocks.release();
    S->scal.release();
    S->iters.release();
    S->sv.release();
    S->lsflag.release();
    S->lsval.release();
    S->lsit.release();
    S->trial_st.release();
    S->trial_e.release();
    S->cand_alpha.release();
    S->plan.release();
    S->dcount.release();
    S->cnt.release();
    for (void* h : {(void*)S->hcount, (void*)S->hcnt, (void*)S->hiters})
        if (h) (void)hipHostFree(h);
    delete S;
    return ABD_OK;
}

}  // extern "C"
