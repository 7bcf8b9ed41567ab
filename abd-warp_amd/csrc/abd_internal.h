// abd_internal.h — host-side internals shared by the libabd_hip.so translation
// units: error handling, the per-device scratch arena, and launchers of the
// generic scan / reduction kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <tuple>

#include "../../include/abd_hip.h"

namespace abd {

// The error code of a failed HIP call (-hipError_t); with ABD_DEBUG_ERRORS set in the
// environment it also prints the call's site and the runtime's message to stderr.
int hip_failure(hipError_t e, const char* file, int line, const char* expr);
#define ABD_CHECK(expr)                                                                  \
    do {                                                                                 \
        hipError_t _e = (expr);                                                          \
        if (_e != hipSuccess) return ::abd::hip_failure(_e, __FILE__, __LINE__, #expr); \
    } while (0)
#define ABD_CHECK_LAUNCH() ABD_CHECK(hipGetLastError())

// A graph recorded by this thread: between graph_record(g) and graph_record_end() every
// launch_kernel and copy_to_host of the thread becomes the next node of g, one after the other,
// and nothing runs.  (Not a stream capture: while a stream of the process is captured the
// runtime refuses device synchronization, which any other thread may be doing.)
// graph_record_end: ABD_OK, or why a node could not be added; the graph then lacks it and all
// that followed, and must not run.
void graph_record(hipGraph_t g);
int graph_record_end();
bool capturing();
void graph_add_kernel(const void* f, dim3 grid, dim3 block, void** args, size_t lds);
int copy_to_host(hipStream_t s, void* dst, const void* src, size_t bytes);

// Launches f on s (a failure is hipGetLastError's), or records the launch (graph_record_end's).
template <typename... P, typename... A>
inline void launch_kernel(void (*f)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t s, A&&... a) {
    std::tuple<P...> vals(static_cast<P>(a)...);
    std::apply(
        [&](P&... v) {
            void* args[] = {(void*)&v...};
            if (capturing())
                graph_add_kernel((const void*)f, grid, block, args, lds);
            else
                (void)hipLaunchKernel((const void*)f, grid, block, args, lds, s);
        },
        vals);
}

inline hipStream_t to_stream(abd_stream_t s) { return reinterpret_cast<hipStream_t>(s); }

// Per-device scratch arena: `slots` independent growable device buffers plus a
// small pinned host buffer for count read-back.  Growing synchronizes the
// device first, so a buffer still in use by queued work is never freed early.
constexpr int kArenaSlots = 41;
enum ArenaSlot {
    kSlotScanA = 0,
    kSlotScanB,
    kSlotReduce,
    kSlotFlags,
    kSlotList,
    kSlotFilter,
    kSlotFilterCount,
    kSlotChunk,
    kSlotChunkCount,
    kSlotContact,
    kSlotMisc,
    kSlotSolver,
    kSlotSpare,
    kSlotSolveBytes,
    kSlotPlan,
    kSlotPrecond,
    // a second primitive-culling workspace (culls run side by side) and the VG culling's
    kSlotFilterB,
    kSlotFilterCountB,
    kSlotScanBB,
    kSlotChunkCountB,
    kSlotChunkB,
    kSlotVgA,
    kSlotVgB,
    kSlotKeep,     // keep_from_superset: block counts and offsets
    kSlotKeepMap,  // keep_from_superset: old -> new pair index
    kSlotKeepCount,
    kSlotLdlt,        // direct solve: the factors of the systems
    kSlotLdltStatus,  // direct solve: per-system status when the caller takes no iteration counts
    kSlotPairChunk,   // contact stage D: per-pair work-item counts and offsets
    kSlotPairPart,    // contact stage D: the work items' partial sums
    kSlotKeepFlags,   // keep_from_superset: each entry's predicate
    kSlotToiQueue,    // CCD: the candidates whose cubic has a bracketed root
    kSlotToiSlots,    // CCD: per-scene minima of the queued candidates and the queue count
    kSlotProfBytes,   // profiling: algorithmic byte counts computed on the device
};
// Launch shapes that change no result (abd_set_tuning); process-wide.
AbdTuning tuning();
// Staged culling (abd_cull.hip): begin / count / fill leave their counts on the device
// (total_chunks, total_pairs, total) so several cullings share one host synchronization;
// `set` 0 or 1 picks one of two independent workspaces.
struct PrimSets {
    const int32_t* off1;  // per-body offsets of set 1 (PT points / EE edges)
    const int32_t* off2;  // set 2 (PT triangles / EE edges)
    const float *lo1, *hi1, *lo2, *hi2;
};
struct PrimCull {
    int set = 0, pt = 0;
    const int32_t* ij = nullptr;
    PrimSets S{};
    int64_t nunits = 0, maxs = 0, T = 0;
    int32_t* flist = nullptr;
    int64_t *fcnt = nullptr, *choff = nullptr, *ccnt = nullptr, *ccoff = nullptr;
    const int64_t* total_chunks = nullptr;  // device, after begin
    const int64_t* total_pairs = nullptr;   // device, after count
    AbdTuning tune{};
    unsigned grid = 0;
};
struct VgCull {
    const AbdScene* sc = nullptr;
    const float *blo = nullptr, *plo = nullptr, *phi = nullptr;
    double yth = 0.0;
    float fg = 0.f;
    int64_t nblk = 0;
    int64_t *bcnt = nullptr, *boff = nullptr;
    const int64_t* total = nullptr;  // device, after begin
};
// total_copy (device, nullable): a second place for the stage's total, so that a caller
// can gather the totals of several cullings into one buffer and read them with one copy.
int prim_cull_begin(hipStream_t s, const AbdScene* sc, int mode, const int32_t* ij, int64_t nij, const float* lo1,
                    const float* hi1, const float* lo2, const float* hi2, int set, PrimCull& C,
                    int64_t* total_copy = nullptr);
int prim_cull_count(hipStream_t s, PrimCull& C, int64_t T, int64_t* total_copy = nullptr);
int prim_cull_fill(hipStream_t s, PrimCull& C, int32_t* out, int64_t cap, int64_t n);
int vg_cull_begin(hipStream_t s, const AbdScene* sc, const float* blo, const float* plo, const float* phi, double dhat,
                  double ground, VgCull& C,
                  int64_t* total_copy = nullptr);
int vg_cull_fill(hipStream_t s, VgCull& C, int32_t* out, int64_t cap, int64_t n);

// Swept boxes dilated at both ends (kind ABD_KIND_*, or -1 for body boxes): the union of
// the dilated boxes at x0 and at x1.
int swept_boxes(hipStream_t s, const AbdScene* sc, int kind, const double* x0, const double* x1, double dil,
                float* lo, float* hi);
// Vertex ranges of a candidate superset (n3 = 3 * vertices): lo = min(x0, x1) - skin,
// hi = max(x0, x1) + skin per coordinate.  Boxes of any positions inside these ranges
// lie inside the swept boxes of (lo, hi) (every box formula is monotone in the
// positions), so their culling output is a subset of that superset's.
int vertex_ranges(hipStream_t s, int64_t n3, const double* x0, const double* x1, double skin, double* lo,
                  double* hi);
// *flag (device, 0 before) becomes 1 when some coordinate of x leaves [lo + margin, hi - margin],
// or of the rest positions r differs from r0.
int within_ranges(hipStream_t s, int64_t n3, const double* x, const double* lo, const double* hi, double margin,
                  const double* r, const double* r0, int64_t* flag);
// dn (here and below, nullable): the lists' sizes on the device, [nij, nij, npt, nee, nvg],
// the counts passed then bounding them.
// What a candidate set keeps beside its tuples (each nullable): the scene vertex ids of each
// PT / EE candidate (4 per tuple, in the order fetch_pt_idx / fetch_ee_idx give them), so
// that a kernel reads them instead of gathering them through the topology; and of each PT /
// EE / VG candidate the step length below which it stays inactive on the step last passed to
// whose CCD was taken (apart_until), written by the filter (KeepSweep) and read by line_chunks and the next filter.
struct CandSide {
    const int32_t* pt = nullptr;
    const int32_t* ee = nullptr;
    float* apart_pt = nullptr;
    float* apart_ee = nullptr;
    float* apart_vg = nullptr;
};
// Line-search trials q - alpha dq of at most kMaxTrials lengths at once (S = 1: the whole
// system as one scene).  trial_states: the bodies' states st [K][nb][12] (16-byte aligned)
// and inertia energies e [K][nb] at alpha [K][S] (device); a negative length is skipped.  line_chunks: the chunks' contact energies at alpha [K][S]
// (negative: 0) over a planned set, scene s's at trial k part[stride k + choff[s] ..
// choff[s + 1]) in the order their sum is taken.
constexpr int kMaxTrials = 12;
struct TrialSums {
    const int64_t* choff;
    const double* part;
    int64_t stride;
};
int trial_states(hipStream_t s, const AbdScene* sc, const AbdParams* P, int S, int K, const double* alpha,
                 const double* A, const double* p, const double* dq, const double* A0, const double* p0,
                 const double* Adot, const double* pdot, double* st, double* e);
int line_chunks(hipStream_t s, const AbdScene* sc, const AbdParams* P, int S, int K, const double* alpha,
                const double* st, const int32_t* pt, int64_t npt, const int32_t* ee, int64_t nee, const int32_t* vg,
                int64_t nvg, const int64_t* plan, const int64_t* dn, CandSide vids, TrialSums* out);
// The per-scene chunk plan of the energy reductions over one set of candidate lists: its size
// (int64); the swept set's is made by its filter (KeepSweep).
size_t reduce_plan_elems(int S);
// Per-scene dot products a.b and c.d (each seg_dot_kernel's) that the TOI's final per-scene
// pass computes after the scene's TOI when out1 is set (the driver's q.g and g.g).
struct SceneDots {
    const int32_t* sboff = nullptr;
    int64_t n = 0;
    const double *a = nullptr, *b = nullptr, *c = nullptr, *d = nullptr;
    double *out1 = nullptr, *out2 = nullptr;
};
// The line search's first step length from a TOI (abd.py:300-302): clamped to [0, 1], x 0.9
// below 1.  sweep_toi's first_alpha (device, nullable) receives it per scene (-1 for the
// scenes not active).
__host__ __device__ inline double first_step_length(double t) {
    t = t < 1.0 ? t : 1.0;  // std::min(1.0, t)
    t = 0.0 < t ? t : 0.0;  // std::max(0.0, t)
    if (t < 1.0) t *= 0.9;
    return t;
}
// The per-body passes of an iteration (abd_body.hip).  body_start: the accepted step lengths
// alpha [ns] taken (A, p in place, Ak, pk alike), x, the body boxes at x dilated by dil, the
// inertia gradient and the diagonal Hessian slots (both written), the scenes' rows
// committed (row 1 of newton, E0, it over row 0), *range_flag and the words zeroed.
struct BodyStart {
    const double* alpha;
    double *A, *p, *Ak, *pk;
    const double* dq;
    double* x;
    double dil;
    float *lo, *hi;
    const double *A0, *p0, *Adot, *pdot;
    double *g, *blocks;
    double* zero;  // nzero words zeroed
    int64_t nzero;
    double* zero2;  // nzero2 more
    int64_t nzero2;
    uint32_t* zero32;  // nzero32 more, of 4 bytes
    int64_t nzero32;
    unsigned long long* slots;  // [ns] set to 1.0
    int32_t* qcount;            // set to 0
    int64_t* counters;          // ncounters set to 0
    int ncounters;
    int ns;
    uint8_t* newton;
    double* E0;
    int32_t* it;
    int64_t* range_flag;
};
// Whether a body's workgroup is one wave (abd_body.hip).
bool small_bodies(const AbdScene* sc);
int body_start(hipStream_t s, const AbdScene* sc, const AbdParams* P, const BodyStart& U);
// body_end: x = x(q - dq) of the scenes in active (x(q) of the others), the union (slo, shi)
// of the body boxes there and blo, bhi; with lo, hi the range test (margin inside them) into
// *flag, which bodies within skin - margin of qref [2][nb][12] (step_states of the step the
// ranges were made around) pass by their rest_max [nb][3].
struct BodyEnd {
    const double *A, *p, *dq;
    const uint8_t* active;
    int ns;
    double* x;
    double dil;
    const float *blo, *bhi;
    float *slo, *shi;
    const double *lo, *hi, *qref, *rest_max;
    double skin, margin;
    int64_t* flag;
    uint8_t* on;  // [nb] active of the body's scene
    float4* ebox;  // nullable: [nv][2] the vertices' boxes at both ends dilated by dil in FP64: lo, hi, 0, 0
};
int body_end(hipStream_t s, const AbdScene* sc, const BodyEnd& U);
// each body's largest |rest coordinate| per axis (out [nb][3]) and a copy of the rest positions
int rest_max(hipStream_t s, const AbdScene* sc, double* out, double* copy);
int step_states(hipStream_t s, const AbdScene* sc, const double* A, const double* p, const double* dq,
                const uint8_t* active, double* qref);
// abd_contact_energy (S = 1) / abd_scene_contact_energy with the lists' sizes on the device.
int contact_energy(hipStream_t s, const AbdScene* sc, const AbdParams* P, int S, const double* xk, const int32_t* pt,
                   int64_t npt, const int32_t* ee, int64_t nee, const int32_t* vg, int64_t nvg, const int64_t* dn,
                   double* E);
// Whether abd_bsr_solve of nb bodies waits for the device between its launches.
bool solve_waits(int32_t method, int nb);
// abd_update_q_scenes writing the result to a second state as well (when A_out2, p_out2 are given).
int update_q_scenes_dual(hipStream_t s, const AbdScene* sc, const double* A, const double* p, const double* dq,
                         const double* alpha, double* A_out, double* p_out, double* A_out2, double* p_out2);
// Collision set from a superset of it (keep_from_superset, abd_cull.hip): the superset's
// body pairs (ij, and ji when given), PT / EE / VG tuples, the current body / point /
// edge / triangle boxes; outputs sized like the inputs (no aliasing).  The five totals
// (nij, nij of ji, npt, nee, nvg) go to dcount (device) and, after one synchronization,
// to hcount (host, pinned).
// dn (nullable): the input sizes on the device in the output layout [nij, nij, npt, nee,
// nvg] (the counts here then bound them).
struct KeepInput {
    const int32_t *ij, *ji, *pt, *ee, *vg;
    int64_t nij, npt, nee, nvg;
    const int64_t* dn = nullptr;
    CandSide vids = {};  // the PT / EE tuples' vertex ids (nullable)
};
struct KeepBoxes {
    const float *blo, *bhi, *plo, *phi, *elo, *ehi, *tlo, *thi;
};
struct KeepOutput {
    int32_t *ij, *ji, *pt, *ee, *vg;
    int32_t *ptv = nullptr, *eev = nullptr;  // the kept tuples' vertex ids (when the input has them)
};
// The vertex ids of n PT (kind 0) or EE (kind 1) tuples into vid [n][4] (CandSide).
int cand_vertex_ids(hipStream_t s, const AbdScene* sc, int kind, const int32_t* tuples, int64_t n, int32_t* vid);
// The primitive boxes of the predicates computed per entry from the vertices x instead of
// read from KeepBoxes (whose point, edge and triangle boxes are then unused): the box
// kernels' own expressions, points (float)x -+ (float)pdil, edges and triangles the FP64
// min / max of their vertices -+ edil / tdil, cast to FP32; with x1 set, the swept boxes'
// (the union of the boxes at x and at x1).
// alpha (nullable): x is the state at step length alpha[scene] of the step the input's
// apart_* were written for; an entry apart at its scene's length is dropped unevaluated (its
// boxes there do not overlap).  body_scene null: one scene.
struct KeepAtX {
    const double *x, *x1;
    double pdil, edil, tdil;
    const double* alpha = nullptr;
    const int32_t* body_scene = nullptr;
    // swept (x1): the vertices' edge boxes at both ends (body_end's ebox), read for the EE
    // entries of an input with vertex ids in place of the positions (nullable)
    const float4* ebox = nullptr;
};
// The CCD of a step taken while its swept set is written (x, x1: the step's ends), over the
// scenes with active[s]: each kept PT / EE / VG entry's apart_until, the PT / EE entries whose
// cubic has a bracketed root queued as (output index << 1 | is EE), the VG entries' TOI min-ed
// into their scene's slot, and the kept entries per list (EE, PT, VG) and scene counted
// (S > 1), from which sweep_toi makes the reduction plan of the output lists.
constexpr int kSweepLists = 3;
struct KeepSweep {
    int S;
    const uint8_t* active;   // [S]
    const uint8_t* body_on;  // [nb], a body's scene's
    const int32_t* body_scene;
    double ground, dhat;
    int32_t* queue;
    int32_t* qcount;            // 0 before
    unsigned long long* slots;  // 1.0 before
    float *apt, *aee, *avg;     // apart_until beside the output lists
    uint32_t* scnt;             // [kSweepLists][S], 0 before
    int use_pt, use_ee, use_vg;  // a list switched off has no TOI
};
// Counters of a filter of lists of these sizes (uint32, an even number of them, 0 before it).
size_t keep_counters(int64_t nij, int64_t npt, int64_t nee, int64_t nvg);
// The arena's CCD scratch of a set of nq PT and EE candidates over S scenes.
int toi_scratch(int S, int64_t nq, unsigned long long** slots, int32_t** qcount, int32_t** queue);
// The reduction plan (int64 [reduce_plan_elems(S)]) of the lists a sweep wrote (dn: their
// sizes on the device in the keep layout; npt, nee bound them), the scene minima from the
// queued candidates, the first step lengths, the scenes' dots, and the states and inertia
// energies (trial_states') of K trials of the first lengths halved k times.
int sweep_toi(hipStream_t s, const AbdScene* sc, const AbdParams* P, int S, const double* x_t0, const double* x_t1,
              const int32_t* pt, int64_t npt, const int32_t* ee, int64_t nee, const int64_t* dn, CandSide side,
              const KeepSweep& W, int64_t* plan, double* toi, double* first_alpha, const SceneDots& dots, int K,
              const double* A, const double* p, const double* dq, const double* A0, const double* p0,
              const double* Adot, const double* pdot, double* st, double* e);
// sync false: the totals reach hcount with the stream's next synchronization (the caller's);
// hcount null: they stay on the device.
// counters (nullable): keep_counters words zeroed before (else the call zeroes its own).
int keep_from_superset(hipStream_t s, const AbdScene* sc, const KeepInput& in, const KeepBoxes& bx, double dhat,
                       double ground, const KeepOutput& out, int64_t* dcount, int64_t* hcount, bool sync = true,
                       const KeepAtX* at = nullptr, uint32_t* counters = nullptr, const KeepSweep* sweep = nullptr);
// abd_bsr_structure; dnij (nullable): the pair count on the device (nij bounds it; cols and
// slots hold nb + 2 nij entries).
int bsr_structure(hipStream_t s, int nb, const int32_t* ij, const int32_t* ji, int64_t nij, const int64_t* dnij,
                  int32_t* row_ptr, int32_t* cols, int32_t* slots);
// abd_cull_bodies without the (j, i) order when ji == nullptr.
int cull_bodies(hipStream_t s, const AbdScene* sc, const float* lo, const float* hi, int32_t* ij, int32_t* ji,
                int64_t cap, int64_t* count);
// The gh stage's candidate lists.  dn (nullable): their sizes on the device, [nij, nij,
// npt, nee, nvg]; the counts here are then upper bounds.
struct GhLists {
    const int32_t* pt;
    int64_t npt;
    const int32_t* ee;
    int64_t nee;
    const int32_t* vg;
    int64_t nvg;
    int64_t nij;
    const int64_t* dn;
};
// row_bodies: the bodies of the largest scene (0: not known, all bodies), which bound a row's pairs.
int contact_gh(hipStream_t s, const AbdScene* sc, const AbdParams* P, const double* x, const GhLists& L,
               const int32_t* row_ptr, const int32_t* slots, double* g, double* blocks, uint8_t* highlight,
               int64_t* n_active, int64_t* n_active_dev, bool zeroed = false, int row_bodies = 0);
// The words (8 bytes) that a contact_gh over these sizes wants 0; with them zeroed before it it
// runs with zeroed = true.
int gh_zero_region(int nb, int64_t nij, int64_t n, void** p, int64_t* words);
// A set of arena buffers.  The stateless entry points share one per device (process-wide);
// each simulator owns one, made the calling thread's arena by an ArenaScope for the length
// of a simulator call, so simulators stepped from different threads or streams never share
// scratch.
struct Arena {
    void* ptr[kArenaSlots] = {};
    size_t size[kArenaSlots] = {};
    void* host = nullptr;
    size_t host_size = 0;
};
class ArenaScope {
  public:
    explicit ArenaScope(Arena* a);
    ~ArenaScope();
    ArenaScope(const ArenaScope&) = delete;
    ArenaScope& operator=(const ArenaScope&) = delete;

  private:
    Arena* prev_;
};
int arena_get(int slot, size_t bytes, void** ptr);
int arena_host(size_t bytes, void** ptr);  // pinned host memory
int arena_release_current();
int arena_free(Arena& a);  // synchronizes the device, then releases every buffer of `a`
// A counter that every (re)allocation of library scratch advances: device pointers baked into
// a recorded HIP graph stay valid while it is unchanged.
uint64_t alloc_generation();
void note_reallocation();
// (While this thread records a graph, scratch that would have to grow returns
// ABD_ERR_CAPACITY instead of allocating.)
// Zeroes `bytes` (a multiple of 8, 8-byte aligned) with a kernel: a fill that may be recorded in
// a HIP graph (memset nodes are avoided there).
int zero_fill(hipStream_t s, void* p, size_t bytes);

// Exclusive scan of n int64 counts (device) in place into `out` (may alias),
// writing the total to *total (device).  Fixed-order, single workgroup passes.
int scan_exclusive_i64(hipStream_t s, const int64_t* in, int64_t* out, int64_t n, int64_t* total,
                       int64_t* total2 = nullptr);
// Several independent exclusive scans in one launch (one workgroup each, same order as
// scan_exclusive_i64); total2 nullable.
struct ScanSeg {
    const int64_t* in;
    int64_t* out;
    int64_t n;
    int64_t *total, *total2;
};
constexpr int kMaxScanSegs = 8;
int scan_exclusive_i64_multi(hipStream_t s, const ScanSeg* segs, int nseg);
// Copies one int64 from device to host (synchronizes `s`).
int read_i64(hipStream_t s, const int64_t* dev, int64_t* host);

constexpr int kBlock = 256;
inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }
inline unsigned grid_for(int64_t n, int block = kBlock, int64_t cap = 65535) {
    int64_t g = ceil_div(n, block);
    if (g < 1) g = 1;
    if (g > cap) g = cap;
    return static_cast<unsigned>(g);
}

}  // namespace abd
