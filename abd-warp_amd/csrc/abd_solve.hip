// abd_solve.hip — Newton linear solve over the body-block sparse matrix:
// unpreconditioned BiCGSTAB (abd.py:244, warp.optim.linear.bicgstab) and the
// Jacobi-preconditioned CG of bsr_utils.py:126-235.
//
// One workgroup runs the whole Krylov loop for one system: matrix and vectors in registers
// where they fit (RegSystem), else the vectors in LDS or the scratch arena; every dot product
// is a fixed-order reduction, and the stopping test is evaluated inside the kernel every
// `check_every` iterations, so a solve is one launch with no host round trips.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "abd_block.h"
#include "abd_internal.h"
#include "abd_profile.h"

namespace abd {

constexpr int kSolveThreads = 1024;
// The direct block LDL^T (ldlt_kernel) takes systems of up to kLdltMaxBodies bodies; it
// marks a system it declines with kLdltFailed in the iteration count, and the block-Jacobi
// CG that follows it solves exactly those.
constexpr int kLdltMaxBodies = 64;
constexpr int kLdltFailed = -2;
// LDS for a system's staged block structure (row offsets and (column, slot) entries).
constexpr size_t kLdsStructBytes = 24 * 1024;

struct Bsr {
    int nb;
    const int32_t* row_ptr;
    const int32_t* cols;
    const int32_t* slots;
    const double* blocks;
};

// One 12x12 block's row (ii, k) against 12 entries of a vector: the three-term sums of
// sub-blocks (ii, jj), jj = 0..3, added to acc in jj order.
__device__ __forceinline__ double block_row_add(double acc, const double (&B)[12], const double* __restrict__ xin) {
#pragma unroll
    for (int jj = 0; jj < 4; ++jj)
        acc += B[3 * jj] * xin[3 * jj] + B[3 * jj + 1] * xin[3 * jj + 1] + B[3 * jj + 2] * xin[3 * jj + 2];
    return acc;
}

__device__ __forceinline__ void load_block_row(const double* __restrict__ blocks, int64_t slot, int ii, int k,
                                               double (&B)[12]) {
    const double* base = blocks + 9 * 16 * slot + 3 * k;
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
        const double* Bj = base + 9 * (ii + 4 * jj);
        B[3 * jj] = Bj[0];
        B[3 * jj + 1] = Bj[1];
        B[3 * jj + 2] = Bj[2];
    }
}

// A system's block structure as its SpMV reads it: from the global CSR (columns outside
// the system filtered on the fly) or from an LDS copy made once per solve by stage_rows
// (local row offsets lrp, entries ent = (local column or -1, slot)), which takes two
// dependent global loads off every block the SpMV visits.
struct Rows {
    int row0, nbs;
    const int* lrp;
    const int2* ent;
    double* part;  // LDS partial products of the entry-parallel SpMV (12 per block)
};

// SpMV modes: rows over the global structure, rows over the staged structure, and
// entry-parallel over the staged structure (systems that fit the LDS budget, entries_fit).
// The first two sum each row over (block, column triple) in one sequence; the third sums
// each block's row first and the block results in column order.  The mode of a system
// depends on its own size only, so a scene gives the same bits alone or in a batch.
enum { kSpmvRows = 0, kSpmvRowsStaged = 1, kSpmvEntries = 2 };

// lrp capacity of the staged structure (bodies + 1)
constexpr int kLrpCap = 2048;
constexpr size_t kLrpBytes = sizeof(int) * (size_t)kLrpCap;
constexpr int kEntCap = (int)((kLdsStructBytes - kLrpBytes) / sizeof(int2));

// Does a system of n rows and nnz blocks take the entry-parallel SpMV?  Its six vectors
// and its partial products must fit the LDS budget beside the structure, counting the
// vectors as if in LDS wherever they live, so that the answer depends on the system
// alone and on the device, never on the other systems of a launch.
__device__ __forceinline__ bool entries_fit(int n, int nnz, int budget) {
    return budget >= 0 && 8 * (6 * (int64_t)n + 12 * (int64_t)nnz) + (int64_t)kLdsStructBytes <= budget;
}

template <int MODE>
__device__ __forceinline__ void row_entry(const Bsr& M, const Rows& R, int e, int& lc, int64_t& slot) {
    if (MODE != kSpmvRows) {
        const int2 v = R.ent[e];
        lc = v.x;
        slot = v.y;
    } else {
        lc = M.cols[e] - R.row0;
        if ((unsigned)lc >= (unsigned)R.nbs) lc = -1;  // a block coupling two scenes is part of neither
        slot = M.slots[e];
    }
}

// (H in)[row (lb, ii, k)] of the system (local body lb), summed over the row's blocks in
// column order.  Two blocks are loaded per step so that their memory latencies overlap;
// the sum order is that of a one-block loop.
template <int MODE>
__device__ __forceinline__ double row_product(const Bsr& M, const Rows& R, int lb, int ii, int k,
                                              const double* __restrict__ in) {
    double acc = 0.0;
    int e = MODE != kSpmvRows ? R.lrp[lb] : M.row_ptr[R.row0 + lb];
    const int e1 = MODE != kSpmvRows ? R.lrp[lb + 1] : M.row_ptr[R.row0 + lb + 1];
    for (; e + 1 < e1; e += 2) {
        int lc0, lc1;
        int64_t s0, s1;
        row_entry<MODE>(M, R, e, lc0, s0);
        row_entry<MODE>(M, R, e + 1, lc1, s1);
        double B0[12], B1[12];
        load_block_row(M.blocks, s0, ii, k, B0);
        load_block_row(M.blocks, s1, ii, k, B1);
        if (lc0 >= 0) acc = block_row_add(acc, B0, in + 12 * (int64_t)lc0);
        if (lc1 >= 0) acc = block_row_add(acc, B1, in + 12 * (int64_t)lc1);
    }
    if (e < e1) {
        int lc;
        int64_t sl;
        row_entry<MODE>(M, R, e, lc, sl);
        if (lc >= 0) {
            double B[12];
            load_block_row(M.blocks, sl, ii, k, B);
            acc = block_row_add(acc, B, in + 12 * (int64_t)lc);
        }
    }
    return acc;
}

// Entry-parallel products: work item (block e, block row ii) multiplies rows 3 ii .. 3 ii + 2
// of block e by its column's 12 entries of `in` (each row's four sub-block sums in
// order) into R.part[12 e + 3 ii + r]; every load of an item is independent of the others.
__device__ __forceinline__ void entry_products(const Bsr& M, const Rows& R, const double* __restrict__ in) {
    const int nnz = R.lrp[R.nbs];
    for (int wi = threadIdx.x; wi < 4 * nnz; wi += blockDim.x) {
        const int e = wi >> 2, ii = wi & 3;
        const int2 en = R.ent[e];
        if (en.x < 0) continue;  // outside the system: skipped by the row sums too
        const double* B = M.blocks + 144 * (int64_t)en.y + 9 * ii;
        const double* xin = in + 12 * en.x;
        double y0 = 0.0, y1 = 0.0, y2 = 0.0;
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
            const double* Bj = B + 36 * jj;  // sub-block (ii, jj), row-major 3x3
            const double x0 = xin[3 * jj], x1 = xin[3 * jj + 1], x2 = xin[3 * jj + 2];
            y0 = y0 + (Bj[0] * x0 + Bj[1] * x1 + Bj[2] * x2);
            y1 = y1 + (Bj[3] * x0 + Bj[4] * x1 + Bj[5] * x2);
            y2 = y2 + (Bj[6] * x0 + Bj[7] * x1 + Bj[8] * x2);
        }
        double* pe = R.part + 12 * e + 3 * ii;
        pe[0] = y0;
        pe[1] = y1;
        pe[2] = y2;
    }
    __syncthreads();
}

// row idx of the entry-parallel SpMV: its blocks' partial products in column order
__device__ __forceinline__ double entry_row_sum(const Rows& R, int idx) {
    const int lb = idx / 12, lr = idx % 12;
    double acc = 0.0;
    for (int e = R.lrp[lb]; e < R.lrp[lb + 1]; ++e)
        if (R.ent[e].x >= 0) acc += R.part[12 * e + lr];
    return acc;
}

// Copies the structure of the system's rows into LDS (lrp: kLrpCap ints, ent: kEntCap
// entries) when the device holds it (budget >= 0) and it fits; returns the SpMV mode of
// the system.  Uniform over the workgroup; ends with a barrier when it stages.
__device__ __forceinline__ int stage_rows(const Bsr& M, Rows& R, int* lrp, int2* ent, int budget) {
    const int e0 = M.row_ptr[R.row0], nnz = M.row_ptr[R.row0 + R.nbs] - e0;
    if (budget < 0 || nnz > kEntCap || R.nbs + 1 > kLrpCap) return kSpmvRows;
    for (int r = threadIdx.x; r <= R.nbs; r += blockDim.x) lrp[r] = M.row_ptr[R.row0 + r] - e0;
    for (int e = threadIdx.x; e < nnz; e += blockDim.x) {
        const int lc = M.cols[e0 + e] - R.row0;
        ent[e] = make_int2((unsigned)lc < (unsigned)R.nbs ? lc : -1, M.slots[e0 + e]);
    }
    __syncthreads();
    R.lrp = lrp;
    R.ent = ent;
    return entries_fit(12 * R.nbs, nnz, budget) ? kSpmvEntries : kSpmvRowsStaged;
}

// out = H in over the system's rows (in / out indexed from its first row); row idx of
// local body idx / 12, sub-row (ii, k) = ((idx % 12) / 3, idx % 3)
template <int MODE>
__device__ __forceinline__ void spmv(const Bsr& M, const Rows& R, const double* __restrict__ in,
                                     double* __restrict__ out, int n) {
    if (MODE == kSpmvEntries) entry_products(M, R, in);
    for (int idx = threadIdx.x; idx < n; idx += blockDim.x) {
        const int lr = idx % 12;
        out[idx] = MODE == kSpmvEntries ? entry_row_sum(R, idx) : row_product<MODE>(M, R, idx / 12, lr / 3, lr % 3, in);
    }
    __syncthreads();
}

// out = H in over this thread's rows (the rows spmv() gives it), returning the
// thread's partial sum of w[idx] * out[idx] in row order; no barrier at the end: the
// caller reduces the partials (which also orders the writes before any cross-thread read).
template <int MODE>
__device__ __forceinline__ double spmv_rows_dot(const Bsr& M, const Rows& R, const double* __restrict__ in,
                                                double* __restrict__ out, int n, const double* __restrict__ w) {
    if (MODE == kSpmvEntries) entry_products(M, R, in);
    double part = 0.0;
    for (int idx = threadIdx.x; idx < n; idx += blockDim.x) {
        const int lr = idx % 12;
        const double acc =
            MODE == kSpmvEntries ? entry_row_sum(R, idx) : row_product<MODE>(M, R, idx / 12, lr / 3, lr % 3, in);
        out[idx] = acc;
        part += w[idx] * acc;
    }
    return part;
}

__device__ __forceinline__ double vdot(const double* __restrict__ a, const double* __restrict__ b, int n,
                                       double* sh) {
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) acc += a[i] * b[i];
    return block_sum_fast(acc, sh);
}

// The Krylov loops of a system whose rows fit one per thread (n <= T) and whose blocks fit
// four threads each (entry-parallel mode): the matrix in registers for the whole solve, K
// rows of one block a thread (K = 1, 2, 3: the least that fits), the vectors too, each thread
// its row; only the multiplied vector and the block rows' partial products pass through LDS.
// Every sum is the one of cg_body / bicgstab_body in entry-parallel mode (a thread there owns
// the same row; absent waves add 0), so the bits are the same.  What bounds these solves is
// the latency of an iteration's dependent steps: hence no matrix reads from L2, one barrier a
// sum, lane moves in place of LDS shuffles, and waves without rows taking part in the
// products only.  Against the memory loops: CG of 61 systems of 2 to 40 bodies 294 -> 116 us,
// CG of 16 uncoupled bodies 33.5 -> 14.8 us, BiCGSTAB of 2 bodies 98 -> 22 us (of which one wave
// in place of 16 about a quarter).
constexpr int kRegRows = 3;
template <int K, int T>
struct RegSystem {
    static constexpr int kPer = 12 / K;  // threads a block
    double B[K][12];
    int xo;      // first entry of the column in the multiplied vector (-1: none)
    int e0, e1;  // the entries of this thread's row
    bool rows;   // this wave has rows
    int nw;      // waves with rows
    double* part;
    double* sums;  // LDS: [2][2][16], the halves in turn
    int turn;
    double one[2];  // the sums of a single wave

    __device__ __forceinline__ RegSystem(const Bsr& M, const Rows& R, int n, double* lds_sums)
        : xo(-1), e0(0), e1(0), nw((n + kWave - 1) / kWave), part(R.part), sums(lds_sums), turn(0) {
        const int t = threadIdx.x, e = t / kPer, r0 = K * (t % kPer);
        rows = T == kWave || __builtin_amdgcn_readfirstlane(wave_id()) < nw;
#pragma unroll
        for (int k = 0; k < K; ++k)
#pragma unroll
            for (int q = 0; q < 12; ++q) B[k][q] = 0.0;
        if (e < R.lrp[R.nbs]) {
            const int2 en = R.ent[e];
            if (en.x >= 0) {
                xo = 12 * en.x;
#pragma unroll
                for (int k = 0; k < K; ++k) load_block_row(M.blocks, en.y, (r0 + k) / 3, (r0 + k) % 3, B[k]);
            } else {
                for (int k = 0; k < K; ++k) part[12 * e + r0 + k] = 0.0;  // outside the system: adds nothing
            }
        }
        if (t < n) {
            e0 = R.lrp[t / 12];
            e1 = R.lrp[t / 12 + 1];
        }
    }
    // the block rows' products with `in` (LDS); then a barrier and row()
    __device__ __forceinline__ void products(const double* __restrict__ in) const {
        if (xo < 0) return;
        double y[K];
#pragma unroll
        for (int k = 0; k < K; ++k) y[k] = 0.0;
#pragma unroll
        for (int q = 0; q < 12; q += 3) {  // block_row_add of every row, the column's entries read once
            const double x0 = in[xo + q], x1 = in[xo + q + 1], x2 = in[xo + q + 2];
#pragma unroll
            for (int k = 0; k < K; ++k) y[k] += B[k][q] * x0 + B[k][q + 1] * x1 + B[k][q + 2] * x2;
        }
#pragma unroll
        for (int k = 0; k < K; ++k) part[K * threadIdx.x + k] = y[k];
    }
    // this thread's row of the product: its blocks' in column order, four loads in flight
    __device__ __forceinline__ double row() const {
        double acc = 0.0;
        const double* pr = part + threadIdx.x % 12;
        for (int e = e0; e < e1; e += 4) {
            double v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = e + j < e1 ? pr[12 * (e + j)] : 0.0;
#pragma unroll
            for (int j = 0; j < 4; ++j) acc += v[j];
        }
        return acc;
    }
    // block_sum_fast's value in three parts: put (waves with rows), a barrier, get; the
    // buffers alternate, so the next put needs no barrier of its own
    __device__ __forceinline__ void put(double v, int which = 0) {
        v = wave_sum(v);
        if (T == kWave)
            one[which] = v + 0.0;
        else if (lane_id() == 0)
            sums[32 * turn + 16 * which + wave_id()] = v;
    }
    __device__ __forceinline__ double get(int which = 0) const {
        return T == kWave ? one[which] : waves_sum(sums + 32 * turn + 16 * which, nw);
    }
    __device__ __forceinline__ void next() { turn ^= 1; }
};

template <int K, int T>
__device__ __forceinline__ void bicgstab_regs(const Bsr& M, const Rows& R, int n, const double* __restrict__ b,
                                              double* __restrict__ xg, double tol, int maxiter, int check_every,
                                              double* V, int32_t* __restrict__ iters, double* __restrict__ resid,
                                              double* sums) {
    double *pl = V, *rl = V + n;
    const int i = threadIdx.x;
    const bool own = i < n;
    double x = own ? xg[i] : 0.0;
    const double bi = own ? b[i] : 0.0;
    if (own) pl[i] = x;
    RegSystem<K, T> H(M, R, n, sums);
    const bool rows = H.rows;
    __syncthreads();
    H.products(pl);
    __syncthreads();
    double r = 0.0;
    if (rows) {
        r = bi - H.row();
        H.put(own ? 0.0 + r * r : 0.0);
        H.put(own ? 0.0 + bi * bi : 0.0, 1);
    }
    __syncthreads();
    double rr = H.get();
    const double atol = tol * sqrt(H.get(1));
    H.next();
    const double atol_sq = atol * atol;
    int it = 0;
    if (rr > atol_sq) {
        const double r0 = r;
        double p = r, rho = rr, v = 0.0, t = 0.0, alpha = 0.0, omega = 0.0;
        if (own) pl[i] = p;
        __syncthreads();
        for (;;) {
            for (int c = 1; c <= check_every; ++c) {
                H.products(pl);
                __syncthreads();
                if (rows) {
                    v = H.row();
                    H.put(own ? 0.0 + r0 * v : 0.0);
                }
                __syncthreads();
                if (rows) {
                    const double r0v = H.get();
                    alpha = r0v != 0.0 ? rho / r0v : 0.0;
                    x += alpha * p;
                    r -= alpha * v;
                    if (own) rl[i] = r;
                }
                H.next();
                __syncthreads();
                H.products(rl);
                __syncthreads();
                if (rows) {
                    t = H.row();
                    H.put(own ? 0.0 + t * r : 0.0);
                    H.put(own ? 0.0 + t * t : 0.0, 1);
                }
                __syncthreads();
                if (rows) {
                    const double tr = H.get(), tt = H.get(1);
                    H.next();
                    omega = tt != 0.0 ? tr / tt : 0.0;
                    x += omega * r;
                    r -= omega * t;
                    H.put(own ? 0.0 + r * r : 0.0);
                    H.put(own ? 0.0 + r0 * r : 0.0, 1);
                } else {
                    H.next();
                }
                __syncthreads();
                if (rows || c == check_every) rr = H.get();
                if (rows) {
                    const double rho_old = rho;
                    rho = H.get(1);
                    const double beta = (rho_old != 0.0 && omega != 0.0) ? (rho / rho_old) * (alpha / omega) : 0.0;
                    p = r + beta * (p - omega * v);
                    if (own) pl[i] = p;
                }
                H.next();
                __syncthreads();
            }
            it += check_every;
            if (rr <= atol_sq || it >= maxiter) break;
        }
    }
    if (own) xg[i] = x;
    if (i == 0) {
        if (iters) *iters = it;
        if (resid) *resid = rr;
    }
}

template <int K, int T>
__device__ __forceinline__ void cg_regs(const Bsr& M, const Rows& R, int n, const double* __restrict__ b,
                                        double* __restrict__ xg, double tol, int maxiter, int check_every, double* V,
                                        int32_t* __restrict__ iters, double* __restrict__ resid, double* sums) {
    double* pl = V;
    const int i = threadIdx.x;
    const bool own = i < n;
    double x = 0.0, bi = 0.0, da = 0.0;
    bool plain = true;  // a zero diagonal sub-block, or no row: z = r
    if (own) {
        const double* D = M.blocks + 9 * (16 * (int64_t)(R.row0 + i / 12) + 5 * (i % 12 / 3));
        const double d0 = D[0], d1 = D[4], d2 = D[8];
        plain = d0 * d0 + d1 * d1 + d2 * d2 == 0.0;
        da = fabs(i % 3 == 0 ? d0 : i % 3 == 1 ? d1 : d2);
        x = xg[i];
        bi = b[i];
        pl[i] = x;
    }
    RegSystem<K, T> H(M, R, n, sums);
    const bool rows = H.rows;
    __syncthreads();
    H.products(pl);
    __syncthreads();
    double r = 0.0, z = 0.0, p = 0.0;
    if (rows) {
        r = bi - H.row();
        z = plain ? r : r / da;
        p = z;
        H.put(own ? 0.0 + r * z : 0.0);
        if (own) pl[i] = p;
    }
    __syncthreads();
    double rz_old = H.get(), rz_new = 0.0;
    H.next();
    const double tol_sq = tol * tol * (double)n;
    double err = rz_old;
    int end_iter = 0;
    if (err > tol_sq) {
        end_iter = maxiter;
        for (int c = 0; c < maxiter; ++c) {
            const bool check = ((c + 1) % check_every) == 0;
            double Ap = 0.0;
            H.products(pl);
            __syncthreads();
            if (rows) {
                Ap = H.row();
                H.put(own ? 0.0 + p * Ap : 0.0);
            }
            __syncthreads();
            if (rows) {
                const double pAp = H.get();
                H.next();
                const double alpha = pAp != 0.0 ? rz_old / pAp : 0.0;
                x += alpha * p;
                r -= alpha * Ap;
                z = plain ? r : r / da;
                H.put(own ? 0.0 + r * z : 0.0);
            } else {
                H.next();
            }
            __syncthreads();
            if (rows || check) rz_new = H.get();
            H.next();
            if (check && rz_new <= tol_sq) {  // uniform: the same sum in every wave
                end_iter = c;
                err = rz_new;
                break;
            }
            if (rows) {
                const double beta = rz_new > tol_sq ? rz_new / rz_old : 0.0;
                p = z + beta * p;
                if (own) pl[i] = p;
            }
            __syncthreads();
            rz_old = rz_new;
            err = rz_old;
        }
    }
    if (own) xg[i] = x;
    if (i == 0) {
        if (iters) *iters = end_iter;
        if (resid) *resid = err;
    }
}

// Dynamic LDS of a solve workgroup: the staged structure (lrp, then ent), the six Krylov
// vectors of the system's n rows when LDS (else in the scratch arena), then the partial
// products of the entry-parallel SpMV.
template <bool LDS>
struct SolveLds {
    double* V;
    double* part;
    int* lrp;
    int2* ent;
    __device__ SolveLds(double* ws, int n) {
        extern __shared__ double lds_dyn[];
        char* base = (char*)lds_dyn;
        lrp = (int*)base;
        ent = (int2*)(base + kLrpBytes);
        double* after = (double*)(base + kLdsStructBytes);
        V = LDS ? after : ws;
        part = LDS ? after + 6 * n : after;
    }
};

template <int MODE>
__device__ __forceinline__ void bicgstab_body(const Bsr& M, const Rows& R, int n, const double* __restrict__ b,
                                              double* __restrict__ xg, double tol, int maxiter, int check_every,
                                              double* V, int32_t* __restrict__ iters, double* __restrict__ resid,
                                              double* sh, double* sh2) {
    double* x = V;
    double* r = V + n;
    double* r0 = V + 2 * n;
    double* p = V + 3 * n;
    double* v = V + 4 * n;
    double* t = V + 5 * n;
    for (int i = threadIdx.x; i < n; i += blockDim.x) x[i] = xg[i];
    __syncthreads();
    spmv<MODE>(M, R, x, t, n);
    for (int i = threadIdx.x; i < n; i += blockDim.x) r[i] = b[i] - t[i];
    __syncthreads();
    double rr = vdot(r, r, n, sh);
    const double bb = vdot(b, b, n, sh);
    const double atol = tol * sqrt(bb);
    const double atol_sq = atol * atol;
    int it = 0;
    if (rr > atol_sq) {
        for (int i = threadIdx.x; i < n; i += blockDim.x) {
            r0[i] = r[i];
            p[i] = r[i];
        }
        __syncthreads();
        double rho = rr;
        for (;;) {
            // fused passes: each dot is accumulated where its operand is produced, in
            // the row order of vdot(), so the iterates match the unfused sequence bit for bit
            for (int c = 0; c < check_every; ++c) {
                const double r0v = block_sum_fast(spmv_rows_dot<MODE>(M, R, p, v, n, r0), sh);
                const double alpha = r0v != 0.0 ? rho / r0v : 0.0;
                for (int i = threadIdx.x; i < n; i += blockDim.x) {
                    x[i] += alpha * p[i];
                    r[i] -= alpha * v[i];
                }
                __syncthreads();
                // t = H r, then t.r and t.t over this thread's rows in row order
                spmv<MODE>(M, R, r, t, n);
                double tr = 0.0, tt = 0.0;
                for (int idx = threadIdx.x; idx < n; idx += blockDim.x) {
                    const double acc = t[idx];
                    tr += acc * r[idx];
                    tt += acc * acc;
                }
                block_sum2_fast(tr, tt, sh2);
                const double omega = tt != 0.0 ? tr / tt : 0.0;
                double rr_p = 0.0, rho_p = 0.0;
                for (int i = threadIdx.x; i < n; i += blockDim.x) {
                    x[i] += omega * r[i];
                    r[i] -= omega * t[i];
                    rr_p += r[i] * r[i];
                    rho_p += r0[i] * r[i];
                }
                block_sum2_fast(rr_p, rho_p, sh2);
                rr = rr_p;
                const double rho_old = rho;
                rho = rho_p;
                const double beta = (rho_old != 0.0 && omega != 0.0) ? (rho / rho_old) * (alpha / omega) : 0.0;
                for (int i = threadIdx.x; i < n; i += blockDim.x) p[i] = r[i] + beta * (p[i] - omega * v[i]);
                __syncthreads();
            }
            it += check_every;
            if (rr <= atol_sq || it >= maxiter) break;
        }
    }
    for (int i = threadIdx.x; i < n; i += blockDim.x) xg[i] = x[i];
    if (threadIdx.x == 0) {
        if (iters) *iters = it;
        if (resid) *resid = rr;
    }
}

// Whether a system takes the register-resident loops of T threads (12 / kRegRows a block).
template <int T>
__device__ __forceinline__ bool regs_fit(const Rows& R, int n) {
    return n <= T && 4 * R.lrp[R.nbs] <= T;
}

// budget: bytes of dynamic LDS (SolveLds; -1: the device holds no staged structure).  T: the
// workgroup's threads (solve_threads).
template <bool LDS, int T>
__global__ __launch_bounds__(T) void bicgstab_kernel(Bsr M, const int32_t* __restrict__ sboff,
                                                                  const uint8_t* __restrict__ active,
                                                                  const double* __restrict__ b,
                                                                  double* __restrict__ xg, double tol, int maxiter,
                                                                  int check_every, int cap_rows, int budget,
                                                                  double* __restrict__ ws,
                                                                  int32_t* __restrict__ iters,
                                                                  double* __restrict__ resid) {
    __shared__ double sh[17];
    __shared__ double sh2[64];
    // one system per workgroup: the bodies of scene blockIdx.x (all bodies without scenes)
    const int sidx = blockIdx.x;
    if (active && !active[sidx]) return;
    const int row0 = sboff ? sboff[sidx] : 0;
    const int n = 12 * ((sboff ? sboff[sidx + 1] : M.nb) - row0);
    b += 12 * (int64_t)row0;
    xg += 12 * (int64_t)row0;
    if (iters) iters += sidx;
    if (resid) resid += sidx;
    if (n > cap_rows) {  // larger than the vector storage sized by the caller: report, touch nothing
        if (threadIdx.x == 0 && iters) *iters = -1;
        return;
    }
    const SolveLds<LDS> S(ws + (LDS ? 0 : 6 * 12 * (int64_t)row0), n);
    if (maxiter <= 0) maxiter = n;  // the system size of this workgroup's system
    Rows R{row0, n / 12, nullptr, nullptr, S.part};
    const int mode = stage_rows(M, R, S.lrp, S.ent, budget);
    if (mode == kSpmvEntries && regs_fit<T>(R, n)) {
        double* Vr = LDS ? S.V : S.part + 12 * R.lrp[R.nbs];  // two of entries_fit's six vectors
        const int nnz = R.lrp[R.nbs];
        if (12 * nnz <= T)
            bicgstab_regs<1, T>(M, R, n, b, xg, tol, maxiter, check_every, Vr, iters, resid, sh2);
        else if (6 * nnz <= T)
            bicgstab_regs<2, T>(M, R, n, b, xg, tol, maxiter, check_every, Vr, iters, resid, sh2);
        else
            bicgstab_regs<kRegRows, T>(M, R, n, b, xg, tol, maxiter, check_every, Vr, iters, resid, sh2);
    } else if (mode == kSpmvEntries)
        bicgstab_body<kSpmvEntries>(M, R, n, b, xg, tol, maxiter, check_every, S.V, iters, resid, sh, sh2);
    else if (mode == kSpmvRowsStaged)
        bicgstab_body<kSpmvRowsStaged>(M, R, n, b, xg, tol, maxiter, check_every, S.V, iters, resid, sh, sh2);
    else
        bicgstab_body<kSpmvRows>(M, R, n, b, xg, tol, maxiter, check_every, S.V, iters, resid, sh, sh2);
}

__device__ __forceinline__ void jacobi(const double* __restrict__ dg, const double* __restrict__ r,
                                       double* __restrict__ z, int n) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const int i3 = i - i % 3;
        const double d0 = dg[i3], d1 = dg[i3 + 1], d2 = dg[i3 + 2];
        z[i] = (d0 * d0 + d1 * d1 + d2 * d2 == 0.0) ? r[i] : r[i] / fabs(dg[i]);
    }
    __syncthreads();
}

// Inverse of each body's 12x12 diagonal block (slot b) by Gauss-Jordan elimination with
// partial pivoting, written to dinv + 144 b; a singular block gives the identity (that
// body stays unpreconditioned).  One 64-thread workgroup per body: the augmented 12x24
// matrix in LDS, the 288 entries of each elimination step updated in parallel, each with
// the arithmetic of the sequential elimination (row c scaled by 1 / pivot, then
// a[r][j] -= a[r][c] a[c][j] for every other row with a[r][c] != 0).
// pending (nullable): per-system status of a direct solve; then only the bodies of the
// systems it declined (kLdltFailed) are inverted, the system of body b found in sboff [nsys + 1].
constexpr int kInvThreads = 64;
__global__ __launch_bounds__(kInvThreads) void invert_blocks_kernel(Bsr M, double* __restrict__ dinv,
                                                                    const int32_t* __restrict__ pending,
                                                                    const int32_t* __restrict__ sboff, int nsys) {
    __shared__ double a[12][24];
    __shared__ double srow[24];
    __shared__ double f[12];
    const int b = blockIdx.x, t = threadIdx.x;
    if (pending) {
        int sys = 0;
        if (sboff) {
            int lo = 0, hi = nsys - 1;  // the last system whose first body is <= b
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (sboff[mid] <= b)
                    lo = mid;
                else
                    hi = mid - 1;
            }
            sys = lo;
        }
        if (pending[sys] != kLdltFailed) return;  // uniform over the workgroup
    }
    for (int e = t; e < 288; e += kInvThreads) {
        const int i = e / 24, j = e % 24;
        a[i][j] = j < 12 ? M.blocks[9 * (16 * (int64_t)b + i / 3 + 4 * (j / 3)) + 3 * (i % 3) + j % 3]
                         : (i == j - 12 ? 1.0 : 0.0);
    }
    __syncthreads();
    bool ok = true;
    for (int c = 0; c < 12; ++c) {
        int piv = c;  // the first row of largest |a[r][c]|, r >= c (every thread alike)
        for (int r = c + 1; r < 12; ++r)
            if (fabs(a[r][c]) > fabs(a[piv][c])) piv = r;
        if (a[piv][c] == 0.0) {
            ok = false;
            break;
        }
        __syncthreads();
        if (piv != c && t < 24) {
            const double u = a[c][t];
            a[c][t] = a[piv][t];
            a[piv][t] = u;
        }
        __syncthreads();
        const double inv = 1.0 / a[c][c];
        if (t < 24) srow[t] = a[c][t] * inv;
        if (t < 12) f[t] = a[t][c];
        __syncthreads();
        for (int e = t; e < 288; e += kInvThreads) {
            const int i = e / 24, j = e % 24;
            if (i == c)
                a[i][j] = srow[j];
            else if (f[i] != 0.0)
                a[i][j] -= f[i] * srow[j];
        }
        __syncthreads();
    }
    double* out = dinv + 144 * (int64_t)b;
    for (int e = t; e < 144; e += kInvThreads) {
        const int i = e / 12, j = e % 12;
        out[e] = ok ? a[i][12 + j] : (i == j ? 1.0 : 0.0);
    }
}

// z = D_b^-1 r for row k of a system whose body-diagonal inverses are in dinv (global body ids)
__device__ __forceinline__ double block_precond(const double* __restrict__ dinv, const double* __restrict__ r,
                                                int row0, int k) {
    const int lb = k / 12, l = k % 12;
    const double* Di = dinv + 144 * (int64_t)(row0 + lb) + 12 * l;
    const double* rb = r + 12 * lb;
    double acc = 0.0;
#pragma unroll
    for (int q = 0; q < 12; ++q) acc += Di[q] * rb[q];
    return acc;
}

template <bool BJ, int MODE>
__device__ __forceinline__ void cg_body(const Bsr& M, const Rows& R, int n, const double* __restrict__ b,
                                        double* __restrict__ xg, double tol, int maxiter, int check_every,
                                        double* V, const double* __restrict__ dinv, int32_t* __restrict__ iters,
                                        double* __restrict__ resid, double* sh) {
    const int row0 = R.row0;
    double* x = V;
    double* r = V + n;
    double* p = V + 2 * n;
    double* Ap = V + 3 * n;
    double* z = V + 4 * n;
    double* dg = V + 5 * n;
    // bsr_get_diag: diagonal of the diagonal 3x3 blocks (sub-block (ii, ii) of slot b)
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const int bb = row0 + i / 12, ii = (i % 12) / 3, a = i % 3;
        dg[i] = M.blocks[9 * (16 * (int64_t)bb + ii + 4 * ii) + 4 * a];
        x[i] = xg[i];
    }
    __syncthreads();
    spmv<MODE>(M, R, x, Ap, n);
    for (int i = threadIdx.x; i < n; i += blockDim.x) r[i] = b[i] - Ap[i];
    __syncthreads();
    if (BJ) {
        for (int i = threadIdx.x; i < n; i += blockDim.x) z[i] = block_precond(dinv, r, row0, i);
        __syncthreads();
    } else {
        jacobi(dg, r, z, n);
    }
    for (int i = threadIdx.x; i < n; i += blockDim.x) p[i] = z[i];
    __syncthreads();
    double rz_old = vdot(r, z, n, sh), rz_new = 0.0;
    const double tol_sq = tol * tol * (double)n;
    double err = rz_old;
    int end_iter = 0;
    if (err > tol_sq) {
        end_iter = maxiter;
        // fused passes (dots accumulated where their operands are produced, in vdot()'s
        // row order: the iterates match the unfused sequence bit for bit)
        for (int i = 0; i < maxiter; ++i) {
            const double pAp = block_sum_fast(spmv_rows_dot<MODE>(M, R, p, Ap, n, p), sh);
            // unguarded in the reference: p = 0 once the residual vanishes exactly between checks
            const double alpha = pAp != 0.0 ? rz_old / pAp : 0.0;
            double rz_p = 0.0;
            if (BJ) {
                // the body's whole residual enters z: update r, then precondition
                for (int k = threadIdx.x; k < n; k += blockDim.x) {
                    x[k] += alpha * p[k];
                    r[k] -= alpha * Ap[k];
                }
                __syncthreads();
                for (int k = threadIdx.x; k < n; k += blockDim.x) {
                    z[k] = block_precond(dinv, r, row0, k);
                    rz_p += r[k] * z[k];
                }
            } else {
                for (int k = threadIdx.x; k < n; k += blockDim.x) {
                    x[k] += alpha * p[k];
                    r[k] -= alpha * Ap[k];
                    const int k3 = k - k % 3;
                    const double d0 = dg[k3], d1 = dg[k3 + 1], d2 = dg[k3 + 2];
                    z[k] = (d0 * d0 + d1 * d1 + d2 * d2 == 0.0) ? r[k] : r[k] / fabs(dg[k]);
                    rz_p += r[k] * z[k];
                }
            }
            rz_new = block_sum_fast(rz_p, sh);
            if (((i + 1) % check_every) == 0 && rz_new <= tol_sq) {
                end_iter = i;
                err = rz_new;
                break;
            }
            const double beta = rz_new > tol_sq ? rz_new / rz_old : 0.0;
            for (int k = threadIdx.x; k < n; k += blockDim.x) p[k] = z[k] + beta * p[k];
            __syncthreads();
            const double tmp = rz_old;
            rz_old = rz_new;
            rz_new = tmp;
            err = rz_old;
        }
    }
    for (int i = threadIdx.x; i < n; i += blockDim.x) xg[i] = x[i];
    if (threadIdx.x == 0) {
        if (iters) *iters = end_iter;
        if (resid) *resid = err;
    }
}

// BJ: the per-body 12x12 block-Jacobi preconditioner (beyond the reference) in place of
// the diagonal one; dinv: [nb][144] workspace of the inverses.  budget as bicgstab_kernel.
template <bool LDS, bool BJ, int T>
__global__ __launch_bounds__(T) void cg_kernel(Bsr M, const int32_t* __restrict__ sboff,
                                                           const uint8_t* __restrict__ active,
                                                           const double* __restrict__ b, double* __restrict__ xg,
                                                           double tol, int maxiter, int check_every, int cap_rows,
                                                           int budget, double* __restrict__ ws,
                                                           double* __restrict__ dinv, int32_t* __restrict__ iters,
                                                           double* __restrict__ resid,
                                                           const int32_t* __restrict__ pending) {
    __shared__ double sh[BJ ? 17 : 64];
    // one system per workgroup: the bodies of scene blockIdx.x (all bodies without scenes);
    // pending (nullable): only the systems the direct solve declined
    const int sidx = blockIdx.x;
    if (active && !active[sidx]) return;
    if (pending && pending[sidx] != kLdltFailed) return;
    const int row0 = sboff ? sboff[sidx] : 0;
    const int n = 12 * ((sboff ? sboff[sidx + 1] : M.nb) - row0);
    b += 12 * (int64_t)row0;
    xg += 12 * (int64_t)row0;
    if (iters) iters += sidx;
    if (resid) resid += sidx;
    if (n > cap_rows) {  // larger than the vector storage sized by the caller: report, touch nothing
        if (threadIdx.x == 0 && iters) *iters = -1;
        return;
    }
    const SolveLds<LDS> S(ws + (LDS ? 0 : 6 * 12 * (int64_t)row0), n);
    if (maxiter <= 0) maxiter = n;  // the system size of this workgroup's system
    Rows R{row0, n / 12, nullptr, nullptr, S.part};
    const int mode = stage_rows(M, R, S.lrp, S.ent, budget);
    if constexpr (!BJ)
        if (mode == kSpmvEntries && regs_fit<T>(R, n)) {
            double* Vr = LDS ? S.V : S.part + 12 * R.lrp[R.nbs];  // one of entries_fit's six vectors
            const int nnz = R.lrp[R.nbs];
            if (12 * nnz <= T)
                cg_regs<1, T>(M, R, n, b, xg, tol, maxiter, check_every, Vr, iters, resid, sh);
            else if (6 * nnz <= T)
                cg_regs<2, T>(M, R, n, b, xg, tol, maxiter, check_every, Vr, iters, resid, sh);
            else
                cg_regs<kRegRows, T>(M, R, n, b, xg, tol, maxiter, check_every, Vr, iters, resid, sh);
            return;
        }
    if (mode == kSpmvEntries)
        cg_body<BJ, kSpmvEntries>(M, R, n, b, xg, tol, maxiter, check_every, S.V, dinv, iters, resid, sh);
    else if (mode == kSpmvRowsStaged)
        cg_body<BJ, kSpmvRowsStaged>(M, R, n, b, xg, tol, maxiter, check_every, S.V, dinv, iters, resid, sh);
    else
        cg_body<BJ, kSpmvRows>(M, R, n, b, xg, tol, maxiter, check_every, S.V, dinv, iters, resid, sh);
}

// ------------------------------------------------------------------ direct solve
// Beyond the reference: the system solved directly by a block LDL^T factorization of its
// 12x12 body blocks (no exchanges between bodies), fill-in kept; one workgroup per system
// of at most kLdltMaxBodies bodies.  Structure: one 64-bit upper row mask per body, its
// fill (eliminating the bodies in their own order), the transposed masks, and the levels
// of that order's elimination tree (parent of k: the first body above k coupled to it;
// level: 0 for a leaf, else one more than the highest child's) -- bodies of one level are
// never coupled to each other and are eliminated together, level after level, in chunks
// of at most kLdltCols columns of [A' | I].  The factor's upper blocks live in the system's
// workspace region (row i's blocks from pos[i], in column order), the chunk's W blocks
// after them.  Elimination of body k: Gauss-Jordan elimination without row exchanges on
// [P | A'_k,j1 .. A'_k,jd | I], P = A'_kk, leaving W_j = P^-1 A'_kj and P^-1.  The pivot
// columns depend on P alone: pivot_columns() finds them for all bodies of the chunk, 16 lanes
// a body, and stores each as the columns take it; then every column of A' and I goes through
// the 12 pivots in registers with no barrier between (64 bodies of one level: 26 k cycles, as
// with one barrier per pivot pair; a level of one body: 5.3 k + 3.9 k instead of 10 k).  Each
// Schur target A'_ij (and each forward-solve target y_i) is updated by its chunk's bodies
// in ascending order, A'_ij -= A'_ki^T W_j, y_i -= W_i^T y_k (12-term sums), by the
// thread of the lowest of them, so a system gives the same bits whatever else a launch
// holds; z_k = P^-1 y_k; W then replaces row k.  Backward solve, levels from the top:
// x_k = z_k - sum_i W_i x_i, each W_i x_i a 12-term sum, added in ascending i.  This is
// the arithmetic, in the same order, of eliminating body by body in (level, body) order.
// A pivot that is not positive (the system is not positive definite as factored) or a
// system above the size limit leaves x untouched and status kLdltFailed; else status 1
// and resid (nullable) = |b - H x|^2.  The factor and the W blocks live in the workgroup's dynamic
// LDS (dyn_blocks 12x12 blocks) when they fit there -- the factor's upper blocks with fill
// and at most min(kLdltWBlocks, off-diagonal blocks) W blocks -- else in the system's
// workspace region, with each chunk's pivot columns, A' and W blocks staged in the LDS where
// those fit; the arithmetic is the same in all places.  Latency bounds it: a level's few
// dependent phases, on one CU.  Against a barrier per pivot pair, one element of a Schur target
// a thread and nothing staged: 64 bodies of two levels 41 -> 32 us, 256 scenes of 2 to 64 bodies
// 60 -> 48 us, 64 bodies of 47 levels (11 blocks a row, in memory) 589 -> 413 us, about half of
// that by the tiles and the staged blocks (12-17 k -> 4.5 k cycles a level).
constexpr int kLdltCols = kSolveThreads;      // one column a thread
constexpr int kLdltWBlocks = kLdltCols / 12;  // bound on a chunk's W blocks
__host__ __device__ inline int64_t ldlt_region(int m) { return 144 * ((int64_t)m * (m + 1) / 2 + kLdltWBlocks); }

// the largest index r in [0, n) with v[r] <= key (v ascending, v[0] <= key)
__device__ __forceinline__ int last_le(const int* v, int n, int key) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (v[mid] <= key) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

__device__ __forceinline__ unsigned long long bits_above(unsigned long long row, int k) {
    return row & ~((2ull << k) - 1ull);
}
__device__ __forceinline__ unsigned long long bits_below(int j) { return (1ull << j) - 1ull; }

// v, recomputed where it is used: comparisons and indices derived from it are not kept in
// registers from an earlier use.
__device__ __forceinline__ int fresh(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

// The pivot columns of a 12x12 block in 16 lanes (a DPP row), row l in p of lane l (lanes 12
// to 15: zeros): for pivot C, out[12 C + q], q < 11, the entries of column C below and then
// above row C (rows C + 1, .., 11, 0, .., C - 1) as pivot C meets them, and out[12 C + 11] the
// reciprocal pivot.  Only the columns above C are still needed.  write: this block exists;
// bad: a pivot was not positive.  Unrolled: as a loop that moves rows and columns up one
// place a pivot it took twice as long (10 k cycles a level, 26 k with 64 bodies).
template <int C, class Out>
__device__ __forceinline__ void pivot_columns(double (&p)[12], Out out, bool write, bool& bad) {
    const int l = fresh(threadIdx.x & 15);
    const double piv = dpp_move<kDppRowBcast + C>(p[C]), f = p[C];
    const double inv = 1.0 / piv;
    bad |= !(piv > 0.0) || !isfinite(piv);
    if (write && l < 12) out[12 * C + l - C + (l > C ? -1 : 11)] = l == C ? inv : f;
    if constexpr (C < 11) {
        double u[12];
#pragma unroll
        for (int j = C + 1; j < 12; ++j) u[j] = dpp_move<kDppRowBcast + C>(p[j]) * inv;
        if (l != C) {
#pragma unroll
            for (int j = C + 1; j < 12; ++j) u[j] = p[j] - f * u[j];
        }
#pragma unroll
        for (int j = C + 1; j < 12; ++j) p[j] = u[j];
        pivot_columns<C + 1>(p, out, write, bad);
    }
}

__global__ __launch_bounds__(kSolveThreads) void ldlt_kernel(Bsr M, const int32_t* __restrict__ sboff,
                                                             const uint8_t* __restrict__ active,
                                                             const double* __restrict__ b, double* __restrict__ xg,
                                                             int64_t region, double* __restrict__ ws,
                                                             int32_t* __restrict__ status, double* __restrict__ resid,
                                                             int dyn_blocks) {
    constexpr int MB = kLdltMaxBodies;
    extern __shared__ __align__(16) double ldlt_dyn[];
    __shared__ unsigned long long adj[MB];   // upper row pattern with fill (bits >= row)
    __shared__ unsigned long long colm[MB];  // colm[i]: the rows k < i whose pattern holds i
    __shared__ unsigned long long levm[MB];  // the bodies of each level
    __shared__ int lvl[MB];                  // the level of each body
    __shared__ unsigned char mlist[MB][MB];  // mlist[k]: the columns above k in row k, ascending
    __shared__ int lrp[MB + 1], pos[MB + 1];
    // the system's CSR entries (at most m^2): slot, and row << 8 | local column, then the
    // factor's block (0xffff: lower, or outside the system)
    __shared__ int eslot[MB * MB];
    __shared__ uint16_t eblk[MB * MB];
    __shared__ int cnode[MB], cstart[MB + 1], sstart[MB + 1], woff[MB];  // the chunk
    __shared__ int nlev, fail, nchunk, nstage;
    __shared__ unsigned long long chunkmask, restm;  // the chunk; the level's bodies not yet eliminated
    __shared__ double y[12 * MB];  // b, then the forward solve, then x
    __shared__ double z[12 * MB];
    __shared__ double sh[17];
    const int sidx = blockIdx.x, t = threadIdx.x, nt = blockDim.x;
    if (active && !active[sidx]) return;
    const int row0 = sboff ? sboff[sidx] : 0;
    const int m = (sboff ? sboff[sidx + 1] : M.nb) - row0;
    if (m > MB) {
        if (t == 0) status[sidx] = kLdltFailed;
        return;
    }
    const int n = 12 * m;
    b += 12 * (int64_t)row0;
    xg += 12 * (int64_t)row0;
    double* U = ws + region * sidx;  // in LDS instead when the factor fits there (below)
    double* W = U + 144 * ((int64_t)m * (m + 1) / 2);
    const int e0 = M.row_ptr[row0];
    if (t <= m) lrp[t] = M.row_ptr[row0 + t] - e0;
    if (t < MB) {
        adj[t] = t < m ? 1ull << t : 0ull;
        levm[t] = 0ull;
    }
    if (t == 0) {
        nlev = 0;
        fail = 0;
    }
    for (int i = t; i < n; i += nt) y[i] = b[i];
    __syncthreads();
    const int nnz = lrp[m];
    if (nnz > MB * MB) {  // more entries than m^2 (blocks coupling other systems): declined
        if (t == 0) status[sidx] = kLdltFailed;
        return;
    }
    for (int e = t; e < nnz; e += nt) {
        const int j = M.cols[e0 + e] - row0;
        const int i = last_le(lrp, m, e);
        eslot[e] = M.slots[e0 + e];
        eblk[e] = j >= i && j < m ? (uint16_t)(i << 8 | j) : (uint16_t)0xffff;
        if (j > i && j < m) atomicOr(&adj[i], 1ull << j);
    }
    __syncthreads();
    // a thread copies element q of blocks e0, e0 + 7, ...; the first kAhead of them are in
    // flight while the structure is found
    constexpr int kAhead = 8, kAtOnce = kSolveThreads / 144;
    const int q0 = t % 144, e0t = t < 144 * kAtOnce ? t / 144 : MB * MB;
    double ahead[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
        const int e = e0t + u * kAtOnce;
        ahead[u] = M.blocks[e < nnz ? 144 * (int64_t)eslot[e] + q0 : 0];
    }
    if (t < 64) {  // wave 0, lane = row: fill, transposed pattern and tree levels, row by row
        unsigned long long mine = t < m ? adj[t] : 0ull, cm = 0ull;
        int h = 0;
        // only rows with entries above the diagonal change anything (fill, colm, a parent's
        // level); fill reaches only later rows, so the rows left are found again after each
        unsigned long long todo = __ballot(t < m && bits_above(mine, t) != 0ull);
        while (todo) {  // uniform
            const int k = __builtin_ctzll(todo);
            // row k is final once k is reached, and so is its level (lane k's values,
            // read by the uniform lane index)
            const unsigned lo32 = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)mine, k);
            const unsigned hi32 = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(mine >> 32), k);
            const unsigned long long ak = ((unsigned long long)hi32 << 32) | lo32;
            const int hk = __builtin_amdgcn_readlane(h, k);
            const unsigned long long above = bits_above(ak, k);
            if ((above >> t) & 1ull) {
                mine |= ak & (~0ull << t);
                cm |= 1ull << k;
            }
            if (above && t == __builtin_ctzll(above) && h < hk + 1) h = hk + 1;
            todo = __ballot(t < m && t > k && bits_above(mine, t) != 0ull);
        }
        if (t < m) {
            adj[t] = mine;
            colm[t] = cm;
            lvl[t] = h;
            atomicOr(&levm[h], 1ull << t);
            atomicMax(&nlev, h + 1);
        }
    }
    __syncthreads();
    if (t < m) {
        int idx = 0;
        for (unsigned long long bt = bits_above(adj[t], t); bt; bt &= bt - 1ull) mlist[t][idx++] = __builtin_ctzll(bt);
    }
    if (t < kWave) {  // wave 0: pos = the exclusive prefix sum of the rows' block counts
        const int cnt = t < m ? __popcll(adj[t]) : 0;
        int incl = cnt;
        for (int off = 1; off < kWave; off <<= 1) {
            const int v = __shfl_up(incl, off, kWave);
            if (t >= off) incl += v;
        }
        if (t < m) pos[t] = incl - cnt;
        const int acc = __shfl(incl, kWave - 1, kWave);
        if (t == 0) {
            pos[m] = acc;
            const int offd = acc - m, wmax = offd < kLdltWBlocks ? offd : kLdltWBlocks;
            fail = acc + wmax <= dyn_blocks ? 2 : 0;  // 2: the factor in LDS (reset below)
        }
    }
    __syncthreads();
    const bool in_lds = fail == 2;  // uniform
    __syncthreads();
    if (t == 0) fail = 0;
    for (int e = t; e < nnz; e += nt)
        if (eblk[e] != 0xffff) {
            const int i = eblk[e] >> 8, j = eblk[e] & 0xff;
            eblk[e] = (uint16_t)(pos[i] + __popcll(adj[i] & bits_below(j)));
        }
    // The factorization and both solves, instantiated for a factor in LDS (its accesses then
    // LDS instructions) and for one in the global workspace; false: a pivot was not positive.
    typedef __attribute__((address_space(3))) double lds_double;
    auto factor_solve = [&](auto U, auto W, auto lds_c) __attribute__((always_inline)) -> bool {
        for (int64_t e = t; e < 144 * (int64_t)pos[m]; e += nt) U[e] = 0.0;
        __syncthreads();
        // the matrix's upper blocks into the factor (row-major 12x12), the lanes reading the
        // slots' 144 doubles in storage order (16 3x3 sub-blocks, sub-block (R/3, C/3) at
        // 9 (R/3 + 4 C/3), row-major inside)
        {
            const int sb = q0 / 9, w9 = q0 % 9;
            auto dst = U + (12 * (3 * (sb & 3) + w9 / 3) + 3 * (sb >> 2) + w9 % 3);
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const int e = e0t + u * kAtOnce;
                if (e < nnz && eblk[e] != 0xffff) dst[144 * (int)eblk[e]] = ahead[u];
            }
            for (int e1 = e0t + kAhead * kAtOnce; e1 < nnz; e1 += 4 * kAtOnce) {
                double v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int e = e1 + u * kAtOnce;
                    v[u] = M.blocks[e < nnz ? 144 * (int64_t)eslot[e] + q0 : 0];
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int e = e1 + u * kAtOnce;
                    if (e < nnz && eblk[e] != 0xffff) dst[144 * (int)eblk[e]] = v[u];
                }
            }
        }
        const int levels = nlev;
        for (int L = 0; L < levels; ++L) {
            if (t == 0) restm = levm[L];
            bool more;
            do {
                __syncthreads();  // the previous chunk is written back, its tables are free
                if (t < kWave) {
                    // wave 0, lane = body: the chunk is the lowest bodies of the level not yet
                    // eliminated whose columns fit kLdltCols and, for a factor in memory, whose
                    // pivot, A' and W blocks fit the LDS (prefix sums in body order; a single
                    // body's columns always fit, one whose blocks do not is a chunk unstaged)
                    const unsigned long long rest = restm;
                    const bool member = t < m && ((rest >> t) & 1ull);
                    const int d = member ? __popcll(bits_above(adj[t], t)) : 0;
                    // columns (16 bits), Schur tiles (24), W blocks (12), bodies
                    const unsigned long long one =
                        member ? (unsigned long long)(12 * (d + 1)) | (unsigned long long)(8 * d * (d + 1)) << 16 |
                                     (unsigned long long)d << 40 | 1ull << 52
                               : 0ull;
                    unsigned long long incl = one;
                    for (int off = 1; off < kWave; off <<= 1) {
                        const unsigned long long v = __shfl_up(incl, off, kWave);
                        if (t >= off) incl += v;
                    }
                    const unsigned long long excl = incl - one;
                    const int ic = (int)(incl & 0xffff), is = (int)(incl >> 16 & 0xffffff), iw = (int)(incl >> 40 & 0xfff);
                    const int c0 = (int)(one & 0xffff), s0 = (int)(one >> 16 & 0xffffff), w0 = d;
                    const int need = (int)(incl >> 52) + 2 * iw;
                    bool take = member && ic <= kLdltCols;
                    if (!in_lds) {
                        const bool first = member && excl == 0;
                        const bool alone = __ballot(first && need > dyn_blocks) != 0;  // unstaged
                        take = take && (alone ? first : need <= dyn_blocks);
                        if (t == 0) nstage = alone ? 0 : 1;
                    }
                    const unsigned long long cmask = __ballot(take);
                    const int nc = __popcll(cmask);
                    if (take) {
                        const int q = __popcll(cmask & bits_below(t));
                        cnode[q] = t;
                        cstart[q] = ic - c0;
                        sstart[q] = is - s0;
                        woff[t] = iw - w0;
                        if (q == nc - 1) {
                            cstart[nc] = ic;
                            sstart[nc] = is;
                        }
                    }
                    if (t == 0) {
                        nchunk = nc;
                        chunkmask = cmask;
                        restm = rest & ~cmask;
                    }
                }
                __syncthreads();
                const int nc = nchunk;
                more = restm != 0ull;  // read here: written again only after the chunk's barriers
                const unsigned long long cmask = chunkmask;
                const int C = cstart[nc];
                // F: the bodies' pivot columns, then P^-1 (over P, or block ln of the stage);
                // Ab: their A' blocks from aoff; Wb: their W blocks from woff
                auto eliminate = [&](auto Fb, auto Wb, auto Ab, auto staged_c) __attribute__((always_inline)) -> bool {
                    constexpr bool staged = decltype(staged_c)::value;
                    auto foff = [&](int ln, int k) { return 144 * (int64_t)(staged ? ln : pos[k]); };
                    auto aoff = [&](int k) { return 144 * (int64_t)(staged ? woff[k] : pos[k] + 1); };
                    if (4 * (t / kWave) < nc) {  // uniform over the wave: its four bodies' pivots
                        const int q = t >> 4, kq = cnode[q < nc ? q : 0], l = t & 15;
                        double p[12];
                        const auto src = U + 144 * (int64_t)pos[kq] + 12 * l;
#pragma unroll
                        for (int j = 0; j < 12; ++j) p[j] = q < nc && l < 12 ? src[j] : 0.0;
                        bool bad = false;
                        pivot_columns<0>(p, Fb + foff(q, kq), q < nc, bad);
                        if (bad && q < nc) fail = 1;
                    }
                    double a[12];
                    const int col = t;
                    int ln = -1, k = 0, g = 0, c = 0, d = 0;
                    if (col < C) {
                        ln = last_le(cstart, nc, col);
                        k = cnode[ln];
                        const int within = col - cstart[ln];
                        g = within / 12;
                        c = within % 12;
                        d = (cstart[ln + 1] - cstart[ln]) / 12 - 1;
                        if (g < d) {
                            const auto src = U + 144 * (int64_t)(pos[k] + 1 + g) + c;
#pragma unroll
                            for (int r = 0; r < 12; ++r) a[r] = src[12 * r];
                            if (staged) {
                                auto dst = Ab + aoff(k) + 144 * g + c;
#pragma unroll
                                for (int r = 0; r < 12; ++r) dst[12 * r] = a[r];
                            }
                        } else {
#pragma unroll
                            for (int r = 0; r < 12; ++r) a[r] = r == c ? 1.0 : 0.0;
                        }
                    }
                    __syncthreads();
                    if (fail) {  // uniform
                        if (t == 0) status[sidx] = kLdltFailed;
                        return false;
                    }
                    if (ln >= 0) {
                        // each pivot's entry is first in turn: the others move up one place
                        auto F = Fb + foff(ln, k);
                        double f[12];
#pragma unroll
                        for (int r = 0; r < 12; ++r) f[r] = F[r];
#pragma unroll 1
                        for (int pc = 0; pc < 12; ++pc) {
                            double next[12];  // the next pivot's column, in flight meanwhile
                            if (pc < 11) F += 12;
#pragma unroll
                            for (int r = 0; r < 12; ++r) next[r] = F[r];
                            const double sc = a[0] * f[11];
#pragma unroll
                            for (int r = 0; r < 11; ++r) a[r] = a[r + 1] - f[r] * sc;
                            a[11] = sc;
#pragma unroll
                            for (int r = 0; r < 12; ++r) f[r] = next[r];
                        }
                        if (g < d) {
                            auto dst = Wb + 144 * (int64_t)(woff[k] + g) + c;
#pragma unroll
                            for (int r = 0; r < 12; ++r) dst[12 * r] = a[r];
                        }
                    }
                    __syncthreads();
                    if (ln >= 0 && g == d) {  // P^-1 over the pivot columns, all read
                        auto dst = Fb + foff(ln, k) + c;
#pragma unroll
                        for (int r = 0; r < 12; ++r) dst[12 * r] = a[r];
                    }
                    // Schur complement: 3x3 tiles of target (i, j), i <= j, updated by the thread of
                    // its lowest contributor in the chunk, the contributors in ascending order
                    for (int w = t; w < sstart[nc]; w += nt) {
                        const int l2 = last_le(sstart, nc, w);
                        const int k1 = cnode[l2], within = w - sstart[l2];
                        const int pidx = within >> 4, ta = 3 * (within >> 2 & 3), tb = 3 * (within & 3);
                        int v = (int)((__builtin_sqrtf(8.0f * pidx + 1.0f) - 1.0f) * 0.5f);
                        while (v * (v + 1) / 2 > pidx) --v;
                        while ((v + 1) * (v + 2) / 2 <= pidx) ++v;
                        const int i = mlist[k1][pidx - v * (v + 1) / 2], j = mlist[k1][v];
                        const unsigned long long contrib = cmask & colm[i] & colm[j];
                        const int rank = __popcll(contrib & bits_below(k1));
                        if (decltype(lds_c)::value && __popcll(contrib) >= 3) {
                            // a row of the tile each for the threads of the three lowest: one
                            // thread's nine sums over many contributors would be the level's
                            // chain (20 bodies coupled to one: 53 us, 40 here).  Only where the
                            // factor is in LDS: the other two instances too would take 40 bodies
                            // coupled so from 95 to 80 us, but every solve 1 us more, in code
                            // and spilled registers (256 scenes 51 to 52)
                            if (rank >= 3) continue;
                            auto tgt = U + 144 * (int64_t)(pos[i] + __popcll(adj[i] & bits_below(j))) +
                                       12 * (ta + rank) + tb;
                            double val[3] = {tgt[0], tgt[1], tgt[2]};
                            for (unsigned long long bt = contrib; bt; bt &= bt - 1ull) {
                                const int k2 = __builtin_ctzll(bt);
                                const unsigned long long ab = bits_above(adj[k2], k2);
                                const auto Aki = Ab + aoff(k2) + 144 * __popcll(ab & bits_below(i)) + ta + rank;
                                const auto Wj = Wb + 144 * (int64_t)(woff[k2] + __popcll(ab & bits_below(j))) + tb;
                                double acc[3] = {0.0, 0.0, 0.0};
#pragma unroll 4
                                for (int r = 0; r < 12; ++r)
#pragma unroll
                                    for (int q = 0; q < 3; ++q) acc[q] += Aki[12 * r] * Wj[12 * r + q];
#pragma unroll
                                for (int q = 0; q < 3; ++q) val[q] -= acc[q];
                            }
#pragma unroll
                            for (int q = 0; q < 3; ++q) tgt[q] = val[q];
                            continue;
                        }
                        if (rank) continue;
                        auto tgt = U + 144 * (int64_t)(pos[i] + __popcll(adj[i] & bits_below(j))) + 12 * ta + tb;
                        double val[9];
#pragma unroll
                        for (int q = 0; q < 9; ++q) val[q] = tgt[12 * (q / 3) + q % 3];
                        for (unsigned long long bt = contrib; bt; bt &= bt - 1ull) {
                            const int k2 = __builtin_ctzll(bt);
                            const unsigned long long ab = bits_above(adj[k2], k2);
                            const auto Aki = Ab + aoff(k2) + 144 * __popcll(ab & bits_below(i)) + ta;
                            const auto Wj = Wb + 144 * (int64_t)(woff[k2] + __popcll(ab & bits_below(j))) + tb;
                            double acc[9];
#pragma unroll
                            for (int q = 0; q < 9; ++q) acc[q] = 0.0;
#pragma unroll 4
                            for (int r = 0; r < 12; ++r) {
                                const double x[3] = {Aki[12 * r], Aki[12 * r + 1], Aki[12 * r + 2]};
                                const double y3[3] = {Wj[12 * r], Wj[12 * r + 1], Wj[12 * r + 2]};
#pragma unroll
                                for (int q = 0; q < 9; ++q) acc[q] += x[q / 3] * y3[q % 3];
                            }
#pragma unroll
                            for (int q = 0; q < 9; ++q) val[q] -= acc[q];
                        }
#pragma unroll
                        for (int q = 0; q < 9; ++q) tgt[12 * (q / 3) + q % 3] = val[q];
                    }
                    // forward solve: y_i -= W_i^T y_k over the chunk's bodies k coupled to i, ascending
                    for (int w = t; w < n; w += nt) {
                        const int i = w / 12, a2 = w % 12;
                        unsigned long long bt = cmask & colm[i];
                        if (!bt) continue;
                        double val = y[w];
                        for (; bt; bt &= bt - 1ull) {
                            const int k2 = __builtin_ctzll(bt);
                            const unsigned long long ab = bits_above(adj[k2], k2);
                            const auto Wi = Wb + 144 * (int64_t)(woff[k2] + __popcll(ab & bits_below(i))) + a2;
                            double acc = 0.0;
#pragma unroll
                            for (int r = 0; r < 12; ++r) acc += Wi[12 * r] * y[12 * k2 + r];
                            val -= acc;
                        }
                        y[w] = val;
                    }
                    __syncthreads();
                    // z_k = P^-1 y_k for the chunk's bodies
                    for (int w = t; w < 12 * nc; w += nt) {
                        const int kz = cnode[w / 12], a2 = w % 12;
                        const auto Di = Fb + foff(w / 12, kz) + 12 * a2;
                        double acc = 0.0;
#pragma unroll
                        for (int r = 0; r < 12; ++r) acc += Di[r] * y[12 * kz + r];
                        z[12 * kz + a2] = acc;
                    }
                    // rows of the factor: W (read back: kept in registers over the tiles it spills)
                    if (ln >= 0 && g < d) {
                        auto dst = U + 144 * (int64_t)(pos[k] + 1 + g) + c;
                        const auto src = Wb + 144 * (int64_t)(woff[k] + g) + c;
#pragma unroll
                        for (int r = 0; r < 12; ++r) dst[12 * r] = src[12 * r];
                    }
                    return true;
                };
                bool ok;
                if constexpr (decltype(lds_c)::value) {
                    ok = eliminate(U, W, U, std::false_type{});
                } else if (nstage) {  // uniform
                    lds_double* St = (lds_double*)ldlt_dyn;
                    const int nw = (C / 12 - nc);
                    ok = eliminate(St, St + 144 * nc, St + 144 * (nc + nw), std::true_type{});
                } else {
                    ok = eliminate(U, W, U, std::false_type{});
                }
                if (!ok) return false;
            } while (more);  // uniform; every level has a body
        }
        // backward solve, levels from the top
        for (int L = levels - 1; L >= 0; --L) {
            __syncthreads();
            for (int w = t; w < n; w += nt) {
                const int k = w / 12, a2 = w % 12;
                if (lvl[k] != L) continue;
                double acc = 0.0;
                int u = 0;
                for (unsigned long long bt = bits_above(adj[k], k); bt; bt &= bt - 1ull, ++u) {
                    const int i = __builtin_ctzll(bt);
                    const auto Wu = U + 144 * (int64_t)(pos[k] + 1 + u) + 12 * a2;
                    double p = 0.0;
    #pragma unroll
                    for (int c = 0; c < 12; ++c) p += Wu[c] * y[12 * i + c];
                    acc += p;
                }
                y[w] = z[w] - acc;
            }
        }
        return true;
    };
    bool ok;
    if (in_lds) {
        lds_double* Ul = (lds_double*)ldlt_dyn;
        ok = factor_solve(Ul, Ul + 144 * (int64_t)pos[m], std::true_type{});
    } else {
        ok = factor_solve(U, W, std::false_type{});
    }
    if (!ok) return;
    __syncthreads();
    for (int i = t; i < n; i += nt) xg[i] = y[i];
    double rr = 0.0;
    if (resid) {  // uniform: the residual's product with H only when asked for
        Rows R{row0, m, nullptr, nullptr, nullptr};
        for (int i = t; i < n; i += nt) {
            const int lr = i % 12;
            const double r = b[i] - row_product<kSpmvRows>(M, R, i / 12, lr / 3, lr % 3, y);
            rr += r * r;
        }
        rr = block_sum_fast(rr, sh);
    }
    if (t == 0) {
        status[sidx] = 1;
        if (resid) resid[sidx] = rr;
    }
}

// Algorithmic bytes of one solve launch, summed over its systems: per iteration
// each SpMV streams the system's blocks (144 doubles), column and slot ids, and
// row pointers; with vectors outside LDS, ~10 vector passes of 12 n doubles too.
__global__ void solve_bytes_kernel(const int32_t* __restrict__ row_ptr, int nb, const int32_t* __restrict__ sboff,
                                   const uint8_t* __restrict__ active, int nsys, const int32_t* __restrict__ iters,
                                   int spmv_per_it, int lds, double precond_per_body, double* __restrict__ out) {
    __shared__ double sh[17];
    double acc = 0.0;
    for (int s = threadIdx.x; s < nsys; s += blockDim.x) {
        if (active && !active[s]) continue;  // not solved in this launch
        const int r0 = sboff ? sboff[s] : 0, r1 = sboff ? sboff[s + 1] : nb;
        const double nnzb = (double)(row_ptr[r1] - row_ptr[r0]);
        const double nbs = (double)(r1 - r0);
        const double per_it = spmv_per_it * (1160.0 * nnzb + 4.0 * (nbs + 1)) + (lds ? 0.0 : 10.0 * 96.0 * nbs) +
                              precond_per_body * nbs;
        const int it = iters[s] > 0 ? iters[s] : 0;
        acc += per_it * it;
    }
    const double r = block_sum_fast(acc, sh);
    if (threadIdx.x == 0) *out = r;
}

// ---------------------------------------------------------------------------
// Jacobi CG of bsr_utils.py:126-235 (or its 12x12 block-Jacobi form) for one system
// too large for one workgroup's LDS (more than kLargeBodies bodies): the rows are split
// over workgroups of kMwThreads (kMwBjThreads, whole bodies, for the block form; one row
// per thread), and each iteration is two launches —
// [beta, p = z + beta p and its SpMV, partial p.Ap], [alpha, x / r / z update + partial r.z]:
// a workgroup forms the directions of the bodies its rows couple to itself (the same
// arithmetic in every workgroup), so the SpMV needs no launch between (1024 bodies, ten
// iterations: 30 launches of 2.2 to 3 us became 20 of 2.9 and 3.3 us and a check; a frame of
// ten such solves 4.05 -> 3.91 ms).
// Every workgroup reduces the per-workgroup partials itself, in workgroup order,
// so all of them hold the same scalars and the sequence is deterministic.  The
// stopping test (every check_every iterations) is a launch of its own at a batch's
// end; the host reads its flag once per batch.
constexpr int kMwThreads = 256;
constexpr int kMwBjThreads = 192;  // 16 bodies of 12 rows
static_assert(kMwBjThreads % 12 == 0 && kMwBjThreads <= kMwThreads, "whole bodies per block-Jacobi workgroup");
constexpr int kLargeBodies = 170;  // from here one workgroup's SpMV is the bottleneck

struct MwState {
    double* x;
    double* r;
    double* p[2];   // the directions of even and odd iterations
    double* Ap;
    double* z;
    double* dg;
    double* part;   // [2][nblk]: partials of p.Ap and r.z
    double* rz;     // [2]: r.z of the current iteration (slot i % 2) and the next
    double* err;    // final r.z
    int32_t* done;  // 1 once stopped
    int32_t* it;    // end_iter
};

// the workgroups' partials as a workgroup of `rows` threads adds them (waves past those add 0)
__device__ __forceinline__ double mw_sum(const double* __restrict__ part, int nblk, double* sh, int rows) {
    double acc = 0.0;
    if ((int)threadIdx.x < rows)
        for (int k = threadIdx.x; k < nblk; k += rows) acc += part[k];
    return block_sum_fast(acc, sh);
}

__device__ __forceinline__ double mw_row(const Bsr& M, const double* __restrict__ in, int idx) {
    const int b = idx / 12, lr = idx % 12, ii = lr / 3, k = lr % 3;
    double acc = 0.0;
    for (int e = M.row_ptr[b]; e < M.row_ptr[b + 1]; ++e) {
        const double* xin = in + 12 * (int64_t)M.cols[e];
        const double* base = M.blocks + 9 * 16 * (int64_t)M.slots[e] + 3 * k;
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
            const double* B = base + 9 * (ii + 4 * jj);
            acc += B[0] * xin[3 * jj] + B[1] * xin[3 * jj + 1] + B[2] * xin[3 * jj + 2];
        }
    }
    return acc;
}

__device__ __forceinline__ double mw_jacobi(const double* __restrict__ dg, const double r, int i) {
    const int i3 = i - i % 3;
    const double d0 = dg[i3], d1 = dg[i3 + 1], d2 = dg[i3 + 2];
    return (d0 * d0 + d1 * d1 + d2 * d2 == 0.0) ? r : r / fabs(dg[i]);
}

// Block-Jacobi preconditioner of row i: z_i = (D_b^-1 r_b)_i with the 12 residuals of body b
// in rs (LDS, the workgroup's rows; a workgroup of kMwBjThreads rows holds whole bodies).
__device__ __forceinline__ double mw_block_precond(const double* __restrict__ dinv, const double* rs, int i) {
    const int lr = i % 12;
    const double* Di = dinv + 144 * (int64_t)(i / 12) + 12 * lr;
    const double* rb = rs + (threadIdx.x - lr);
    double acc = 0.0;
#pragma unroll
    for (int q = 0; q < 12; ++q) acc += Di[q] * rb[q];
    return acc;
}

// setup: diagonal, x = x0, r = b - H x, z, p = z, partial r.z
template <bool BJ>
__global__ __launch_bounds__(kMwThreads) void mw_init_kernel(Bsr M, const double* __restrict__ b,
                                                             const double* __restrict__ xg, MwState W,
                                                             const double* __restrict__ dinv) {
    __shared__ double sh[17];
    __shared__ double rs[BJ ? kMwThreads : 1];
    const int n = 12 * M.nb;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    double part = 0.0, r = 0.0, z = 0.0;
    if (i < n) {
        // bsr_get_diag: the three diagonal entries of this row's 3x3 diagonal sub-block (a
        // 3-row group may straddle two workgroups, so each thread reads all three itself)
        const int bb = i / 12, ii = (i % 12) / 3, a = i % 3;
        const double* D = M.blocks + 9 * (16 * (int64_t)bb + ii + 4 * ii);
        const double d[3] = {D[0], D[4], D[8]};
        W.dg[i] = d[a];
        W.x[i] = xg[i];
        r = b[i] - mw_row(M, xg, i);
        W.r[i] = r;
        if (!BJ) z = (d[0] * d[0] + d[1] * d[1] + d[2] * d[2] == 0.0) ? r : r / fabs(d[a]);
    }
    if (BJ) {
        rs[threadIdx.x] = r;
        __syncthreads();
        if (i < n) z = mw_block_precond(dinv, rs, i);
    }
    if (i < n) {
        W.z[i] = z;
        W.p[0][i] = z;
        part = r * z;
    }
    const double t = block_sum_fast(part, sh);
    if (threadIdx.x == 0) W.part[gridDim.x + blockIdx.x] = t;
}

__global__ __launch_bounds__(kMwThreads) void mw_start_kernel(int nblk, double tol_sq, int maxiter, MwState W) {
    __shared__ double sh[17];
    const double rz = mw_sum(W.part + nblk, nblk, sh, blockDim.x);
    if (threadIdx.x == 0) {
        W.rz[0] = rz;
        *W.err = rz;
        *W.it = rz > tol_sq ? maxiter : 0;
        *W.done = rz > tol_sq ? 0 : 1;
    }
}

// What one of a row's two lanes takes of kMwEntries entries from e on: six of the multiplied
// vector's values, from q0 on (as it stands, or z and p_old), and the rows of their sub-blocks.
constexpr int kMwLanes = 2, kMwEntries = 3;
struct MwPart {
    double z[6], p[6], B[6];
};
template <bool STORED>
__device__ __forceinline__ void mw_load(const Bsr& M, const double* __restrict__ z, const double* __restrict__ p_old,
                                        int e, int e1, int at, int q0, MwPart (&E)[kMwEntries]) {
    if (e >= e1) return;
    int col[kMwEntries], slot[kMwEntries];
#pragma unroll
    for (int u = 0; u < kMwEntries; ++u) {
        const int q = e + u < e1 ? e + u : e;
        col[u] = M.cols[q];
        slot[u] = M.slots[q];
    }
#pragma unroll
    for (int u = 0; u < kMwEntries; ++u)
        if (e + u < e1) {
            const int64_t c = 12 * (int64_t)col[u] + q0;
            const double* B = M.blocks + 144 * (int64_t)slot[u] + at;
#pragma unroll
            for (int q = 0; q < 6; ++q) {
                E[u].z[q] = z[c + q];
                if (!STORED) E[u].p[q] = p_old[c + q];
                E[u].B[q] = B[36 * (q / 3) + q % 3];
            }
        }
}

// iteration i, part 1: the beta of iteration i - 1, this iteration's direction (FIRST: z
// already), its SpMV (mw_row's sums) and partial p.Ap.  Two lanes a row, each with two of an
// entry's four 3x3 sub-blocks, whose parts both add in order; kRows rows a workgroup: those of
// the other launches, whose sums it shares.
// Bound by the latency of a row's entries: three are in flight (242 VGPRs: a workgroup a CU is
// all there is to run), the first three while the partials of r.z are summed.  An iteration of
// 600 bodies with 4, 24 and 100 couplings each (block form) 17, 31 and 84 us, the product of a
// plate under 400 cubes 91.  One thread a row with an entry at a time took 20, 43, 184 and 157;
// four lanes a row with four entries 17, 34, 93 and 71, but 8 to 28 % more in the Jacobi form,
// whose registers hold two; a direction kernel before a product that then reads one vector for
// two 19, 33, 104 and 90.
template <int kRows, bool FIRST>
__global__ __launch_bounds__(kMwLanes * kRows) void mw_spmv_kernel(Bsr M, int iter, double tol_sq, MwState W) {
    __shared__ double sh[17];
    __shared__ double parts[kRows];
    if (*W.done) return;
    const int n = 12 * M.nb, nblk = gridDim.x, t = threadIdx.x;
    const int row = t / kMwLanes, l = t % kMwLanes, i = blockIdx.x * kRows + row, b = i / 12, lr = i % 12;
    const int q0 = 6 * l, at = 9 * (lr / 3) + 3 * (lr % 3) + 12 * q0;
    const double* z = FIRST ? W.p[0] : W.z;
    const double* p_old = W.p[(iter - 1) & 1];
    const int e0 = i < n ? M.row_ptr[b] : 0, e1 = i < n ? M.row_ptr[b + 1] : 0;
    MwPart E[kMwEntries];
    mw_load<FIRST>(M, z, p_old, e0, e1, at, q0, E);
    double beta = 0.0;
    if (!FIRST) {
        const double rz_new = mw_sum(W.part + nblk, nblk, sh, kRows);
        beta = rz_new > tol_sq ? rz_new / W.rz[(iter - 1) & 1] : 0.0;
        if (blockIdx.x == 0 && t == 0) {
            W.rz[iter & 1] = rz_new;
            *W.err = rz_new;
        }
    }
    double acc = 0.0;
    for (int e = e0; e < e1; e += kMwEntries) {
        if (e != e0) mw_load<FIRST>(M, z, p_old, e, e1, at, q0, E);
#pragma unroll
        for (int u = 0; u < kMwEntries; ++u)
            if (e + u < e1) {
                double v[2];
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    double x[3];
#pragma unroll
                    for (int q = 0; q < 3; ++q)
                        x[q] = FIRST ? E[u].z[3 * k + q] : E[u].z[3 * k + q] + beta * E[u].p[3 * k + q];
                    v[k] = E[u].B[3 * k] * x[0] + E[u].B[3 * k + 1] * x[1] + E[u].B[3 * k + 2] * x[2];
                }
                acc += dpp_move<kDppPair0>(v[0]);
                acc += dpp_move<kDppPair0>(v[1]);
                acc += dpp_move<kDppPair1>(v[0]);
                acc += dpp_move<kDppPair1>(v[1]);
            }
    }
    if (l == 0) {
        double part = 0.0;
        if (i < n) {
            const double p = FIRST ? z[i] : z[i] + beta * p_old[i];
            if (!FIRST) W.p[iter & 1][i] = p;
            W.Ap[i] = acc;
            part = p * acc;
        }
        parts[row] = part;
    }
    __syncthreads();
    const double sum = block_sum_fast(t < kRows ? parts[t] : 0.0, sh);
    if (t == 0) W.part[blockIdx.x] = sum;
}

// part 2: alpha, x / r / z update, partial r.z
template <bool BJ>
__global__ __launch_bounds__(kMwThreads) void mw_update_kernel(int n, int iter, MwState W,
                                                               const double* __restrict__ dinv) {
    __shared__ double sh[17];
    __shared__ double rs[BJ ? kMwThreads : 1];
    if (*W.done) return;  // uniform over the grid
    const int nblk = gridDim.x;
    const double pAp = mw_sum(W.part, nblk, sh, blockDim.x);
    const double rz_old = W.rz[iter & 1];
    // unguarded in the reference: p = 0 once the residual vanishes exactly between checks
    const double alpha = pAp != 0.0 ? rz_old / pAp : 0.0;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    double part = 0.0, r = 0.0, z = 0.0;
    if (i < n) {
        W.x[i] += alpha * W.p[iter & 1][i];
        r = W.r[i] - alpha * W.Ap[i];
        W.r[i] = r;
        if (!BJ) z = mw_jacobi(W.dg, r, i);
    }
    if (BJ) {
        rs[threadIdx.x] = r;
        __syncthreads();
        if (i < n) z = mw_block_precond(dinv, rs, i);
    }
    if (i < n) {
        W.z[i] = z;
        part = r * z;
    }
    const double t = block_sum_fast(part, sh);
    if (threadIdx.x == 0) W.part[nblk + blockIdx.x] = t;
}

// the end of a batch, whose last iteration is `iter`: its stopping test (every check_every
// iterations), for the host.  One workgroup of the iterations' own size, so that the sum it
// decides by is the one they take; no launch that reads *W.done across workgroups writes it.
__global__ __launch_bounds__(kMwThreads) void mw_check_kernel(int nblk, int iter, int check_every, double tol_sq,
                                                              MwState W) {
    __shared__ double sh[17];
    if (*W.done) return;
    const double rz_new = mw_sum(W.part + nblk, nblk, sh, blockDim.x);
    if (threadIdx.x != 0) return;
    *W.err = rz_new;
    if ((iter + 1) % check_every == 0 && rz_new <= tol_sq) {
        *W.done = 1;
        *W.it = iter;
    }
}

__global__ void mw_finish_kernel(int n, MwState W, double* __restrict__ xg, int32_t* __restrict__ iters,
                                 double* __restrict__ resid) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) xg[i] = W.x[i];
    if (i == 0) {
        if (iters) *iters = *W.it;
        if (resid) *resid = *W.err;
    }
}

bool solve_waits(int32_t method, int nb) {
    return nb > kLargeBodies && method != ABD_SOLVER_BICGSTAB;  // solve_cg_multi
}

}  // namespace abd

using namespace abd;

extern "C" {

namespace {
// Workgroup size of a solve of systems of up to max_bodies bodies: the smallest whose
// threads hold every row and a matrix with all its max_bodies^2 blocks (regs_fit); else 16 waves, which keep enough loads in flight where a matrix stays in
// memory.  A system's sums are the same for every size (each thread owns at most the rows
// it has in the largest; absent waves add 0), so a scene gives the same bits on its own or
// in a batch.
int solve_threads(int max_bodies) {
    for (int t : {kWave, 4 * kWave})
        if (12 * (int64_t)max_bodies <= t && 4 * (int64_t)max_bodies * max_bodies <= t) return t;
    return kSolveThreads;
}

int launch_solve(hipStream_t s, int32_t method, const Bsr& M, int nsys, const int32_t* sboff, const uint8_t* active,
                 int max_rows, const double* b, double* x, double tol, int32_t maxiter, int32_t check_every,
                 int32_t* iters, double* resid, int threads, const int32_t* pending = nullptr) {
    const int n_all = 12 * M.nb;
    double* ws;
    int rc = arena_get(kSlotSolver, sizeof(double) * 6 * (size_t)n_all, (void**)&ws);
    if (rc) return rc;
    const bool bj = method == ABD_SOLVER_CG_BLOCK;
    double* dinv = nullptr;
    if (bj && (rc = arena_get(kSlotPrecond, sizeof(double) * 144 * (size_t)M.nb, (void**)&dinv))) return rc;
    if (bj) {
        // every body's diagonal-block inverse, one 64-thread workgroup per body (inactive scenes
        // included: cheap)
        if (M.nb > 0) {
            // algorithmic bytes: each diagonal block read, its inverse written
            const int ph_inv = pending ? -1 : prof_start(kProfPrecond, s, 2304.0 * M.nb);
            launch_kernel(invert_blocks_kernel, dim3(M.nb), dim3(kInvThreads), 0, s, M, dinv, pending, sboff,
                               nsys);
            ABD_CHECK_LAUNCH();
            prof_stop(ph_inv, s);
        }
    }
    // the fallback of a direct solve is timed with it (its launch returns at once unless a
    // system was declined)
    int ph = pending ? -1 : prof_start(kProfSolve, s, 1.0);
    const size_t vec_bytes = sizeof(double) * 6 * (size_t)max_rows;
    // dynamic LDS: the whole budget of the device (beside the kernels' static LDS) when it
    // holds the structure region, the vectors in it when they fit beside the structure
    int dev = 0, max_lds = 0;
    ABD_CHECK(hipGetDevice(&dev));
    ABD_CHECK(hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    const size_t usable = (size_t)max_lds > 1024 ? (size_t)max_lds - 1024 : 0;
    const bool staged = usable >= kLdsStructBytes + 8 * 1024;
    const int budget = staged ? (int)usable : -1;
    const bool lds = staged && kLdsStructBytes + vec_bytes <= usable;
    const size_t dyn = staged ? usable : 0;
    static bool attr_set = false;
    static std::mutex attr_mu;  // the first calls of several threads
    std::unique_lock<std::mutex> attr_lock(attr_mu);
    if (!attr_set) {
        const int cap = (int)usable;
        const void* fns[] = {(const void*)bicgstab_kernel<true, kWave>,
                             (const void*)bicgstab_kernel<true, 4 * kWave>,
                             (const void*)bicgstab_kernel<true, kSolveThreads>,
                             (const void*)bicgstab_kernel<false, kSolveThreads>,
                             (const void*)cg_kernel<true, false, kWave>,
                             (const void*)cg_kernel<true, false, 4 * kWave>,
                             (const void*)cg_kernel<true, false, kSolveThreads>,
                             (const void*)cg_kernel<true, true, kSolveThreads>,
                             (const void*)cg_kernel<false, false, kSolveThreads>,
                             (const void*)cg_kernel<false, true, kSolveThreads>};
        for (const void* f : fns) ABD_CHECK(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, cap));
        attr_set = true;
    }
    attr_lock.unlock();
    if (bj || !lds) threads = kSolveThreads;
    auto bicgstab = bicgstab_kernel<false, kSolveThreads>;
    auto cg = cg_kernel<false, false, kSolveThreads>;
    if (lds && threads == kWave) {
        bicgstab = bicgstab_kernel<true, kWave>;
        cg = cg_kernel<true, false, kWave>;
    } else if (lds && threads == 4 * kWave) {
        bicgstab = bicgstab_kernel<true, 4 * kWave>;
        cg = cg_kernel<true, false, 4 * kWave>;
    } else if (lds) {
        bicgstab = bicgstab_kernel<true, kSolveThreads>;
        cg = bj ? cg_kernel<true, true, kSolveThreads> : cg_kernel<true, false, kSolveThreads>;
    } else if (bj) {
        cg = cg_kernel<false, true, kSolveThreads>;
    }
    if (method == ABD_SOLVER_BICGSTAB)
        launch_kernel(bicgstab, dim3(nsys), dim3(threads), dyn, s, M, sboff, active, b, x, tol, maxiter,
                           check_every, max_rows, budget, ws, iters, resid);
    else
        launch_kernel(cg, dim3(nsys), dim3(threads), dyn, s, M, sboff, active, b, x, tol, maxiter, check_every,
                           max_rows, budget, ws, dinv, iters, resid, pending);
    ABD_CHECK_LAUNCH();
    prof_stop(ph, s);
    if (ph >= 0 && iters) {
        // the byte count needs the iteration counts: computed behind the solve, on its stream
        double* dbytes;
        if ((rc = arena_get(kSlotSolveBytes, sizeof(double), (void**)&dbytes))) return rc;
        launch_kernel(solve_bytes_kernel, dim3(1), dim3(256), 0, s, M.row_ptr, M.nb, sboff, active, nsys, iters,
                           method == ABD_SOLVER_BICGSTAB ? 2 : 1, lds ? 1 : 0, bj ? 1152.0 : 0.0, dbytes);
        ABD_CHECK_LAUNCH();
        prof_stop(ph, s, nullptr, dbytes);
    } else {
        prof_stop(ph, s);
    }
    return ABD_OK;
}
// The direct solve (ldlt_kernel) of every system of at most kLdltMaxBodies bodies, then
// the block-Jacobi CG of the systems it declined (status kLdltFailed in iters).
int launch_ldlt(hipStream_t s, const Bsr& M, int nsys, const int32_t* sboff, const uint8_t* active, int max_bodies,
                const double* b, double* x, double tol, int32_t maxiter, int32_t check_every, int32_t* iters,
                double* resid) {
    int rc;
    int32_t* status = iters;
    if (!status && (rc = arena_get(kSlotLdltStatus, sizeof(int32_t) * (size_t)nsys, (void**)&status))) return rc;
    const int cap = max_bodies < kLdltMaxBodies ? max_bodies : kLdltMaxBodies;
    const int64_t region = ldlt_region(cap);
    double* ws;
    if ((rc = arena_get(kSlotLdlt, sizeof(double) * (size_t)region * (size_t)nsys, (void**)&ws))) return rc;
    // dynamic LDS: the device's budget beside the kernel's static LDS, in whole blocks
    static int dyn_bytes = -1;
    static std::mutex dyn_mu;  // the first calls of several threads
    std::unique_lock<std::mutex> dyn_lock(dyn_mu);
    if (dyn_bytes < 0) {
        int dev = 0, max_lds = 0;
        ABD_CHECK(hipGetDevice(&dev));
        ABD_CHECK(hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
        hipFuncAttributes fa;
        ABD_CHECK(hipFuncGetAttributes(&fa, (const void*)ldlt_kernel));
        const int avail = max_lds - (int)fa.sharedSizeBytes - 256;
        dyn_bytes = avail > 0 ? (avail / 1152) * 1152 : 0;
        if (dyn_bytes > 0)
            ABD_CHECK(hipFuncSetAttribute((const void*)ldlt_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                          dyn_bytes));
    }
    dyn_lock.unlock();
    const int ph = prof_start_ext(kProfSolve, 1.0);
    prof_launch(ph, ldlt_kernel, dim3(nsys), dim3(kSolveThreads), (uint32_t)dyn_bytes, s, M, sboff, active, b, x,
                region, ws, status, resid, dyn_bytes / 1152);
    ABD_CHECK_LAUNCH();
    if (ph >= 0) {
        // algorithmic bytes of the systems solved directly: each block, b and x once
        double* dbytes;
        if ((rc = arena_get(kSlotSolveBytes, sizeof(double), (void**)&dbytes))) return rc;
        launch_kernel(solve_bytes_kernel, dim3(1), dim3(256), 0, s, M.row_ptr, M.nb, sboff, active, nsys,
                           (const int32_t*)status, 1, 1, 192.0, dbytes);
        ABD_CHECK_LAUNCH();
        prof_stop(ph, s, nullptr, dbytes);
    }
    if ((rc = launch_solve(s, ABD_SOLVER_CG_BLOCK, M, nsys, sboff, active, 12 * max_bodies, b, x, tol, maxiter,
                           check_every, status, resid, solve_threads(max_bodies), status)))
        return rc;
    return ABD_OK;
}
}  // namespace

// Jacobi (bj: 12x12 block-Jacobi) CG over several workgroups (systems of more than
// kLargeBodies bodies).  The block-Jacobi form runs kMwBjThreads rows per workgroup so that
// every body's 12 rows share one.
int solve_cg_multi(hipStream_t s, const Bsr& M, const double* b, double* x, double tol, int32_t maxiter,
                   int32_t check_every, int32_t* iters, double* resid, bool bj) {
    const int n = 12 * M.nb;
    const int threads = bj ? kMwBjThreads : kMwThreads;
    const int nblk = (n + threads - 1) / threads;
    if (maxiter <= 0) maxiter = n;
    double* ws;
    const size_t nd = 7 * (size_t)n + 2 * (size_t)nblk + 3;
    int rc = arena_get(kSlotSolver, sizeof(double) * nd + 2 * sizeof(int32_t) + 16, (void**)&ws);
    if (rc) return rc;
    MwState W;
    W.x = ws;
    W.r = ws + n;
    W.p[0] = ws + 2 * (size_t)n;
    W.p[1] = ws + 6 * (size_t)n;
    W.Ap = ws + 3 * (size_t)n;
    W.z = ws + 4 * (size_t)n;
    W.dg = ws + 5 * (size_t)n;
    W.part = ws + 7 * (size_t)n;
    W.rz = W.part + 2 * nblk;
    W.err = W.rz + 2;
    W.done = reinterpret_cast<int32_t*>(W.err + 1);
    W.it = W.done + 1;
    int32_t* hdone;
    if ((rc = arena_host(sizeof(int32_t), (void**)&hdone))) return rc;
    double* dinv = nullptr;
    if (bj) {
        if ((rc = arena_get(kSlotPrecond, sizeof(double) * 144 * (size_t)M.nb, (void**)&dinv))) return rc;
        const int ph_inv = prof_start(kProfPrecond, s, 2304.0 * M.nb);
        launch_kernel(invert_blocks_kernel, dim3(M.nb), dim3(kInvThreads), 0, s, M, dinv,
                           (const int32_t*)nullptr, (const int32_t*)nullptr, 1);
        ABD_CHECK_LAUNCH();
        prof_stop(ph_inv, s);
    }
    const double tol_sq = tol * tol * (double)n;
    int ph = prof_start(kProfSolve, s, 0.0);
    if (bj)
        launch_kernel(mw_init_kernel<true>, dim3(nblk), dim3(threads), 0, s, M, b, (const double*)x, W,
                           (const double*)dinv);
    else
        launch_kernel(mw_init_kernel<false>, dim3(nblk), dim3(threads), 0, s, M, b, (const double*)x, W,
                           (const double*)dinv);
    ABD_CHECK_LAUNCH();
    launch_kernel(mw_start_kernel, dim3(1), dim3(kMwThreads), 0, s, nblk, tol_sq, maxiter, W);
    ABD_CHECK_LAUNCH();
    const auto first = bj ? mw_spmv_kernel<kMwBjThreads, true> : mw_spmv_kernel<kMwThreads, true>;
    const auto next = bj ? mw_spmv_kernel<kMwBjThreads, false> : mw_spmv_kernel<kMwThreads, false>;
    for (int i0 = 0; i0 < maxiter; i0 += check_every) {
        const int i1 = i0 + check_every < maxiter ? i0 + check_every : maxiter;
        for (int i = i0; i < i1; ++i) {
            launch_kernel(i == 0 ? first : next, dim3(nblk), dim3(kMwLanes * threads), 0, s, M, i, tol_sq, W);
            if (bj)
                launch_kernel(mw_update_kernel<true>, dim3(nblk), dim3(threads), 0, s, n, i, W, (const double*)dinv);
            else
                launch_kernel(mw_update_kernel<false>, dim3(nblk), dim3(threads), 0, s, n, i, W, (const double*)dinv);
        }
        launch_kernel(mw_check_kernel, dim3(1), dim3(threads), 0, s, nblk, i1 - 1, (int)check_every, tol_sq, W);
        ABD_CHECK_LAUNCH();
        ABD_CHECK(hipMemcpyAsync(hdone, W.done, sizeof(int32_t), hipMemcpyDeviceToHost, s));
        ABD_CHECK(hipStreamSynchronize(s));
        if (*hdone) break;
    }
    launch_kernel(mw_finish_kernel, dim3(nblk), dim3(kMwThreads), 0, s, n, W, x, iters, resid);
    ABD_CHECK_LAUNCH();
    prof_stop(ph, s);
    return ABD_OK;
}

int abd_bsr_solve(abd_stream_t stream, int32_t method, int32_t nb, const int32_t* row_ptr, const int32_t* cols,
                  const int32_t* slots, const double* blocks, const double* b, double* x, double tol, int32_t maxiter,
                  int32_t check_every, int32_t* iters, double* resid) {
    if (nb <= 0 || !row_ptr || !cols || !slots || !blocks || !b || !x || check_every <= 0) return ABD_ERR_ARG;
    if (method != ABD_SOLVER_BICGSTAB && method != ABD_SOLVER_CG_JACOBI && method != ABD_SOLVER_CG_BLOCK &&
        method != ABD_SOLVER_LDLT)
        return ABD_ERR_ARG;
    Bsr M{nb, row_ptr, cols, slots, blocks};
    if (method == ABD_SOLVER_LDLT) {
        if (nb <= kLdltMaxBodies)
            return launch_ldlt(to_stream(stream), M, 1, nullptr, nullptr, nb, b, x, tol, maxiter, check_every, iters,
                               resid);
        method = ABD_SOLVER_CG_BLOCK;  // above the direct solve's size: its fallback
    }
    if ((method == ABD_SOLVER_CG_JACOBI || method == ABD_SOLVER_CG_BLOCK) && nb > kLargeBodies)
        return solve_cg_multi(to_stream(stream), M, b, x, tol, maxiter, check_every, iters, resid,
                              method == ABD_SOLVER_CG_BLOCK);
    return launch_solve(to_stream(stream), method, M, 1, nullptr, nullptr, 12 * nb, b, x, tol, maxiter, check_every,
                        iters, resid, solve_threads(nb));
}

int abd_bsr_solve_scenes(abd_stream_t stream, int32_t method, const AbdScene* sc, int32_t max_scene_bodies,
                         const int32_t* row_ptr, const int32_t* cols, const int32_t* slots, const double* blocks,
                         const double* b, double* x, double tol, int32_t maxiter, int32_t check_every,
                         const uint8_t* active, int32_t* iters, double* resid) {
    if (!sc || sc->n_scenes <= 0 || !sc->scene_boff || max_scene_bodies <= 0 || !row_ptr || !cols || !slots ||
        !blocks || !b || !x || check_every <= 0)
        return ABD_ERR_ARG;
    if (method != ABD_SOLVER_BICGSTAB && method != ABD_SOLVER_CG_JACOBI && method != ABD_SOLVER_CG_BLOCK &&
        method != ABD_SOLVER_LDLT)
        return ABD_ERR_ARG;
    Bsr M{sc->n_bodies, row_ptr, cols, slots, blocks};
    if (method == ABD_SOLVER_LDLT)
        return launch_ldlt(to_stream(stream), M, sc->n_scenes, sc->scene_boff, active, max_scene_bodies, b, x, tol,
                           maxiter, check_every, iters, resid);
    return launch_solve(to_stream(stream), method, M, sc->n_scenes, sc->scene_boff, active, 12 * max_scene_bodies, b,
                        x, tol, maxiter, check_every, iters, resid, solve_threads(max_scene_bodies));
}

}  // extern "C"
