// abd_body.hip — the per-body passes of a Newton iteration: one workgroup per body places
// its vertices and does everything else that needs only that body's state.
//
// What bounds them: the vertices' bytes for large scenes (24 read, 24 written each), the
// number of launches for small ones.  As separate kernels the start of an iteration
// (update_q, the rows' commit, projection, body boxes, fills, inertia terms) and the step's end
// (projection with the range test, swept body boxes) took 8 launches and read the vertices
// again for the boxes and, for the range test, 72 bytes of ranges and start positions: 108 us
// an iteration for 1.06M vertices of 8217 bodies, against 48 us here (29 + 19; 59 where the
// step's end also writes the vertices' swept boxes for the filter after it).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "abd_block.h"
#include "abd_inertia.h"
#include "abd_internal.h"

namespace abd {

namespace {

// x_c = ((p_c + r_0 A[0][c]) + r_1 A[1][c]) + r_2 A[2][c] (abd.py:313-316); q = A, then p
__device__ __forceinline__ double place(const double* q, const double (&r)[3], int c) {
    double v = q[9 + c] + r[0] * q[c];
    v = v + r[1] * q[3 + c];
    return v + r[2] * q[6 + c];
}

// The start of an iteration for body blockIdx.x: the accepted step taken (q and (Ak, pk), a
// scene with step length 0 keeping its state bit for bit), x = x(q), the body box at x, the
// inertia gradient (written) and Hessian (the diagonal slot written).  The workgroups past
// the bodies commit the scenes' rows and zero the words given.
template <int T>
__global__ __launch_bounds__(T) void body_start_kernel(AbdScene sc, AbdParams P, BodyStart U) {
    __shared__ double q[12];
    __shared__ double sh[6 * (T / kWave)];
    const int b = blockIdx.x, t = threadIdx.x, nb = sc.n_bodies;
    if (b >= nb) {
        const int64_t i0 = (int64_t)(b - nb) * T + t, step = (int64_t)(gridDim.x - nb) * T;
        for (int64_t i = i0; i < U.nzero; i += step) U.zero[i] = 0;
        for (int64_t i = i0; i < U.nzero2; i += step) U.zero2[i] = 0;
        for (int64_t i = i0; i < U.nzero32; i += step) U.zero32[i] = 0;
        for (int64_t s = i0; s < U.ns; s += step) {
            U.newton[s] = U.newton[U.ns + s];
            U.E0[s] = U.E0[U.ns + s];
            U.it[s] = U.it[U.ns + s];
            if (U.slots) U.slots[s] = 0x3FF0000000000000ull;  // 1.0
        }
        if (i0 < U.ncounters) U.counters[i0] = 0;
        if (i0 == 0) {
            *U.range_flag = 0;
            if (U.qcount) *U.qcount = 0;
        }
        return;
    }
    const double al = U.alpha[U.ns > 1 ? sc.body_scene[b] : 0];
    if (t < 12) {
        const double v = t < 9 ? U.A[9 * b + t] : U.p[3 * b + t - 9];
        const double d = t < 9 ? U.dq[3 * (4 * b + 1 + t / 3) + t % 3] : U.dq[12 * b + t - 9];
        q[t] = al == 0.0 ? v : v - d * al;
    }
    __syncthreads();
    if (t < 9)
        U.A[9 * b + t] = U.Ak[9 * b + t] = q[t];
    else if (t < 12)
        U.p[3 * b + t - 9] = U.pk[3 * b + t - 9] = q[t];
    double mn[3], mx[3];
    for (int k = 0; k < 3; ++k) {
        mn[k] = 1.0 / 0.0;
        mx[k] = -1.0 / 0.0;
    }
    const int v1 = sc.voff[b + 1];
    for (int64_t v = sc.voff[b] + t; v < v1; v += T) {
        const double r[3] = {sc.x0[3 * v], sc.x0[3 * v + 1], sc.x0[3 * v + 2]};
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const double c = place(q, r, k);
            U.x[3 * v + k] = c;
            mn[k] = c < mn[k] ? c : mn[k];
            mx[k] = c > mx[k] ? c : mx[k];
        }
    }
    if (t < 16) {
        const double m = sc.mass ? sc.mass[b] : P.mass, i0 = sc.I0 ? sc.I0[b] : P.I0;
        if (t < 4) {
            double g[3];
            inertia_gradient_row(P, t, q, q + 9, U.A0 + 9 * b, U.p0 + 3 * b, U.Adot + 9 * b, U.pdot + 3 * b, m, i0, g);
            for (int k = 0; k < 3; ++k) U.g[3 * (4 * b + t) + k] = g[k];
        }
        double dh[9];
        inertia_hessian_block(P, t % 4, t / 4, q, m, i0, dh);
        double* B = U.blocks + 9 * (16 * (int64_t)b + t);
        for (int k = 0; k < 9; ++k) B[k] = 0.0 + dh[k];
    }
    body_extrema<T>(mn, mx, sh);
    if (t == 0)
        for (int k = 0; k < 3; ++k) {
            U.lo[3 * b + k] = (float)(mn[k] - U.dil);
            U.hi[3 * b + k] = (float)(mx[k] + U.dil);
        }
}

// The end of a step for body blockIdx.x: x = x(q - dq) for the scenes in `active` (x(q) for
// the others), the union of the body boxes at both ends, and the range test: *flag = 1 when a
// vertex may have left the superset's ranges.  A body whose state lies within the skin of one
// of the two states the ranges were widened around, coordinate by coordinate (the largest
// rest coordinates bound every vertex's move), is inside without reading them.  (The start
// of the step lies between positions tested before: every test leaves a margin of 1e-6 of the
// skin, far above the rounding of positions.)
template <int T>
__global__ __launch_bounds__(T) void body_end_kernel(AbdScene sc, BodyEnd U) {
    __shared__ double q[12], q0[12];
    __shared__ double sh[6 * (T / kWave)];
    const int b = blockIdx.x, t = threadIdx.x;
    const double al = U.active[U.ns > 1 ? sc.body_scene[b] : 0] ? 1.0 : 0.0;
    if (t < 12) {
        const double v = t < 9 ? U.A[9 * b + t] : U.p[3 * b + t - 9];
        const double d = t < 9 ? U.dq[3 * (4 * b + 1 + t / 3) + t % 3] : U.dq[12 * b + t - 9];
        q[t] = al == 0.0 ? v : v - d * al;
        q0[t] = v;
    }
    __syncthreads();
    bool test = U.lo != nullptr;
    if (test) {
        const double* rm = U.rest_max + 3 * b;
        bool in[2];
        for (int e = 0; e < 2; ++e) {
            const double* qr = U.qref + 12 * ((int64_t)e * sc.n_bodies + b);
            in[e] = true;
            for (int k = 0; k < 3; ++k) {
                double d = fabs(q[9 + k] - qr[9 + k]);
                for (int r = 0; r < 3; ++r) d += rm[r] * fabs(q[3 * r + k] - qr[3 * r + k]);
                in[e] &= d <= U.skin - U.margin;  // NaN: not inside
            }
        }
        test = !(in[0] || in[1]);
    }
    double mn[3], mx[3];
    for (int k = 0; k < 3; ++k) {
        mn[k] = 1.0 / 0.0;
        mx[k] = -1.0 / 0.0;
    }
    bool out = false;
    const int v1 = sc.voff[b + 1];
    for (int64_t v = sc.voff[b] + t; v < v1; v += T) {
        const double r[3] = {sc.x0[3 * v], sc.x0[3 * v + 1], sc.x0[3 * v + 2]};
        float e[6];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const double c = place(q, r, k), c0 = place(q0, r, k);
            U.x[3 * v + k] = c;
            e[k] = fminf((float)(c0 - U.dil), (float)(c - U.dil));
            e[3 + k] = fmaxf((float)(c0 + U.dil), (float)(c + U.dil));
            if (!(c - c0 == c - c0)) {  // not finite: a box that overlaps every other
                e[k] = -INFINITY;
                e[3 + k] = INFINITY;
            }
            mn[k] = c < mn[k] ? c : mn[k];
            mx[k] = c > mx[k] ? c : mx[k];
            if (test)
                out |= !(c - U.margin >= U.lo[3 * v + k] && c + U.margin <= U.hi[3 * v + k]);  // NaN: outside
        }
        if (U.ebox) {
            U.ebox[2 * v] = make_float4(e[0], e[1], e[2], e[3]);
            U.ebox[2 * v + 1] = make_float4(e[4], e[5], 0.0f, 0.0f);
        }
    }
    if (__any(out) && lane_id() == 0) *U.flag = 1;  // every writer stores 1
    body_extrema<T>(mn, mx, sh);
    if (t == 0)
        for (int k = 0; k < 3; ++k) {
            U.slo[3 * b + k] = fminf(U.blo[3 * b + k], (float)(mn[k] - U.dil));
            U.shi[3 * b + k] = fmaxf(U.bhi[3 * b + k], (float)(mx[k] + U.dil));
        }
    if (t == 0) U.on[b] = al != 0.0;
}

// The largest |rest coordinate| of each body, per axis (one wave per body), and a copy of the
// rest positions.
__global__ __launch_bounds__(kWave) void rest_max_kernel(AbdScene sc, double* __restrict__ out,
                                                          double* __restrict__ copy) {
    const int b = blockIdx.x;
    double m[3] = {0.0, 0.0, 0.0};
    for (int64_t v = sc.voff[b] + threadIdx.x; v < sc.voff[b + 1]; v += kWave)
        for (int k = 0; k < 3; ++k) {
            const double c = sc.x0[3 * v + k];
            copy[3 * v + k] = c;
            m[k] = fmax(m[k], fabs(c));
        }
    for (int k = 0; k < 3; ++k) {
        for (int off = kWave / 2; off > 0; off >>= 1) m[k] = fmax(m[k], __shfl_xor(m[k], off, kWave));
        if (threadIdx.x == 0) out[3 * b + k] = m[k];
    }
}

// The two ends of the step the superset's ranges are made around: q, and q - dq for the
// scenes in `active` (q for the others).
__global__ __launch_bounds__(kBlock) void step_states_kernel(int nb, const int32_t* __restrict__ body_scene,
                                                              const double* __restrict__ A,
                                                              const double* __restrict__ p,
                                                              const double* __restrict__ dq,
                                                              const uint8_t* __restrict__ active,
                                                              double* __restrict__ qref) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= 12 * nb) return;
    const int b = i / 12, t = i % 12;
    const double v = t < 9 ? A[9 * b + t] : p[3 * b + t - 9];
    const double d = t < 9 ? dq[3 * (4 * b + 1 + t / 3) + t % 3] : dq[12 * b + t - 9];
    qref[i] = v;
    qref[12 * (int64_t)nb + i] = active[body_scene ? body_scene[b] : 0] ? v - d : v;
}

}  // namespace

// threads of a body's workgroup: a wave where the scene's largest body keeps it to a few
// vertices a lane (a cube fills an eighth of it), else four
bool small_bodies(const AbdScene* sc) { return sc->max_verts <= 4 * kWave; }

int body_start(hipStream_t s, const AbdScene* sc, const AbdParams* P, const BodyStart& U) {
    if (sc->n_bodies == 0) return ABD_OK;
    const bool small = small_bodies(sc);
    const int T = small ? kWave : kBlock;
    // workgroups for the rows and the fill: about 16 words a thread
    const int64_t words = U.nzero + U.nzero2 + U.nzero32 / 2;
    const int64_t extra = std::min<int64_t>(4096, 1 + ceil_div(std::max<int64_t>(words, U.ns), 16 * (int64_t)T));
    const dim3 grid((unsigned)(sc->n_bodies + extra));
    if (small)
        launch_kernel(body_start_kernel<kWave>, grid, dim3(T), 0, s, *sc, *P, U);
    else
        launch_kernel(body_start_kernel<kBlock>, grid, dim3(T), 0, s, *sc, *P, U);
    ABD_CHECK_LAUNCH();
    return ABD_OK;
}

int body_end(hipStream_t s, const AbdScene* sc, const BodyEnd& U) {
    if (sc->n_bodies == 0) return ABD_OK;
    if (small_bodies(sc))
        launch_kernel(body_end_kernel<kWave>, dim3(sc->n_bodies), dim3(kWave), 0, s, *sc, U);
    else
        launch_kernel(body_end_kernel<kBlock>, dim3(sc->n_bodies), dim3(kBlock), 0, s, *sc, U);
    ABD_CHECK_LAUNCH();
    return ABD_OK;
}

int rest_max(hipStream_t s, const AbdScene* sc, double* out, double* copy) {
    if (sc->n_bodies == 0) return ABD_OK;
    launch_kernel(rest_max_kernel, dim3(sc->n_bodies), dim3(kWave), 0, s, *sc, out, copy);
    ABD_CHECK_LAUNCH();
    return ABD_OK;
}

int step_states(hipStream_t s, const AbdScene* sc, const double* A, const double* p, const double* dq,
                const uint8_t* active, double* qref) {
    if (sc->n_bodies == 0) return ABD_OK;
    launch_kernel(step_states_kernel, dim3(grid_for(12 * (int64_t)sc->n_bodies, kBlock, INT32_MAX)), dim3(kBlock),
                       0, s, sc->n_bodies, sc->n_scenes > 1 ? sc->body_scene : nullptr, A, p, dq, active, qref);
    ABD_CHECK_LAUNCH();
    return ABD_OK;
}

}  // namespace abd
