// abd_dense.h — the dense contact modes (psd = 2 exact Hessian, psd = 3 full IPC): one
// wave per contact, the 24x24 block and gradient of one contact formed by its 64 lanes.
//
// What bounds it: the projection of the 12x12 Hessian (psd = 3) is a chain of some 66
// rotations a sweep, each waiting for two square roots and three divisions, so a contact
// takes its chain's latency however many others there are.  With one thread per contact
// the 144-entry matrices lived in scratch memory and every entry of a rotation, of the
// derivatives and of the 24x24 map was another step of that chain: 2.72 ms a launch for the
// ~50 active contacts of 24 scenes (4 to 32 bodies).  With one wave per contact the matrices live in LDS and an
// entry is a lane's work: 189 us.  Every entry keeps the operations, and the order, of the sequential
// formulas, so the results are theirs bit for bit.
#pragma once
#include "abd_device.h"

namespace abd {

// The 12 coordinates' derivatives of one contact, shared by the lanes of its wave.
struct DenseLds {
    double H[144];      // d2s/dx2, then the contact's Hessian
    double V[144];      // the projection's eigenvectors
    double He[81];      // d2s of the plane / line distance over (u, v, w)
    double Hc[36];      // d2C, C = |a x b|^2 (point-edge; the mollifier)
    double L[12];       // point coefficients of (u, v, w)
    double t[9], n[9];  // dT, dN
    double e[12];       // u, v, w, c = u x v
    double ab[6], gC[6], gN[6], gs6[6];
    double gs[12], gc[12], gx[12];
};

// One wave per workgroup: orders the lanes' LDS accesses.
__device__ __forceinline__ void dense_sync() { __syncthreads(); }

// Entry (r, k) of s [a]x ([a]x b = a x b); the diagonal's is not added by the callers.
__device__ __forceinline__ double skew_entry(const double* a, int r, int k, double s) {
    const double v = a[3 - r - k];
    return ((k - r + 3) % 3 == 2 ? v : -v) * s;
}

// s = T^2 / N with T = w.(u x v) and N = |u x v|^2 over the edge vectors u, v, w:
//   dT = (v x w, w x u, u x v),  d2T: uv = -[w]x, uw = [v]x, vw = -[u]x (transposes below),
//   dN = (2 v x c, 2 c x u, 0),  d2N: uu = 2(|v|^2 I - v v^T), vv = 2(|u|^2 I - u u^T),
//                                  uv = 2(u v^T - (u.v) I) - 2[c]x   (c = u x v),
//   ds  = (2T/N) dT - (T^2/N^2) dN,
//   d2s = (2/N) dT dT^T + (2T/N) d2T - (2T/N^2)(dT dN^T + dN dT^T) - (T^2/N^2) d2N
//         + (2T^2/N^3) dN dN^T,
// with u, v, w = L x: ds to D.gs and d2s to D.H in the point coordinates; scale_h maps an
// entry's sum to the stored value.  D.L holds the point coefficients.
template <class ScaleH>
__device__ __forceinline__ void wave_plane_dist2(int lane, d3 u, d3 v, d3 w, DenseLds& D, ScaleH scale_h) {
    const d3 c = cross(u, v);
    const double T = dot(w, c), N = dot(c, c);
    if (lane == 0) {
        st3(D.e, u);
        st3(D.e + 3, v);
        st3(D.e + 6, w);
        st3(D.e + 9, c);
        st3(D.t, cross(v, w));
        st3(D.t + 3, cross(w, u));
        st3(D.t + 6, c);
        st3(D.n, cross(v, c) * 2.0);
        st3(D.n + 3, cross(c, u) * 2.0);
        st3(D.n + 6, mk(0.0, 0.0, 0.0));
    }
    dense_sync();
    const double a1 = 2.0 * T / N, a2 = T * T / (N * N);
    const double b0 = 2.0 / N, b1 = 2.0 * T / (N * N), b2 = 2.0 * T * T / (N * N * N);
    const double uu = dot(u, u), vv = dot(v, v), uv = dot(u, v);
    for (int q = lane; q < 81; q += kWave) {
        const int i = q / 9, j = q % 9, bi = i / 3, bj = j / 3, r = i % 3, k = j % 3;
        const double ti = D.t[i], tj = D.t[j], ni = D.n[i], nj = D.n[j];
        double h = b0 * (ti * tj) - b1 * (ti * nj + ni * tj) + b2 * (ni * nj);
        if (bi != bj && r != k)  // (2T/N) d2T: the block's third edge vector
            h += skew_entry(D.e + 3 * (3 - bi - bj), r, k, (bj - bi + 3) % 3 == 1 ? -a1 : a1);
        const double I = r == k ? 1.0 : 0.0;
        if (bi < 2 && bj < 2) {  // -(T^2/N^2) d2N
            const double* eu = D.e;
            const double* ev = D.e + 3;
            if (bi == bj)
                h -= bi == 0 ? a2 * (2.0 * (vv * I - ev[r] * ev[k])) : a2 * (2.0 * (uu * I - eu[r] * eu[k]));
            else
                h -= bi == 0 ? a2 * (2.0 * (eu[r] * ev[k] - uv * I)) : a2 * (2.0 * (ev[r] * eu[k] - uv * I));
            if (bi != bj && r != k) h += skew_entry(D.e + 9, r, k, bi == 0 ? 2.0 * a2 : -2.0 * a2);
        }
        D.He[q] = h;
    }
    if (lane < 12) {
        double acc = 0.0;
        for (int e = 0; e < 3; ++e) {
            const int i = 3 * e + lane % 3;
            acc += D.L[4 * e + lane / 3] * (a1 * D.t[i] - a2 * D.n[i]);
        }
        D.gs[lane] = acc;
    }
    dense_sync();
    for (int q = lane; q < 144; q += kWave) {
        const int i = q / 12, j = q % 12, a = i / 3, k = i % 3, b = j / 3, m = j % 3;
        double acc = 0.0;
        for (int e = 0; e < 3; ++e)
            for (int f = 0; f < 3; ++f) acc += D.L[4 * e + a] * D.L[4 * f + b] * D.He[9 * (3 * e + k) + 3 * f + m];
        D.H[q] = scale_h(i, j, acc);
    }
    dense_sync();
}

// C = |a x b|^2 and its derivatives in (a, b): D.gC (6) = (2 b x c, 2 c x a) with c = a x b
// (the cross-product form keeps full relative accuracy when a and b are nearly parallel),
// D.Hc (36, row-major) from C = |a|^2 |b|^2 - (a.b)^2.
__device__ __forceinline__ double wave_cross2(int lane, d3 a, d3 b, DenseLds& D) {
    const double aa = dot(a, a), bb = dot(b, b), ab = dot(a, b);
    const d3 c = cross(a, b);
    if (lane == 0) {
        st3(D.ab, a);
        st3(D.ab + 3, b);
        st3(D.gC, cross(b, c) * 2.0);
        st3(D.gC + 3, cross(c, a) * 2.0);
    }
    dense_sync();
    if (lane < 36) {
        const int i = lane / 6, j = lane % 6, r = i % 3, k = j % 3;
        const double* va = D.ab;
        const double* vb = D.ab + 3;
        const double I = r == k ? 1.0 : 0.0;
        double h;
        if (i < 3)
            h = j < 3 ? 2.0 * bb * I - 2.0 * vb[r] * vb[k] : 4.0 * va[r] * vb[k] - 2.0 * vb[r] * va[k] - 2.0 * ab * I;
        else
            h = j >= 3 ? 2.0 * aa * I - 2.0 * va[r] * va[k] : 4.0 * vb[r] * va[k] - 2.0 * va[r] * vb[k] - 2.0 * ab * I;
        D.Hc[lane] = h;
    }
    dense_sync();
    return dot(c, c);
}

// The point coefficients of (u, v, w) to D.L.  IPC: the triangle's edges from t0 (PT), the
// segments and their start points (EE); else the edge vectors of cmap_pt / cmap_ee.
template <bool IPC>
__device__ __forceinline__ void wave_coefficients(int lane, int kind, DenseLds& D) {
    if (lane == 0) {
        const double pt_ipc[12] = {0, -1, 1, 0, 0, -1, 0, 1, 1, -1, 0, 0};
        const double pt_c[12] = {0, 1, -1, 0, 0, 0, -1, 1, 1, 0, -1, 0};
        const double ee[12] = {-1, 1, 0, 0, 0, 0, -1, 1, -1, 0, 1, 0};
#pragma unroll
        for (int q = 0; q < 12; ++q) D.L[q] = kind == 1 ? ee[q] : IPC ? pt_ipc[q] : pt_c[q];
    }
    dense_sync();
}

// The squared distance s of the feature pair f, ds (D.gs) and d2s (D.H) in the 12 point
// coordinates.
__device__ __forceinline__ double wave_feature_dist2(int lane, int kind, const Feat& f, const d3 x[4], DenseLds& D) {
    // the feature's points by selects: its indices are uniform but not constants
    auto pnt = [&](int i) { return i == 0 ? x[0] : i == 1 ? x[1] : i == 2 ? x[2] : x[3]; };
    if (f.kind == kFeatPP) {
        const d3 dlt = pnt(f.i) - pnt(f.j);
        if (lane < 12) {
            const int a = lane / 3;
            const double c = comp(dlt, lane % 3);
            D.gs[lane] = a == f.i ? 2.0 * c : a == f.j ? -2.0 * c : 0.0;
        }
        for (int q = lane; q < 144; q += kWave) {
            const int i = q / 12, j = q % 12, a = i / 3, b = j / 3;
            const bool on = (a == f.i || a == f.j) && (b == f.i || b == f.j) && i % 3 == j % 3;
            D.H[q] = on ? (a == b ? 2.0 : -2.0) : 0.0;
        }
        dense_sync();
        return dot(dlt, dlt);
    }
    if (f.kind == kFeatPE) {
        // s = C / N, C = |a x b|^2 with a = e0 - p, b = e1 - p; N = |e1 - e0|^2
        const d3 p = pnt(f.i), e0 = pnt(f.j), e1 = pnt(f.k);
        const d3 e = e1 - e0;
        const double C = wave_cross2(lane, e0 - p, e1 - p, D);
        const double N = dot(e, e);
        if (lane < 6) {
            const double gN = (lane < 3 ? -2.0 : 2.0) * comp(e, lane % 3);
            D.gN[lane] = gN;
            D.gs6[lane] = D.gC[lane] / N - C * gN / (N * N);
        }
        dense_sync();
        if (lane < 36) {
            const int i = lane / 6, j = lane % 6;
            const double d2N = ((i < 3) == (j < 3) ? 2.0 : -2.0) * (i % 3 == j % 3 ? 1.0 : 0.0);
            D.He[lane] = D.Hc[lane] / N - (D.gC[i] * D.gN[j] + D.gN[i] * D.gC[j]) / (N * N) - C * d2N / (N * N) +
                         2.0 * C * D.gN[i] * D.gN[j] / (N * N * N);
        }
        dense_sync();
        // (a, b) = (e0 - p, e1 - p): coefficients of p, e0, e1 in a and b (a point outside
        // the pair: none)
        auto ca = [&](int a) { return a == f.i ? -1.0 : a == f.j ? 1.0 : 0.0; };
        auto cb = [&](int a) { return a == f.i ? -1.0 : a == f.k ? 1.0 : 0.0; };
        auto in = [&](int a) { return a == f.i || a == f.j || a == f.k; };
        if (lane < 12) {
            const int a = lane / 3, k = lane % 3;
            D.gs[lane] = in(a) ? 0.0 + (ca(a) * D.gs6[k] + cb(a) * D.gs6[3 + k]) : 0.0;
        }
        for (int q = lane; q < 144; q += kWave) {
            const int i = q / 12, j = q % 12, a = i / 3, k = i % 3, b = j / 3, m = j % 3;
            double h = 0.0;
            if (in(a) && in(b))
                h += ca(a) * ca(b) * D.He[6 * k + m] + ca(a) * cb(b) * D.He[6 * k + 3 + m] +
                     cb(a) * ca(b) * D.He[6 * (3 + k) + m] + cb(a) * cb(b) * D.He[6 * (3 + k) + 3 + m];
            D.H[q] = h;
        }
        dense_sync();
        return C / N;
    }
    // plane / line: s = (w.(u x v))^2 / |u x v|^2 over edge vectors with point coefficients L
    wave_coefficients<true>(lane, kind, D);
    const d3 u = kind == 0 ? x[2] - x[1] : x[1] - x[0];
    const d3 v = kind == 0 ? x[3] - x[1] : x[3] - x[2];
    const d3 w = kind == 0 ? x[0] - x[1] : x[2] - x[0];
    wave_plane_dist2(lane, u, v, w, D, [](int, int, double h) { return h; });
    const d3 cuv = cross(u, v);
    const double T = dot(w, cuv);
    return T * T / dot(cuv, cuv);
}

// In-place projection of the symmetric 12x12 D.H onto the PSD cone (negative eigenvalues
// set to zero) by cyclic Jacobi rotations (Golub & Van Loan, Matrix Computations, 4th ed.,
// sec. 8.5.2-8.5.3), to a relative off-diagonal norm of 1e-15 or 30 sweeps.  A rotation
// (p, q) combines pairs of entries: (A[k][p], A[k][q]) of the columns (lanes 0..11 by k),
// (A[p][k], A[q][k]) of the rows (lanes 16..27) and (V[k][p], V[k][q]) (lanes 32..43), all
// with the same two sums, independent of each other except for the four entries of rows
// and columns p, q, which lane 48 takes through the columns, then the rows.
__device__ __forceinline__ void wave_psd_project12(int lane, DenseLds& D) {
    double* A = D.H;
    double* V = D.V;
    for (int q = lane; q < 144; q += kWave) V[q] = q / 12 == q % 12 ? 1.0 : 0.0;
    double fro = 0.0;  // every lane the same sums (broadcast reads)
    for (int q = 0; q < 144; ++q) fro += A[q] * A[q];
    if (fro == 0.0) return;
    dense_sync();
    const int k = lane & 15, role = lane >> 4;
    double* const mat = role == 2 ? V : A;
    const int ks = role == 1 ? 1 : 12, ps = role == 1 ? 12 : 1;  // strides of k and of p, q
    for (int sweep = 0; sweep < 30; ++sweep) {
        double off = 0.0;
        for (int p = 0; p < 12; ++p)
            for (int q = p + 1; q < 12; ++q) off += A[12 * p + q] * A[12 * p + q];
        if (off <= 1e-30 * fro) break;
        for (int p = 0; p < 11; ++p)
            for (int q = p + 1; q < 12; ++q) {
                const double app = A[13 * p], aqq = A[13 * q], apq = A[12 * p + q], aqp = A[12 * q + p];
                if (apq == 0.0) continue;  // uniform
                const bool mine = role < 3 && k < 12 && (role == 2 || (k != p && k != q));
                const double m0 = mine ? mat[ks * k + ps * p] : 0.0, m1 = mine ? mat[ks * k + ps * q] : 0.0;
                const double tau = (aqq - app) / (2.0 * apq);
                const double t = (tau >= 0.0 ? 1.0 : -1.0) / (fabs(tau) + sqrt(1.0 + tau * tau));
                const double c = 1.0 / sqrt(1.0 + t * t), s = t * c;
                dense_sync();
                if (mine) {
                    mat[ks * k + ps * p] = c * m0 - s * m1;
                    mat[ks * k + ps * q] = s * m0 + c * m1;
                }
                if (lane == 48) {
                    const double bpp = c * app - s * apq, bpq = s * app + c * apq;  // columns p, q
                    const double bqp = c * aqp - s * aqq, bqq = s * aqp + c * aqq;
                    A[13 * p] = c * bpp - s * bqp;  // rows p, q
                    A[12 * p + q] = c * bpq - s * bqq;
                    A[12 * q + p] = s * bpp + c * bqp;
                    A[13 * q] = s * bpq + c * bqq;
                }
                dense_sync();
            }
    }
    double acc[3];
#pragma unroll
    for (int w = 0; w < 3; ++w) {
        const int q = lane + kWave * w;
        acc[w] = 0.0;
        if (q < 144)
            for (int e = 0; e < 12; ++e) {
                const double lam = A[13 * e] > 0.0 ? A[13 * e] : 0.0;
                acc[w] += V[12 * (q / 12) + e] * lam * V[12 * (q % 12) + e];
            }
    }
    dense_sync();  // the diagonal has been read
#pragma unroll
    for (int w = 0; w < 3; ++w)
        if (lane + kWave * w < 144) A[lane + kWave * w] = acc[w];
    dense_sync();
}

// The dense 24x24 block J^T H J and gradient gscale J^T gx of one contact (out[0..575]
// row-major, bodies [I | J]; out[576..599]): vertex t of body half h(t) maps through
// [1, r_t^T] (x) I3; PT has one vertex on body I, EE two.
constexpr int kDenseStride = 600;
constexpr int kDenseGOff = 576;
__device__ __forceinline__ void wave_body_map(int lane, int kind, const d3 r[4], const double* gx, double gscale,
                                              const double* Hx, double* __restrict__ out) {
    const int nI = kind == 0 ? 1 : 2;
    for (int q = lane; q < kDenseStride; q += kWave) {
        const bool isg = q >= kDenseGOff;
        const int i = isg ? q - kDenseGOff : q / 24, j = isg ? 0 : q % 24;
        const int hi = i / 12, ai = (i % 12) / 3, ki = i % 3;
        const int hj = j / 12, aj = (j % 12) / 3, kj = j % 3;
        double acc = 0.0;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            if ((t < nI ? 0 : 1) != hi) continue;
            const double Ji = ai == 0 ? 1.0 : comp(r[t], ai - 1);
            if (isg) {
                acc += Ji * gx[3 * t + ki];
                continue;
            }
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                if ((p < nI ? 0 : 1) != hj) continue;
                const double Jj = aj == 0 ? 1.0 : comp(r[p], aj - 1);
                acc += Ji * Jj * Hx[12 * (3 * t + ki) + 3 * p + kj];
            }
        }
        out[q] = isg ? gscale * acc : acc;
    }
}

// Exact mode (psd = 2, beyond the reference): J^T (b' d2s/dx2 + b'' ds/dx ds/dx^T) J and the
// gradient b' J^T ds/dx.  False: not active.
__device__ __forceinline__ bool wave_contact_exact(int lane, int kind, const d3 v[4], const d3 r[4], double d2hat,
                                                   double kappa, DenseLds& D, double* __restrict__ out) {
    const CMap c = kind == 0 ? cmap_pt(v[0], v[1], v[2], v[3]) : cmap_ee(v[0], v[1], v[2], v[3]);
    const bool valid = kind == 0 ? valid_pt(c.beta, c.gamma) : valid_ee(c.beta, c.gamma);
    const double l = signed_distance(c.e0, c.e1p, c.e2p);
    const double s = kind == 0 ? l * l : dot(c.e2p, c.e2p);
    if (!(s < d2hat && valid)) return false;
    const double b1 = barrier_d1(s, d2hat, kappa);
    const double b2 = barrier_d2(s, d2hat, kappa);
    wave_coefficients<false>(lane, kind, D);
    const d3 u = kind == 0 ? v[1] - v[2] : v[1] - v[0];
    const d3 vv = v[3] - v[2];
    const d3 w = kind == 0 ? v[0] - v[2] : v[2] - v[0];
    const double* gs = D.gs;
    wave_plane_dist2(lane, u, vv, w, D, [=](int i, int j, double h) { return h * b1 + (gs[i] * gs[j]) * b2; });
    wave_body_map(lane, kind, r, D.gs, b1, D.H, out);
    dense_sync();
    return true;
}

// Full-IPC mode (psd = 3, beyond the reference): the barrier of the squared distance to the
// closest feature pair (no validity gate), times the edge-edge mollifier for EE; the 12x12
// Hessian in the points' coordinates projected onto the PSD cone, then mapped to the two
// bodies like the exact mode's.  False: not active.
__device__ __forceinline__ bool wave_contact_full(int lane, int kind, const d3 v[4], const d3 r[4], double d2hat,
                                                  double kappa, DenseLds& D, double* __restrict__ out) {
    const Feat f = kind == 0 ? pt_feature(v) : ee_feature(v);
    const double s = wave_feature_dist2(lane, kind, f, v, D);
    if (!(s < d2hat)) return false;
    const double b0 = barrier(s, d2hat, kappa), b1 = barrier_d1(s, d2hat, kappa), b2 = barrier_d2(s, d2hat, kappa);
    // mollifier m(c), c = |u x v|^2, u = x1 - x0, v = x3 - x2 (EE below eps only)
    double m = 1.0, m1 = 0.0, m2 = 0.0;
    const double eps = kind == 1 ? ee_mollifier_eps(r) : 0.0;
    const double c = kind == 1 ? wave_cross2(lane, v[1] - v[0], v[3] - v[2], D) : 0.0;
    const bool moll = kind == 1 && c < eps;
    if (moll) {
        m = mollifier(c, eps);
        m1 = (2.0 - 2.0 * c / eps) / eps;
        m2 = -2.0 / (eps * eps);
    }
    // point coefficients of u (points 0, 1) and v (points 2, 3)
    auto cu = [](int a) { return a == 0 ? -1.0 : a == 1 ? 1.0 : 0.0; };
    auto cv = [](int a) { return a == 2 ? -1.0 : a == 3 ? 1.0 : 0.0; };
    if (lane < 12) {
        const int a = lane / 3, k = lane % 3;
        const double gc = moll ? cu(a) * D.gC[k] + cv(a) * D.gC[3 + k] : 0.0;
        D.gc[lane] = gc;
        D.gx[lane] = m * b1 * D.gs[lane] + b0 * m1 * gc;
    }
    dense_sync();
    for (int q = lane; q < 144; q += kWave) {
        const int i = q / 12, j = q % 12;
        double h = m * (b1 * D.H[q] + b2 * (D.gs[i] * D.gs[j]));
        if (moll) {
            const int a = i / 3, k = i % 3, b = j / 3, mm = j % 3;
            double hc = 0.0;
            hc += cu(a) * cu(b) * D.Hc[6 * k + mm];
            hc += cu(a) * cv(b) * D.Hc[6 * k + 3 + mm];
            hc += cv(a) * cu(b) * D.Hc[6 * (3 + k) + mm];
            hc += cv(a) * cv(b) * D.Hc[6 * (3 + k) + 3 + mm];
            h += b0 * (m2 * (D.gc[i] * D.gc[j]) + m1 * hc) + b1 * m1 * (D.gs[i] * D.gc[j] + D.gc[i] * D.gs[j]);
        }
        D.H[q] = h;
    }
    dense_sync();
    wave_psd_project12(lane, D);
    wave_body_map(lane, kind, r, D.gx, 1.0, D.H, out);
    dense_sync();
    return true;
}

}  // namespace abd
