// abd_device.h — device-side math of the contact path (gfx950, FP64).
//
// Operation order follows the reference Warp functions cited on each helper so
// that validity predicates (strict inequalities on barycentric coordinates)
// and FP32 boxes come out bit-identical to a CPU evaluation of the same
// formulas; the library is compiled with -ffp-contract=off for that reason.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace abd {

struct d3 {
    double x, y, z;
};
__device__ __forceinline__ d3 mk(double x, double y, double z) { return d3{x, y, z}; }
__device__ __forceinline__ d3 operator+(d3 a, d3 b) { return mk(a.x + b.x, a.y + b.y, a.z + b.z); }
__device__ __forceinline__ d3 operator-(d3 a, d3 b) { return mk(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ __forceinline__ d3 operator*(d3 a, double s) { return mk(a.x * s, a.y * s, a.z * s); }
__device__ __forceinline__ d3 operator/(d3 a, double s) { return mk(a.x / s, a.y / s, a.z / s); }
// wp.dot: (a.x*b.x + a.y*b.y) + a.z*b.z
__device__ __forceinline__ double dot(d3 a, d3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ d3 cross(d3 a, d3 b) {
    return mk(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x);
}
__device__ __forceinline__ double comp(d3 a, int k) { return k == 0 ? a.x : (k == 1 ? a.y : a.z); }
__device__ __forceinline__ d3 ld3(const double* p) { return mk(p[0], p[1], p[2]); }
__device__ __forceinline__ void st3(double* p, d3 a) {
    p[0] = a.x;
    p[1] = a.y;
    p[2] = a.z;
}

// ipcsk/barrier.py:4-15 barrier(s), s = squared distance
__device__ __forceinline__ double barrier(double d, double d2hat, double kappa) {
    double ret = 0.0;
    if (d < d2hat) {
        double r = d / d2hat;
        double t = r - 1.0;
        ret = kappa * -(t * t) * log(r);
    }
    return ret;
}
// ipcsk/barrier.py:18-24 barrier_derivative
__device__ __forceinline__ double barrier_d1(double d, double d2hat, double kappa) {
    double ret = 0.0;
    if (d < d2hat) ret = kappa * (d2hat - d) * (2.0 * log(d / d2hat) + (d - d2hat) / d) / (d2hat * d2hat);
    return ret;
}
// ipcsk/barrier.py:34-39 barrier_derivative2
__device__ __forceinline__ double barrier_d2(double d, double d2hat, double kappa) {
    double ret = 0.0;
    if (d < d2hat)
        ret = -kappa * (2.0 * log(d / d2hat) + (d - d2hat) / d + (d - d2hat) * (2.0 / d + d2hat / (d * d))) /
              (d2hat * d2hat);
    return ret;
}

// Warp mat22 inverse (adjugate * 1/det, zero matrix for det == 0) applied to b.
__device__ __forceinline__ void inv22_mul(double m00, double m01, double m10, double m11, double b0, double b1,
                                          double& r0, double& r1) {
    double det = m00 * m11 - m10 * m01;
    double i00 = 0.0, i01 = 0.0, i10 = 0.0, i11 = 0.0;
    if (fabs(det) > 0.0) {
        double s = 1.0 / det;
        i00 = m11 * s;
        i01 = -m01 * s;
        i10 = -m10 * s;
        i11 = m00 * s;
    }
    r0 = i00 * b0 + i01 * b1;
    r1 = i10 * b0 + i11 * b1;
}

// Contact-space coordinates c = (e0, e1perp, e2perp) with (alpha, beta, gamma):
// psd/vf.py:4-41 (PT: x0 point, x1..x3 triangle) and psd/ee.py:6-31,119-133
// (EE: edges x0x1, x2x3).  The two maps differ only in the edge vectors.
struct CMap {
    d3 e0, e1p, e2p;
    double alpha, beta, gamma;
};
__device__ __forceinline__ CMap cmap_from_edges(d3 e0, d3 e1, d3 e2) {
    CMap c;
    double e0e0 = dot(e0, e0), e0e1 = dot(e0, e1), e1e1 = dot(e1, e1);
    c.alpha = e0e1 / e0e0;
    c.e0 = e0;
    c.e1p = e1 - e0 * c.alpha;
    inv22_mul(e0e0, e0e1, e0e1, e1e1, dot(e0, e2), dot(e1, e2), c.beta, c.gamma);
    c.e2p = (e2 - e0 * c.beta) - e1 * c.gamma;
    return c;
}
__device__ __forceinline__ CMap cmap_pt(d3 x0, d3 x1, d3 x2, d3 x3) {
    return cmap_from_edges(x1 - x2, x3 - x2, x0 - x2);
}
__device__ __forceinline__ CMap cmap_ee(d3 x0, d3 x1, d3 x2, d3 x3) {
    return cmap_from_edges(x1 - x0, x3 - x2, x2 - x0);
}
// ccd.py:45-54 verify_root_pt / verify_root_ee (strict)
__device__ __forceinline__ bool valid_pt(double b, double g) {
    return 0.0 < b && b < 1.0 && 0.0 < g && g < 1.0 && 0.0 < b + g && b + g < 1.0;
}
__device__ __forceinline__ bool valid_ee(double b, double g) { return 0.0 < b && b < 1.0 && 0.0 < -g && -g < 1.0; }
// psd/hl.py:16-17
__device__ __forceinline__ double signed_distance(d3 e0p, d3 e1p, d3 e2p) {
    d3 n = cross(e0p, e1p);
    return dot(e2p, n) / sqrt(dot(n, n));
}

// ------------------------------------------------------------------ CCD
// cubic_roots.py:6-19
__device__ __forceinline__ double evaluate(const double c[4], double x) {
    return c[0] + x * (c[1] + x * (c[2] + x * c[3]));
}
__device__ __forceinline__ double multi_sign(double a, double b) { return b < 0.0 ? -a : a; }
__device__ __forceinline__ bool diff_sign(double y0, double yr) { return y0 * yr < 0.0; }
__device__ __forceinline__ double wmin(double a, double b) { return a < b ? a : b; }
__device__ __forceinline__ double wmax(double a, double b) { return a > b ? a : b; }

constexpr double kXError = 1e-10;
// Bound on the Newton/bisection loop; the reference loop is unbounded, and the
// bracket shrinks strictly every step, so real inputs stop long before this.
constexpr int kFindClosedMaxIt = 1000;

// cubic_roots.py:29-62 find_closed
__device__ inline double find_closed(const double c[4], const double dv[4], double x0, double x1, double y0) {
    double xr = (x0 + x1) / 2.0;
    double yr = evaluate(c, xr);
    double xb0 = x0, xb1 = x1;
    if (!(x1 - x0 <= kXError * 2.0)) {
        for (int it = 0; it < kFindClosedMaxIt; ++it) {
            bool side = diff_sign(y0, yr);
            if (side)
                xb1 = xr;
            else
                xb0 = xr;
            double dy = evaluate(dv, xr);
            double dx = yr / dy;
            double xn = xr - dx;
            if (xn > xb0 && xn < xb1) {
                double stepsize = fabs(xr - xn);
                xr = xn;
                if (stepsize > kXError)
                    yr = evaluate(c, xr);
                else
                    break;
            } else {
                xr = (xb0 + xb1) / 2.0;
                yr = evaluate(c, xr);
                if (xb0 == xr || xb1 == xr || xb1 - xb0 <= 2.0 * kXError) break;
            }
        }
    }
    return xr;
}
// cubic_roots.py:63-93 quadratic_roots (constant-first)
__device__ inline int quadratic_roots(const double coef[3], double x0, double x1, double roots[2]) {
    roots[0] = roots[1] = 0.0;
    double c = coef[0], b = coef[1], a = coef[2];
    double delta = b * b - 4.0 * a * c;
    int ret = 0;
    if (delta > 0.0) {
        double d = sqrt(delta);
        double q = -(b + multi_sign(d, b)) * 0.5;
        double rv0 = q / a, rv1 = c / q;
        double xa = wmin(rv0, rv1), xb = wmax(rv0, rv1);
        if (xa >= x0 && xa <= x1) roots[ret++] = xa;
        if (xb >= x0 && xb <= x1) roots[ret++] = xb;
    } else if (delta < 0.0) {
        ret = 0;
    } else {
        double r0 = -0.5 * b / a;
        roots[0] = r0;
        if (r0 >= x0 && r0 <= x1) ret = 1;
    }
    return ret;
}
// cubic_roots.py:21-27 deflate
__device__ __forceinline__ void deflate(const double c[4], double root, double d[3]) {
    d[2] = c[3];
    d[1] = c[2] + root * d[2];
    d[0] = c[1] + root * d[1];
}
// cubic_roots.py:95-193 cubic_roots, split into its bracketing decisions (which interval
// the Newton / bisection search runs on, and whether the deflated quadratic follows) and
// the searches themselves: a candidate whose bracket is kNone has no root in [x0, x1]
// without any search.
struct CubicBracket {
    int kind;  // kNone: no root; kOne: one root in [lo, hi]; kDeflate: it, then the
               // deflated quadratic's roots in [qlo, x1]
    double lo, hi, ylo, qlo;
    static constexpr int kNone = 0, kOne = 1, kDeflate = 2;
};
__device__ inline CubicBracket cubic_bracket(const double coef[4], double x0, double x1) {
    const double y0 = evaluate(coef, x0), y1 = evaluate(coef, x1);
    const double a = coef[3] * 3.0, b_2 = coef[2], c = coef[1];
    const double delta_4 = b_2 * b_2 - a * c;
    if (delta_4 > 0.0) {
        const double d_2 = sqrt(delta_4);
        const double q = -(b_2 + multi_sign(d_2, b_2));
        const double rv0 = q / a, rv1 = c / q;
        const double xa = wmin(rv0, rv1), xb = wmax(rv0, rv1);
        const bool outside = xa >= x1 || xb <= x0 || (xa <= x0 && xb >= x1);
        if (diff_sign(y0, y1)) {
            if (outside) return {CubicBracket::kOne, x0, x1, y0, 0.0};
        } else if (outside) {
            return {CubicBracket::kNone, 0.0, 0.0, 0.0, 0.0};
        }
        if (xa > x0) {
            const double ya = evaluate(coef, xa);
            if (diff_sign(y0, ya)) {
                const bool more = diff_sign(ya, y1) || (xb < x1 && diff_sign(ya, evaluate(coef, xb)));
                return {more ? CubicBracket::kDeflate : CubicBracket::kOne, x0, xa, y0, xa};
            }
            if (xb < x1) {
                const double yb = evaluate(coef, xb);
                if (diff_sign(ya, yb))
                    return {diff_sign(yb, y1) ? CubicBracket::kDeflate : CubicBracket::kOne, xa, xb, ya, xb};
                if (diff_sign(yb, y1)) return {CubicBracket::kOne, xb, x1, yb, 0.0};
            } else if (diff_sign(ya, y1)) {
                return {CubicBracket::kOne, xa, x1, ya, 0.0};
            }
        } else {
            const double yb = evaluate(coef, xb);
            if (diff_sign(y0, yb))
                return {diff_sign(yb, y1) ? CubicBracket::kDeflate : CubicBracket::kOne, x0, xb, y0, xb};
            if (diff_sign(yb, y1)) return {CubicBracket::kOne, xb, x1, yb, 0.0};
        }
        return {CubicBracket::kNone, 0.0, 0.0, 0.0, 0.0};
    }
    if (diff_sign(y0, y1)) return {CubicBracket::kOne, x0, x1, y0, 0.0};
    return {CubicBracket::kNone, 0.0, 0.0, 0.0, 0.0};
}
// the searches of a bracket (one pass of the reference's while-True block)
__device__ inline int cubic_roots(const double coef[4], double x0, double x1, double roots[3]) {
    roots[0] = roots[1] = roots[2] = 0.0;
    const CubicBracket br = cubic_bracket(coef, x0, x1);
    if (br.kind == CubicBracket::kNone) return 0;
    const double deriv[4] = {coef[1], 2.0 * coef[2], coef[3] * 3.0, 0.0};
    roots[0] = find_closed(coef, deriv, br.lo, br.hi, br.ylo);
    if (br.kind == CubicBracket::kOne) return 1;
    double qr[2], dp[3];
    deflate(coef, roots[0], dp);
    const int r = quadratic_roots(dp, br.qlo, x1, qr);
    roots[1] = qr[0];
    roots[2] = qr[1];
    return r + 1;
}

// ccd.py:122-129 cubic_binomial: prod_k (b_k + t a_k), constant first, accumulated into acc
__device__ __forceinline__ void cubic_binomial_acc(double a0, double a1, double a2, double b0, double b1, double b2,
                                                   double acc[4]) {
    acc[0] += b0 * b1 * b2;
    acc[1] += a0 * b1 * b2 + b0 * b1 * a2 + b0 * a1 * b2;
    acc[2] += a0 * a1 * b2 + a0 * b1 * a2 + b0 * a1 * a2;
    acc[3] += a0 * a1 * a2;
}
// ccd.py:82-119 det_polynomial of M(t) = b + t a, with a, b given by their columns
// (R1: mat33(u, v, w) has columns u, v, w, so m[r][c] = col_c[r]).
__device__ inline void det_polynomial(const d3 ac[3], const d3 bc[3], double out[4]) {
#define M_(m, r, c) comp(m[c], r)
    double pos[4] = {0.0, 0.0, 0.0, 0.0}, neg[4] = {0.0, 0.0, 0.0, 0.0};
    cubic_binomial_acc(M_(ac, 0, 0), M_(ac, 1, 1), M_(ac, 2, 2), M_(bc, 0, 0), M_(bc, 1, 1), M_(bc, 2, 2), pos);
    cubic_binomial_acc(M_(ac, 0, 1), M_(ac, 1, 2), M_(ac, 2, 0), M_(bc, 0, 1), M_(bc, 1, 2), M_(bc, 2, 0), pos);
    cubic_binomial_acc(M_(ac, 0, 2), M_(ac, 1, 0), M_(ac, 2, 1), M_(bc, 0, 2), M_(bc, 1, 0), M_(bc, 2, 1), pos);
    cubic_binomial_acc(M_(ac, 0, 0), M_(ac, 1, 2), M_(ac, 2, 1), M_(bc, 0, 0), M_(bc, 1, 2), M_(bc, 2, 1), neg);
    cubic_binomial_acc(M_(ac, 0, 1), M_(ac, 1, 0), M_(ac, 2, 2), M_(bc, 0, 1), M_(bc, 1, 0), M_(bc, 2, 2), neg);
    cubic_binomial_acc(M_(ac, 0, 2), M_(ac, 1, 1), M_(ac, 2, 0), M_(bc, 0, 2), M_(bc, 1, 1), M_(bc, 2, 0), neg);
#undef M_
    for (int k = 0; k < 4; ++k) out[k] = pos[k] - neg[k];
}
// ccd.py:56-79 build_and_solve_4_points_coplanar: coefficients of the coplanarity cubic
__device__ inline void coplanar_poly(const d3 p0[4], const d3 p1[4], double coef[4]) {
    static constexpr int sel[4][3] = {{1, 2, 3}, {0, 2, 3}, {0, 1, 3}, {0, 1, 2}};
    double d[4][4];
    for (int m = 0; m < 4; ++m) {
        d3 ac[3], bc[3];
        for (int k = 0; k < 3; ++k) {
            bc[k] = p0[sel[m][k]];
            ac[k] = p1[sel[m][k]] - bc[k];
        }
        det_polynomial(ac, bc, d[m]);
    }
    for (int k = 0; k < 4; ++k) coef[k] = d[0][k] - d[1][k] + d[2][k] - d[3][k];
}
// wp.lerp(a, b, t) = a*(1-t) + b*t
__device__ __forceinline__ d3 lerp(d3 a, d3 b, double t) { return a * (1.0 - t) + b * t; }
// ccd.py:133-186 pt_collision_time (kind 0) / ee_collision_time (kind 1)
__device__ inline double collision_time(int kind, const d3 t0[4], const d3 t1[4]) {
    double coef[4], roots[3];
    coplanar_poly(t0, t1, coef);
    int n = cubic_roots(coef, 0.0, 1.0, roots);
    double root = 1.0;
    bool true_root = false;
    for (int i = 0; i < n; ++i) {
        root = roots[i];
        d3 p[4];
        for (int k = 0; k < 4; ++k) p[k] = lerp(t0[k], t1[k], root);
        CMap c = kind == 0 ? cmap_pt(p[0], p[1], p[2], p[3]) : cmap_ee(p[0], p[1], p[2], p[3]);
        true_root = kind == 0 ? valid_pt(c.beta, c.gamma) : valid_ee(c.beta, c.gamma);
        if (true_root) break;
    }
    if (!true_root) root = 1.0;
    return root;
}

// ------------------------------------------------------------- fetchers
// affine_body.py:106-234 fetch_pt / fetch_ee over the flattened scene.
struct SceneView {
    const int32_t* voff;
    const int32_t* foff;
    const int32_t* eoff;
    const int32_t* tris;
    const int32_t* edges;
    const double* x0;
};
__device__ __forceinline__ void fetch_pt_idx(const SceneView& S, const int32_t* t5, int64_t v[4]) {
    int I = t5[0], J = t5[1];
    const int32_t* T = S.tris + 3 * (int64_t)(S.foff[J] + t5[4]);
    int vj = S.voff[J];
    v[0] = S.voff[I] + t5[3];
    v[1] = vj + T[0];
    v[2] = vj + T[1];
    v[3] = vj + T[2];
}
__device__ __forceinline__ void fetch_ee_idx(const SceneView& S, const int32_t* t5, int64_t v[4]) {
    int I = t5[0], J = t5[1];
    const int32_t* EI = S.edges + 2 * (int64_t)(S.eoff[I] + t5[3]);
    const int32_t* EJ = S.edges + 2 * (int64_t)(S.eoff[J] + t5[4]);
    int vi = S.voff[I], vj = S.voff[J];
    v[0] = vi + EI[0];
    v[1] = vi + EI[1];
    v[2] = vj + EJ[0];
    v[3] = vj + EJ[1];
}
// The four scene vertex ids of a PT (kind 0) / EE (kind 1) candidate: from `vid` (the ids
// fetch_pt_idx / fetch_ee_idx give, stored beside the list; nullable) or fetched through
// the topology.
__device__ __forceinline__ void cand_idx(int kind, const SceneView& S, const int32_t* t5, const int32_t* vid,
                                         int64_t v[4]) {
    if (vid) {
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = vid[q];
    } else if (kind == 0) {
        fetch_pt_idx(S, t5, v);
    } else {
        fetch_ee_idx(S, t5, v);
    }
}

}  // namespace abd

namespace abd {
// Per-candidate barrier energy (ipcsk/energy.py:10-48) and TOI (ccd.py:9-40), shared
// by the whole-list and the per-scene kernels.
// Vertex positions of the candidate functions: read from an array (Verts), or computed
// on the fly by another source with the same interface (load4: vertices vi[0..nI) of
// body I, the rest of body J; y: the y coordinate of vertex vid of body b).
struct Verts {
    const double* x;
    __device__ __forceinline__ void load4(int, int, const int64_t vi[4], int, d3 v[4]) const {
        for (int k = 0; k < 4; ++k) v[k] = ld3(x + 3 * vi[k]);
    }
    __device__ __forceinline__ double y(int, int64_t vid) const { return x[3 * vid + 1]; }
};

template <class Src>
__device__ __forceinline__ double cand_energy_ee(const SceneView& S, const Src& X, const int32_t* t5, double d2hat,
                                                 double kappa, const int32_t* vid = nullptr) {
    int64_t vi[4];
    cand_idx(1, S, t5, vid, vi);
    d3 v[4];
    X.load4(t5[0], t5[1], vi, 2, v);
    CMap c = cmap_ee(v[0], v[1], v[2], v[3]);
    double d = signed_distance(c.e0, c.e1p, c.e2p);
    return valid_ee(c.beta, c.gamma) ? barrier(d * d, d2hat, kappa) : 0.0;
}
template <class Src>
__device__ __forceinline__ double cand_energy_pt(const SceneView& S, const Src& X, const int32_t* t5, double d2hat,
                                                 double kappa, const int32_t* vid = nullptr) {
    int64_t vi[4];
    cand_idx(0, S, t5, vid, vi);
    d3 v[4];
    X.load4(t5[0], t5[1], vi, 1, v);
    CMap c = cmap_pt(v[0], v[1], v[2], v[3]);
    return valid_pt(c.beta, c.gamma) ? barrier(dot(c.e2p, c.e2p), d2hat, kappa) : 0.0;
}
template <class Src>
__device__ __forceinline__ double cand_energy_vg(const int32_t* __restrict__ voff, const Src& X, const int32_t* t2,
                                                 double ground, double d2hat, double kappa) {
    const int64_t vid = voff[t2[0]] + t2[1];
    const double d = X.y(t2[0], vid) - ground;
    return barrier(d * d, d2hat, kappa);
}
__device__ __forceinline__ double cand_toi(int kind, const SceneView& S, const double* __restrict__ x0,
                                           const double* __restrict__ x1, const int32_t* t,
                                           const int32_t* vid = nullptr) {
    int64_t vi[4];
    cand_idx(kind, S, t, vid, vi);
    d3 a[4], b[4];
    for (int q = 0; q < 4; ++q) {
        a[q] = ld3(x0 + 3 * vi[q]);
        b[q] = ld3(x1 + 3 * vi[q]);
    }
    return collision_time(kind, a, b);
}
// The four vertices of a PT (kind 0) / EE (kind 1) candidate at both ends of the step.
__device__ __forceinline__ void cand_verts(int kind, const SceneView& S, const double* __restrict__ x0,
                                           const double* __restrict__ x1, const int32_t* t, d3 a[4], d3 b[4],
                                           const int32_t* vid = nullptr) {
    int64_t vi[4];
    cand_idx(kind, S, t, vid, vi);
    for (int q = 0; q < 4; ++q) {
        a[q] = ld3(x0 + 3 * vi[q]);
        b[q] = ld3(x1 + 3 * vi[q]);
    }
}
// Whether collision_time of the step a -> b of a candidate's vertices can be below 1: its
// coplanarity cubic has a bracketed root in [0, 1] (cubic_bracket); otherwise it has no root
// and its TOI is 1.
__device__ __forceinline__ bool toi_bracketed(const d3 a[4], const d3 b[4]) {
    double coef[4];
    coplanar_poly(a, b, coef);
    return cubic_bracket(coef, 0.0, 1.0).kind != CubicBracket::kNone;
}
// A lower bound of the step lengths at which a PT (kind 0) / EE (kind 1) candidate can be
// active on the step a -> b of its vertices: below it some axis separates the two
// primitives by more than dhat, so the barrier is zero, and their boxes dilated as the
// collision set's (FP32 rounding included) do not overlap; above 1 they are apart on the
// whole step.  Along an axis the gap between the boxes
// is concave in the step length (a minimum of linear functions minus a maximum), so from a
// positive gap at the start it stays above the chord to the gap at the end.  In FP32 on the
// differences to one vertex.  The margins: 1e-3 dhat for the rounding of positions on the
// step, 1e-6 of the differences for FP32, 5e-7 of the coordinates for the boxes' casts (four
// roundings of 2^-24).  NaN or infinite coordinates give 0.
__device__ __forceinline__ float chord_zero(float u0, float u1, float best) {
    if (!(u0 > 0.0f)) return best;
    const float t = u1 > 0.0f ? 2.0f : u0 / (u0 - u1);
    return t > best ? t : best;
}
constexpr float kApartShrink = 1.0f - 4e-6f;  // below the chord's zero whatever its roundings
__device__ __forceinline__ float apart_until(int kind, const d3 a[4], const d3 b[4], double dhat) {
    float best = 0.0f;
    const float dh = 1.001f * (float)dhat;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const double ref = comp(a[0], k);
        float l[2][2], h[2][2];  // [end][primitive]
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const d3* v = e ? b : a;
            const float c0 = (float)(comp(v[0], k) - ref), c1 = (float)(comp(v[1], k) - ref),
                        c2 = (float)(comp(v[2], k) - ref), c3 = (float)(comp(v[3], k) - ref);
            const float m23 = fminf(c2, c3), x23 = fmaxf(c2, c3);
            l[e][0] = kind == 0 ? c0 : fminf(c0, c1);
            h[e][0] = kind == 0 ? c0 : fmaxf(c0, c1);
            l[e][1] = kind == 0 ? fminf(c1, m23) : m23;
            h[e][1] = kind == 0 ? fmaxf(c1, x23) : x23;
        }
        float m = 0.0f;
#pragma unroll
        for (int p = 0; p < 2; ++p)
            m = fmaxf(m, fmaxf(fmaxf(-l[0][p], h[0][p]), fmaxf(-l[1][p], h[1][p])));
        const float d = dh + 1e-6f * m + 5e-7f * (fabsf((float)ref) + m);
        best = chord_zero((l[0][1] - h[0][0]) - d, (l[1][1] - h[1][0]) - d, best);
        best = chord_zero((l[0][0] - h[0][1]) - d, (l[1][0] - h[1][1]) - d, best);
    }
    return best * kApartShrink;
}
// The same of a vertex above the ground (its height y0 -> y1).
__device__ __forceinline__ float apart_until_vg(double y0, double y1, double ground, double dhat) {
    const float u0 = (float)(y0 - ground), u1 = (float)(y1 - ground);
    const float m = fmaxf(fabsf(u0), fabsf(u1));
    const float d = 1.001f * (float)dhat + 1e-6f * m + 5e-7f * (fabsf((float)ground) + m);
    return chord_zero(u0 - d, u1 - d, 0.0f) * kApartShrink;
}
__device__ __forceinline__ double cand_toi_vg(const int32_t* __restrict__ voff, const double* __restrict__ x0,
                                              const double* __restrict__ x1, const int32_t* t2, double ground) {
    const int64_t vid = voff[t2[0]] + t2[1];
    const double d1 = x1[3 * vid + 1] - ground;
    double t = 1.0;
    if (d1 < 0) {
        const double d0 = x0[3 * vid + 1] - ground;
        t = d0 / (d0 - d1);
    }
    return t;
}
}  // namespace abd

namespace abd {
// ------------------------------------------------------------------ full IPC
// psd = 3 (beyond the reference, which has no distance types): the squared distance of
// a PT / EE candidate to its closest feature pair (Li et al. 2020, Incremental Potential
// Contact), the edge-edge mollifier, and their exact derivatives in the 12 coordinates
// of the contact's four points x0..x3 (PT: point, triangle t0 t1 t2; EE: a0 a1, b0 b1).

// Feature pairs: kFeatPlane (PT: point-plane; EE: line-line), kFeatPE (point x[i] against
// edge x[j] x[k]), kFeatPP (x[i] against x[j]).
enum { kFeatPlane = 0, kFeatPE = 1, kFeatPP = 2 };
struct Feat {
    int kind, i, j, k;
};

// Closest feature of point x0 to triangle x1 x2 x3 by the Voronoi regions of the
// triangle (Ericson, Real-Time Collision Detection, 2005, sec. 5.1.5).
__device__ __forceinline__ Feat pt_feature(const d3 x[4]) {
    const d3 a = x[1], b = x[2], c = x[3], p = x[0];
    const d3 ab = b - a, ac = c - a, ap = p - a;
    const double d1 = dot(ab, ap), d2 = dot(ac, ap);
    if (d1 <= 0.0 && d2 <= 0.0) return Feat{kFeatPP, 0, 1, 0};
    const d3 bp = p - b;
    const double d3_ = dot(ab, bp), d4 = dot(ac, bp);
    if (d3_ >= 0.0 && d4 <= d3_) return Feat{kFeatPP, 0, 2, 0};
    const double vc = d1 * d4 - d3_ * d2;
    if (vc <= 0.0 && d1 >= 0.0 && d3_ <= 0.0) return Feat{kFeatPE, 0, 1, 2};
    const d3 cp = p - c;
    const double d5 = dot(ab, cp), d6 = dot(ac, cp);
    if (d6 >= 0.0 && d5 <= d6) return Feat{kFeatPP, 0, 3, 0};
    const double vb = d5 * d2 - d1 * d6;
    if (vb <= 0.0 && d2 >= 0.0 && d6 <= 0.0) return Feat{kFeatPE, 0, 1, 3};
    const double va = d3_ * d6 - d5 * d4;
    if (va <= 0.0 && d4 - d3_ >= 0.0 && d5 - d6 >= 0.0) return Feat{kFeatPE, 0, 2, 3};
    return Feat{kFeatPlane, 0, 0, 0};
}

// Closest feature pair of segments x0 x1 and x2 x3: the line parameters of the closest
// points, clamped to the segments in turn (Sunday, "Distance between 3D lines and
// segments", geomalgorithms.com); (near-)parallel segments start from s = 0.
__device__ __forceinline__ Feat ee_feature(const d3 x[4]) {
    const d3 u = x[1] - x[0], v = x[3] - x[2], w = x[0] - x[2];
    const double a = dot(u, u), b = dot(u, v), c = dot(v, v), d = dot(u, w), e = dot(v, w);
    const double D = a * c - b * b;
    double sN, sD = D, tN, tD = D;
    int s_end = -1, t_end = -1;  // -1: interior, 0 / 1: that end
    if (D <= 1e-12 * a * c) {
        sN = 0.0;
        sD = 1.0;
        tN = e;
        tD = c;
        s_end = 0;
    } else {
        sN = b * e - c * d;
        tN = a * e - b * d;
        if (sN <= 0.0) {
            sN = 0.0;
            tN = e;
            tD = c;
            s_end = 0;
        } else if (sN >= sD) {
            sN = sD;
            tN = e + b;
            tD = c;
            s_end = 1;
        }
    }
    if (tN <= 0.0) {
        t_end = 0;
        if (-d <= 0.0)
            s_end = 0;
        else if (-d >= a)
            s_end = 1;
        else
            s_end = -1;
    } else if (tN >= tD) {
        t_end = 1;
        if (-d + b <= 0.0)
            s_end = 0;
        else if (-d + b >= a)
            s_end = 1;
        else
            s_end = -1;
    }
    if (s_end < 0 && t_end < 0) return Feat{kFeatPlane, 0, 0, 0};
    if (s_end >= 0 && t_end >= 0) return Feat{kFeatPP, s_end, 2 + t_end, 0};
    if (s_end >= 0) return Feat{kFeatPE, s_end, 2, 3};
    return Feat{kFeatPE, 2 + t_end, 0, 1};
}

// Squared distance of the feature pair alone (no derivatives).
__device__ __forceinline__ double feature_dist2_value(int ckind, const Feat& f, const d3 x[4]) {
    if (f.kind == kFeatPP) {
        const d3 dlt = x[f.i] - x[f.j];
        return dot(dlt, dlt);
    }
    if (f.kind == kFeatPE) {
        const d3 c = cross(x[f.j] - x[f.i], x[f.k] - x[f.i]), e = x[f.k] - x[f.j];
        return dot(c, c) / dot(e, e);
    }
    const d3 u = ckind == 0 ? x[2] - x[1] : x[1] - x[0];
    const d3 v = ckind == 0 ? x[3] - x[1] : x[3] - x[2];
    const d3 w = ckind == 0 ? x[0] - x[1] : x[2] - x[0];
    const d3 cuv = cross(u, v);
    const double T = dot(w, cuv);
    return T * T / dot(cuv, cuv);
}

// Edge-edge mollifier (Li et al. 2020): eps_x = 1e-3 |a1 - a0|^2 |b1 - b0|^2 at rest,
// m(c) = (2 - c / eps_x) c / eps_x for c = |(a1 - a0) x (b1 - b0)|^2 < eps_x, else 1.
__device__ __forceinline__ double ee_mollifier_eps(const d3 r[4]) {
    const d3 ua = r[1] - r[0], ub = r[3] - r[2];
    return 1e-3 * dot(ua, ua) * dot(ub, ub);
}
__device__ __forceinline__ double ee_cross2(const d3 x[4]) {
    const d3 c = cross(x[1] - x[0], x[3] - x[2]);
    return dot(c, c);
}
__device__ __forceinline__ double mollifier(double c, double eps) {
    if (c >= eps) return 1.0;
    const double t = c / eps;
    return (2.0 - t) * t;
}

// Full-IPC barrier energy of one candidate (kind 0 PT, 1 EE) at points x, rest points r.
__device__ __forceinline__ double ipc_full_energy(int kind, const d3 x[4], const d3 r[4], double d2hat,
                                                  double kappa) {
    const Feat f = kind == 0 ? pt_feature(x) : ee_feature(x);
    const double s = feature_dist2_value(kind, f, x);
    if (!(s < d2hat)) return 0.0;
    const double b = barrier(s, d2hat, kappa);
    return kind == 0 ? b : mollifier(ee_cross2(x), ee_mollifier_eps(r)) * b;
}

// Full-IPC energy of a PT (ckind 0) or EE (1) candidate tuple, points from X, rest points
// from the scene's rest positions.
template <class Src>
__device__ __forceinline__ double cand_energy_full(int ckind, const SceneView& S, const Src& X, const int32_t* t5,
                                                   double d2hat, double kappa) {
    int64_t vi[4];
    if (ckind == 0)
        fetch_pt_idx(S, t5, vi);
    else
        fetch_ee_idx(S, t5, vi);
    d3 v[4], r[4];
    X.load4(t5[0], t5[1], vi, ckind == 0 ? 1 : 2, v);
    for (int k = 0; k < 4; ++k) r[k] = ld3(S.x0 + 3 * vi[k]);
    return ipc_full_energy(ckind, v, r, d2hat, kappa);
}
}  // namespace abd
