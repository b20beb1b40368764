// The closed form of one column of a Wigner-D basis and of its gradient, and the
// edge frame (see wigner.hip): shared by the kernels of wigner.hip (degrees up to
// kLaneL) and wigner_high.h (the rest).
#pragma once

#include "feq_internal.h"

#include <cfloat>
#include <cmath>
#include <type_traits>

namespace feq {

struct WignerArgs {
    int32_t nirr;
    int32_t dim;
    int32_t lvals[FEQ_MAX_IRREPS];
    int32_t off[FEQ_MAX_IRREPS];       // component offset of every irrep
    int32_t plan_off[FEQ_MAX_IRREPS];  // offset of every irrep's plan block (doubles)
};

// The other form (wigner_high.h).
constexpr int kLaneL = 6;
template <class T>
int wigner_high_fwd(const WignerArgs& A, const double* plan, const int32_t* perm, int64_t E, const T* dirs, T* out,
                    hipStream_t s);
template <class T>
int wigner_high_bwd(const WignerArgs& A, const double* plan, const int32_t* perm, int64_t E, const T* dirs,
                    const T* grad_out, T* grad_dirs, hipStream_t s);

// Representations whose matrix exceeds 64 KB are refused (dimensions over 128 in
// float32, 90 in float64), whatever kernel the call would take: the column kernel
// stages whole matrices, and every kernel holds perm in FEQ_MAX_SLOTS entries.
constexpr size_t kMatrixBytes = 64 * 1024;
template <class T>
int check_dim(const WignerArgs& A) {
    static_assert(kMatrixBytes / sizeof(float) <= FEQ_MAX_SLOTS * FEQ_MAX_SLOTS, "perm's LDS copy");
    if (sizeof(T) * static_cast<size_t>(A.dim) * A.dim > kMatrixBytes)
        return fail(FEQ_ERR_UNSUPPORTED, "representation dimension %d too large", A.dim);
    return FEQ_OK;
}

inline int max_degree(const WignerArgs& A) {
    int lmax = 0;
    for (int i = 0; i < A.nirr; ++i) lmax = A.lvals[i] > lmax ? A.lvals[i] : lmax;
    return lmax;
}
// Edges per workgroup of the column kernels: one thread per (edge, column) of 256, the
// edges' matrices (dim x dim values of T) staged in at most kMatrixBytes of LDS.
template <class T>
int column_edges(const WignerArgs& A) {
    const int e = 256 / A.dim;
    const int cap = static_cast<int>(kMatrixBytes / (sizeof(T) * static_cast<size_t>(A.dim) * A.dim));
    return e < cap ? e : cap;
}

// The lane kernels take degrees up to kLaneL, where the column kernels' workgroups do
// not all run at once: a thread per column has all columns of its edges at once, a
// wave of the lane kernels one after the other (and degrees 5 and 6, whose unrolled code is
// fetched anew in each launch, twice as many).  Float32, forward and backward in us,
// column kernels and these: lvals 0..4, 2000 edges (200 workgroups) 11.5 and 13.7,
// 13.5 and 21.3; 4500 edges (450) 15.4 and 24.9, 14.4 and 21.4; lvals 0..3, 3300 edges
// (207) 8.6 and 10.5, 9.6 and 11.8; 4500 (282) 10.5 and 18.3, 9.7 and 11.8; lvals 0..6,
// 2000 edges (400) 28.8 and 62.5, 34.2 and 62.3; 2600 (520) 40.7 and 87, 34.6 and 62.4.
// In float64 the lines are the same, but forward at degrees 5 and 6: lvals 0..6, 2000
// edges (667) 34 and 47, 3300 (1100) 50 and 47.  Matrices of up to 4 columns leave most of
// a lane kernel's waves without one: degree 0, 640 000 edges 9.1 and 18.7, 32.4 and
// 47.6; degrees 0 and 1 34.9 and 60.5, 37.2 and 63.2 (two of degree 1 51 and 100, 44 and 85).
template <class T>
bool lane_form(const WignerArgs& A, int64_t E, bool backward) {
    const int lmax = max_degree(A);
    if (lmax > kLaneL || A.dim <= 4) return false;
    const int at_once = lmax <= 4 ? 256 : sizeof(T) == 8 && !backward ? 768 : 512;
    return ceil_div(E, column_edges<T>(A)) > at_once;
}

namespace {

// nan_to_num(x, 0.0) in the output type: NaN -> 0, +-inf -> +-max
template <class T>
__device__ __forceinline__ T sanitize(double v) {
    if (v != v) return T(0);
    if constexpr (std::is_same_v<T, float>) {
        if (v > static_cast<double>(FLT_MAX)) return FLT_MAX;
        if (v < -static_cast<double>(FLT_MAX)) return -FLT_MAX;
        return static_cast<float>(v);
    } else {
        if (v > DBL_MAX) return DBL_MAX;
        if (v < -DBL_MAX) return -DBL_MAX;
        return v;
    }
}

// Cosines and sines of an edge's angles phi and ang = theta rho.
struct Trig {
    double cp, sp, ca, sa;
};
__device__ __forceinline__ Trig trig_of(double phi, double ang) {
    Trig t;
    sincos(phi, &t.sp, &t.cp);
    sincos(ang, &t.sa, &t.ca);
    return t;
}

// cos(q x), sin(q x) for q = 0..L.
template <int L>
__device__ __forceinline__ void multiples(double c1, double s1, double (&c)[L + 1], double (&s)[L + 1]) {
    c[0] = 1.0;
    s[0] = 0.0;
#pragma unroll
    for (int q = 1; q <= L; ++q) {
        c[q] = c[q - 1] * c1 - s[q - 1] * s1;
        s[q] = s[q - 1] * c1 + c[q - 1] * s1;
    }
}

// Column c of D for an irrep of degree L (n = 2L + 1) and edge angles (phi,
// ang = theta rho): D = Z(phi) V Z(ang) V^T Z(-phi), where Z(x) rotates the
// (r, 2L - r) pair by (L - r) x -- the structure of the m-diagonal generator,
// which the host checks when it builds V.  All indices are compile-time, so
// the vectors live in registers.
template <int L>
__device__ __forceinline__ void wigner_column(const double* __restrict__ V, int c, const Trig& t,
                                              double (&y)[2 * L + 1]) {
    constexpr int n = 2 * L + 1;
    double cp[L + 1], sp[L + 1], ca[L + 1], sa[L + 1];
    multiples<L>(t.cp, t.sp, cp, sp);
    multiples<L>(t.ca, t.sa, ca, sa);
    // v1 = Z(-phi) e_c: entries at c (cos) and its partner n-1-c (sin of the
    // partner's coupling), then w = V^T v1
    const int pc = n - 1 - c;
    const int mc = L - c;                         // coupling of row c
    const int amc = mc < 0 ? -mc : mc;
    double cphi = 1.0, sphi = 0.0;
#pragma unroll
    for (int q = 0; q <= L; ++q)
        if (q == amc) {
            cphi = cp[q];
            sphi = sp[q];
        }
    const double v_c = cphi;
    const double v_p = pc != c ? (mc < 0 ? -sphi : sphi) : 0.0;
    double w[n], u[n];
#pragma unroll
    for (int q = 0; q < n; ++q) w[q] = V[c * n + q] * v_c + V[pc * n + q] * v_p;
    // u = Z(ang) w
#pragma unroll
    for (int r = 0; r < n; ++r) {
        const int m = L - r, am = m < 0 ? -m : m;
        u[r] = ca[am] * w[r] + (r != L ? (m < 0 ? -sa[am] : sa[am]) * w[n - 1 - r] : 0.0);
    }
    // x = V u, y = Z(phi) x
    double xv[n];
#pragma unroll
    for (int r = 0; r < n; ++r) {
        double acc = 0.0;
#pragma unroll
        for (int q = 0; q < n; ++q) acc += V[r * n + q] * u[q];
        xv[r] = acc;
    }
#pragma unroll
    for (int r = 0; r < n; ++r) {
        const int m = L - r, am = m < 0 ? -m : m;
        y[r] = cp[am] * xv[r] + (r != L ? (m < 0 ? -sp[am] : sp[am]) * xv[n - 1 - r] : 0.0);
    }
}

template <int L, class T>
__device__ __forceinline__ void column_into(const double* __restrict__ V, int c, const Trig& t,
                                            bool ident, T* dst, int stride) {
    constexpr int n = 2 * L + 1;
    double y[n];
    if (L == 0) {
        y[0] = 1.0;
    } else if (ident) {
#pragma unroll
        for (int r = 0; r < n; ++r) y[r] = r == c ? 1.0 : 0.0;
    } else {
        wigner_column<L>(V, c, t, y);
    }
#pragma unroll
    for (int r = 0; r < n; ++r) dst[r * stride] = sanitize<T>(y[r]);
}

struct EdgeFrame {
    double phi, ang;
    int ident;   // axis of zero length: D = I
};

// The edge frame in T like rot_to_ez: d = v/(|v|+eps), axis = (-d_y, d_x, 0)/(|.|+eps),
// theta = acos(clamp(d_z, -1 + eps, 1 - eps)); a = rho (cos phi, sin phi).
// T = float: as the reference's float32 rot_to_ez (whose clamp bounds
// +-(1 - eps) round to +-1); T = double: the frame in float64 with the clamp as
// written (a float64 module runs rot_to_ez in float64).
template <class T>
__device__ __forceinline__ EdgeFrame edge_frame(const T* __restrict__ v) {
    const T eps = T(1e-8);
    const T vx = v[0], vy = v[1], vz = v[2];
    const T nv = sqrt(vx * vx + vy * vy + vz * vz) + eps;
    const T dx = vx / nv, dy = vy / nv, dz = vz / nv;
    const T a0r = -dy, a1r = dx;
    const T na = sqrt(a0r * a0r + a1r * a1r) + eps;
    const T a0 = a0r / na, a1 = a1r / na;
    const T theta = acos(fmin(fmax(dz, T(-1) + eps), T(1) - eps));
    const double rho = sqrt(static_cast<double>(a0) * a0 + static_cast<double>(a1) * a1);
    EdgeFrame f;
    f.ident = rho == 0.0;
    f.phi = f.ident ? 0.0 : atan2(static_cast<double>(a1), static_cast<double>(a0));
    f.ang = static_cast<double>(theta) * rho;
    return f;
}

// ---- backward: gradient with respect to the edge directions --------------------------
//
// With X(phi) = cos(phi) G0 + sin(phi) G1 = Z(phi) V G2 V^T Z(-phi) and the
// exponent theta (a0 G0 + a1 G1) = ang X(phi) (a = rho (cos phi, sin phi),
// ang = theta rho), the derivatives of D = exp(ang X(phi)) are exact and cheap:
//     dD/dang = X D,        dD/dphi = G2 D - D G2
// (phi enters as a conjugation by the z-rotation Z(phi) = exp(phi G2)).  Each
// thread takes one column c of an irrep block of D and adds, with G = dL/dD
// (the columns of dL/dM moved back through perm):
//     <G[:,c], X D[:,c]>                                 to dL/dang,
//     <G[:,c], G2 D[:,c]> - z_c <G[:,pc], D[:,c]>        to dL/dphi
// (z_c = L - c: G2's coupling of row c to its partner row pc = n-1-c).  At
// rho = 0 (the forward's D = I) the exponent is theta (a0 G0 + a1 G1) at a = 0,
// whose derivative is dD/da_k = theta G_k: the threads add <G[:,c], G_k e_c>.
// One thread per edge then chains (phi, ang) -- or (a0, a1) -- back through
// a = a_raw/(|a_raw|+eps), a_raw = (-d_y, d_x), theta = acos(d_z) and
// d = v/(|v|+eps), the operations of rot_to_ez (wigner.py:220-238), with
// torch's conventions (the norm's gradient is 0 at 0).

// out = X(phi) y for one irrep: Z(phi) V G2 V^T Z(-phi) y, with cos(q phi),
// sin(q phi) for q = 0..L in cpm, spm.
template <int L>
__device__ __forceinline__ void apply_axis_generator(const double* __restrict__ V,
                                                     const double (&cpm)[L + 1],
                                                     const double (&spm)[L + 1],
                                                     const double (&y)[2 * L + 1],
                                                     double (&out)[2 * L + 1]) {
    constexpr int n = 2 * L + 1;
    double u[n], w[n], x[n];
    // u = Z(-phi) y
#pragma unroll
    for (int r = 0; r < n; ++r) {
        const int m = L - r, am = m < 0 ? -m : m;
        u[r] = cpm[am] * y[r] - (r != L ? (m < 0 ? -spm[am] : spm[am]) * y[n - 1 - r] : 0.0);
    }
    // w = V^T u
#pragma unroll
    for (int q = 0; q < n; ++q) {
        double acc = 0.0;
#pragma unroll
        for (int r = 0; r < n; ++r) acc += V[r * n + q] * u[r];
        w[q] = acc;
    }
    // w <- G2 w: (G2 w)[r] = (L - r) w[n-1-r]
#pragma unroll
    for (int r = 0; r < n; ++r) u[r] = static_cast<double>(L - r) * w[n - 1 - r];
    // x = V u
#pragma unroll
    for (int r = 0; r < n; ++r) {
        double acc = 0.0;
#pragma unroll
        for (int q = 0; q < n; ++q) acc += V[r * n + q] * u[q];
        x[r] = acc;
    }
    // out = Z(phi) x
#pragma unroll
    for (int r = 0; r < n; ++r) {
        const int m = L - r, am = m < 0 ? -m : m;
        out[r] = cpm[am] * x[r] + (r != L ? (m < 0 ? -spm[am] : spm[am]) * x[n - 1 - r] : 0.0);
    }
}

// Contributions of column c of one irrep block.  gcol / gpar: columns c and
// n-1-c of dL/dD restricted to the block's rows.  t0/t1: (dL/dang, dL/dphi), or
// at rho = 0 (ident) (dL/da0, dL/da1) without the factor theta.
template <int L, class T>
__device__ __forceinline__ void column_grad(const double* __restrict__ V, int c, const Trig& t,
                                            bool ident, const T* gcol, const T* gpar,
                                            int stride, double& t0, double& t1) {
    constexpr int n = 2 * L + 1;
    t0 = 0.0;
    t1 = 0.0;
    if (L == 0) return;                       // D = 1 is constant
    double g[n], gp[n], y[n], xy[n];
#pragma unroll
    for (int r = 0; r < n; ++r) {
        g[r] = gcol[r * stride];
        gp[r] = gpar[r * stride];
    }
    if (ident) {
        double cz[L + 1], sz[L + 1], c9[L + 1], s9[L + 1];
        double c1, s1;
        sincos(0.5 * M_PI, &s1, &c1);
        multiples<L>(1.0, 0.0, cz, sz);
        multiples<L>(c1, s1, c9, s9);
#pragma unroll
        for (int r = 0; r < n; ++r) y[r] = r == c ? 1.0 : 0.0;
        apply_axis_generator<L>(V, cz, sz, y, xy);      // G0 e_c
#pragma unroll
        for (int r = 0; r < n; ++r) t0 += g[r] * xy[r];
        apply_axis_generator<L>(V, c9, s9, y, xy);      // G1 e_c
#pragma unroll
        for (int r = 0; r < n; ++r) t1 += g[r] * xy[r];
        return;
    }
    wigner_column<L>(V, c, t, y);
    double cp[L + 1], sp[L + 1];
    multiples<L>(t.cp, t.sp, cp, sp);
    apply_axis_generator<L>(V, cp, sp, y, xy);
#pragma unroll
    for (int r = 0; r < n; ++r) {
        t0 += g[r] * xy[r];
        t1 += g[r] * static_cast<double>(L - r) * y[n - 1 - r] - static_cast<double>(L - c) * gp[r] * y[r];
    }
}

// The frame in double from the float32 directions: near the poles (|d_z| -> 1)
// d theta / d d_z = -1/sqrt(1 - d_z^2) amplifies the float32 rounding of d_z
// (1 - |d_z| = 3e-6 loses 2% to it), while the forward's matrices are
// insensitive to it; the gradient is therefore formed from an exact frame.
struct ExactFrame {
    double dx, dy, dz, nv, na, a0, a1, th;
    EdgeFrame f;
};
template <class T>
__device__ __forceinline__ ExactFrame exact_frame(const T* __restrict__ v) {
    const double eps = 1e-8;
    ExactFrame X;
    const double vx = v[0], vy = v[1], vz = v[2];
    X.nv = sqrt(vx * vx + vy * vy + vz * vz);
    const double nv = X.nv + eps;
    X.dx = vx / nv;
    X.dy = vy / nv;
    X.dz = vz / nv;
    const double a0r = -X.dy, a1r = X.dx;
    X.na = sqrt(a0r * a0r + a1r * a1r);
    const double na = X.na + eps;
    X.a0 = a0r / na;
    X.a1 = a1r / na;
    // the reference's clamp to [-1 + eps, 1 - eps] (wigner.py:235), which
    // binds in float64 (within ~1.4e-4 rad of the poles; in float32 its
    // bounds round to +-1, as the forward's float32 frame has them)
    X.th = acos(fmin(fmax(X.dz, -1.0 + eps), 1.0 - eps));
    const double rho = sqrt(X.a0 * X.a0 + X.a1 * X.a1);
    X.f.ident = rho == 0.0;
    X.f.phi = X.f.ident ? 0.0 : atan2(X.a1, X.a0);
    X.f.ang = X.th * rho;
    return X;
}

// The direction's gradient from s0, s1: the sums of t0, t1 over all columns.
template <class T>
__device__ __forceinline__ void frame_grad(const ExactFrame& X, double s0, double s1,
                                           const T* __restrict__ v, T* __restrict__ g) {
    const double eps = 1e-8;
    const EdgeFrame& f = X.f;
    const double th = X.th, a0 = X.a0, a1 = X.a1;
    double ga0, ga1, gth;
    if (f.ident) {
        ga0 = th * s0;
        ga1 = th * s1;
        gth = 0.0;                            // the exponent theta * (a . G) vanishes with a
    } else {
        const double rho = sqrt(a0 * a0 + a1 * a1);
        const double cph = a0 / rho, sph = a1 / rho;
        const double grho = th * s0;          // ang = theta rho
        gth = rho * s0;
        ga0 = cph * grho - sph / rho * s1;
        ga1 = sph * grho + cph / rho * s1;
    }
    // a = a_raw / (|a_raw| + eps), a_raw = (-d_y, d_x)
    const double ar0 = -X.dy, ar1 = X.dx, na = X.na, ta = na + eps;
    double gr0 = ga0 / ta, gr1 = ga1 / ta;
    if (na > 0.0) {
        const double dotp = (ga0 * ar0 + ga1 * ar1) / (na * ta * ta);
        gr0 -= dotp * ar0;
        gr1 -= dotp * ar1;
    }
    double gd0 = gr1, gd1 = -gr0, gd2 = 0.0;
    // theta = acos(clamp(d_z, -1 + eps, 1 - eps)): -1/sqrt(1 - d_z^2) where the
    // clamp passes d_z, 0 where it binds (torch's clamp gradient), so the
    // directions along +-e_z get finite gradients, the float64 values of the
    // reference's formula (its float32 autograd has 0 * -inf = NaN there)
    const double dz = X.dz;
    if (gth != 0.0 && dz >= -1.0 + eps && dz <= 1.0 - eps) gd2 = -gth / sqrt(1.0 - dz * dz);
    // d = v / (|v| + eps)
    const double vx = v[0], vy = v[1], vz = v[2];
    const double nv = X.nv, tv = nv + eps;
    double gv0 = gd0 / tv, gv1 = gd1 / tv, gv2 = gd2 / tv;
    if (nv > 0.0) {
        const double dotv = (gd0 * vx + gd1 * vy + gd2 * vz) / (nv * tv * tv);
        gv0 -= dotv * vx;
        gv1 -= dotv * vy;
        gv2 -= dotv * vz;
    }
    g[0] = static_cast<T>(gv0);
    g[1] = static_cast<T>(gv1);
    g[2] = static_cast<T>(gv2);
}

}  // namespace
}  // namespace feq
