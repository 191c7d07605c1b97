// nls_core.h -- device-side building blocks shared by the kernels of
// libnls_amd: complex load/store types, the pointwise right-hand side and
// the RK4 stage bookkeeping.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "nls_stencil.h"

namespace nls {

// BC_SLAB (2-D fused kernel only): one row slab of a grid that is periodic
// along its rows, with the 4R ghost rows above and below supplied in the
// buffers; x wraps, y reads the ghost rows.
enum { BC_REF = 0, BC_PERIODIC = 1, BC_SLAB = 2 };

template <typename T> struct cvec;
template <> struct cvec<float> { using type = float2; };
template <> struct cvec<double> { using type = double2; };
template <typename T> using cplx_t = typename cvec<T>::type;

template <typename T> __device__ __forceinline__ cplx_t<T> mk(T a, T b) {
    cplx_t<T> r; r.x = a; r.y = b; return r;
}

// Coefficients of the model actually read by the core (reference c(k)).
template <typename T> struct Coeffs {
    T c3, c4, c5, c6;        // gain, loss, self-interaction, reservoir coupling
    T c11, c12, c13, c14;    // reservoir: d/dt, pumping, decay, depletion
    T d12, d13, d14;         // c12/c11, c13/c11, c14/c11 (formed in double, rounded once); 0 when c11 = 0
};

template <typename T> inline Coeffs<T> make_coeffs(const double *c) {
    Coeffs<T> r;
    r.c3 = (T)c[2]; r.c4 = (T)c[3]; r.c5 = (T)c[4]; r.c6 = (T)c[5];
    r.c11 = (T)c[10]; r.c12 = (T)c[11]; r.c13 = (T)c[12]; r.c14 = (T)c[13];
    const bool dyn = c[10] != 0.0;
    r.d12 = dyn ? (T)(c[11] / c[10]) : (T)0;
    r.d13 = dyn ? (T)(c[12] / c[10]) : (T)0;
    r.d14 = dyn ? (T)(c[13] / c[10]) : (T)0;
    return r;
}

// Right-hand side at one point, given the stage input (y, yn), pumping P and
// the Laplacian of y.  Mirrors hamiltonian / revervoir of the reference
// (nls/nls.f90:570-581, :637-647):
//   r      = c12 P / (c13 + c14 |y|^2)   (adiabatic)   or yn (dynamic)
//   k.re   = (c3 r - c4) y.re + (c5 |y|^2 + c6 r) y.im - (L y).im
//   k.im   = (c3 r - c4) y.im - (c5 |y|^2 + c6 r) y.re + (L y).re
//   kn     = (c12 P - (c13 + c14 |y|^2) yn) / c11        (dynamic only)
// The reservoir's 1/c11 is folded into its coefficients once
// (kn = d12 P - (d13 + d14 |y|^2) yn), and each psi component is two fused
// multiply-adds; both regroupings move results by rounding only.
//
// rhs_point_cp takes the pumping term already formed as cP = c12 P
// (adiabatic) or d12 P (dynamic), so kernels that keep a point's pumping in
// a register across the four stages form it once (pump_term).
template <typename T, bool DYN> __device__ __forceinline__ T pump_term(const Coeffs<T> &c, T P) {
    return DYN ? c.d12 * P : c.c12 * P;
}

template <typename T, bool DYN>
__device__ __forceinline__ void rhs_point_cp(const Coeffs<T> &c, T cP, cplx_t<T> y, T yn, cplx_t<T> lap,
                                             cplx_t<T> &k, T &kn) {
    const T s = y.x * y.x + y.y * y.y;
    const T r = DYN ? yn : cP / (c.c13 + c.c14 * s);
    const T g = c.c3 * r - c.c4;
    const T q = c.c5 * s + c.c6 * r;
    k.x = fma(g, y.x, fma(q, y.y, -lap.y));
    k.y = fma(g, y.y, fma(-q, y.x, lap.x));
    if (DYN) kn = fma(-fma(c.d14, s, c.d13), yn, cP);
}

template <typename T, bool DYN>
__device__ __forceinline__ void rhs_point(const Coeffs<T> &c, T P, cplx_t<T> y, T yn, cplx_t<T> lap,
                                          cplx_t<T> &k, T &kn) {
    rhs_point_cp<T, DYN>(c, pump_term<T, DYN>(c, P), y, yn, lap, k, kn);
}

// Cartesian Laplacian of a point with value c from its neighbours at
// distance d = 1..R (weights w_d of nls_stencil.h).
//   double precision: the stencil sum as written, the centre weight times c
//     (lap_centre) plus w_d times the sum of the neighbours at distance d;
//   single precision: the centre weight is folded into the neighbour terms
//     (the weights of a stencil sum to zero).  For d = 1 the differences to c
//     are formed first -- exact when the values are close, as on a smooth
//     field on a fine grid -- so the largest weights (w_1 ~ 1/h^2) no longer
//     amplify the rounding of c; for d >= 2 the neighbour sum less 2c (1-D,
//     line_lap) or 4c (2-D, lap_quad).  This keeps the single-precision Laplacian accurate where the
//     stencil sum cancels to a small result.
// The two forms are equal up to rounding.
template <typename T> __device__ __forceinline__ T lap_centre(T wc, T c) {
    return sizeof(T) == 8 ? wc * c : (T)0;
}

template <typename T> __device__ __forceinline__ T lap_quad(T w, T c, T a0, T a1, T b0, T b1, int d) {
    if (sizeof(T) == 8) return w * ((a0 + a1) + (b0 + b1));
    if (d == 1) return w * (((a0 - c) + (a1 - c)) + ((b0 - c) + (b1 - c)));
    return w * (((a0 + a1) + (b0 + b1)) - (T)4 * c);
}

// Coefficients of the fused 2-D step: the slopes of psi are kept in a unit, the
// step sizes take it back (dt unit), the centre weight joins the point's own
// factor.  A coefficient, a weight or a step that is rounded is rounded alike at
// every point and step: a drift, beside which the points' own roundings average out.
//   Order 5, single precision: the unit is the first neighbour weight w_1, and the
// weights 1, -1/16 and -3.75 are exact; rounded they cost the 2048^2 grid 3.3e-6
// against 64 bits after 300 steps instead of 5.8e-7, the 512-grid sweep 2.1e-6 after
// 500 instead of 5.9e-7.  It is moved by what dt w_1 / 6 is rounded by, so that the
// step of the new state is exact and the weights take its rounding.
//   Orders 3 and 7, and grid_ring1_from's sums at every order: the one of 32 units
// whose coefficients, weights and step round least together.  The weights still sum to
// zero: of order 3 as they are, of order 7 in units of w_1, with a product of the sum
// (grid_sum).  A product or two a point and stage, 1 to 3% of a step (2 to 5% up to
// 64^2), against units of w_1, in which long solves ended up to 3.5 times further from
// 64 bits than with coefficients, weights and dt as they are, and against those as they
// are, up to 5 times further than in units of w_1.  Of 3000 random problems of 20^2 to
// 1200^2 nine in ten are now at most 1.03 times as far as with either, one is more than
// 1.5 times as far as with the coefficients as they are and four as in units of w_1.
//   Double precision takes everything as it is (unit 1).  The reservoir's slope
// keeps its own units.
constexpr float GRID_CENTRE_7 = (float)(-98.0 / 27.0);    // 2 w_0 / w_1 at order 7
template <typename T> struct GridCoeffs {
    T c3, c4, c5, c6, wc;    // c_k / unit, 2 w_0 / unit (order 7, single precision: 0)
    T r1, r2, r3;            // w_d / unit (single precision, order 5: r1 = 1, order 7: r2, r3 of w_1)
    T dtw, dtw6, dt6;        // dt unit, dt unit / 6, dt / 6
};
template <typename T>
inline GridCoeffs<T> make_grid_coeffs(const double *c, int order, double dt, double dx, T *lo = nullptr) {
    // where the Laplacian's weights vanish beside the coefficients (a spacing
    // beyond 1e14 or so), the unit is held at 2^-100 of the largest
    // coefficient, so that the quotients stay in range; the Laplacian then
    // stays far below rounding
    double cmax = 0.0;
    for (int k = 2; k < 6; ++k) cmax = c[k] > cmax ? c[k] : -c[k] > cmax ? -c[k] : cmax;
    const double w = stencil_s2(order, 1, dx), least = cmax * 0x1p-100;
    double unit = sizeof(T) == 8 ? 1.0 : w > least ? w : least, h = dx, per = 1.0;
    GridCoeffs<T> g;
    auto weights = [&] {
        if (sizeof(T) == 4 && order == 7 && !lo) {
            g.wc = (T)0;
            g.r1 = (T)(stencil_s2(order, 1, dx) / per);
            g.r2 = (T)-0.1;
            g.r3 = (T)(-0.25 * (double)GRID_CENTRE_7 - 1.0 - (double)g.r2);
            return;
        }
        g.wc = (T)(2.0 * stencil_s2(order, 0, h) / per);
        g.r1 = (T)(stencil_s2(order, 1, h) / per);
        g.r2 = order > 3 ? (T)(stencil_s2(order, 2, h) / per) : (T)0;
        g.r3 = order > 5 ? (T)(stencil_s2(order, 3, h) / per) : (T)0;
    };
    if (sizeof(T) == 4 && order == 5 && !lo) {
        // in units of w_1 the ratios do not depend on the spacing
        h = 1.0;
        per = stencil_s2(order, 1, h);
        const float step = (float)(dt * unit / 6.0);
        if (std::isnormal(step)) unit = 6.0 * step / dt;
    } else if (sizeof(T) == 4) {
        // the unit's place between two powers of two: where the roundings of the
        // coefficients and the Laplacian (its second moment), each with the step's, are
        // least together
        const double base = std::ldexp(1.0, std::ilogb(unit));
        const double moment = w + 4.0 * (order > 3 ? stencil_s2(order, 2, dx) : 0.0) +
                              9.0 * (order > 5 ? stencil_s2(order, 3, dx) : 0.0);
        double best = HUGE_VAL;
        unit = per = base;
        for (int j = 0; j < 32; ++j) {
            const double u = base * (1.0 + j / 32.0), step = dt * u / 6.0, es = lo ? 0.0 : (float)step / step - 1.0;
            per = u;
            weights();
            double e = order == 7 && !lo ? g.r1 * u / w : (g.r1 + 4.0 * g.r2 + 9.0 * g.r3) * u / moment, sum;
            e += es - 1.0;
            sum = e * e;
            for (int k = 2; k < 6; ++k) {
                const double x = c[k] / u;
                e = x != 0.0 ? (float)x / x - 1.0 + es : 0.0;
                sum += e * e;
            }
            if (sum < best) { best = sum; unit = u; }
        }
        per = unit;
    }
    weights();
    g.c3 = (T)(c[2] / unit); g.c4 = (T)(c[3] / unit); g.c5 = (T)(c[4] / unit); g.c6 = (T)(c[5] / unit);
    g.dtw = (T)(dt * unit);
    g.dtw6 = (T)(dt * unit / 6.0);
    g.dt6 = (T)(dt / 6.0);
    if (lo) {
        lo[0] = (T)(dt * unit / 6.0 - g.dtw6);
        lo[1] = (T)(dt / 6.0 - g.dt6);
    }
    return g;
}

// Arithmetic of one point of the fused 2-D step, shared by its kernels, with
// every fused multiply-add written out and contraction off: a grid's result
// has the same bits in every form, tile shape and row slab.
// The neighbour sum, ring by ring: sum of r_d ((left + right) + (up + down)),
// r_1 = 1 in single precision of order 5.
template <int R, typename T> __device__ __forceinline__ T grid_ring1(const GridCoeffs<T> &g, T l, T r, T u, T d) {
#pragma clang fp contract(off)
    const T s = (l + r) + (u + d);
    return sizeof(T) == 4 && R > 1 ? s : g.r1 * s;
}
template <typename T> __device__ __forceinline__ T grid_ring(T S, T ratio, T l, T r, T u, T d) {
#pragma clang fp contract(off)
    return fma(ratio, (l + r) + (u + d), S);
}
// Order 7 in single precision: the centre's share joins the sum, in units of w_1.
template <int R, typename T>
__device__ __forceinline__ cplx_t<T> grid_sum(const GridCoeffs<T> &g, cplx_t<T> y, T sr, T sm) {
#pragma clang fp contract(off)
    if constexpr (sizeof(T) == 4 && R == 3)
        return mk<T>(g.r1 * fma(GRID_CENTRE_7, y.x, sr), g.r1 * fma(GRID_CENTRE_7, y.y, sm));
    return mk<T>(sr, sm);
}
// The same sums less the centre's share, for the kernels of grids of up to 64
// points a side in single precision: neighbours close to the centre c differ
// from it exactly, and neither the sum nor the point's factor is rounded at
// the size of the centre weight.  Eight operations a point and stage more than
// with the centre weight in the factor; those kernels wait for latency.
// The sixth of the step carries what its rounding leaves (grid_new_from), so that the
// unit need not suit it.
__device__ __forceinline__ float grid_ring1_from(float w, float c, float l, float r, float u, float d) {
#pragma clang fp contract(off)
    return w * (((l - c) + (r - c)) + ((u - c) + (d - c)));
}
__device__ __forceinline__ float grid_ring_from(float S, float ratio, float c, float l, float r, float u, float d) {
#pragma clang fp contract(off)
    return fma(ratio, fma(-4.0f, c, (l + r) + (u + d)), S);
}
// Slopes at a point (y, yn) from its neighbour sum S.  FROM: of those sums.
template <typename T, bool DYN, bool FROM = false>
__device__ __forceinline__ void grid_rhs(const GridCoeffs<T> &g, const Coeffs<T> &c, T cP, cplx_t<T> y, T yn,
                                         cplx_t<T> S, cplx_t<T> &k, T &kn) {
#pragma clang fp contract(off)
    const T s = fma(y.x, y.x, y.y * y.y);
    const T r = DYN ? yn : cP / fma(c.c14, s, c.c13);
    const T a = fma(g.c3, r, -g.c4);
    T q;
    if constexpr (FROM) {
        q = fma(g.c5, s, g.c6 * r);
    } else if constexpr (sizeof(T) == 4) {
        q = fma(g.c5, s, fma(g.c6, r, -g.wc));
    } else {
        q = fma(g.c5, s, g.c6 * r);
        S.x = fma(g.wc, y.x, S.x);
        S.y = fma(g.wc, y.y, S.y);
    }
    k.x = fma(a, y.x, fma(q, y.y, -S.y));
    k.y = fma(a, y.y, fma(-q, y.x, S.x));
    kn = DYN ? fma(-fma(c.d14, s, c.d13), yn, cP) : (T)0;
}
// Accumulator after stage s = 1..3, the next stage's input u + k step, and
// the new state u + (acc + k4) dt/6.
template <typename T> __device__ __forceinline__ void grid_acc(T &acc, T k, bool first) {
    acc = first ? k : fma((T)2, k, acc);
}
template <typename T> __device__ __forceinline__ T grid_input(T u, T k, T step) { return fma(k, step, u); }
template <typename T> __device__ __forceinline__ T grid_new(T u, T acc, T k, T step6) {
    return fma(acc + k, step6, u);
}
// The same with the sixth of the step in two terms (beside grid_ring1_from).  The
// second, lo, is added to the increment; to u it would be lost.
template <typename T> __device__ __forceinline__ T grid_new_from(T u, T acc, T k, T step6, T lo) {
#pragma clang fp contract(off)
    const T s = acc + k;
    return u + fma(s, step6, s * lo);
}

// Arithmetic of one point of a 1-D line, shared by the resident and the line
// kernels, with every fused multiply-add written out and contraction off:
// both kernels round each operation alike, so a line solved alone and in a
// batch gives the same bits whichever of them runs it.
// Periodic Laplacian from the neighbours e[-R..R] (e[0] the point), in the
// forms above.
template <typename T, int R> __device__ __forceinline__ T line_lap(const T *w, const T *e) {
#pragma clang fp contract(off)
    T l;
    if constexpr (sizeof(T) == 8) {
        l = w[0] * e[0];
#pragma unroll
        for (int d = 1; d <= R; ++d) l = fma(w[d], e[-d] + e[d], l);
    } else {
        l = w[1] * ((e[-1] - e[0]) + (e[1] - e[0]));
#pragma unroll
        for (int d = 2; d <= R; ++d) l = fma(w[d], fma((T)-2, e[0], e[-d] + e[d]), l);
    }
    return l;
}
// Radial Laplacian: the row's weights on e[-R..R]; points outside the grid
// are zero and their weights too.
template <typename T, int R> __device__ __forceinline__ T line_lap_row(const T *w, const T *e) {
#pragma clang fp contract(off)
    T l = w[0] * e[-R];
#pragma unroll
    for (int d = 1 - R; d <= R; ++d) l = fma(w[d + R], e[d], l);
    return l;
}
// Right-hand side of rhs_point_cp.
template <typename T, bool DYN>
__device__ __forceinline__ void line_rhs(const Coeffs<T> &c, T cP, cplx_t<T> y, T yn, T lr, T li, cplx_t<T> &k,
                                         T &kn) {
#pragma clang fp contract(off)
    const T s = fma(y.x, y.x, y.y * y.y);
    const T r = DYN ? yn : cP / fma(c.c14, s, c.c13);
    const T g = fma(c.c3, r, -c.c4);
    const T q = fma(c.c5, s, c.c6 * r);
    k.x = fma(g, y.x, fma(q, y.y, -li));
    k.y = fma(g, y.y, fma(-q, y.x, lr));
    kn = DYN ? fma(-fma(c.d14, s, c.d13), yn, cP) : (T)0;
}
// Step sizes of a line: dt, dt/2 and dt/6 = dt6 + dt6lo.  In single precision
// dt6 alone would stretch every step by its rounding, the same way each time:
// 2000 steps of the 256-point line end 2.1e-6 from the exact solution with it
// and 1.7e-6 with dt6lo, as with a division by 6.
template <typename T> struct LineStep {
    T dt, dt2, dt6, dt6lo;
};
template <typename T> __device__ __forceinline__ LineStep<T> line_step(T dt) {
#pragma clang fp contract(off)
    LineStep<T> h;
    h.dt = dt;
    h.dt2 = dt * (T)0.5;
    h.dt6 = dt / (T)6;
    h.dt6lo = fma((T)-6, h.dt6, dt) / (T)6;
    return h;
}
// Stage S = 1..4 of the combination: acc := k1 + 2 k2 + 2 k3 + k4 so far;
// returns the next stage input u + k (dt/2, dt/2, dt), at S = 4 the new
// state u + acc dt/6.
template <typename T, int S> __device__ __forceinline__ T line_combine(T &acc, T k, T u, const LineStep<T> &h) {
#pragma clang fp contract(off)
    acc = S == 1 ? k : S == 4 ? acc + k : fma((T)2, k, acc);
    if (S < 4) return fma(k, S == 3 ? h.dt : h.dt2, u);
    if (sizeof(T) == 8) return fma(acc, h.dt6, u);
    return u + fma(acc, h.dt6, acc * h.dt6lo);
}

// Periodic index wrap for offsets that may exceed one period.
__device__ __forceinline__ int wrap_index(int g, int n) {
    while (g < 0) g += n;
    while (g >= n) g -= n;
    return g;
}

// Periodic index wrap for -n <= g < 2n as one three-way unsigned minimum:
// of g, g + n and g - n exactly one lies in [0, n) and the others, as
// unsigned values, are larger.
__device__ __forceinline__ int wrap_near3(int g, int n) {
    const unsigned a = (unsigned)g, b = (unsigned)(g + n), c = (unsigned)(g - n);
    return (int)min(min(a, b), c);
}

// Linear index gy * n + gx of a point of an n x n grid whose index fits 32
// bits (so gy, n < 2^24): one 24-bit multiply-add.  Written as a 32-bit
// product the compiler emits a 64-bit multiply-add whose high addend half
// it may take from any register -- in the fused kernels, one a ring-table
// load is still filling, so the first field loads waited for that load.
__device__ __forceinline__ unsigned grid_index(int gy, int n, int gx) {
    return __umul24((unsigned)gy, (unsigned)n) + (unsigned)gx;
}

// Periodic index wrap for -n <= g < 2n.
__device__ __forceinline__ int wrap_near(int g, int n) {
    g += g < 0 ? n : 0;
    g -= g >= n ? n : 0;
    return g;
}

}  // namespace nls
