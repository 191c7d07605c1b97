// nls_line.hip -- plain RK4 solves of one 1-D line of any length: waves that
// step overlapping pieces of the line in registers.
//
// A wave of 64 lanes holds Q consecutive points a lane: 64 Q points of which
// the inner S = 64 Q - 2H are its own and H = 4R on each side (R the stencil
// radius, four stages of R points) are copies of its neighbours'.  All four
// stages of a step run without leaving the wave -- neighbours come from the
// lane's own registers and from the next lanes by wave shifts (DPP) -- while
// the copies go stale from the outside in, by R points a stage.  After the
// step every wave writes its own points to LDS, and after one barrier the
// copies are read back: one barrier and one LDS round trip a step, where the
// resident kernel has four.
//
// A workgroup of NW waves holds NW S points.  A line that fits runs all the
// steps of a call (up to 4096 a launch) in one workgroup.  A longer one is
// cut into chunks: a workgroup runs K steps of B = NW S - 2H (K - 1) points,
// its region going stale by H points a step from both ends, so no workgroup
// waits for another; launches alternate between the caller's arrays and the
// workspace.
//
// Bound: a wave's chain of VALU instructions (about 200 for the four stages
// of a point at order 5, at four cycles each) and the LDS round trip; memory
// is read once in K steps.  Measured, us per step (the resident kernel, or
// beyond 4096 points the per-stage kernels, before): n = 256 FP32 dynamic
// 0.56 (0.88), n = 1000 radial FP32 0.61 (3.6), n = 4096 FP64 0.65 (6.3).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "nls_amd.h"
#include "nls_internal.h"
#include "nls_rk4.h"

namespace nls {

constexpr int LINE_WAVES = 8;            // waves per workgroup, at most

template <typename T> struct LineArgs {
    int n, steps;
    int B;                               // points a workgroup writes; 0: the whole line in one workgroup
    T dt, w0, w1, w2, w3;
    Coeffs<T> c;
    const T *wtab;                       // radial rows (n x order), reference boundaries only
    const cplx_t<T> *u; const T *un;
    cplx_t<T> *uo; T *uno;
    const T *P;
};

// Value of the previous (next) lane; lane 0 (63) gets zero.
template <bool NEXT> __device__ __forceinline__ int lane_shift(int v) {
    return __builtin_amdgcn_update_dpp(0, v, NEXT ? 0x130 : 0x138, 0xf, 0xf, true);
}
template <bool NEXT> __device__ __forceinline__ float lane_shift(float v) {
    return __builtin_bit_cast(float, lane_shift<NEXT>(__builtin_bit_cast(int, v)));
}
template <bool NEXT> __device__ __forceinline__ double lane_shift(double v) {
    typedef int I2 __attribute__((ext_vector_type(2)));
    I2 p = __builtin_bit_cast(I2, v);
    p.x = lane_shift<NEXT>(p.x);
    p.y = lane_shift<NEXT>(p.y);
    return __builtin_bit_cast(double, p);
}

template <typename T, int ORDER, int BC, bool DYN, int Q>
__global__ void __launch_bounds__(64 * LINE_WAVES) k_line(const LineArgs<T> a) {
    using C = cplx_t<T>;
    constexpr int R = (ORDER - 1) / 2, H = 4 * R, S = 64 * Q - 2 * H;
    static_assert(S > 0, "a wave owns points");
    __shared__ C ly[2][LINE_WAVES * S];
    __shared__ T ln[DYN ? 2 : 1][DYN ? LINE_WAVES * S : 1];
    const int n = a.n;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const bool whole = a.B == 0;
    // grid index of the workgroup's local position 0
    const int g0 = whole ? 0 : (int)blockIdx.x * a.B - H * (a.steps - 1);
    const int olo = whole ? 0 : (int)blockIdx.x * a.B, ohi = whole ? n : min(n, olo + a.B);
    const LineStep<T> h = line_step(a.dt);
    const T wc[4] = {a.w0, a.w1, a.w2, a.w3};

    C u[Q], y[Q], acc[Q];
    T un[Q], yn[Q], accn[Q], cp[Q];
    T wr[BC == BC_REF ? Q : 1][BC == BC_REF ? ORDER : 1];
    int lds[Q];                          // the point's place in LDS
    unsigned inside = 0, own = 0, copy = 0, out = 0;   // bit q: of point q
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int i = lane * Q + q, x = wave * S - H + i;
        int g = g0 + x;
        bool in = true;
        if (BC == BC_PERIODIC) {
            g %= n;
            g += g < 0 ? n : 0;
        } else {
            in = g >= 0 && g < n;
        }
        const bool edge = i < H || i >= 64 * Q - H;
        u[q] = mk<T>(0, 0); un[q] = 0; cp[q] = 0;
        if (in) {
            u[q] = a.u[g];
            cp[q] = pump_term<T, DYN>(a.c, a.P[g]);
            if (DYN) un[q] = a.un[g];
            inside |= 1u << q;
        }
        if constexpr (BC == BC_REF) {
#pragma unroll
            for (int k = 0; k < ORDER; ++k) wr[q][k] = in ? a.wtab[(size_t)g * ORDER + k] : (T)0;
        }
        lds[q] = whole ? g : x;
        if (!edge && (!whole || x < n)) own |= 1u << q;
        if (edge && (whole ? in : x >= 0 && x < nw * S)) copy |= 1u << q;
        // g0 + x, not its wrapped index: a chunk longer than the line holds
        // some points twice
        if (!edge && g0 + x >= olo && g0 + x < ohi) out |= 1u << q;
        y[q] = u[q]; yn[q] = un[q]; acc[q] = mk<T>(0, 0); accn[q] = 0;
    }

    auto stage = [&](auto s_) {
        constexpr int s = decltype(s_)::value;
        // the lane's points and R on each side, from the lanes before and after
        T ex[Q + 2 * R], ey[Q + 2 * R];
#pragma unroll
        for (int q = 0; q < Q; ++q) { ex[R + q] = y[q].x; ey[R + q] = y[q].y; }
#pragma unroll
        for (int d = 1; d <= R; ++d) {
            ex[R - d] = lane_shift<false>(ex[R - d + Q]);
            ey[R - d] = lane_shift<false>(ey[R - d + Q]);
            ex[R + Q - 1 + d] = lane_shift<true>(ex[R - 1 + d]);
            ey[R + Q - 1 + d] = lane_shift<true>(ey[R - 1 + d]);
        }
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            T lr, li;
            if constexpr (BC == BC_REF) {
                lr = line_lap_row<T, R>(wr[q], ex + R + q);
                li = line_lap_row<T, R>(wr[q], ey + R + q);
            } else {
                lr = line_lap<T, R>(wc, ex + R + q);
                li = line_lap<T, R>(wc, ey + R + q);
            }
            C k;
            T kn;
            line_rhs<T, DYN>(a.c, cp[q], mk<T>(ex[R + q], ey[R + q]), yn[q], lr, li, k, kn);
            y[q].x = line_combine<T, s>(acc[q].x, k.x, u[q].x, h);
            y[q].y = line_combine<T, s>(acc[q].y, k.y, u[q].y, h);
            if (DYN) yn[q] = line_combine<T, s>(accn[q], kn, un[q], h);
            if (BC == BC_REF && !((inside >> q) & 1u)) y[q] = mk<T>(0, 0);
        }
    };

    for (int it = 0; it < a.steps; ++it) {
        stage(std::integral_constant<int, 1>{});
        stage(std::integral_constant<int, 2>{});
        stage(std::integral_constant<int, 3>{});
        stage(std::integral_constant<int, 4>{});
        if (it + 1 < a.steps) {
            // two buffers: a wave writes one again only after the next
            // step's barrier, which every wave reaches after reading it
            C *const b = ly[it & 1];
            T *const bn = ln[DYN ? it & 1 : 0];
#pragma unroll
            for (int q = 0; q < Q; ++q)
                if ((own >> q) & 1u) {
                    b[lds[q]] = y[q];
                    if (DYN) bn[lds[q]] = yn[q];
                }
            __syncthreads();
#pragma unroll
            for (int q = 0; q < Q; ++q)
                if ((copy >> q) & 1u) {
                    y[q] = b[lds[q]];
                    if (DYN) yn[q] = bn[lds[q]];
                }
        }
#pragma unroll
        for (int q = 0; q < Q; ++q) { u[q] = y[q]; un[q] = yn[q]; }
    }
    // in place (whole lines): every wave has loaded the line before the first
    // barrier; a launch of one step has none of its own
    if (whole) __syncthreads();
#pragma unroll
    for (int q = 0; q < Q; ++q)
        if ((out >> q) & 1u) {
            const int g = g0 + wave * S - H + lane * Q + q;
            a.uo[g] = u[q];
            if (DYN) a.uno[g] = un[q];
        }
}

template <typename T, int Q>
static void launch_line_q(int order, int bc, bool dyn, int blocks, int nw, const LineArgs<T> &a, hipStream_t s) {
#define NLS_CASE(O, B, D)                                                                                    \
    if (order == O && bc == B && dyn == D) {                                                                 \
        hipLaunchKernelGGL((k_line<T, O, B, D, Q>), dim3(blocks), dim3(64 * nw), 0, s, a);                   \
        return;                                                                                              \
    }
    NLS_CASE(3, 0, false) NLS_CASE(3, 0, true) NLS_CASE(3, 1, false) NLS_CASE(3, 1, true)
    NLS_CASE(5, 0, false) NLS_CASE(5, 0, true) NLS_CASE(5, 1, false) NLS_CASE(5, 1, true)
    NLS_CASE(7, 0, false) NLS_CASE(7, 0, true) NLS_CASE(7, 1, false) NLS_CASE(7, 1, true)
#undef NLS_CASE
}
template <typename T>
static void launch_line(int q, int order, int bc, bool dyn, int blocks, int nw, const LineArgs<T> &a, hipStream_t s) {
    if (q == 1) launch_line_q<T, 1>(order, bc, dyn, blocks, nw, a, s);
    else if (q == 2) launch_line_q<T, 2>(order, bc, dyn, blocks, nw, a, s);
    else launch_line_q<T, 4>(order, bc, dyn, blocks, nw, a, s);
}

// How a line is cut.
struct LinePlan {
    int q, nw;                           // points a lane, waves a workgroup
    int k;                               // steps a launch
    int B;                               // points a workgroup writes; 0: the whole line
};

static int wave_points(int order, int q) { return 64 * q - 4 * (order - 1); }

// The plan with the least estimated time for `iters` steps, from what the
// kernel measured (MI355X, us; FP32 and FP64, algebraic and dynamic alike
// within 15%): a launch costs 2.0 beside its steps, a copy back from the workspace
// (chunks whose launches cannot be even) as much, a step 0.16 for the LDS
// round trip, the barrier and the latency of its four stages and 0.26 for
// each point a SIMD's lane steps (points a lane x waves on the SIMD).  So few
// points a lane and a wave on every SIMD are worth more than little overlap:
// n = 4096 runs 0.65 us a step as 256 workgroups of 16 points over 12 steps
// and 1.25 as 11 workgroups of 400; 16 is the least a chunk writes.  Wide
// lanes (Q = 4: 6 to 12% overlap instead of 25%) come in when the waves fill
// the device, beyond about 60,000 points.
static LinePlan line_plan(const nls_problem *p, int iters, int cus) {
    const double LAUNCH = 2.0, STEP = 0.16, POINT = 0.26;
    const int H = 2 * (p->order - 1);
    if (cus <= 0) cus = 256;
    LinePlan best = {4, LINE_WAVES, 1, 0};
    double least = -1;
    auto consider = [&](int q, int nw, int k, int B) {
        const double blocks = B ? (p->n + B - 1) / B : 1, launches = (iters + k - 1) / k;
        const double waves = (nw + 3) / 4 * ceil(blocks / cus);
        const bool copy = B && (int)launches % 2 && iters <= launches;
        const double t = (launches + copy) * LAUNCH + iters * (STEP + POINT * q * waves);
        if (least < 0 || t < least) { least = t; best = LinePlan{q, nw, k, B}; }
    };
    for (int q = 1; q <= 4; q *= 2) {
        const int S = wave_points(p->order, q);
        const int nw = (p->n + S - 1) / S;
        if (nw <= LINE_WAVES) consider(q, nw, 4096, 0);
        for (int k = 1; k <= std::min(iters, 64); ++k)
            for (int w = 4; w <= LINE_WAVES; w += 4) {
                const int B = w * S - 2 * H * (k - 1);
                if (B >= 16) consider(q, w, k, B);
            }
    }
    return best;
}

static size_t align256l(size_t b) { return (b + 255) & ~(size_t)255; }

template <typename T>
static int line_run(const nls_problem *p, const LinePlan &pl, int iters, const T *P, cplx_t<T> *psi, T *nres,
                    char *ws, hipStream_t s) {
    using C = cplx_t<T>;
    const int n = p->n;
    const bool dyn = p->coeffs[10] != 0.0;
    LineArgs<T> a;
    a.n = n;
    a.B = pl.B;
    a.dt = (T)p->dt;
    T w[4] = {0, 0, 0, 0};
    for (int d = 0; d <= (p->order - 1) / 2; ++d) w[d] = (T)stencil_s2(p->order, d, p->dx);
    a.w0 = w[0]; a.w1 = w[1]; a.w2 = w[2]; a.w3 = w[3];
    a.c = make_coeffs<T>(p->coeffs);
    a.wtab = nullptr;
    a.P = P;
    C *alt = (C *)ws;
    T *altn = (T *)(ws + align256l(n * sizeof(C)));
    if (p->bc == NLS_BC_REF) {
        T *tab = (T *)(ws + align256l(n * sizeof(C)) + (dyn ? align256l(n * sizeof(T)) : 0));
        launch_radial_table<T>(n, p->order, p->dx, tab, s);
        a.wtab = tab;
    }
    C *cur = psi;
    T *curn = nres;
    int launches = (iters + pl.k - 1) / pl.k;
    // chunks: an even count of launches ends in the caller's arrays
    if (pl.B && launches % 2 && iters > launches) ++launches;
    for (int l = 0, done = 0; l < launches; ++l) {
        a.steps = (iters - done + launches - l - 1) / (launches - l);
        done += a.steps;
        a.u = cur; a.un = curn;
        if (pl.B) { std::swap(cur, alt); std::swap(curn, altn); }
        a.uo = cur; a.uno = curn;
        launch_line<T>(pl.q, p->order, p->bc, dyn, pl.B ? (n + pl.B - 1) / pl.B : 1, pl.nw, a, s);
    }
    int rc = hip_check(hipGetLastError(), "line launch");
    if (rc) return rc;
    return cur == psi ? rc : copy_state<T>(n, cur, psi, dyn ? curn : nullptr, dyn ? nres : nullptr, s);
}

size_t line_workspace_bytes(const nls_problem *p) {
    const size_t rs = p->dtype == NLS_F64 ? 8 : 4;
    return align256l((size_t)p->n * 2 * rs) + (p->coeffs[10] != 0.0 ? align256l((size_t)p->n * rs) : 0) +
           (p->bc == NLS_BC_REF ? align256l((size_t)p->n * p->order * rs) : 0);
}

int line_advance(const nls_problem *p, int iters, const void *pumping, void *psi, void *nres, void *ws,
                 hipStream_t s) {
    const LinePlan pl = line_plan(p, iters, device_cus());
    if (p->dtype == NLS_F64)
        return line_run<double>(p, pl, iters, (const double *)pumping, (double2 *)psi, (double *)nres, (char *)ws, s);
    return line_run<float>(p, pl, iters, (const float *)pumping, (float2 *)psi, (float *)nres, (char *)ws, s);
}

}  // namespace nls
