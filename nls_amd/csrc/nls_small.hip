// nls_small.hip -- RK4 on small 2-D grids: several steps of one grid per
// launch, and grids of up to 64 x 64 held by one workgroup each.
#include <type_traits>

#include "nls_march.h"
#include "nls_internal.h"

namespace nls {

// ---------------------------------------------------------------------------
// Several steps per launch.  A small grid leaves most of the device idle and a
// launch that steps it once is mostly its own latency (dispatch, first loads,
// last stores: about 3 us of the 5.3 us that a 256^2 grid's step took).  Here
// a workgroup takes a small output tile with the halo of K steps around it
// (4R K rings, R the stencil radius), steps the shrinking region K times on
// chip -- the fused step's stages, arithmetic and ring order (nls_batch.hip)
// -- and writes the tile: more halo arithmetic on compute units that were
// idle, for 1/K of the launches.
// Bound: the stages one after another, each an LDS round trip, a barrier and
// the vector instructions of three or four waves a SIMD (0.4 us each).
// Measured, us per step before -> after: 256^2 order 5 FP32 5.28 -> 3.70, FP64
// 6.27 -> 4.51; 128^2 FP32 5.19 -> 3.04; 40^2 order 3 zero-outside (one
// workgroup before) 2.6 -> 1.76; order 7 256^2 FP64, one step of smaller tiles,
// 8.37 -> 6.39.
// ---------------------------------------------------------------------------

// Region points in ring order (innermost first), S stages of R rings: LDS
// index in bits 0..15, x in 16..23, y in 24..31.
template <int W, int HH, int R, int S, int WS> struct StepMap {
    unsigned v[W * HH];
    constexpr StepMap() : v() {
        int k = 0;
        for (int s = S; s >= 0; --s) {
            const int a = s * R, b = (s + 1) * R;
            for (int y = a; y < HH - a; ++y)
                for (int x = a; x < W - a; ++x)
                    if (s == S || y < b || y >= HH - b || x < b || x >= W - b)
                        v[k++] = (unsigned)(y * WS + x) | (unsigned)x << 16 | (unsigned)y << 24;
        }
    }
};
template <int W, int HH, int R, int S, int WS> __device__ const StepMap<W, HH, R, S, WS> step_map{};

// LDS row stride: as the fused kernel's, the lanes of a side band (2R points
// a row) spread over the banks.
constexpr int multi_stride(int W, int R) { return W + (R == 1 ? 2 : R == 2 ? 4 : 14); }

// FROM: grid_ring1_from's sums.
template <typename T, int ORDER, int BC, bool DYN, int TX, int TY, int K, bool FROM>
__global__ void __launch_bounds__(1024) k_multi(const MultiArgs<T> f) {
    using C = cplx_t<T>;
    constexpr int R = (ORDER - 1) / 2, NT = 1024, S = 4 * K, H = S * R;
    constexpr int W = TX + 2 * H, HH = TY + 2 * H, NP = W * HH, NOUT = TX * TY;
    constexpr int WS = multi_stride(W, R), PAD = R * WS + R;
    constexpr int J = (NP + NT - 1) / NT;
    static_assert(W < 256 && HH < 256 && HH * WS < 65536 && J <= 32, "region shape");
    __shared__ C mem[2][HH * WS + 2 * PAD];

    const MemberDev<T> m = f.grid;
    const int n = m.n, tid = threadIdx.x;
    const int x0 = (int)(blockIdx.x % f.ntx) * TX, y0 = (int)(blockIdx.x / f.ntx) * TY;
    const unsigned *map = step_map<W, HH, R, S, WS>.v;
    unsigned ent[J];
#pragma unroll
    for (int j = 0; j < J; ++j) ent[j] = (NP % NT == 0 || j < J - 1 || tid + NT * j < NP) ? map[tid + NT * j] : 0u;

    const T dt = m.dt, dt2 = dt * (T)0.5;
    const Coeffs<T> c = m.c;
    const GridCoeffs<T> g = m.g;
    T dtw6lo = 0, dt6lo = 0;
    if constexpr (FROM) { dtw6lo = m.lo[0]; dt6lo = m.lo[1]; }
    const T dtw = g.dtw, dtw2 = dtw * (T)0.5, dtw6 = g.dtw6;

    C uu[J], acc[J];
    T cp[J], nn[J], yn[J], accn[J];
    int li[J];
    unsigned inside = 0;                 // bit j: the point lies on the region and the grid
#pragma unroll
    for (int j = 0; j < J; ++j) {
        uu[j] = acc[j] = mk<T>(0, 0);
        cp[j] = nn[j] = accn[j] = 0;
        li[j] = ent[j] & 0xffff;
        int gx = x0 - H + (int)((ent[j] >> 16) & 255), gy = y0 - H + (int)(ent[j] >> 24);
        bool ok = NP % NT == 0 || j < J - 1 || tid + NT * j < NP;
        if (BC == BC_PERIODIC) {
            gx = wrap_index(gx, n);      // (the halo may exceed the grid)
            gy = wrap_index(gy, n);
        } else {
            ok = ok && gx >= 0 && gx < n && gy >= 0 && gy < n;
        }
        if (ok) {
            const int gi = gy * n + gx;
            inside |= 1u << j;
            uu[j] = f.u[gi];
            cp[j] = f.P[gi];
            if (DYN) nn[j] = f.un[gi];
        }
    }
#pragma unroll
    for (int j = 0; j < J; ++j) {
        if (NP % NT == 0 || j < J - 1 || tid + NT * j < NP) {
            mem[0][PAD + li[j]] = uu[j];
            // points outside the reference's grid stay zero in both buffers
            if (BC == BC_REF && !((inside >> j) & 1u)) mem[1][PAD + li[j]] = uu[j];
        }
        cp[j] = pump_term<T, DYN>(c, cp[j]);
        yn[j] = nn[j];
    }
    __syncthreads();

    typedef T V2 __attribute__((ext_vector_type(2)));
    using LV = __attribute__((address_space(3))) const V2;
    auto slopes = [&](const C *yin, int j, C &k, T &kn) {
        unsigned a = (unsigned)(size_t)((LV *)yin + li[j]);   // R rows and R points before the point
        asm volatile("" : "+v"(a));
        LV *ys = (LV *)(size_t)a;
        auto rd = [&](int i) { const V2 v = ys[PAD + i]; return mk<T>(v.x, v.y); };
        const C y = rd(0);
        T sr, sm;
#pragma unroll
        for (int d = 1; d <= R; ++d) {
            const C l = rd(-d), r = rd(d), u = rd(-d * WS), b = rd(d * WS);
            if constexpr (FROM) {
                const float q = d == 2 ? g.r2 : g.r3;
                sr = d == 1 ? grid_ring1_from(g.r1, y.x, l.x, r.x, u.x, b.x) : grid_ring_from(sr, q, y.x, l.x, r.x, u.x, b.x);
                sm = d == 1 ? grid_ring1_from(g.r1, y.y, l.y, r.y, u.y, b.y) : grid_ring_from(sm, q, y.y, l.y, r.y, u.y, b.y);
            } else if (d == 1) {
                sr = grid_ring1<R>(g, l.x, r.x, u.x, b.x);
                sm = grid_ring1<R>(g, l.y, r.y, u.y, b.y);
            } else {
                sr = grid_ring(sr, d == 2 ? g.r2 : g.r3, l.x, r.x, u.x, b.x);
                sm = grid_ring(sm, d == 2 ? g.r2 : g.r3, l.y, r.y, u.y, b.y);
            }
        }
        grid_rhs<T, DYN, FROM>(g, c, cp[j], y, yn[j], FROM ? mk<T>(sr, sm) : grid_sum<R, T>(g, y, sr, sm), k, kn);
    };

    // stage st of S: points with at least st R rings around them, a prefix of
    // the list (the count opaque, so that each point's body stays a block of
    // its own)
#pragma unroll
    for (int st = 1; st <= S; ++st) {
        if (FROM && st <= 4 * (K - f.steps)) continue;      // fewer steps than K: the outer rings stay out
        const int s = (st - 1) % 4 + 1;
        const int cnt = (W - 2 * st * R) * (HH - 2 * st * R);
        int lim = cnt;
        asm volatile("" : "+s"(lim));
        const C *yin = mem[(st - 1) & 1];
        C *yout = mem[st & 1] + PAD;
        const T dta = s == 3 ? dt : dt2, dtwa = s == 3 ? dtw : dtw2;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            if (NT * j >= cnt) break;
            if (tid + NT * j >= lim) continue;
            if (BC == BC_REF && !((inside >> j) & 1u)) continue;
            C k;
            T kn;
            slopes(yin, j, k, kn);
            C y;
            if (s < 4) {
                grid_acc(acc[j].x, k.x, s == 1);
                grid_acc(acc[j].y, k.y, s == 1);
                if (DYN) grid_acc(accn[j], kn, s == 1);
                y = mk<T>(grid_input(uu[j].x, k.x, dtwa), grid_input(uu[j].y, k.y, dtwa));
                if (DYN) yn[j] = grid_input(nn[j], kn, dta);
            } else {
                if constexpr (FROM) {
                    y = mk<T>(grid_new_from(uu[j].x, acc[j].x, k.x, dtw6, dtw6lo),
                              grid_new_from(uu[j].y, acc[j].y, k.y, dtw6, dtw6lo));
                    if (DYN) nn[j] = yn[j] = grid_new_from(nn[j], accn[j], kn, g.dt6, dt6lo);
                } else {
                    y = mk<T>(grid_new(uu[j].x, acc[j].x, k.x, dtw6), grid_new(uu[j].y, acc[j].y, k.y, dtw6));
                    if (DYN) nn[j] = yn[j] = grid_new(nn[j], accn[j], kn, g.dt6);
                }
                uu[j] = y;
            }
            if (st < S) yout[li[j]] = y;
        }
        if (st < S) __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < J; ++j) {
        if (NT * j >= NOUT) break;
        const int gx = x0 - H + (int)((ent[j] >> 16) & 255), gy = y0 - H + (int)(ent[j] >> 24);
        if ((NOUT % NT && tid + NT * j >= NOUT) || gx >= n || gy >= n) continue;
        const size_t gi = (size_t)gy * n + gx;
        f.uo[gi] = uu[j];
        if (DYN) f.uno[gi] = nn[j];
    }
}

// Tiles: as small as keeps a launch within one workgroup a compute unit; K
// steps while their halo is not much wider than the tile.  Order 5, us per
// step: 256^2 as 256 tiles of 32 x 8 over two steps 3.68, 16 x 16 3.80, 32 x 16
// 4.08, three steps 4.36, one step 4.49; 128^2 as 16 x 8 2.96, 8 x 8 3.00, three
// steps 3.37; 512^2 as 256 tiles of 32 x 32 6.20 against 5.7 of the fused
// kernel, which keeps it.  Order 3 (half the halo): 256^2 as 16 x 16 over four
// steps 2.32, two 2.50; 40^2 as 8 x 8 over four 1.68, six 1.98.  Order 7: one
// step of 16 x 16 tiles (256^2 FP64 6.4; two steps do not fit the LDS).
struct MultiShape {
    int tx, ty, k;
};
static MultiShape multi_shape(int n, int order, int cus) {
    const MultiShape shapes[2] = {order == 3 ? MultiShape{8, 8, 4} : order == 5 ? MultiShape{16, 8, 2} : MultiShape{16, 16, 1},
                                  order == 3 ? MultiShape{16, 16, 4} : order == 5 ? MultiShape{32, 8, 2} : MultiShape{16, 16, 1}};
    for (const MultiShape &s : shapes)
        if ((long long)((n + s.tx - 1) / s.tx) * ((n + s.ty - 1) / s.ty) <= cus) return s;
    return MultiShape{0, 0, 0};
}
int multi_steps(int n, int order, int cus) { return multi_shape(n, order, cus).k; }

template <typename T, int O, int B, bool D, int TX, int TY, int K, bool FROM = false>
static void launch_multi_t(MultiArgs<T> a, hipStream_t s) {
    const int n = a.grid.n;
    a.ntx = (n + TX - 1) / TX;
    hipLaunchKernelGGL((k_multi<T, O, B, D, TX, TY, K, FROM>), dim3(a.ntx * ((n + TY - 1) / TY)), dim3(1024), 0, s, a);
}
template <typename T, int B, bool D> static void launch_multi_o(int order, const MultiArgs<T> &a, int tx, hipStream_t s) {
    if constexpr (sizeof(T) == 4)
        if (a.steps) {                   // up to 64 points a side: the first shapes
            if (order == 3) launch_multi_t<T, 3, B, D, 8, 8, 4, true>(a, s);
            else if (order == 5) launch_multi_t<T, 5, B, D, 16, 8, 2, true>(a, s);
            else launch_multi_t<T, 7, B, D, 16, 16, 1, true>(a, s);
            return;
        }
    if (order == 3) {
        if (tx == 8) launch_multi_t<T, 3, B, D, 8, 8, 4>(a, s);
        else launch_multi_t<T, 3, B, D, 16, 16, 4>(a, s);
    } else if (order == 5) {
        if (tx == 16) launch_multi_t<T, 5, B, D, 16, 8, 2>(a, s);
        else launch_multi_t<T, 5, B, D, 32, 8, 2>(a, s);
    } else {
        launch_multi_t<T, 7, B, D, 16, 16, 1>(a, s);
    }
}
template <typename T> void launch_multi(int order, int bc, bool dyn, MultiArgs<T> a, int cus, hipStream_t s) {
    const int tx = multi_shape(a.grid.n, order, cus).tx;
    if (bc == NLS_BC_REF) {
        if (dyn) launch_multi_o<T, BC_REF, true>(order, a, tx, s);
        else launch_multi_o<T, BC_REF, false>(order, a, tx, s);
    } else {
        if (dyn) launch_multi_o<T, BC_PERIODIC, true>(order, a, tx, s);
        else launch_multi_o<T, BC_PERIODIC, false>(order, a, tx, s);
    }
}
template void launch_multi<float>(int, int, bool, MultiArgs<float>, int, hipStream_t);
template void launch_multi<double>(int, int, bool, MultiArgs<double>, int, hipStream_t);

// ---------------------------------------------------------------------------
// One workgroup per grid of up to 64 x 64 (the RESIDENT engine in 2-D), all
// steps of a call in one launch.  A thread holds V points below one another:
// it knows its own column, so a point costs 2R horizontal LDS reads and its
// share of 2R vertical ones, 5 a point at order 5 instead of 9, all at
// constant offsets (rows of 64 + 2R points whatever n is, the border holding
// zeros, or on periodic grids copies that the edge threads write).  Two
// buffers, one barrier a stage.  The arithmetic is the fused step's, in single
// precision with grid_ring1_from's sums.
// Bound: vector instructions of one compute unit; few grids, the latency of a
// thread's points in turn.  us per step, order 5, one point a thread slot with all
// its reads -> strips: FP32, one grid, zero-outside 16^2 1.46 -> 0.98, 32^2 2.2 -> 1.65,
// 64^2 7.5 -> 5.2; periodic 32^2 1.8 -> 1.5, 48^2 3.6 -> 3.2, 56^2 4.7 -> 4.8, dynamic
// 64^2 5.1 -> 4.9; 1000 grids of 16^2 periodic 4.5 -> 2.0.  FP64, one grid, zero-outside
// 64^2 14.8 -> 7.9, periodic 48^2 6.6 -> 6.0, 64^2 10.9 -> 9.0; 1000 of 16^2 8.9 -> 4.2.
// Behind are periodic algebraic grids of 33 to 36 points (33^2 order 7 2.8 -> 3.3), where
// strips of two points fill nine waves, so that one SIMD steps three of them.
// ---------------------------------------------------------------------------
constexpr int square_v(int bytes) { return bytes == 4 ? 4 : 8; }      // V of 64 x 64 grids

template <typename T, int ORDER, int BC, bool DYN, int V>
__global__ void __launch_bounds__((V > 4 ? 512 : 1024)) k_resident_2d(const ResidentArgs<T> r) {
    using C = cplx_t<T>;
    constexpr int R = (ORDER - 1) / 2, WS = 64 + 2 * R;
    __shared__ C mem[2][WS * WS];
    const MemberDev<T> m = r.mem[blockIdx.x];
    const int n = m.n, tid = threadIdx.x;
    const int steps = min(r.iters, m.steps);
    // (the host plans no larger grid, nor one with more strips than threads)
    if (n > 64 || n * ((n + V - 1) / V) > (int)blockDim.x || steps <= 0) return;
    C *psi = r.psi + m.off;
    T *nres = DYN ? r.nres + m.off : nullptr;
    const T *P = r.P + m.off;
    const T dt = m.dt, dt2 = dt * (T)0.5;
    const Coeffs<T> c = m.c;
    const GridCoeffs<T> g = m.g;
    T dtw6lo = 0, dt6lo = 0;
    if constexpr (sizeof(T) == 4) { dtw6lo = m.lo[0]; dt6lo = m.lo[1]; }
    const T dtw = g.dtw, dtw2 = dtw * (T)0.5, dtw6 = g.dtw6;

    const int strip = tid / n, col = tid - strip * n, r0 = strip * V;
    const int rows = min(V, n - r0);     // points of this thread; none if <= 0
    const int li = (r0 + R) * WS + col + R;
    // copies across the border of a periodic grid: of the thread's column, and
    // of its rows (bit v: the row is copied past the bottom, past the top)
    const int cx = BC != BC_PERIODIC ? 0 : col < R ? n : col >= n - R ? -n : 0;
    const bool top = BC == BC_PERIODIC && r0 < R, bottom = BC == BC_PERIODIC && r0 + rows > n - R;

    // KEEP: the thread's own stage inputs stay in registers; double precision
    // has none to spare and reads its column from LDS as it goes down
    constexpr bool KEEP = sizeof(T) == 4;
    // WRAP: the points of a periodic grid read their neighbours from the places they
    // wrap to, held in registers, and nothing is copied (56^2 FP32 6.2 -> 4.8 us a
    // step); eight points in double precision with a reservoir would spill
    constexpr bool WRAP = BC == BC_PERIODIC && (V < 8 || !DYN);
    unsigned ry[WRAP ? V + 2 * R : 1], hx[WRAP ? V : 1][2 * R];     // LDS byte addresses in the first buffer
    typedef T V2 __attribute__((ext_vector_type(2)));
    using LV = __attribute__((address_space(3))) const V2;
    if constexpr (WRAP) {
        auto at = [&](int y, int x) {
            return (unsigned)(size_t)((LV *)mem[0] + (wrap_near(y, n) + R) * WS + wrap_near(x, n) + R);
        };
#pragma unroll
        for (int d = 0; d < V + 2 * R; ++d) ry[d] = at(r0 - R + d, col);
#pragma unroll
        for (int v = 0; v < V; ++v)
#pragma unroll
            for (int d = 1; d <= R; ++d) {
                hx[v][d - 1] = at(r0 + v, col - d);
                hx[v][R + d - 1] = at(r0 + v, col + d);
            }
    }
    if constexpr (!WRAP) {               // the border
        for (int i = tid; i < WS * WS; i += blockDim.x) mem[0][i] = mem[1][i] = mk<T>(0, 0);
        __syncthreads();
    }
    C u[V], y[KEEP ? V : 1], acc[V];
    T cp[V], un[V], yn[V], accn[V];
    // copies of the thread's points, just written to out, across the border
    auto copy_edges = [&](C *out) {
        if constexpr (WRAP) {
        } else if constexpr (KEEP) {
#pragma unroll
            for (int v = 0; v < V; ++v) {
                if (v >= rows) continue;
                if (cx) out[li + v * WS + cx] = y[v];
                if (top && r0 + v < R) out[li + (v + n) * WS] = y[v];
                if (bottom && r0 + v >= n - R) out[li + (v - n) * WS] = y[v];
            }
        } else {
            if (cx)
#pragma clang loop unroll(disable)
                for (int v = 0; v < rows; ++v) out[li + v * WS + cx] = out[li + v * WS];
            if (top)
#pragma clang loop unroll(disable)
                for (int v = 0; v < rows && r0 + v < R; ++v) out[li + (v + n) * WS] = out[li + v * WS];
            if (bottom)
#pragma clang loop unroll(disable)
                for (int v = max(0, n - R - r0); v < rows; ++v) out[li + (v - n) * WS] = out[li + v * WS];
        }
    };
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const bool ok = v < rows;
        const int idx = (r0 + v) * n + col;
        u[v] = ok ? psi[idx] : mk<T>(0, 0);
        cp[v] = pump_term<T, DYN>(c, ok ? P[idx] : (T)0);
        un[v] = yn[v] = DYN && ok ? nres[idx] : (T)0;
        if (KEEP) y[KEEP ? v : 0] = u[v];
        acc[v] = mk<T>(0, 0);
        accn[v] = 0;
        if (ok) mem[0][li + v * WS] = u[v];
    }
    if (rows > 0) copy_edges(mem[0]);
    __syncthreads();

    auto stage = [&](auto s_) {
        constexpr int s = decltype(s_)::value;
        const T dta = s == 3 ? dt : dt2, dtwa = s == 3 ? dtw : dtw2;
        if (rows > 0) {
            unsigned a = (unsigned)(size_t)((LV *)mem[(s - 1) & 1] + (li - R * WS - R));
            asm volatile("" : "+v"(a));
            LV *in = (LV *)(size_t)a;
            auto rd = [&](int row, int x) {
                V2 z;
                if constexpr (WRAP)
                    z = *(LV *)(size_t)((x == 0 ? ry[row + R] : hx[row][x < 0 ? -x - 1 : R + x - 1]) +
                                        (s - 1) % 2 * (unsigned)sizeof(mem[0]));
                else z = in[(row + R) * WS + x + R];
                return mk<T>(z.x, z.y);
            };
            C *const out = mem[s & 1];
            // the column from R above to R below (past the last row of a
            // short strip the rows read are the grid's next, or its border)
            C w[V + 2 * R];
#pragma unroll
            for (int d = 0; d < V + 2 * R; ++d) {
                const bool own = KEEP && d >= R && d < V + R;
                if (own) w[d] = d - R < rows ? y[KEEP ? d - R : 0] : rd(d - R, 0);
                else if (KEEP || d < 2 * R) w[d] = rd(d - R, 0);
            }
#pragma unroll
            for (int v = 0; v < V; ++v) {
                // double precision: a point's reads do not wait in registers
                // for the points before it
                if (!KEEP) {
                    __builtin_amdgcn_sched_barrier(0);
                    w[v + 2 * R] = rd(v + R, 0);
                }
                T sr, sm;
#pragma unroll
                for (int d = 1; d <= R; ++d) {
                    const C l = rd(v, -d), q = rd(v, d), up = w[R + v - d], dn = w[R + v + d];
                    if constexpr (KEEP) {
                        const C &y0 = w[R + v];
                        const float rt = d == 2 ? g.r2 : g.r3;
                        sr = d == 1 ? grid_ring1_from(g.r1, y0.x, l.x, q.x, up.x, dn.x)
                                    : grid_ring_from(sr, rt, y0.x, l.x, q.x, up.x, dn.x);
                        sm = d == 1 ? grid_ring1_from(g.r1, y0.y, l.y, q.y, up.y, dn.y)
                                    : grid_ring_from(sm, rt, y0.y, l.y, q.y, up.y, dn.y);
                    } else if (d == 1) {
                        sr = grid_ring1<R>(g, l.x, q.x, up.x, dn.x);
                        sm = grid_ring1<R>(g, l.y, q.y, up.y, dn.y);
                    } else {
                        sr = grid_ring(sr, d == 2 ? g.r2 : g.r3, l.x, q.x, up.x, dn.x);
                        sm = grid_ring(sm, d == 2 ? g.r2 : g.r3, l.y, q.y, up.y, dn.y);
                    }
                }
                C k;
                T kn;
                grid_rhs<T, DYN, KEEP>(g, c, cp[v], w[R + v], yn[v], mk<T>(sr, sm), k, kn);
                C z;
                if (s < 4) {
                    grid_acc(acc[v].x, k.x, s == 1);
                    grid_acc(acc[v].y, k.y, s == 1);
                    if (DYN) grid_acc(accn[v], kn, s == 1);
                    z = mk<T>(grid_input(u[v].x, k.x, dtwa), grid_input(u[v].y, k.y, dtwa));
                    if (DYN) yn[v] = grid_input(un[v], kn, dta);
                } else {
                    if constexpr (KEEP) {
                        z = mk<T>(grid_new_from(u[v].x, acc[v].x, k.x, dtw6, dtw6lo),
                                  grid_new_from(u[v].y, acc[v].y, k.y, dtw6, dtw6lo));
                        if (DYN) un[v] = yn[v] = grid_new_from(un[v], accn[v], kn, g.dt6, dt6lo);
                    } else {
                        z = mk<T>(grid_new(u[v].x, acc[v].x, k.x, dtw6), grid_new(u[v].y, acc[v].y, k.y, dtw6));
                        if (DYN) un[v] = yn[v] = grid_new(un[v], accn[v], kn, g.dt6);
                    }
                    u[v] = z;
                }
                if (KEEP) y[KEEP ? v : 0] = z;
                if (v < rows) out[li + v * WS] = z;
            }
            copy_edges(out);
        }
        // a thread writes a buffer again only after the next barrier, which
        // every thread reaches after its reads of it
        __syncthreads();
    };
    for (int it = 0; it < steps; ++it) {
        stage(std::integral_constant<int, 1>{});
        stage(std::integral_constant<int, 2>{});
        stage(std::integral_constant<int, 3>{});
        stage(std::integral_constant<int, 4>{});
    }
#pragma unroll
    for (int v = 0; v < V; ++v)
        if (v < rows) {
            const int idx = (r0 + v) * n + col;
            psi[idx] = u[v];
            if (DYN) nres[idx] = un[v];
        }
}

// Points a thread of grids of up to n x n: as few as 1024 threads hold in single
// precision, in double 512 (256 registers; three and four points of 1024 threads
// would spill, and with 8 whatever the size 48^2 took 9.8 us a step instead of 6.0).
// A step's length is the points a thread times the waves of a SIMD, and small
// grids keep it short for each of many as for one: with V of the largest for more
// grids than CUs, 1000 grids of 16^2 FP32 took 12.3 us a step instead of 2.0.  Only
// zero-outside FP32 grids of more than 48 points do better so: two workgroups of V = 4
// share a CU's registers, those of 3 do not (300 of 52^2 8.2 -> 7.3, 300 of 48^2 6.7
// against 5.0).
template <typename T>
void launch_resident_2d(int order, int bc, bool dyn, int count, int n, const ResidentArgs<T> &r, hipStream_t s) {
    constexpr int VM = square_v(sizeof(T));
    auto strips = [&](int v) { return n * ((n + v - 1) / v); };
    int v = strips(1) <= 1024 ? 1 : strips(2) <= 1024 ? 2 : VM;
    if (sizeof(T) == 8 && v == VM) v = strips(5) <= 512 ? 5 : strips(6) <= 512 ? 6 : VM;
    if (sizeof(T) == 4 && v == VM && strips(3) <= 1024) v = 3;
    if (sizeof(T) == 4 && bc == NLS_BC_REF && n > 48 && count > device_cus()) v = VM;
    const int nt = v == VM ? 64 * 64 / VM : (strips(v) + 63) / 64 * 64;
    // Grids of a hybrid batch on up to half the CUs keep them to themselves, by unused
    // LDS: a tile of the other members on the same CU steps at half the rate, and the
    // batch's step waits for it (20 of 64^2 beside 20 of 128^2 FP32 zero-outside 9.9
    // us a step sharing, 6.7 apart; 256 of 64^2, on every CU, 10.3 and 12.1)
    constexpr int ALONE = 120 * 1024;    // leaves less than the smallest tile takes
    const int row = 64 + order - 1, own = 2 * row * row * (int)sizeof(cplx_t<T>);
    const int pad = 2 * count <= device_cus() && own < ALONE ? ALONE - own : 0;
#define NLS_V(O, B, D, V) \
    if (v == V) hipLaunchKernelGGL((k_resident_2d<T, O, B, D, V>), dim3(count), dim3(nt), pad, s, r);
#define NLS_CASE(O, B, D)                                  \
    if (order == O && bc == B && dyn == D) {               \
        NLS_V(O, B, D, 1) NLS_V(O, B, D, 2)                \
        NLS_V(O, B, D, VM)                                 \
        if constexpr (sizeof(T) == 4) { NLS_V(O, B, D, 3) } \
        else { NLS_V(O, B, D, 5) NLS_V(O, B, D, 6) }       \
        return;                                            \
    }
    NLS_CASE(3, 0, false) NLS_CASE(3, 0, true) NLS_CASE(3, 1, false) NLS_CASE(3, 1, true)
    NLS_CASE(5, 0, false) NLS_CASE(5, 0, true) NLS_CASE(5, 1, false) NLS_CASE(5, 1, true)
    if constexpr (sizeof(T) == 4) {
        NLS_CASE(7, 0, false) NLS_CASE(7, 0, true) NLS_CASE(7, 1, false) NLS_CASE(7, 1, true)
    }
#undef NLS_CASE
#undef NLS_V
}
template void launch_resident_2d<float>(int, int, bool, int, int, const ResidentArgs<float> &, hipStream_t);
template void launch_resident_2d<double>(int, int, bool, int, int, const ResidentArgs<double> &, hipStream_t);

}  // namespace nls
