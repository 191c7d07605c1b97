// nls_march.hip -- one RK4 step of large 2-D grids and batches (order 5,
// periodic), by workgroups that march down the rows.
//
// A workgroup takes a strip of 256 columns, a thread each, and steps down a
// piece of its rows: as row r comes in, stage s computes row r - 2 s, so all
// four stages advance together.  A thread keeps what its column needs in
// registers -- nine rows of the state, five of each stage input, the
// accumulators, pumping and reservoir on their way down, rings that unrolling
// ten rows indexes statically -- and takes only the four horizontal
// neighbours of each stage's row from LDS, where that row was written two
// rows before, so one barrier serves two rows and no wait is on the way from
// a stage to the next.  The tile kernels (nls_batch.hip) compute 1.31 stage
// points for each of the tile's, wait at a barrier every stage and load,
// compute and store one after another; here the halo's stages cost 6 rows a
// piece and 16 columns a strip (none where a strip is a whole row of up to
// 256 points), and loads and stores run along with the arithmetic.
//
// Bound: on a 2048^2 grid in single precision VALU issue (134 vector instructions
// a row and wave, 77% of a launch's issue slots, where the strips and pieces add
// 1.31 of redundancy) and traffic together, in double precision the traffic behind
// the L2s (284 MiB for 224 of fields, 6.3 TB/s); for batches beyond the 256 MB cache
// HBM (131 grids of 128^2 and 109 of 256^2, 300 MB a step, at 5.1 TB/s).  Per step,
// against the tile kernels on the same box: 2048^2 FP32 31.8 -> 25.1 us, FP64 58.8 ->
// 45.6; 4096^2 162 -> 115 and 286 -> 213; those 240 grids FP32 88 -> 67.
// Measured and left: deeper prefetch (three rows, ten rows at the start) and
// stages guarded at run time instead of an unrolled start (10% slower).
#include <algorithm>
#include <type_traits>

#include "nls_march.h"
#include "nls_internal.h"

namespace nls {

constexpr int MARCH_NT = 256;            // columns a workgroup steps, a thread each
constexpr int MARCH_R = 2;               // stencil radius
constexpr int MARCH_H = 4 * MARCH_R;     // halo columns and rows of one step
constexpr int MARCH_WS = 272;            // columns of an LDS row: up to four pieces with 2R pads

template <typename T> __device__ __forceinline__ cplx_t<T> load_c(__amdgpu_buffer_rsrc_t r, unsigned off);
template <> __device__ __forceinline__ float2 load_c<float>(__amdgpu_buffer_rsrc_t r, unsigned off) {
    return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0));
}
template <> __device__ __forceinline__ double2 load_c<double>(__amdgpu_buffer_rsrc_t r, unsigned off) {
    return __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0));
}
template <typename T> __device__ __forceinline__ T load_r(__amdgpu_buffer_rsrc_t r, unsigned off);
template <> __device__ __forceinline__ float load_r<float>(__amdgpu_buffer_rsrc_t r, unsigned off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0));
}
template <> __device__ __forceinline__ double load_r<double>(__amdgpu_buffer_rsrc_t r, unsigned off) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0));
}

// Stores at a byte offset; those at or past the buffer's end are dropped.
__device__ __forceinline__ void put(__amdgpu_buffer_rsrc_t r, unsigned off, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, (int)off, 0, 0);
}
typedef unsigned U2 __attribute__((ext_vector_type(2)));
typedef unsigned U4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void put(__amdgpu_buffer_rsrc_t r, unsigned off, double v) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, v), r, (int)off, 0, 0);
}
__device__ __forceinline__ void put(__amdgpu_buffer_rsrc_t r, unsigned off, float2 v) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, v), r, (int)off, 0, 0);
}
__device__ __forceinline__ void put(__amdgpu_buffer_rsrc_t r, unsigned off, double2 v) {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(U4, v), r, (int)off, 0, 0);
}

// One piece of a member.
template <typename T, bool DYN, bool FULL>
__device__ __forceinline__ void march_piece(const MarchArgs<T> &f, const StripDesc &sd, const MemberDev<T> &m, char *lds) {
    using C = cplx_t<T>;
    constexpr int R = MARCH_R, H = MARCH_H, U = 10;
    constexpr bool AHEAD = sizeof(T) == 4;
    constexpr int SS = MARCH_WS * (int)sizeof(C), SL = 4 * SS;   // bytes of an LDS row, of a slot of four
    const int n = m.n, N = n * n;
    const int tid = threadIdx.x;
    const int cw = FULL ? n : MARCH_NT;  // columns of a piece
    const int sub = FULL ? tid / cw : 0, col = tid - sub * cw;
    const bool active = sub < sd.subs;
    int gx = FULL ? col : sd.x0 - H + col;
    gx += gx < 0 ? n : 0;
    gx -= gx >= n ? n : 0;
    const int ys = sd.y0 + (active ? sub : 0) * sd.E;    // first row this thread writes
    const int rows = min(sd.L, n - ys);                  // rows it writes (none if <= 0)
    const bool store = active && (FULL || (col >= H && col < H + sd.wd && gx >= sd.x0));
    const long long off = m.off;
    const C *u = f.u + off;
    const T *un = DYN ? f.un + off : nullptr, *P = f.P + off;
    C *uo = f.uo + off;
    T *uno = DYN ? f.uno + off : nullptr;

    if (f.it >= m.steps) {               // budget used up: pass the state through
        for (int y = 0; store && y < rows; ++y) {
            const size_t gi = (size_t)(ys + y) * n + gx;
            uo[gi] = u[gi];
            if (DYN) uno[gi] = un[gi];
        }
        return;
    }

    const unsigned cbytes = (unsigned)((unsigned long long)N * sizeof(C));
    auto rsrc = [](const void *p, unsigned bytes) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes, 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t ru = rsrc(u, cbytes), rp = rsrc(P, cbytes / 2), rn = rsrc(DYN ? un : P, cbytes / 2),
                                 wu = rsrc(uo, cbytes), wn = rsrc(DYN ? uno : nullptr, DYN ? cbytes / 2 : 0);

    const T dt = m.dt, dt2 = dt * (T)0.5, dt6 = m.g.dt6;
    const T dtw = m.g.dtw, dtw2 = dtw * (T)0.5, dtw6 = m.g.dtw6;
    Coeffs<T> c = m.c;
    GridCoeffs<T> g = m.g;
    if constexpr (sizeof(T) == 4) asm volatile("" : "+v"(g.c4), "+v"(g.wc), "+v"(c.d13), "+v"(c.c13));

    // LDS byte address of the column's leftmost neighbour; A: slots 0, 1, B: 2, 3
    unsigned A = (unsigned)(size_t)(__attribute__((address_space(3))) char *)lds + (tid + 2 * R * sub) * sizeof(C);
    unsigned B = A + 2 * SL;
    // whole rows: the first and last R columns are copied past the other end
    const int wrap = !FULL || !active ? 0 : col < R ? cw : col >= cw - R ? -cw : 0;

    // row rings, indexed by row modulo their length
    C w1[U], w2[5], w3[5], w4[5], a1[2], a2[2], a3[2];
    T cp[U], nn[U], n3[2], n4[2], b1[2], b2[2], b3[2];
    // state rows on their way, loaded D rows ahead (pumping and reservoir are
    // first used two rows after the state)
    constexpr int D = AHEAD ? 2 : 1;
    C in[5];

    // byte offset of the newest row (of the complex arrays)
    const unsigned pitch = (unsigned)n * sizeof(C);
    int r0 = ys - H;
    r0 += r0 < 0 ? n : 0;
    r0 -= r0 >= n ? n : 0;
    unsigned lp = ((unsigned)r0 * n + gx) * sizeof(C);
    // byte offset of the row being written; rows past the grid's end, and
    // lanes that write nothing, lie past the buffer (such stores are dropped)
    unsigned so = store && ys < n ? ((unsigned)ys * n + gx) * sizeof(C) : cbytes;

    // the next state row, and the next row's fields into ring place k; each
    // offset then wraps past the last row
    unsigned lf = lp;
    auto load = [&](C &to) {
        to = load_c<T>(ru, lp);
        lp += pitch;
        lp = min(lp, lp - cbytes);
    };
    auto load_field = [&](int k) {
        cp[k] = load_r<T>(rp, lf >> 1);
        if (DYN) nn[k] = load_r<T>(rn, lf >> 1);
        lf += pitch;
        lf = min(lf, lf - cbytes);
    };
    typedef T V2 __attribute__((ext_vector_type(2)));
    using LV = __attribute__((address_space(3))) V2;
    // LDS row s (stage input s + 1) of the slot of iteration k
    auto at = [&](int k, int s, int x) {
        return (LV *)(size_t)((k & 2) ? B : A) + ((k & 1) * SL + s * SS) / (int)sizeof(C) + x;
    };

    // The four neighbours in a row of stage input s + 1 that LDS holds, of the
    // slot written two iterations before iteration k
    struct Row4 { C l2, l1, q1, q2; };
    auto beside = [&](int k, int s) {
        auto rd = [&](int x) { const V2 v = *at(k + 2, s, R + x); return mk<T>(v.x, v.y); };
        return Row4{rd(-2), rd(-1), rd(1), rd(2)};
    };
    // Slopes at a point from the five rows of its column and those.
    auto slopes = [&](const Row4 &h, const C &ym2, const C &ym1, const C &y, const C &yp1, const C &yp2, T cP, T yn,
                      C &kk, T &kn) {
        T sr = grid_ring1<R>(g, h.l1.x, h.q1.x, ym1.x, yp1.x), sm = grid_ring1<R>(g, h.l1.y, h.q1.y, ym1.y, yp1.y);
        sr = grid_ring(sr, g.r2, h.l2.x, h.q2.x, ym2.x, yp2.x);
        sm = grid_ring(sm, g.r2, h.l2.y, h.q2.y, ym2.y, yp2.y);
        grid_rhs<T, DYN>(g, c, cP, y, yn, mk<T>(sr, sm), kk, kn);
    };

    // Iteration k of a block of U rows; stages 1 .. S run (fewer while the
    // column's first rows come in).  Each stage's LDS reads are issued before
    // the arithmetic of the stage before it.
    auto row = [&](auto k_, auto S_) {
        constexpr int k = decltype(k_)::value, S = decltype(S_)::value;
        auto u1 = [&](int d) -> C & { return w1[(k + U - d) % U]; };      // row d above the newest
        auto m5 = [&](C(&w)[5], int d) -> C & { return w[(k + U - d) % 5]; };
        constexpr int now = k & 1;                                          // rings of two
        auto fence = [] { __builtin_amdgcn_sched_barrier(0); };
        C kk;
        T kn;
        Row4 h1, h2;
        if constexpr (S >= 1) h1 = beside(k, 0);
        u1(0) = in[k % 5];
        load(in[(k + D) % 5]);
        if (AHEAD) load_field(k);
        if constexpr (S >= 1) {          // centre: 2 rows above the newest
            if constexpr (AHEAD && S >= 2) h2 = beside(k, 1);
            fence();
            const T yn = nn[(k + U - 2) % U];
            // the row's pumping becomes its pump term at its first use, two
            // rows after its load
            T &cP = cp[(k + U - 2) % U];
            cP = pump_term<T, DYN>(c, cP);
            slopes(h1, u1(4), u1(3), u1(2), u1(1), u1(0), cP, yn, kk, kn);
            m5(w2, 2) = mk<T>(grid_input(u1(2).x, kk.x, dtw2), grid_input(u1(2).y, kk.y, dtw2));
            C acc = a1[now];
            T bcc = b1[now], old = DYN ? grid_input(nn[(k + U - 4) % U], bcc, dt2) : (T)0;
            a1[now] = kk;
            if (DYN) b1[now] = kn;
            if constexpr (S >= 2) {      // 4 rows above
                fence();
                if constexpr (!AHEAD) h2 = beside(k, 1);
                else if constexpr (S >= 3) h1 = beside(k, 2);
                if (AHEAD) fence();
                slopes(h2, m5(w2, 6), m5(w2, 5), m5(w2, 4), m5(w2, 3), m5(w2, 2), cp[(k + U - 4) % U], old, kk, kn);
                grid_acc(acc.x, kk.x, false);
                grid_acc(acc.y, kk.y, false);
                if (DYN) grid_acc(bcc, kn, false);
                m5(w3, 4) = mk<T>(grid_input(u1(4).x, kk.x, dtw2), grid_input(u1(4).y, kk.y, dtw2));
                C acc3 = a2[now];
                T bcc3 = b2[now];
                old = n3[now];
                a2[now] = acc;
                if (DYN) { b2[now] = bcc; n3[now] = grid_input(nn[(k + U - 4) % U], kn, dt2); }
                if constexpr (S >= 3) {  // 6 rows above
                    fence();
                    if constexpr (!AHEAD) h1 = beside(k, 2);
                    else if constexpr (S >= 4) h2 = beside(k, 3);
                    if (AHEAD) fence();
                    slopes(h1, m5(w3, 8), m5(w3, 7), m5(w3, 6), m5(w3, 5), m5(w3, 4), cp[(k + U - 6) % U], old, kk, kn);
                    grid_acc(acc3.x, kk.x, false);
                    grid_acc(acc3.y, kk.y, false);
                    if (DYN) grid_acc(bcc3, kn, false);
                    m5(w4, 6) = mk<T>(grid_input(u1(6).x, kk.x, dtw), grid_input(u1(6).y, kk.y, dtw));
                    acc = a3[now];
                    bcc = b3[now];
                    old = n4[now];
                    a3[now] = acc3;
                    if (DYN) { b3[now] = bcc3; n4[now] = grid_input(nn[(k + U - 6) % U], kn, dt); }
                    if constexpr (S >= 4) {   // 8 rows above: the new state
                        fence();
                        if constexpr (!AHEAD) h2 = beside(k, 3);
                        slopes(h2, m5(w4, 10), m5(w4, 9), m5(w4, 8), m5(w4, 7), m5(w4, 6), cp[(k + U - 8) % U], old, kk,
                               kn);
                        put(wu, so, mk<T>(grid_new(u1(8).x, acc.x, kk.x, dtw6), grid_new(u1(8).y, acc.y, kk.y, dtw6)));
                        if (DYN) put(wn, so >> 1, grid_new(nn[(k + U - 8) % U], bcc, kn, dt6));
                        so += pitch;
                    }
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        // this iteration's rows of the stage inputs, for the neighbours two
        // iterations on
        auto share = [&](int x) {
            *at(k, 0, R + x) = V2{u1(0).x, u1(0).y};
            if constexpr (S >= 1) *at(k, 1, R + x) = V2{m5(w2, 2).x, m5(w2, 2).y};
            if constexpr (S >= 2) *at(k, 2, R + x) = V2{m5(w3, 4).x, m5(w3, 4).y};
            if constexpr (S >= 3) *at(k, 3, R + x) = V2{m5(w4, 6).x, m5(w4, 6).y};
        };
        share(0);
        // (double precision: a branch here would spill; the other lanes
        // write their own place again)
        if (FULL && (!AHEAD || wrap)) share(wrap);
        if (!AHEAD) load_field(k);
        if constexpr (k & 1) __syncthreads();
    };
#define NLS_I(v) std::integral_constant<int, v>{}
    auto swap = [&] { const unsigned x = A; A = B; B = x; };
#pragma unroll
    for (int k = 0; k < D; ++k) load(in[k]);
    // the first 16 rows: stage s starts 4 s rows in
    row(NLS_I(0), NLS_I(0)); row(NLS_I(1), NLS_I(0));
    row(NLS_I(2), NLS_I(0)); row(NLS_I(3), NLS_I(0));
    row(NLS_I(4), NLS_I(1)); row(NLS_I(5), NLS_I(1));
    row(NLS_I(6), NLS_I(1)); row(NLS_I(7), NLS_I(1));
    row(NLS_I(8), NLS_I(2)); row(NLS_I(9), NLS_I(2));
    swap();                              // ten rows on, slots k & 3 are two places on
    row(NLS_I(0), NLS_I(2)); row(NLS_I(1), NLS_I(2));
    row(NLS_I(2), NLS_I(3)); row(NLS_I(3), NLS_I(3));
    row(NLS_I(4), NLS_I(3)); row(NLS_I(5), NLS_I(3));
    int o = 0;                           // rows written
    const int L = sd.L;
    for (;;) {
        row(NLS_I(6), NLS_I(4)); row(NLS_I(7), NLS_I(4)); o += 2; if (o >= L) break;
        row(NLS_I(8), NLS_I(4)); row(NLS_I(9), NLS_I(4)); o += 2;
        swap();
        if (o >= L) break;
        row(NLS_I(0), NLS_I(4)); row(NLS_I(1), NLS_I(4)); o += 2; if (o >= L) break;
        row(NLS_I(2), NLS_I(4)); row(NLS_I(3), NLS_I(4)); o += 2; if (o >= L) break;
        row(NLS_I(4), NLS_I(4)); row(NLS_I(5), NLS_I(4)); o += 2; if (o >= L) break;
    }
#undef NLS_I
}

// Workgroup t of a launch steps pieces first[t] .. first[t + 1] - 1, or the
// t-th piece of one grid, pieces across first.
template <typename T, bool DYN, bool FULL>
__global__ void __launch_bounds__(MARCH_NT, sizeof(T) == 4 ? 3 : 2) k_march(const MarchArgs<T> f, const MemberDev<T> *__restrict__ mem, const StripDesc *__restrict__ strips,
        const int *__restrict__ first) {
    __shared__ __align__(16) char lds[16 * MARCH_WS * sizeof(cplx_t<T>)];
    // workgroups are dispatched to the 8 XCDs round-robin; each XCD takes a
    // contiguous range, so that neighbouring pieces share its L2
    const int b = blockIdx.x, t = (b & 7) * f.chunk + (b >> 3);
    if (t >= f.groups) return;
    if (!FULL && f.grid_nx > 0) {        // (one grid this small stays on tiles)
        const int n = f.grid.n, row = t / f.grid_nx, col = t - row * f.grid_nx, y = row * f.grid_L;
        const StripDesc sd = {0, col * f.grid_wd, f.grid_wd, y, min(f.grid_L, n - y), n, 1};
        march_piece<T, DYN, FULL>(f, sd, f.grid, lds);
    } else {
        for (int i = first[t]; i < first[t + 1]; ++i) {
            const StripDesc sd = strips[i];
            march_piece<T, DYN, FULL>(f, sd, mem[sd.m], lds);
            __syncthreads();
        }
    }
}

// percu workgroups a CU share the launch: the dispatcher may fill a CU with
// as many as it holds before another has one, so unused LDS keeps each CU to
// its share.
template <typename T, bool DYN> static void launch(bool full, int percu, const MarchArgs<T> &a, hipStream_t s) {
    constexpr int CU_LDS = 160 * 1024, OWN = 16 * MARCH_WS * (int)sizeof(cplx_t<T>);
    const dim3 grid(8 * a.chunk);
    const int pad = percu < CU_LDS / OWN ? std::max(0, CU_LDS / (percu + 1) + 1024 - OWN) : 0;
    if (full) hipLaunchKernelGGL((k_march<T, DYN, true>), grid, dim3(MARCH_NT), pad, s, a, a.mem, a.strips, a.first);
    else hipLaunchKernelGGL((k_march<T, DYN, false>), grid, dim3(MARCH_NT), pad, s, a, a.mem, a.strips, a.first);
}
template <typename T> void launch_march(bool dyn, bool full, int percu, const MarchArgs<T> &a, hipStream_t s) {
    if (dyn) launch<T, true>(full, percu, a, s);
    else launch<T, false>(full, percu, a, s);
}
template void launch_march<float>(bool, bool, int, const MarchArgs<float> &, hipStream_t);
template void launch_march<double>(bool, bool, int, const MarchArgs<double> &, hipStream_t);

}  // namespace nls
