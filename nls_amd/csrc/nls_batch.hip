// nls_batch.hip -- batched solves: many independent instances (members) of
// mixed sizes packed into shared device arrays and advanced together, one
// launch covering the tiles of every member.
//
// Members share dim, order, boundary family, reservoir mode and dtype; each
// has its own n, dt, dx, coefficients and step budget.  A member whose
// budget is used up passes its state through unchanged, so a batch can hold
// solves of different lengths (the serving loop relies on this).
//
// Engines:
//   NLS_ENGINE_STAGE    one launch per RK4 stage (bodies in nls_stage.h), 15 S
//                       + 4 r bytes per point and step; any dim/boundary/order.
//   NLS_ENGINE_FUSED    one launch per RK4 step, 2-D only.  A workgroup loads
//                       its output tile plus a halo of 4R points (R = stencil
//                       radius) into registers and LDS once, runs the four
//                       stages on the shrinking region on chip, and writes the
//                       new state of the tile: 2 S + r bytes per point and
//                       step from HBM plus the halo re-reads, at the price of
//                       recomputing the halo's stages.
//   NLS_ENGINE_RESIDENT a workgroup per member holds the member on chip and
//                       runs every step of a call (1-D n <= 4096, 2-D n <= 64).
//   NLS_ENGINE_HYBRID   the members that fit the resident engine on it, on a
//                       stream of the batch, beside the others on the fused
//                       (2-D) or per-stage (1-D) engine.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <type_traits>
#include <cstring>
#include <vector>

#include "nls_amd.h"
#include "nls_internal.h"
#include "nls_march.h"
#include "nls_rk4.h"

namespace nls {

constexpr int BATCH_STAGE_TY = 16;    // tile height of the STAGE engine's 2-D tiles

template <typename T> struct BatchArgs {
    const MemberDev<T> *mem;
    const TileDesc *tiles;
    int ntiles, chunk;      // XCD-aware mapping: blocks of one XCD take a contiguous tile range
    int it;                 // step index within this advance call
    int stage;
    T scale;
    const T *wtab;
    const cplx_t<T> *u; const T *un;
    const cplx_t<T> *kin; const T *kin_n;
    cplx_t<T> *kout; T *kout_n;
    cplx_t<T> *acc; T *acc_n;
    const T *P;
};

// Workgroups are dispatched to the 8 XCDs round-robin; give each XCD a
// contiguous range of tiles so neighbouring tiles share its L2.
__device__ __forceinline__ int xcd_tile(int ntiles, int chunk) {
    const int b = blockIdx.x;
    const int t = (b & 7) * chunk + (b >> 3);
    return t < ntiles ? t : -1;
}

template <typename T>
__device__ __forceinline__ StageArgs<T> member_view(const BatchArgs<T> &b, const MemberDev<T> &m) {
    StageArgs<T> a;
    a.n = m.n; a.stage = b.stage; a.dt = m.dt; a.scale = b.scale; a.c = m.c;
    a.w0 = m.w0; a.w1 = m.w1; a.w2 = m.w2; a.w3 = m.w3;
    a.wtab = m.tab >= 0 ? b.wtab + m.tab : nullptr;
    const long long o = m.off;
    a.u = b.u + o; a.un = b.un ? b.un + o : nullptr;
    a.kin = b.kin ? b.kin + o : nullptr; a.kin_n = b.kin_n ? b.kin_n + o : nullptr;
    a.kout = b.kout ? b.kout + o : nullptr; a.kout_n = b.kout_n ? b.kout_n + o : nullptr;
    a.acc = b.acc + o; a.acc_n = b.acc_n ? b.acc_n + o : nullptr;
    a.P = b.P + o;
    return a;
}

// ---------------------------------------------------------------------------
// Engine STAGE
// ---------------------------------------------------------------------------

template <typename T, int ORDER, int BC, bool DYN, int DIM>
__global__ void __launch_bounds__(256) k_batch_stage(const BatchArgs<T> b) {
    constexpr int R = (ORDER - 1) / 2;
    constexpr int LDS = DIM == 2 ? (BATCH_STAGE_TY + 2 * R) * (TILE2_X + 2 * R) : TILE1 + 2 * R;
    __shared__ cplx_t<T> tile[LDS];
    const int t = xcd_tile(b.ntiles, b.chunk);
    if (t < 0) return;
    const TileDesc td = b.tiles[t];
    const MemberDev<T> m = b.mem[td.m];
    const StageArgs<T> a = member_view(b, m);
    if (b.it >= m.steps) {
        // budget used up: carry the state into the buffer that becomes u
        if (b.stage == 4) {
            const int n = m.n;
            if (DIM == 2) {
                const int gx = td.x0 + (threadIdx.x & 63);
                for (int j = 0; j < BATCH_STAGE_TY / 4 && gx < n; ++j) {
                    const int gy = td.y0 + (threadIdx.x >> 6) + 4 * j;
                    if (gy >= n) break;
                    const size_t gi = (size_t)gy * n + gx;
                    a.acc[gi] = a.u[gi];
                    if (DYN) a.acc_n[gi] = a.un[gi];
                }
            } else {
                const int gx = td.x0 + threadIdx.x;
                if (gx < n) { a.acc[gx] = a.u[gx]; if (DYN) a.acc_n[gx] = a.un[gx]; }
            }
        }
        return;
    }
    if (DIM == 2) stage_tile_2d<T, ORDER, BC, DYN, BATCH_STAGE_TY>(a, td.x0, td.y0, tile);
    else stage_tile_1d<T, ORDER, BC, DYN>(a, td.x0, tile);
}

// ---------------------------------------------------------------------------
// Engine FUSED (2-D): one RK4 step per launch, halo recomputation.
// Output tile 64 x TY, halo H = 4R, region W x HH = (64 + 2H) x (TY + 2H).
// Stage s (1..4) computes the rectangle of points with at least sR halo rings
// around them.  The region's points are listed in ring order (RingMap): the
// output tile row-major, then the ring only stages 1..3 compute, then stage
// 1..2's ring, stage 1's ring and the outermost ring that is only loaded.
// Every stage's rectangle is then a prefix of the list; with 256 threads
// owning list entries t + 256 j, a stage's active lanes fill whole
// wavefronts but for one, and inactive wavefronts skip the stage entirely.
// Per owned point the state u, reservoir, pumping (as its pump_term), the
// reservoir's stage input and the RK4 accumulators stay in registers; the
// psi stage input sits in LDS so the stencil can read the neighbours.
// ---------------------------------------------------------------------------

// Buffer loads at a 32-bit byte offset from a buffer resource (base address,
// size in bytes); offsets at or past the size read zero.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void *base, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes, 0x00020000);
}
template <typename T> __device__ __forceinline__ cplx_t<T> buffer_load_c(__amdgpu_buffer_rsrc_t r, unsigned off);
template <> __device__ __forceinline__ float2 buffer_load_c<float>(__amdgpu_buffer_rsrc_t r, unsigned off) {
    return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0));
}
template <> __device__ __forceinline__ double2 buffer_load_c<double>(__amdgpu_buffer_rsrc_t r, unsigned off) {
    return __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0));
}
template <typename T> __device__ __forceinline__ T buffer_load_r(__amdgpu_buffer_rsrc_t r, unsigned off);
template <> __device__ __forceinline__ float buffer_load_r<float>(__amdgpu_buffer_rsrc_t r, unsigned off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0));
}
template <> __device__ __forceinline__ double buffer_load_r<double>(__amdgpu_buffer_rsrc_t r, unsigned off) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0));
}

// Grids (members, row slabs) the fused kernel holds.  In single precision it
// addresses a member's arrays with 32-bit byte offsets from buffer
// resources: complex arrays smaller than 4 GiB.  In double precision it takes
// 64-bit addresses from a 32-bit point index: fewer than 2^32 points.
bool fused_holds(long long points, int dtype) {
    return dtype == NLS_F64 ? points <= 0xffffffffLL : points * 8LL <= 0xffffffffLL;
}

template <typename T> struct FusedArgs {
    const MemberDev<T> *mem;
    const TileDesc *tiles;
    int ntiles, chunk;
    int it;
    const cplx_t<T> *u; const T *un;     // state at the start of the step
    cplx_t<T> *uo; T *uno;               // state at its end
    const T *P;
    // One grid instead of a member table: grid_ntx > 0 tiles per row of the
    // grid described by `grid`; tile t sits at (t % grid_ntx, t / grid_ntx).
    int grid_ntx;
    MemberDev<T> grid;
    // BC_SLAB: buffer rows 0..4R-1 and slab_end..slab_end+4R-1 are ghost
    // rows; rows 4R..slab_end-1 are the slab's own (the only ones written)
    int slab_end;
};

// Tile shape and launch shape of the fused kernel.  TY: output rows.  NT:
// threads per workgroup; each thread owns ceil(region / NT) points, so NT
// trades registers per thread against waves per SIMD (the kernel is bound by
// latency, and waves per SIMD hide it).  DB: the psi stage input is
// double-buffered in LDS (stage s reads one buffer and writes the next
// stage's input into the other: one barrier per stage and no registers
// holding the next input).  WAVES: waves per SIMD the register budget is
// sized for.
//
// FORM, chosen per launch by fused_form():
//  - FORM_TALL: 64 x 32 tiles of 1024 threads (order 7: 64 x 24 tiles of 768
//    threads), for launches of several rounds, where the tall tile's smaller
//    halo per output point pays, or whose tall tiles fit one per compute unit.
//    Single precision of order 5 runs the pair kernel, double precision of
//    order 5 and order 7 the group kernel, order 3 this one.
//  - FORM_SHORT: 64 x 16 tiles of 1024 threads, for launches with no more
//    such tiles than the device has compute units (a lone grid, a few small
//    members): the step is then one workgroup's critical path, which grows
//    with the region points per thread (2.5 instead of 3.75).
//  - FORM_HALF (double precision, periodic grids and row slabs): 64 x 16
//    tiles of 512 threads with a single stage buffer, 48 KB of LDS, so a CU
//    holds two workgroups (the 1024-thread 64 x 32 tile needs 137 KB and a
//    CU holds one) and one workgroup's loads overlap the other's arithmetic,
//    which outweighs the larger halo when the launch runs more than two
//    rounds.
//    With reflecting boundaries this form would spill registers.
//  - FORM_TALL512 (single precision, order 5, periodic: the pair kernel):
//    64 x 32 tiles of 512 threads, four pairs a thread.  A stage's pairs then
//    fill 87% of the lanes of its passes instead of 75% (the stages step
//    1672, 1440, 1224 and 1024 pairs), at half the waves per SIMD; chosen by
//    the autotuner (batches of all-fused 2-D members: 92.8 -> 90.8 us on
//    sweep512; a lone 2048^2 grid: 33.1 -> 35.2 us).
// (A 64 x 64 single-precision form, 1.20 region points per output point
// instead of 1.31 but 110 KB of LDS and so one workgroup per CU, measured
// 111 us against 81 us per step on the sweep512 batch: with one workgroup a
// CU idles at every stage barrier.)
enum { FORM_TALL = 0, FORM_SHORT = 1, FORM_HALF = 2, FORM_TALL512 = 3 };
template <typename T, int ORDER, int FORM> struct FusedTile;
template <int ORDER, int FORM> struct FusedTile<float, ORDER, FORM> {
    static_assert(FORM != FORM_HALF, "single precision has no half-size form");
    static constexpr int TY = FORM == FORM_SHORT ? 16 : 32;
    static constexpr int NT = FORM == FORM_TALL512 ? 512 : 1024;
    static constexpr bool DB = true;
    static constexpr int WAVES = FORM == FORM_TALL512 ? 4 : 8;
};
template <int ORDER, int FORM> struct FusedTile<double, ORDER, FORM> {
    static constexpr bool HALF = FORM == FORM_HALF;
    static constexpr int TY = FORM != FORM_TALL ? 16 : 32;
    static constexpr int NT = HALF ? 512 : 1024;
    static constexpr bool DB = !HALF;
    static constexpr int WAVES = 4;
};
// LDS row stride of the region (W + pad), chosen so that the lanes of the
// ring order's side bands (2R points per row over consecutive rows) fall in
// distinct banks.
constexpr int fused_lds_stride(int W, int R) { return W + (R == 1 ? 2 : R == 2 ? 4 : 14); }
static int fused_ty(int order, int form) {
    if (order == 7) return form == FORM_SHORT ? 16 : 24;
    return form != FORM_TALL && form != FORM_TALL512 ? 16 : 32;
}

// Region points in ring order, built at compile time: entry k holds the
// point's LDS index y WS + x in bits 0..15, x in bits 16..23, y in 24..31.
template <int W, int HH, int R, int WS> struct RingMap {
    unsigned v[W * HH];
    constexpr RingMap() : v() {
        int k = 0;
        for (int s = 4; s >= 0; --s) {           // rectangle s minus rectangle s + 1
            const int a = s * R, b = (s + 1) * R;
            for (int y = a; y < HH - a; ++y)
                for (int x = a; x < W - a; ++x) {
                    const bool inner = s < 4 && y >= b && y < HH - b && x >= b && x < W - b;
                    if (!inner) v[k++] = (unsigned)(y * WS + x) | (unsigned)x << 16 | (unsigned)y << 24;
                }
        }
    }
};
static_assert(RingMap<80, 48, 2, 84>().v[0] == (8 * 84 + 8 | 8 << 16 | 8 << 24), "ring order starts at the output tile");
static_assert(RingMap<80, 48, 2, 84>().v[2048] == (6 * 84 + 6 | 6 << 16 | 6 << 24), "stage-3 ring follows the 64 x 32 tile");
static_assert(RingMap<80, 32, 2, 84>().v[1024] == (6 * 84 + 6 | 6 << 16 | 6 << 24), "stage-3 ring follows the 64 x 16 tile");
template <int W, int HH, int R, int WS> __device__ const RingMap<W, HH, R, WS> ring_map{};

// A tile whose waves hold few columns of the grid: double-precision arithmetic of a
// wave with eight active lanes or fewer takes longer than of one with all (8 grids of
// order 3 zero-outside: 73^2 4.4 us a step, 72^2, whose last tile is eight columns
// wide, 5.4, as all lanes 5.0), so there every lane runs and the stores are masked.
template <typename T> __device__ __forceinline__ bool few_columns(int n, int x0) {
    return sizeof(T) == 8 && n - x0 <= 8;
}

// S32 (double precision only): the fields sit in HBM in single precision --
// state, reservoir and pumping are widened on load and the new state rounded
// once on store -- and everything else is the double-precision step: FP64
// stage arithmetic and LDS at FP32 storage bytes.  The FusedArgs pointers
// then hold the single-precision arrays.
template <typename T, int ORDER, int BC, bool DYN, int FORM, bool S32 = false>
__global__ void __launch_bounds__((FusedTile<T, ORDER, FORM>::NT), (FusedTile<T, ORDER, FORM>::WAVES))
k_fused_step_2d(const FusedArgs<T> f) {
    static_assert(!S32 || sizeof(T) == 8, "single-precision storage under double-precision arithmetic");
    using C = cplx_t<T>;
    using FT = FusedTile<T, ORDER, FORM>;
    constexpr int R = (ORDER - 1) / 2, H = 4 * R;
    constexpr int TX = 64, TY = FT::TY, NT = FT::NT;
    constexpr bool DB = FT::DB;
    constexpr int W = TX + 2 * H, HH = TY + 2 * H, NP = W * HH;
    constexpr int WS = fused_lds_stride(W, R);
    constexpr int J = (NP + NT - 1) / NT;
    constexpr int JOUT = TX * TY / NT;    // list entries t + NT j, j < JOUT, are the output tile
    static_assert(TX * TY % NT == 0 && W < 256 && HH < 256, "fused tile shape");
    static_assert(DB || BC != BC_REF, "points outside the grid are written once per buffer");
    // psi stage input, point (x, y) of the region at ys_mem[b][PAD + y WS + x]:
    // the front pad makes every stencil read a non-negative constant offset
    // from the point's own index, so each read is one LDS instruction with an
    // immediate offset from a single per-point base register
    constexpr int PAD = R * WS + R;
    __shared__ C ys_mem[DB ? 2 : 1][HH * WS + 2 * PAD];
    C *const ya = ys_mem[0] + PAD;            // input of stages 1 and 3 (and 2, 4 unless DB)
    C *const yb = ys_mem[DB ? 1 : 0] + PAD;   // input of stages 2 and 4

    const int t = xcd_tile(f.ntiles, f.chunk);
    if (t < 0) return;
    TileDesc td;
    MemberDev<T> m;
    if (f.grid_ntx > 0) {
        td.m = 0; td.x0 = (t % f.grid_ntx) * TX; td.y0 = (t / f.grid_ntx) * TY + (BC == BC_SLAB ? H : 0);
        m = f.grid;
    } else {
        td = f.tiles[t];
        m = f.mem[td.m];
    }
    const int n = m.n;
    const int ylim = BC == BC_SLAB ? f.slab_end : n;   // output rows end here
    const long long off = m.off;
    using SC = std::conditional_t<S32, float2, C>;      // storage types
    using SR = std::conditional_t<S32, float, T>;
    const SC *u = (const SC *)f.u + off;
    const SR *un = DYN ? (const SR *)f.un + off : nullptr;
    const SR *P = (const SR *)f.P + off;
    SC *uo = (SC *)f.uo + off;
    SR *uno = DYN ? (SR *)f.uno + off : nullptr;
    const int tid = threadIdx.x;
    // single precision: the region loads take 32-bit byte offsets from
    // buffer resources over the member's arrays (fused_holds: under 4 GiB)
    const unsigned cbytes = (unsigned)((unsigned long long)(BC == BC_SLAB ? f.slab_end + H : n) * n * sizeof(C));
    const __amdgpu_buffer_rsrc_t ru = buffer_of(u, cbytes), rp = buffer_of(P, cbytes / 2),
                                 rn = buffer_of(DYN ? un : P, cbytes / 2);

    if (f.it >= m.steps) {            // budget used up: pass the state through
#pragma unroll
        for (int j = 0; j < JOUT; ++j) {
            const int k = tid + NT * j;
            const int gx = td.x0 + (k & (TX - 1)), gy = td.y0 + k / TX;
            if (gx >= n || gy >= ylim) continue;
            const size_t gi = (size_t)gy * n + gx;
            uo[gi] = u[gi];
            if (DYN) uno[gi] = un[gi];
        }
        return;
    }

    // single precision, zero-outside: to skip the points outside costs each of the
    // others a test and a branch (25 grids of 296^2 order 5 with a reservoir 23.8 us a
    // step with all lanes, 25.4 skipping; 257^2 22.9 and 23.6; order 3 16.8 and 17.3)
    const bool few = (sizeof(T) == 4 && BC == BC_REF) || few_columns<T>(n, td.x0);
    const T dt = m.dt, dt2 = dt * (T)0.5, dt6 = m.g.dt6;                   // of the reservoir
    const T dtw = m.g.dtw, dtw2 = dtw * (T)0.5, dtw6 = m.g.dtw6;           // of psi
    Coeffs<T> c = m.c;
    GridCoeffs<T> g = m.g;
    if constexpr (sizeof(T) == 4) {
        // coefficients that meet another coefficient in one fused
        // multiply-add of the right-hand side (c3 r - c4, c6 r - wc,
        // d13 + d14 s, c13 + c14 s): a VALU instruction reads one scalar
        // register, so held in scalar registers each would be copied to a
        // vector register per point and stage; kept in vector registers for
        // the whole kernel
        asm volatile("" : "+v"(g.c4), "+v"(g.wc), "+v"(c.d13), "+v"(c.c13));
    }
    const unsigned *map = ring_map<W, HH, R, WS>.v;

    C uu[J], acc[J], ynext[DB ? 1 : J];
    T cp[J], nn[J], yn[J], accn[J];
    int li[J];                         // LDS index of the point
    unsigned inside = 0;               // BC_REF, bit j: point j lies on the grid
    static_assert(J <= 32, "inside mask");

    const bool near = n >= TX + H;     // region offsets stay within one period of the grid

    // load the state, reservoir and pumping of the whole region once.  In
    // single precision the ring-order table entries of all this thread's
    // points are loaded first, then the fields of all its points, then the
    // LDS stores follow, so that each group of loads is in flight together
    // and waited for once (point by point, each thread waits out the memory
    // latency once per point: 2.5% slower).  In double precision the 512-thread
    // form, two workgroups per CU, groups its loads too (4% at 2048^2); with
    // one 1024-thread workgroup per CU point by point is 7% faster and is kept.
    constexpr bool GROUPED = sizeof(T) == 4 || FORM == FORM_HALF;
    unsigned ent[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int k = tid + NT * j;
        // the first TX*TY list entries are the output tile, row-major: their
        // coordinates need no table entry
        ent[j] = (GROUPED && j >= JOUT && (NP % NT == 0 || j < J - 1 || k < NP)) ? map[k] : 0u;
    }
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int k = tid + NT * j;
        uu[j] = mk<T>(0, 0); cp[j] = 0; nn[j] = 0;
        acc[j] = mk<T>(0, 0); accn[j] = 0;
        if (!DB) ynext[j] = mk<T>(0, 0);
        li[j] = 0;
        if (NP % NT == 0 || j < J - 1 || k < NP) {
            int lx, ly;
            if (j < JOUT) {
                lx = H + (k & (TX - 1));
                ly = H + k / TX;
                li[j] = ly * WS + lx;
            } else {
                const unsigned e = GROUPED ? ent[j] : map[k];
                li[j] = e & 0xffff;
                lx = (int)((e >> 16) & 255);
                ly = (int)(e >> 24);
            }
            int gx = td.x0 - H + lx, gy = td.y0 - H + ly;
            bool ok = true;
            if (BC == BC_PERIODIC) {
                if (near) {
                    if constexpr (sizeof(T) == 4) { gx = wrap_near3(gx, n); gy = wrap_near3(gy, n); }
                    else { gx = wrap_near(gx, n); gy = wrap_near(gy, n); }
                } else {
                    gx = wrap_index(gx, n);
                    gy = wrap_index(gy, n);
                }
            } else if (BC == BC_SLAB) {
                // rows from 0 (the tile rows start at 4R); rows past the
                // bottom ghost rows reach no written point within 4R rows
                gx = near ? (sizeof(T) == 4 ? wrap_near3(gx, n) : wrap_near(gx, n)) : wrap_index(gx, n);
                ok = gy < ylim + H;
            } else {
                ok = gx >= 0 && gx < n && gy >= 0 && gy < n;
            }
            if (ok) {
                const unsigned gi = grid_index(gy, n, gx);
                if (BC == BC_REF) inside |= 1u << j;
                if constexpr (sizeof(T) == 4) {
                    uu[j] = buffer_load_c<T>(ru, gi * (unsigned)sizeof(C));
                    cp[j] = buffer_load_r<T>(rp, gi * (unsigned)sizeof(T));   // the pump term is formed at the store
                    if (DYN) nn[j] = buffer_load_r<T>(rn, gi * (unsigned)sizeof(T));
                } else {
                    // double precision keeps 64-bit addresses: its 512-thread
                    // form has no registers to spare for the buffer resources
                    const SC v = u[gi];
                    uu[j] = mk<T>((T)v.x, (T)v.y);
                    cp[j] = (T)P[gi];
                    if (DYN) nn[j] = (T)un[gi];
                }
            }
            if (!GROUPED) {
                ya[li[j]] = uu[j];
                if (BC == BC_REF && !ok) yb[li[j]] = uu[j];
            }
        }
        if (!GROUPED) {
            cp[j] = pump_term<T, DYN>(c, cp[j]);
            yn[j] = nn[j];
        }
    }
    if (GROUPED) {
#pragma unroll
        for (int j = 0; j < J; ++j) {
            if (NP % NT == 0 || j < J - 1 || tid + NT * j < NP) {
                ya[li[j]] = uu[j];
                if (BC == BC_REF && !((inside >> j) & 1u)) yb[li[j]] = uu[j];
            }
            cp[j] = pump_term<T, DYN>(c, cp[j]);
            yn[j] = nn[j];
        }
    }
    __syncthreads();

    // Laplacian and right-hand side of the stage input yin at point j
    typedef T V2 __attribute__((ext_vector_type(2)));
    using LV = __attribute__((address_space(3))) const V2;
    auto stage_rhs = [&](const C *yin, int j, C &k, T &kn) {
        // LDS byte address of the stencil's lowest point (R rows up), kept
        // opaque to the compiler: every read is then an immediate offset of
        // at most 2 R WS + R elements from this one register.  Folded into
        // the offsets, the buffer's own LDS address pushes the paired reads
        // out of their 8-bit offset range and costs a base add per pair.
        unsigned a = (unsigned)(size_t)((LV *)yin + (li[j] - R * WS));
        asm volatile("" : "+v"(a));
        LV *ys = (LV *)(size_t)a;
        auto rd = [&](int i) { const V2 v = ys[i]; return mk<T>(v.x, v.y); };
        const int idx = R * WS;
        const C y = rd(idx);
        // the neighbour sum (the difference form of lap_quad
        // costs 8 more operations per point and stage, and this kernel is
        // bound by its arithmetic)
        T sr, sm;
#pragma unroll
        for (int d = 1; d <= R; ++d) {
            const C a0 = rd(idx - d), a1 = rd(idx + d);
            const C b0 = rd(idx - d * WS), b1 = rd(idx + d * WS);
            if (d == 1) {
                sr = grid_ring1<R>(g, a0.x, a1.x, b0.x, b1.x);
                sm = grid_ring1<R>(g, a0.y, a1.y, b0.y, b1.y);
            } else {
                sr = grid_ring(sr, d == 2 ? g.r2 : g.r3, a0.x, a1.x, b0.x, b1.x);
                sm = grid_ring(sm, d == 2 ? g.r2 : g.r3, a0.y, a1.y, b0.y, b1.y);
            }
        }
        grid_rhs<T, DYN>(g, c, cp[j], y, yn[j], grid_sum<R, T>(g, y, sr, sm), k, kn);
    };

    // stages 1..3 on the shrinking rectangles.  Stage s computes the points
    // with at least sR halo rings around them: the first cnt list entries.
    // Points outside the reference's grid hold zero in both buffers from the
    // start and are skipped, or stepped and not written (few).
    // The test against cnt is made opaque to the compiler so that each
    // point's body stays a block of its own; resolved at compile time, the
    // stage's bodies would merge and all their LDS reads be hoisted together.
#pragma unroll
    for (int s = 1; s <= 3; ++s) {
        const int cnt = (W - 2 * s * R) * (HH - 2 * s * R);
        int lim = cnt;
        asm volatile("" : "+s"(lim));
        // y_{s+1} = u + k_s dt (1/2, 1/2, 1)
        const T dta = (s == 3) ? dt : dt2, dtwa = (s == 3) ? dtw : dtw2;
        const C *yin = (s == 2) ? yb : ya;
        C *yout = (s == 2) ? ya : yb;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            if (NT * j >= cnt) break;
            if (tid + NT * j >= lim) continue;
            const bool in = BC != BC_REF || ((inside >> j) & 1u);
            if (BC == BC_REF && !in && !few) continue;
            C k;
            T kn;
            stage_rhs(yin, j, k, kn);
            grid_acc(acc[j].x, k.x, s == 1);
            grid_acc(acc[j].y, k.y, s == 1);
            if (DYN) grid_acc(accn[j], kn, s == 1);
            const C yv = mk<T>(grid_input(uu[j].x, k.x, dtwa), grid_input(uu[j].y, k.y, dtwa));
            if (!DB) ynext[j] = yv;
            else if (in) yout[li[j]] = yv;
            if (DYN) yn[j] = grid_input(nn[j], kn, dta);
        }
        __syncthreads();
        if (!DB) {
            // stage s+1 reads its input on the stage-s rectangle
#pragma unroll
            for (int j = 0; j < J; ++j) {
                if (NT * j >= cnt) break;
                if (tid + NT * j >= lim) continue;
                ya[li[j]] = ynext[DB ? 0 : j];
            }
            __syncthreads();
        }
    }

    // stage 4 on the output tile, where it lies on the grid, and
    // u_new = u + (k1 + 2 k2 + 2 k3 + k4) dt/6
#pragma unroll
    for (int j = 0; j < JOUT; ++j) {
        const int k0 = tid + NT * j;
        const int gx = td.x0 + (k0 & (TX - 1)), gy = td.y0 + k0 / TX;
        const bool in = gx < n && gy < ylim;
        if (!in && !few) continue;
        C k;
        T kn;
        stage_rhs(yb, j, k, kn);
        if (!in) continue;
        const size_t gi = (size_t)gy * n + gx;
        uo[gi] = SC{(SR)grid_new(uu[j].x, acc[j].x, k.x, dtw6), (SR)grid_new(uu[j].y, acc[j].y, k.y, dtw6)};
        if (DYN) uno[gi] = (SR)grid_new(nn[j], accn[j], kn, dt6);
    }
}

// Single precision, order 5, periodic grids: the same step with each thread
// owning vertical pairs of points, (x, y) and (x, y + 1).  Every ring of the region is two
// rows tall and every stage's rectangle starts on an even row, so pairs tile
// all of them; listed in ring order (PairMap) each stage's rectangle is still
// a prefix.  The two points of a pair share the column of six values their
// stencils read (rows y - 2 .. y + 3): 14 LDS reads a pair instead of 18, and
// one address.  A point's arithmetic is the same expression as in
// k_fused_step_2d, so results are the same bit for bit.
#ifndef NLS_FUSED_PAIRS
#define NLS_FUSED_PAIRS 1
#endif
// LDS row stride of the pair kernel's region: W + 2.  In ring order a
// 16-lane group of the side bands spans four row pairs; a row pair is
// 2 WS complex values = 4 WS banks apart, which at W + 2 = 82 puts the four
// in distinct banks (at W + 4 every second one collides: a model of the
// kernel's reads and writes gives 0.07 against 0.40 conflict cycles per LDS
// instruction; sweep512 on the hybrid engine 81.7 -> 81.4 us per step).
#ifndef NLS_PAIR_WS_PAD
#define NLS_PAIR_WS_PAD 2
#endif
constexpr int pair_lds_stride(int W) { return W + NLS_PAIR_WS_PAD; }

template <int W, int HH, int WS> struct PairMap {
    unsigned v[W * HH / 2];
    constexpr PairMap() : v() {
        int k = 0;
        constexpr int R = 2;
        for (int s = 4; s >= 0; --s) {
            const int a = s * R, b = (s + 1) * R;
            for (int y = a; y < HH - a; y += 2)
                for (int x = a; x < W - a; ++x) {
                    const bool inner = s < 4 && y >= b && y < HH - b && x >= b && x < W - b;
                    if (!inner) v[k++] = (unsigned)(y * WS + x) | (unsigned)x << 16 | (unsigned)y << 24;
                }
        }
    }
};
static_assert(PairMap<80, 48, 82>().v[0] == (8 * 82 + 8 | 8 << 16 | 8 << 24), "pair order starts at the output tile");
static_assert(PairMap<80, 48, 82>().v[1024] == (6 * 82 + 6 | 6 << 16 | 6 << 24), "stage-3 ring follows the tile");
static_assert(PairMap<80, 32, 82>().v[512] == (6 * 82 + 6 | 6 << 16 | 6 << 24), "stage-3 ring follows the short tile");
template <int W, int HH, int WS> __device__ const PairMap<W, HH, WS> pair_map{};

template <int BC, bool DYN, int FORM>
__global__ void __launch_bounds__((FusedTile<float, 5, FORM>::NT), (FusedTile<float, 5, FORM>::WAVES))
k_fused_pairs_2d(const FusedArgs<float> f) {
    using T = float;
    using C = float2;
    using FT = FusedTile<float, 5, FORM>;
    constexpr int R = 2, H = 4 * R;
    constexpr int TX = 64, TY = FT::TY, NT = FT::NT;
    constexpr int W = TX + 2 * H, HH = TY + 2 * H, NPP = W * HH / 2;
    constexpr int WS = pair_lds_stride(W);
    constexpr int J = (NPP + NT - 1) / NT;          // pairs per thread
    constexpr int NOUT = TX * TY / 2;              // output pairs: the first NOUT entries
    static_assert(TY % 2 == 0 && HH % 2 == 0 && W < 256 && HH < 256, "pair tile shape");
    constexpr int PAD = R * WS + R;
    __shared__ C ys_mem[2][HH * WS + 2 * PAD];
    C *const ya = ys_mem[0] + PAD;
    C *const yb = ys_mem[1] + PAD;

    const int t = xcd_tile(f.ntiles, f.chunk);
    if (t < 0) return;
    TileDesc td;
    MemberDev<T> m;
    if (f.grid_ntx > 0) {
        td.m = 0; td.x0 = (t % f.grid_ntx) * TX; td.y0 = (t / f.grid_ntx) * TY + (BC == BC_SLAB ? H : 0);
        m = f.grid;
    } else {
        td = f.tiles[t];
        m = f.mem[td.m];
    }
    const int n = m.n;
    const int ylim = BC == BC_SLAB ? f.slab_end : n;
    const long long off = m.off;
    const C *u = f.u + off;
    const T *un = DYN ? f.un + off : nullptr;
    const T *P = f.P + off;
    C *uo = f.uo + off;
    T *uno = DYN ? f.uno + off : nullptr;
    const int tid = threadIdx.x;
    const unsigned cbytes = (unsigned)((unsigned long long)(BC == BC_SLAB ? f.slab_end + H : n) * n * sizeof(C));
    const __amdgpu_buffer_rsrc_t ru = buffer_of(u, cbytes), rp = buffer_of(P, cbytes / 2),
                                 rn = buffer_of(DYN ? un : P, cbytes / 2);

    if (f.it >= m.steps) {            // budget used up: pass the state through
        for (int k = tid; k < TX * TY; k += NT) {
            const int gx = td.x0 + (k & (TX - 1)), gy = td.y0 + k / TX;
            if (gx >= n || gy >= ylim) continue;
            const size_t gi = (size_t)gy * n + gx;
            uo[gi] = u[gi];
            if (DYN) uno[gi] = un[gi];
        }
        return;
    }

    const T dt = m.dt, dt2 = dt * (T)0.5, dt6 = m.g.dt6;
    const T dtw = m.g.dtw, dtw2 = dtw * (T)0.5, dtw6 = m.g.dtw6;
    Coeffs<T> c = m.c;
    GridCoeffs<T> g = m.g;
    asm volatile("" : "+v"(g.c4), "+v"(g.wc), "+v"(c.d13), "+v"(c.c13));
    const unsigned *map = pair_map<W, HH, WS>.v;

    C uu[J][2], acc[J][2];
    T cp[J][2], nn[J][2], yn[J][2], accn[J][2];
    int li[J];                         // LDS index of the pair's upper point
    unsigned inside = 0;               // BC_REF, bit 2 j + q: point q of pair j lies on the grid
    static_assert(2 * J <= 32, "inside mask");
    const bool near = n >= TX + H;

    unsigned ent[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int k = tid + NT * j;
        ent[j] = (k >= NOUT && (NPP % NT == 0 || j < J - 1 || k < NPP)) ? map[k] : 0u;
    }
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int k = tid + NT * j;
        li[j] = 0;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            uu[j][q] = mk<T>(0, 0); cp[j][q] = 0; nn[j][q] = 0; acc[j][q] = mk<T>(0, 0); accn[j][q] = 0;
        }
        if (NPP % NT == 0 || j < J - 1 || k < NPP) {
            int lx, ly;
            if (k < NOUT) {
                lx = H + (k & (TX - 1));
                ly = H + 2 * (k / TX);
                li[j] = ly * WS + lx;
            } else {
                const unsigned e = ent[j];
                li[j] = e & 0xffff;
                lx = (int)((e >> 16) & 255);
                ly = (int)(e >> 24);
            }
            int gx = td.x0 - H + lx;
            if (BC == BC_PERIODIC || BC == BC_SLAB) gx = near ? wrap_near3(gx, n) : wrap_index(gx, n);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                int gy = td.y0 - H + ly + q;
                bool ok = true;
                if (BC == BC_PERIODIC) gy = near ? wrap_near3(gy, n) : wrap_index(gy, n);
                else if (BC == BC_SLAB) ok = gy < ylim + H;
                else ok = gx >= 0 && gx < n && gy >= 0 && gy < n;
                if (ok) {
                    const unsigned gi = grid_index(gy, n, gx);
                    if (BC == BC_REF) inside |= 1u << (2 * j + q);
                    uu[j][q] = buffer_load_c<T>(ru, gi * (unsigned)sizeof(C));
                    cp[j][q] = buffer_load_r<T>(rp, gi * (unsigned)sizeof(T));
                    if (DYN) nn[j][q] = buffer_load_r<T>(rn, gi * (unsigned)sizeof(T));
                }
            }
        }
    }
#pragma unroll
    for (int j = 0; j < J; ++j) {
        if (NPP % NT == 0 || j < J - 1 || tid + NT * j < NPP) {
            ya[li[j]] = uu[j][0];
            ya[li[j] + WS] = uu[j][1];
            // outside the reference's grid both buffers hold zero throughout
            if (BC == BC_REF && !((inside >> (2 * j)) & 1u)) yb[li[j]] = mk<T>(0, 0);
            if (BC == BC_REF && !((inside >> (2 * j + 1)) & 1u)) yb[li[j] + WS] = mk<T>(0, 0);
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            cp[j][q] = pump_term<T, DYN>(c, cp[j][q]);
            yn[j][q] = nn[j][q];
        }
    }
    __syncthreads();

    typedef T V2 __attribute__((ext_vector_type(2)));
    using LV = __attribute__((address_space(3))) const V2;
    // right-hand sides of the pair's two points from stage input yin
    auto pair_rhs = [&](const C *yin, int j, C k[2], T kn[2]) {
        // LDS byte address of the column's top (R rows above the upper point),
        // kept opaque: every read is an immediate offset from it
        unsigned a = (unsigned)(size_t)((LV *)yin + (li[j] - R * WS));
        asm volatile("" : "+v"(a));
        LV *ys = (LV *)(size_t)a;
        auto rd = [&](int i) { const V2 v = ys[i]; return mk<T>(v.x, v.y); };
        const C c0 = rd(0), c1 = rd(WS), yA = rd(2 * WS), yB = rd(3 * WS), c4 = rd(4 * WS), c5 = rd(5 * WS);
        const C a1m = rd(2 * WS - 1), a1p = rd(2 * WS + 1), a2m = rd(2 * WS - 2), a2p = rd(2 * WS + 2);
        T sr = grid_ring1<R>(g, a1m.x, a1p.x, c1.x, yB.x), sm = grid_ring1<R>(g, a1m.y, a1p.y, c1.y, yB.y);
        sr = grid_ring(sr, g.r2, a2m.x, a2p.x, c0.x, c4.x);
        sm = grid_ring(sm, g.r2, a2m.y, a2p.y, c0.y, c4.y);
        grid_rhs<T, DYN>(g, c, cp[j][0], yA, yn[j][0], mk<T>(sr, sm), k[0], kn[0]);
        // the lower point's row after the upper point is done, so that its
        // reads do not all live in registers at once
        __builtin_amdgcn_sched_barrier(0);
        const C b1m = rd(3 * WS - 1), b1p = rd(3 * WS + 1), b2m = rd(3 * WS - 2), b2p = rd(3 * WS + 2);
        sr = grid_ring1<R>(g, b1m.x, b1p.x, yA.x, c4.x);
        sm = grid_ring1<R>(g, b1m.y, b1p.y, yA.y, c4.y);
        sr = grid_ring(sr, g.r2, b2m.x, b2p.x, c1.x, c5.x);
        sm = grid_ring(sm, g.r2, b2m.y, b2p.y, c1.y, c5.y);
        grid_rhs<T, DYN>(g, c, cp[j][1], yB, yn[j][1], mk<T>(sr, sm), k[1], kn[1]);
    };

#pragma unroll
    for (int s = 1; s <= 3; ++s) {
        const int cnt = (W - 2 * s * R) * (HH - 2 * s * R) / 2;
        int lim = cnt;
        asm volatile("" : "+s"(lim));
        const T dta = (s == 3) ? dt : dt2, dtwa = (s == 3) ? dtw : dtw2;
        const C *yin = (s == 2) ? yb : ya;
        C *yout = (s == 2) ? ya : yb;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            if (NT * j >= cnt) break;
            if (tid + NT * j >= lim) continue;
            C k[2];
            T kn[2];
            pair_rhs(yin, j, k, kn);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                grid_acc(acc[j][q].x, k[q].x, s == 1);
                grid_acc(acc[j][q].y, k[q].y, s == 1);
                if (DYN) grid_acc(accn[j][q], kn[q], s == 1);
                const C yv = mk<T>(grid_input(uu[j][q].x, k[q].x, dtwa), grid_input(uu[j][q].y, k[q].y, dtwa));
                if (BC != BC_REF || ((inside >> (2 * j + q)) & 1u)) yout[li[j] + q * WS] = yv;
                if (DYN) yn[j][q] = grid_input(nn[j][q], kn[q], dta);
            }
        }
        __syncthreads();
    }

    // stage 4 on the output tile and u_new = u + (k1 + 2 k2 + 2 k3 + k4) dt/6
#pragma unroll
    for (int j = 0; j < (NOUT + NT - 1) / NT; ++j) {
        const int k0 = tid + NT * j;
        if (k0 >= NOUT) break;
        const int gx = td.x0 + (k0 & (TX - 1)), gy = td.y0 + 2 * (k0 / TX);
        if (gx >= n || gy >= ylim) continue;
        C k[2];
        T kn[2];
        pair_rhs(yb, j, k, kn);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            if (gy + q >= ylim) break;
            const size_t gi = (size_t)(gy + q) * n + gx;
            uo[gi] = mk<T>(grid_new(uu[j][q].x, acc[j][q].x, k[q].x, dtw6),
                           grid_new(uu[j][q].y, acc[j][q].y, k[q].y, dtw6));
            if (DYN) uno[gi] = grid_new(nn[j][q], accn[j][q], kn[q], dt6);
        }
    }
}

// Double precision of order 5, and order 7, on tall tiles: the same step with
// each thread owning vertical groups of R points (x, y .. y + R - 1).  Every
// ring of the region is R rows tall, so groups tile all of them; listed in ring
// order (GroupMap) each stage's rectangle is a prefix, and the outermost ring,
// which no stage computes, only has its state written to LDS.  The points of a
// group share a column of 3R values: 9 LDS reads a point at order 7 instead of 13,
// 7 at order 5 instead of 9, and the groups need one address.  A point's arithmetic is the same
// expression as in k_fused_step_2d, so results are the same bit for bit.
//
// Bound, order 7 in double precision: one workgroup a CU (its two stage buffers fill
// the LDS), 8.6 us a round of 256 tiles, of which loads and stores are 3 and the
// stages 5.7, 4.6 of them LDS bandwidth (9816 stage points of 9 reads of 16 bytes); the two
// do not overlap.  Order 7, us per step, 64 x 16 tiles -> these: 777^2 zero-outside
// FP64 22.2 -> 20.0, FP32 15.0 -> 12.8; 2048^2 116 -> 104 and 68 -> 58; but 640^2 (two
// rounds of either) 16.0 -> 19.2, so such launches stay on short tiles (fused_form).
// Order 5 in double precision, against single points: 640^2 10.5 -> 10.1, 1024^2
// 24.6 -> 22.8, zero-outside 2048^2 with a reservoir 85.1 -> 80.6.  Measured and left: order 7 on
// 64 x 18 tiles (one group a thread of 1024: 24.0 at 777^2) and 640 threads (20.8).
template <int W, int HH, int R, int WS> struct GroupMap {
    unsigned v[W * HH / R];
    constexpr GroupMap() : v() {
        int k = 0;
        for (int s = 4; s >= 0; --s) {
            const int a = s * R, b = (s + 1) * R;
            for (int y = a; y < HH - a; y += R)
                for (int x = a; x < W - a; ++x) {
                    const bool inner = s < 4 && y >= b && y < HH - b && x >= b && x < W - b;
                    if (!inner) v[k++] = (unsigned)(y * WS + x) | (unsigned)x << 16 | (unsigned)y << 24;
                }
        }
    }
};
template <int W, int HH, int R, int WS> __device__ const GroupMap<W, HH, R, WS> group_map{};

// Tile rows, threads and waves per SIMD: one workgroup a CU in double precision,
// two in single.
template <typename T, int ORDER> struct GroupTile;
template <> struct GroupTile<double, 5> { static constexpr int TY = 32, NT = 1024, WAVES = 4; };
template <> struct GroupTile<double, 7> { static constexpr int TY = 24, NT = 768, WAVES = 3; };
template <> struct GroupTile<float, 7> { static constexpr int TY = 24, NT = 768, WAVES = 6; };

template <typename T, int ORDER, int BC, bool DYN, bool S32 = false>
__global__ void __launch_bounds__((GroupTile<T, ORDER>::NT), (GroupTile<T, ORDER>::WAVES))
k_fused_groups_2d(const FusedArgs<T> f) {
    using C = cplx_t<T>;
    using GT = GroupTile<T, ORDER>;
    constexpr int R = (ORDER - 1) / 2, H = 4 * R;
    constexpr int TX = 64, TY = GT::TY, NT = GT::NT;
    constexpr int W = TX + 2 * H, HH = TY + 2 * H, WS = W + 2;
    constexpr int NG = W * HH / R, NA = (W - 2 * R) * (HH - 2 * R) / R;     // groups; those of stage 1
    constexpr int J = (NA + NT - 1) / NT;          // groups per thread
    constexpr int NOUT = TX * TY / R;              // output groups: the first entries
    static_assert(TY % R == 0 && W < 256 && HH < 256 && HH * WS < 65536, "group tile shape");
    constexpr int PAD = R * WS + R;
    __shared__ C ys_mem[2][HH * WS + 2 * PAD];
    C *const ya = ys_mem[0] + PAD;
    C *const yb = ys_mem[1] + PAD;

    const int t = xcd_tile(f.ntiles, f.chunk);
    if (t < 0) return;
    TileDesc td;
    MemberDev<T> m;
    if (f.grid_ntx > 0) {
        td.m = 0; td.x0 = (t % f.grid_ntx) * TX; td.y0 = (t / f.grid_ntx) * TY + (BC == BC_SLAB ? H : 0);
        m = f.grid;
    } else {
        td = f.tiles[t];
        m = f.mem[td.m];
    }
    const int n = m.n;
    const int ylim = BC == BC_SLAB ? f.slab_end : n;
    const long long off = m.off;
    using SC = std::conditional_t<S32, float2, C>;      // storage types
    using SR = std::conditional_t<S32, float, T>;
    const SC *u = (const SC *)f.u + off;
    const SR *un = DYN ? (const SR *)f.un + off : nullptr;
    const SR *P = (const SR *)f.P + off;
    SC *uo = (SC *)f.uo + off;
    SR *uno = DYN ? (SR *)f.uno + off : nullptr;
    const int tid = threadIdx.x;

    if (f.it >= m.steps) {            // budget used up: pass the state through
        for (int k = tid; k < TX * TY; k += NT) {
            const int gx = td.x0 + (k & (TX - 1)), gy = td.y0 + k / TX;
            if (gx >= n || gy >= ylim) continue;
            const size_t gi = (size_t)gy * n + gx;
            uo[gi] = u[gi];
            if (DYN) uno[gi] = un[gi];
        }
        return;
    }

    const bool few = few_columns<T>(n, td.x0);
    const T dt = m.dt, dt2 = dt * (T)0.5, dt6 = m.g.dt6;
    const T dtw = m.g.dtw, dtw2 = dtw * (T)0.5, dtw6 = m.g.dtw6;
    Coeffs<T> c = m.c;
    GridCoeffs<T> g = m.g;
    // coefficients as in k_fused_step_2d (with a reservoir and reflecting
    // boundaries there are no registers for them)
    if constexpr (sizeof(T) == 4 && !(BC == BC_REF && DYN))
        asm volatile("" : "+v"(g.c4), "+v"(g.wc), "+v"(c.d13), "+v"(c.c13));
    const unsigned *map = group_map<W, HH, R, WS>.v;

    C uu[J][R], acc[J][R];
    T cp[J][R], nn[J][R], yn[J][R], accn[J][R];
    int li[J];                         // LDS index of the group's uppermost point
    unsigned inside = 0;               // BC_REF, bit R j + q: point q of group j lies on the grid
    static_assert(R * J <= 32, "inside mask");
    const bool near = n >= TX + H && n >= TY + H;
    // grid index of region point (lx, ly); false: outside
    auto locate = [&](int lx, int ly, unsigned &gi) {
        int gx = td.x0 - H + lx, gy = td.y0 - H + ly;
        bool ok = true;
        if (BC == BC_PERIODIC || BC == BC_SLAB) gx = near ? wrap_near3(gx, n) : wrap_index(gx, n);
        if (BC == BC_PERIODIC) gy = near ? wrap_near3(gy, n) : wrap_index(gy, n);
        else if (BC == BC_SLAB) ok = gy < ylim + H;
        else ok = gx >= 0 && gx < n && gy >= 0 && gy < n;
        gi = grid_index(gy, n, gx);
        return ok;
    };

    // the outermost ring's state
#pragma unroll
    for (int j = 0; j < (NG - NA + NT - 1) / NT; ++j) {
        const int k = NA + tid + NT * j;
        if (k < NG) {
            const unsigned e = map[k];
#pragma unroll
            for (int q = 0; q < R; ++q) {
                unsigned gi;
                const bool ok = locate((int)((e >> 16) & 255), (int)(e >> 24) + q, gi);
                ya[(int)(e & 0xffff) + q * WS] = ok ? mk<T>((T)u[gi].x, (T)u[gi].y) : mk<T>(0, 0);
            }
        }
    }
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int k = tid + NT * j;
        li[j] = 0;
#pragma unroll
        for (int q = 0; q < R; ++q) {
            uu[j][q] = mk<T>(0, 0); cp[j][q] = 0; nn[j][q] = 0; acc[j][q] = mk<T>(0, 0); accn[j][q] = 0;
        }
        if (NA % NT == 0 || j < J - 1 || k < NA) {
            const unsigned e = map[k];
            li[j] = e & 0xffff;
#pragma unroll
            for (int q = 0; q < R; ++q) {
                unsigned gi;
                if (locate((int)((e >> 16) & 255), (int)(e >> 24) + q, gi)) {
                    if (BC == BC_REF) inside |= 1u << (R * j + q);
                    uu[j][q] = mk<T>((T)u[gi].x, (T)u[gi].y);
                    cp[j][q] = (T)P[gi];
                    if (DYN) nn[j][q] = (T)un[gi];
                }
            }
        }
    }
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
        for (int q = 0; q < R; ++q) {
            if (NA % NT == 0 || j < J - 1 || tid + NT * j < NA) {
                ya[li[j] + q * WS] = uu[j][q];
                // outside the reference's grid both buffers hold zero throughout
                if (BC == BC_REF && !((inside >> (R * j + q)) & 1u)) yb[li[j] + q * WS] = mk<T>(0, 0);
            }
            cp[j][q] = pump_term<T, DYN>(c, cp[j][q]);
            yn[j][q] = nn[j][q];
        }
    __syncthreads();

    typedef T V2 __attribute__((ext_vector_type(2)));
    using LV = __attribute__((address_space(3))) const V2;
    // right-hand sides of the group's points from stage input yin, the points
    // one after another: done(q, k, kn)
    auto group_rhs = [&](const C *yin, int j, auto done) {
        unsigned a = (unsigned)(size_t)((LV *)yin + (li[j] - R * WS));
        asm volatile("" : "+v"(a));
        LV *ys = (LV *)(size_t)a;
        auto rd = [&](int i) { const V2 v = ys[i]; return mk<T>(v.x, v.y); };
        C col[3 * R];                  // rows y - R .. y + 2R - 1
#pragma unroll
        for (int i = 0; i < 2 * R; ++i) col[i] = rd(i * WS);
#pragma unroll
        for (int q = 0; q < R; ++q) {
            col[2 * R + q] = rd((2 * R + q) * WS);
            T sr, sm;
#pragma unroll
            for (int d = 1; d <= R; ++d) {
                const C l = rd((R + q) * WS - d), r = rd((R + q) * WS + d), &up = col[R + q - d], &dn = col[R + q + d];
                if (d == 1) {
                    sr = grid_ring1<R>(g, l.x, r.x, up.x, dn.x);
                    sm = grid_ring1<R>(g, l.y, r.y, up.y, dn.y);
                } else {
                    sr = grid_ring(sr, d == 2 ? g.r2 : g.r3, l.x, r.x, up.x, dn.x);
                    sm = grid_ring(sm, d == 2 ? g.r2 : g.r3, l.y, r.y, up.y, dn.y);
                }
            }
            C k;
            T kn;
            grid_rhs<T, DYN>(g, c, cp[j][q], col[R + q], yn[j][q], grid_sum<R, T>(g, col[R + q], sr, sm), k, kn);
            done(q, k, kn);
            // the next row's reads after this point is done, so that they do
            // not all live in registers at once
            __builtin_amdgcn_sched_barrier(0);
        }
    };

#pragma unroll
    for (int s = 1; s <= 3; ++s) {
        const int cnt = (W - 2 * s * R) * (HH - 2 * s * R) / R;
        int lim = cnt;
        asm volatile("" : "+s"(lim));
        const T dta = (s == 3) ? dt : dt2, dtwa = (s == 3) ? dtw : dtw2;
        const C *yin = (s == 2) ? yb : ya;
        C *yout = (s == 2) ? ya : yb;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            if (NT * j >= cnt) break;
            if (tid + NT * j >= lim) continue;
            group_rhs(yin, j, [&](int q, const C &k, T kn) {
                grid_acc(acc[j][q].x, k.x, s == 1);
                grid_acc(acc[j][q].y, k.y, s == 1);
                if (DYN) grid_acc(accn[j][q], kn, s == 1);
                const C yv = mk<T>(grid_input(uu[j][q].x, k.x, dtwa), grid_input(uu[j][q].y, k.y, dtwa));
                if (BC != BC_REF || ((inside >> (R * j + q)) & 1u)) yout[li[j] + q * WS] = yv;
                if (DYN) yn[j][q] = grid_input(nn[j][q], kn, dta);
            });
        }
        __syncthreads();
    }

    // stage 4 on the output tile and u_new = u + (k1 + 2 k2 + 2 k3 + k4) dt/6
#pragma unroll
    for (int j = 0; j < (NOUT + NT - 1) / NT; ++j) {
        const int k0 = tid + NT * j;
        if (k0 >= NOUT) break;
        const int gx = td.x0 + (k0 & (TX - 1)), gy = td.y0 + R * (k0 / TX);
        if (!few && (gx >= n || gy >= ylim)) continue;
        group_rhs(yb, j, [&](int q, const C &k, T kn) {
            if (gx < n && gy + q < ylim) {
                const size_t gi = (size_t)(gy + q) * n + gx;
                uo[gi] = SC{(SR)grid_new(uu[j][q].x, acc[j][q].x, k.x, dtw6),
                            (SR)grid_new(uu[j][q].y, acc[j][q].y, k.y, dtw6)};
                if (DYN) uno[gi] = (SR)grid_new(nn[j][q], accn[j][q], kn, dt6);
            }
        });
    }
}

// ---------------------------------------------------------------------------
// Engine RESIDENT: one workgroup per member holds the member's whole grid on
// chip and runs all of the call's steps in one launch -- a persistent kernel
// per step block.  HBM is touched only to load the state at the start and
// store it at the end.  1-D lines (n <= 4096) here; 2-D grids (n <= 64) in
// nls_small.hip.
// ---------------------------------------------------------------------------

constexpr int RES_MAXP = 4096;
// threads per workgroup: 1024 in single precision (4 points each); 512 in
// double precision (8 points each) so the register budget stays at 256
template <typename T> struct ResShape;
template <> struct ResShape<float> { static constexpr int THREADS = 1024; };
template <> struct ResShape<double> { static constexpr int THREADS = 512; };

// Laplacian of point idx of a line (wrow: its row of the radial table; outside
// the reference's grid the line is zero) and of a 2-D grid.
template <typename T, int ORDER, int BC>
__device__ __forceinline__ cplx_t<T> lap_line(const cplx_t<T> *Y, int idx, int n, const T *w, const T *wrow) {
    constexpr int R = (ORDER - 1) / 2;
    T ex[2 * R + 1], ey[2 * R + 1];
#pragma unroll
    for (int d = -R; d <= R; ++d) {
        cplx_t<T> v;
        if constexpr (BC == BC_PERIODIC) {
            int j = idx + d;
            if (d < 0 && j < 0) j += n;
            if (d > 0 && j >= n) j -= n;
            v = Y[j];
        } else {
            v = idx + d >= 0 && idx + d < n ? Y[idx + d] : mk<T>(0, 0);
        }
        ex[R + d] = v.x;
        ey[R + d] = v.y;
    }
    if (BC == BC_PERIODIC) return mk<T>(line_lap<T, R>(w, ex + R), line_lap<T, R>(w, ey + R));
    return mk<T>(line_lap_row<T, R>(wrow, ex + R), line_lap_row<T, R>(wrow, ey + R));
}

template <typename T, int ORDER, int BC>
__device__ __forceinline__ cplx_t<T> lap_grid(const cplx_t<T> *Y, int idx, int n, const T *w) {
    constexpr int R = (ORDER - 1) / 2;
    const cplx_t<T> c = Y[idx];
    const int row = idx / n, col = idx - row * n;
    T lr = lap_centre<T>((T)2 * w[0], c.x), li = lap_centre<T>((T)2 * w[0], c.y);
#pragma unroll
    for (int d = 1; d <= R; ++d) {
        int cm = col - d, cp = col + d, rm = row - d, rp = row + d;
        cplx_t<T> a0 = mk<T>(0, 0), a1 = mk<T>(0, 0), b0 = mk<T>(0, 0), b1 = mk<T>(0, 0);
        if (BC == BC_PERIODIC) {
            if (cm < 0) cm += n;
            if (cp >= n) cp -= n;
            if (rm < 0) rm += n;
            if (rp >= n) rp -= n;
            a0 = Y[row * n + cm]; a1 = Y[row * n + cp]; b0 = Y[rm * n + col]; b1 = Y[rp * n + col];
        } else {
            if (cm >= 0) a0 = Y[row * n + cm];
            if (cp < n) a1 = Y[row * n + cp];
            if (rm >= 0) b0 = Y[rm * n + col];
            if (rp < n) b1 = Y[rp * n + col];
        }
        lr += lap_quad<T>(w[d], c.x, a0.x, a1.x, b0.x, b1.x, d);
        li += lap_quad<T>(w[d], c.y, a0.y, a1.y, b0.y, b1.y, d);
    }
    return mk<T>(lr, li);
}

// Waves a SIMD: in single precision two workgroups share a CU's LDS, and its
// registers where a thread needs no more than 64, which zero-outside order 5
// without a reservoir does by two.  Order 3 with one needs 71, of which twelve are
// the weights of a thread's points; for more lines than CUs (MANY) those are loaded
// every stage, so that two workgroups share one (us per step, 256 points each: 512 lines
// 1.64 -> 1.08; 64 lines, one a CU either way, 0.82 -> 1.05).
template <typename T, int ORDER, int BC, bool DYN>
constexpr bool res_many = sizeof(T) == 4 && ORDER == 3 && BC == BC_REF && DYN;
template <typename T, int ORDER, int BC, bool DYN, bool MANY>
constexpr int res_waves = sizeof(T) == 8 ? 2 : MANY || (ORDER == 5 && BC == BC_REF && !DYN) ? 8 : 4;
template <typename T, int ORDER, int BC, bool DYN, bool MANY>
__global__ void __launch_bounds__(ResShape<T>::THREADS, (res_waves<T, ORDER, BC, DYN, MANY>)) k_resident(const ResidentArgs<T> r) {
    using C = cplx_t<T>;
    constexpr int RES_THREADS = ResShape<T>::THREADS, RES_PPT = RES_MAXP / RES_THREADS;
    // Y[b] is the psi stage input, double-buffered -- stage s reads Y[b] and
    // writes the next stage's input into Y[b ^ 1], so one barrier per stage
    // suffices (a thread writes Y[b] again only after the next barrier, which
    // every thread reaches after its reads of Y[b]); the state at the start of
    // the step is read at the thread's own points only and stays in registers.
    // Double precision of order 7 has no registers to spare for that state (it
    // would spill): Y[0] is the stage input, Y[1] the state, and each stage
    // waits for all reads of Y[0] before writing it.
    constexpr bool PINGPONG = sizeof(T) == 4 || ORDER < 7;
    __shared__ C Y[2][RES_MAXP];
    const MemberDev<T> m = r.mem[blockIdx.x];
    const int n = m.n, N = n;
    const int steps = r.iters < m.steps ? r.iters : m.steps;
    if (N > RES_MAXP || steps <= 0) return;        // the host never plans such members
    C *psi = r.psi + m.off;
    T *nres = DYN ? r.nres + m.off : nullptr;
    const T *P = r.P + m.off;
    const T *wtab = BC == BC_REF ? r.wtab + m.tab : nullptr;
    const T w[4] = {m.w0, m.w1, m.w2, m.w3};
    const int tid = threadIdx.x;
    T pp[RES_PPT], un[RES_PPT], yn[RES_PPT], accn[RES_PPT];
    C acc[RES_PPT], uu[PINGPONG ? RES_PPT : 1];
#pragma unroll
    for (int q = 0; q < RES_PPT; ++q) {
        const int idx = tid + RES_THREADS * q;
        pp[q] = 0; un[q] = 0; yn[q] = 0; accn[q] = 0; acc[q] = mk<T>(0, 0);
        if (PINGPONG) uu[PINGPONG ? q : 0] = mk<T>(0, 0);
        if (idx < N) {
            const C v = psi[idx];
            if (PINGPONG) uu[PINGPONG ? q : 0] = v;
            else Y[1][idx] = v;
            pp[q] = P[idx];
            if (DYN) { un[q] = nres[idx]; yn[q] = un[q]; }
        }
    }
#pragma unroll
    for (int q = 0; q < RES_PPT; ++q) {
        const int idx = tid + RES_THREADS * q;
        if (idx < N) Y[0][idx] = PINGPONG ? uu[PINGPONG ? q : 0] : Y[1][idx];
    }
    __syncthreads();
    int b = 0;
    LineStep<T> h = line_step(m.dt);
    if constexpr (MANY) {                // into scalar registers: the same for all lanes
        auto uniform = [](T v) { return __builtin_bit_cast(T, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v))); };
        h = LineStep<T>{uniform(h.dt), uniform(h.dt2), uniform(h.dt6), uniform(h.dt6lo)};
    }
    auto run_stage = [&](auto s_) {
        constexpr int s = decltype(s_)::value;
        // the next stage input, or at stage 4 the new state; returns the state
        auto advance_point = [&](int q, int idx, const C &kk, T kn, const C &u, C *Yout) {
            const C v = mk<T>(line_combine<T, s>(acc[q].x, kk.x, u.x, h), line_combine<T, s>(acc[q].y, kk.y, u.y, h));
            Yout[idx] = v;
            if (DYN) yn[q] = line_combine<T, s>(accn[q], kn, un[q], h);
            if (s == 4 && DYN) un[q] = yn[q];
            return s == 4 ? v : u;
        };
        auto slopes = [&](const C *Yin, int q, int idx, C &kk, T &kn) {
            unsigned row = idx * ORDER;
            if (MANY) asm volatile("" : "+v"(row));  // (loop-invariant loads otherwise)
            const C lap = lap_line<T, ORDER, BC>(Yin, idx, n, w, BC == BC_REF ? wtab + row : nullptr);
            line_rhs<T, DYN>(m.c, pump_term<T, DYN>(m.c, pp[q]), Yin[idx], yn[q], lap.x, lap.y, kk, kn);
        };
        if constexpr (PINGPONG) {
            const C *Yin = Y[b];
            C *Yout = Y[b ^ 1];
#pragma unroll
            for (int q = 0; q < RES_PPT; ++q) {
                const int idx = tid + RES_THREADS * q;
                if (idx >= N) continue;
                C kk;
                T kn = 0;
                slopes(Yin, q, idx, kk, kn);
                uu[PINGPONG ? q : 0] = advance_point(q, idx, kk, kn, uu[PINGPONG ? q : 0], Yout);
            }
            __syncthreads();
            b ^= 1;
        } else {
            C kk[RES_PPT];
            T kn[RES_PPT];
#pragma unroll
            for (int q = 0; q < RES_PPT; ++q) {
                const int idx = tid + RES_THREADS * q;
                kk[q] = mk<T>(0, 0); kn[q] = 0;
                if (idx < N) slopes(Y[0], q, idx, kk[q], kn[q]);
            }
            __syncthreads();                     // every read of Y[0] for this stage is done
#pragma unroll
            for (int q = 0; q < RES_PPT; ++q) {
                const int idx = tid + RES_THREADS * q;
                if (idx < N) Y[1][idx] = advance_point(q, idx, kk[q], kn[q], Y[1][idx], Y[0]);
            }
            __syncthreads();
        }
    };
    for (int it = 0; it < steps; ++it) {
        run_stage(std::integral_constant<int, 1>{});
        run_stage(std::integral_constant<int, 2>{});
        run_stage(std::integral_constant<int, 3>{});
        run_stage(std::integral_constant<int, 4>{});
    }
#pragma unroll
    for (int q = 0; q < RES_PPT; ++q) {
        const int idx = tid + RES_THREADS * q;
        if (idx < N) {
            psi[idx] = PINGPONG ? uu[PINGPONG ? q : 0] : Y[1][idx];
            if (DYN) nres[idx] = un[q];
        }
    }
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------

template <typename T, int ORDER, int BC, bool DYN>
static void launch_batch_stage_t(int dim, const BatchArgs<T> &b, hipStream_t s) {
    const dim3 grid(8 * b.chunk);
    if (dim == 2) hipLaunchKernelGGL((k_batch_stage<T, ORDER, BC, DYN, 2>), grid, dim3(256), 0, s, b);
    else hipLaunchKernelGGL((k_batch_stage<T, ORDER, BC, DYN, 1>), grid, dim3(256), 0, s, b);
}

template <typename T>
static void launch_batch_stage(int dim, int order, int bc, bool dyn, const BatchArgs<T> &b, hipStream_t s) {
#define NLS_CASE(O, B, D) \
    if (order == O && bc == B && dyn == D) return launch_batch_stage_t<T, O, B, D>(dim, b, s);
    NLS_CASE(3, 0, false) NLS_CASE(3, 0, true) NLS_CASE(3, 1, false) NLS_CASE(3, 1, true)
    NLS_CASE(5, 0, false) NLS_CASE(5, 0, true) NLS_CASE(5, 1, false) NLS_CASE(5, 1, true)
    NLS_CASE(7, 0, false) NLS_CASE(7, 0, true) NLS_CASE(7, 1, false) NLS_CASE(7, 1, true)
#undef NLS_CASE
}

// One fused step launch in the given form; forms a configuration does not
// build (FORM_HALF is double precision without reflecting boundaries, not of
// order 7; FORM_TALL512 is the single-precision pair kernel)
// fall back to FORM_TALL, which fused_form never asks otherwise.
template <typename T, int O, int B, bool D, bool S32 = false>
static void launch_fused_form(int form, const FusedArgs<T> &f, hipStream_t s) {
    const dim3 grid(8 * f.chunk);
    if constexpr (sizeof(T) == 4 && O == 5 && NLS_FUSED_PAIRS) {
        // zero-outside grids with a reservoir field would spill at 1024
        // threads (64 registers) and run the tall tile on 512
        constexpr int TALL = B == BC_REF && D ? FORM_TALL512 : FORM_TALL;
        // (up to one tile a CU, and past two, one point a thread at 1024 threads is the
        // faster: us per step, pairs / points, 30 grids of 70^2 7.5 / 7.0, 700^2 8.4 / 8.2,
        // 12 of 300^2 15.7 / 15.2; between 8 of 296^2 10.8 / 11.0, 1000^2 12.1 / 12.3)
        if constexpr (B == BC_REF && D)
            if (form != FORM_SHORT && (f.ntiles > 2 * device_cus() || f.ntiles <= device_cus())) {
                hipLaunchKernelGGL((k_fused_step_2d<T, O, B, D, FORM_TALL, S32>), grid,
                                   dim3(FusedTile<T, O, FORM_TALL>::NT), 0, s, f);
                return;
            }
        if (form == FORM_SHORT)
            hipLaunchKernelGGL((k_fused_pairs_2d<B, D, FORM_SHORT>), grid, dim3(1024), 0, s, f);
        else if (form == FORM_TALL512 && B == BC_PERIODIC)
            hipLaunchKernelGGL((k_fused_pairs_2d<B, D, FORM_TALL512>), grid, dim3(512), 0, s, f);
        else
            hipLaunchKernelGGL((k_fused_pairs_2d<B, D, TALL>), grid, dim3(FusedTile<T, O, TALL>::NT), 0, s, f);
        return;
    }
    if (form == FORM_SHORT) {
        hipLaunchKernelGGL((k_fused_step_2d<T, O, B, D, FORM_SHORT, S32>), grid,
                           dim3(FusedTile<T, O, FORM_SHORT>::NT), 0, s, f);
        return;
    }
    if constexpr (O != 7 && sizeof(T) == 8 && B != BC_REF)
        if (form == FORM_HALF) {
            hipLaunchKernelGGL((k_fused_step_2d<T, O, B, D, FORM_HALF, S32>), grid,
                               dim3(FusedTile<T, O, FORM_HALF>::NT), 0, s, f);
            return;
        }
    if constexpr (O == 7 || (O == 5 && sizeof(T) == 8))
        hipLaunchKernelGGL((k_fused_groups_2d<T, O, B, D, S32>), grid, dim3(GroupTile<T, O>::NT), 0, s, f);
    else
        hipLaunchKernelGGL((k_fused_step_2d<T, O, B, D, FORM_TALL, S32>), grid, dim3(FusedTile<T, O, FORM_TALL>::NT),
                           0, s, f);
}

// Double-precision arithmetic on single-precision fields (NLS_FLAG_F64_ARITH):
// periodic grids, the double-precision forms.
static void launch_fused_s32(int order, bool dyn, int form, const FusedArgs<double> &f, hipStream_t s) {
#define NLS_CASE(O, D) \
    if (order == O && dyn == D) return launch_fused_form<double, O, BC_PERIODIC, D, true>(form, f, s);
    NLS_CASE(3, false) NLS_CASE(3, true) NLS_CASE(5, false) NLS_CASE(5, true) NLS_CASE(7, false) NLS_CASE(7, true)
#undef NLS_CASE
}

template <typename T>
static void launch_fused(int order, int bc, bool dyn, int form, const FusedArgs<T> &f, hipStream_t s) {
#define NLS_CASE(O, B, D) \
    if (order == O && bc == B && dyn == D) return launch_fused_form<T, O, B, D>(form, f, s);
    NLS_CASE(3, 0, false) NLS_CASE(3, 0, true) NLS_CASE(3, 1, false) NLS_CASE(3, 1, true)
    NLS_CASE(5, 0, false) NLS_CASE(5, 0, true) NLS_CASE(5, 1, false) NLS_CASE(5, 1, true)
    NLS_CASE(7, 0, false) NLS_CASE(7, 0, true) NLS_CASE(7, 1, false) NLS_CASE(7, 1, true)
    NLS_CASE(3, 2, false) NLS_CASE(3, 2, true) NLS_CASE(5, 2, false) NLS_CASE(5, 2, true)
    NLS_CASE(7, 2, false) NLS_CASE(7, 2, true)
#undef NLS_CASE
}

// Compute units of the current device, read once per device.
int device_cus() {
    static std::atomic<int> cache[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
    int v = cache[dev].load(std::memory_order_relaxed);
    if (v > 0) return v;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    cache[dev].store(v, std::memory_order_relaxed);
    return v;
}

// The fused kernel's form for a launch over grids (or row slabs) of the
// given sizes, from the count of its tiles against the compute units.
// Measured on MI355X, order 5:
//  - 64 x 16 tiles <= CUs, FORM_SHORT: a lone 256^2 grid 7.1 -> 5.2 us per step in
//    single precision and 8.8 -> 6.2 us in double; 512^2 (256 tiles)
//    7.3 -> 5.7 and 9.4 -> 7.1 us.
//  - otherwise FORM_TALL: where CUs would hold two short tiles the tall
//    ones are as fast or faster (a 2048 x 256 row slab: 9.7 us short, 9.5 us
//    tall), and launches of several rounds are faster tall (a batch of
//    512^2-class grids: 94.6 us tall, 112.4 us short);
//  - except in double precision without reflecting boundaries, FORM_HALF where
//    the tall tiles take more than two rounds of the CUs (2048^2, 8 rounds: 89
//    -> 82 us, the sweep512 batch 196 -> 190 us), or more than one while a CU
//    has fewer than three half tiles on average: 777^2 18.0 -> 16.4 us,
//    850^2 18.7 -> 17.5, order 3 at 800^2 15.1 -> 13.1; between them the tall
//    tiles are as fast or faster (900^2: 19.9 us tall, 20.7 us half; 1024^2
//    22.2 and 21.9; a 2048 x 256 slab, one round: 13.1 us tall, 14.9 us half);
//  - order 7: a CU's 64 x 24 tiles cost 1.2 to 1.3 of its 64 x 16 ones (9.0 against 6.9 us
//    a round in double precision, 5.0 against 4.1 a tile of a CU in single), so the
//    tall tiles are taken where a CU has fewer than 0.8 as many of them.
// A process-wide choice of form per dtype (nls_tune_fused_form, set by the
// autotuner), -1: the rule below.
static std::atomic<int> g_fused_form[2] = {{-1}, {-1}};

int set_fused_form(int dtype, int form) {
    if (form < -1 || form > FORM_TALL512) return -1;
    g_fused_form[dtype == NLS_F64 ? 1 : 0].store(form);
    return 0;
}
int get_fused_form(int dtype) { return g_fused_form[dtype == NLS_F64 ? 1 : 0].load(); }

// Tiles of a launch by their rows.
struct TileCounts {
    long long t16 = 0, t24 = 0, t32 = 0;
    void add(int n, int rows) {
        const long long nx = (n + 63) / 64;
        t16 += nx * ((rows + 15) / 16);
        t24 += nx * ((rows + 23) / 24);
        t32 += nx * ((rows + 31) / 32);
    }
};
static TileCounts tiles_of(int n, int rows) {
    TileCounts t;
    t.add(n, rows);
    return t;
}
static int fused_form(int dtype, int order, int bc, const TileCounts &t) {
    const int forced = get_fused_form(dtype);
    if (forced >= 0) {
        // forms a configuration does not build run tall (launch_fused_form)
        if (forced == FORM_HALF && (order == 7 || dtype != NLS_F64 || bc == BC_REF)) return FORM_TALL;
        if (forced == FORM_TALL512 && !(dtype == NLS_F32 && order == 5 && bc == BC_PERIODIC && NLS_FUSED_PAIRS))
            return FORM_TALL;
        return forced;
    }
    const int cus = device_cus();
    if (cus <= 0) return FORM_TALL;
    if (t.t16 <= cus) return FORM_SHORT;
    if (order == 7) return 5 * ((t.t24 + cus - 1) / cus) < 4 * ((t.t16 + cus - 1) / cus) ? FORM_TALL : FORM_SHORT;
    if (dtype == NLS_F64 && bc != BC_REF && (t.t32 > 2LL * cus || (t.t32 > cus && t.t16 < 3LL * cus))) return FORM_HALF;
    return FORM_TALL;
}

// ---- marching strips or tiles ------------------------------------------------
// The marching kernel (nls_march.hip: order 5, periodic) runs the step of
// launches that fill the device; its strips are cut for that.  Times in us on
// MI355X, from 380 grids and batches of 64 to 4096 points a side timed both ways:
//  - a piece costs its rows and MARCH_PIECE more (its halo's stages and first
//    loads), and a CU's workgroups add up: 0.37 a row for one on the CU (one
//    wave a SIMD does not hide its latency), 0.21 for each of several, 0.28
//    without a reservoir (each stage divides); double precision 0.55 and 0.43;
//  - a round of tiles (512 of the pair kernel's 64 x 32, 512 of double
//    precision's 64 x 16) costs 7.4 and 7.7, short tiles that fit one per CU
//    5.4 and 6.7 in all; past the first round the next one's tiles start as CUs
//    come free, and the time grows with the tiles.
// With these the slower of the two is taken by 3% at most; with whole rounds and
// one rate a row for both reservoirs, grids without one marched up to 1.3 times
// slower than on tiles (12 of 300^2 FP32 16.9 against 13.0, 30 of 512^2 64 against 53).
// us per step, tiles -> strips: 2048^2 FP32 32.5 -> 26.5, FP64 58.6 -> 49; 154
// grids of 128^2 and 102 of 256^2 FP32 73 -> 52, FP64 175 -> 117; 64 of 200^2
// FP32 28.1 -> 21.9, FP64 52.4 -> 40.8; one 1024^2 grid stays on tiles (11.7; FP64
// 19.8 as strips and tiles).
constexpr double MARCH_LAUNCH = 3.0;
constexpr int MARCH_PIECE = 16;
static double march_us(int dtype, bool dyn, int percu, int rows) {
    if (dtype == NLS_F64) return percu * rows * (percu > 1 ? 0.43 : 0.55);
    return percu * rows * (percu == 1 ? 0.37 : dyn ? 0.21 : 0.28);
}
static double tiles_us(int dtype, bool dyn, const TileCounts &t, int cus) {
    const bool f64 = dtype == NLS_F64;
    if (t.t16 <= cus) return f64 ? 6.7 : 5.4;
    const double r = (f64 ? t.t16 : t.t32) / 512.0, round = f64 ? 7.7 : 7.4, whole = MARCH_LAUNCH + round * ceil(r);
    if (r <= 1) return whole;
    return std::min(whole, f64 ? (dyn ? 5.5 + 7.7 * r : 5.0 + 7.2 * r) : (dyn ? 6.5 + 7.4 * r : 6.0 + 6.4 * r));
}
// Members the kernel takes: rows of at least one wave, and byte offsets that
// stay below 2^32 when they run past the grid's end by up to its size.
static bool march_holds(int n, int dtype) {
    return n >= 64 && (long long)n * n * (dtype == NLS_F64 ? 16 : 8) < (1ll << 31);
}
static bool march_applies(int dtype, int order, int bc) {
    return order == 5 && bc == NLS_BC_PERIODIC && get_fused_form(dtype) < 0;   // a form asked for is a tile form
}
// Columns of a strip, strips across and pieces side by side for an n x n grid.
struct StripShape {
    int wd, nx, subs;
};
static StripShape strip_shape(int n) {
    if (n <= 256) return StripShape{n, 1, 256 / n};
    const int nx = (n + 239) / 240;
    return StripShape{(n + nx - 1) / nx, nx, 1};
}
// Workgroups a CU holds at once: registers (three waves a SIMD in single
// precision, two in double), or LDS.
static int march_slots(int dtype) { return dtype == NLS_F64 ? 2 : 3; }

// A plain n x n grid: each of its strips cut into equal pieces, one for each of
// at most `percu` workgroups a CU; no groups where tiles are faster.
struct MarchGrid {
    int groups, percu, nx, wd, rows;
};
static MarchGrid march_grid(const nls_problem *p) {
    MarchGrid best = {0, 0, 0, 0, 0};
    const int n = p->n, cus = device_cus();
    if (n <= 256 || !march_applies(p->dtype, p->order, p->bc) || !march_holds(n, p->dtype) || cus <= 0) return best;
    const bool dyn = p->coeffs[10] != 0.0;
    double least = tiles_us(p->dtype, dyn, tiles_of(n, n), cus);
    const StripShape sh = strip_shape(n);
    for (int per = 1; per <= march_slots(p->dtype); ++per) {
        const int pieces = std::max(1, per * cus / sh.nx);
        const int L = (n + pieces - 1) / pieces, groups = sh.nx * ((n + L - 1) / L);
        const double t = MARCH_LAUNCH + march_us(p->dtype, dyn, per, L + MARCH_PIECE) * ((groups + per * cus - 1) / (per * cus));
        if (t < least) { least = t; best = MarchGrid{groups, per, sh.nx, sh.wd, L}; }
    }
    return best;
}

// The pieces of a batch's members of up to 256 points a side (full) or of the
// others: the members' strips laid end to end and cut into pieces of equal
// cost, one run of pieces for each of `percu` workgroups a CU.
struct MarchCut {
    std::vector<StripDesc> strips;
    std::vector<int> first;              // of each workgroup, and the end
    int percu = 0;
    double us = 0;
};
static MarchCut march_cut(int dtype, bool dyn, const nls_member *members, int count, bool full, int cus) {
    MarchCut best;
    // cuts for workgroups of at most `cost` rows, MARCH_PIECE of them a piece's;
    // returns the number of workgroups
    auto cut = [&](int cost, MarchCut *out) {
        int groups = 1, left = cost;
        if (out) { out->strips.clear(); out->first.assign(1, 0); }
        for (int i = 0; i < count; ++i) {
            const int n = members[i].n;
            if ((n <= 256) != full) continue;
            const StripShape sh = strip_shape(n);
            const int E = (n + sh.subs - 1) / sh.subs;
            for (int k = 0; k < sh.nx; ++k)
                for (int y = 0; y < E;) {
                    if (left < MARCH_PIECE + 12 && left < cost) {     // not for a few rows
                        ++groups;
                        left = cost;
                        if (out) out->first.push_back((int)out->strips.size());
                    }
                    const int L = std::min(E - y, left - MARCH_PIECE);
                    if (out) out->strips.push_back(StripDesc{i, k * sh.wd, sh.wd, y, L, E, sh.subs});
                    y += L;
                    left -= L + MARCH_PIECE;
                }
        }
        if (out) out->first.push_back((int)out->strips.size());
        return groups;
    };
    long long rows = 0;
    for (int i = 0; i < count; ++i) {
        const StripShape sh = strip_shape(members[i].n);
        if ((members[i].n <= 256) == full) rows += (long long)sh.nx * ((members[i].n + sh.subs - 1) / sh.subs);
    }
    if (rows == 0) return best;
    for (int per = 1; per <= march_slots(dtype); ++per) {
        const int groups = per * cus;
        int lo = std::max(MARCH_PIECE + 11, (int)(rows / groups)), hi = lo + 64;
        while (cut(hi, nullptr) > groups) { lo = hi; hi += hi / 2; }
        while (hi - lo > 1) {
            const int mid = (lo + hi) / 2;
            if (cut(mid, nullptr) > groups) lo = mid;
            else hi = mid;
        }
        const double us = MARCH_LAUNCH + march_us(dtype, dyn, per, hi);
        if (best.percu && us >= best.us) continue;
        cut(hi, &best);
        best.percu = per;
        best.us = us;
    }
    return best;
}

template <typename T>
static void launch_resident(int dim, int order, int bc, bool dyn, int count, int n, const ResidentArgs<T> &r, hipStream_t s) {
    if (dim == 2) return launch_resident_2d<T>(order, bc, dyn, count, n, r, s);
#define NLS_CASE(O, B, D)                                                                                     \
    if (order == O && bc == B && dyn == D) {                                                                 \
        if constexpr (res_many<T, O, B, D>)                                                                   \
            if (count > device_cus()) {                                                                       \
                hipLaunchKernelGGL((k_resident<T, O, B, D, true>), dim3(count), dim3(ResShape<T>::THREADS), 0, s, r); \
                return;                                                                                       \
            }                                                                                                 \
        hipLaunchKernelGGL((k_resident<T, O, B, D, false>), dim3(count), dim3(ResShape<T>::THREADS), 0, s, r); \
        return;                                                                                               \
    }
    NLS_CASE(3, 0, false) NLS_CASE(3, 0, true) NLS_CASE(3, 1, false) NLS_CASE(3, 1, true)
    NLS_CASE(5, 0, false) NLS_CASE(5, 0, true) NLS_CASE(5, 1, false) NLS_CASE(5, 1, true)
    NLS_CASE(7, 0, false) NLS_CASE(7, 0, true) NLS_CASE(7, 1, false) NLS_CASE(7, 1, true)
#undef NLS_CASE
}

template <typename T>
__global__ void k_batch_radial_tables(const MemberDev<T> *mem, int count, int order, const double *dx, T *wtab) {
    // one workgroup per member, rows strided over its threads
    const int mi = blockIdx.x;
    if (mi >= count) return;
    const MemberDev<T> m = mem[mi];
    if (m.tab < 0) return;
    for (int i = threadIdx.x; i < m.n; i += blockDim.x)
        for (int k = 0; k < order; ++k)
            wtab[m.tab + (long long)i * order + k] = (T)radial_weight(i, k, m.n, order, dx[mi]);
}

static size_t align256b(size_t b) { return (b + 255) & ~(size_t)255; }

// Plain 2-D RK4 solve of one n x n grid on the fused kernel.  The member
// descriptor and the tile grid travel in the kernel arguments; the workspace
// holds the other half of the state ping-pong.
size_t fused_grid_workspace_bytes(const nls_problem *p) {
    const size_t N = (size_t)p->n * p->n, rs = p->dtype == NLS_F64 ? 8 : 4;
    return align256b(N * 2 * rs) + (p->coeffs[10] != 0.0 ? align256b(N * rs) : 0);
}

// Coefficients of a 2-D grid's step; from: for the kernels of grid_ring1_from's sums.
template <typename T>
static void set_grid_coeffs(MemberDev<T> &d, const double *c, int order, double dt, double dx, bool from) {
    if constexpr (sizeof(T) == 4) {
        if (from) {
            d.g = make_grid_coeffs<T>(c, order, dt, dx, d.lo);
            return;
        }
    }
    d.g = make_grid_coeffs<T>(c, order, dt, dx);
}

// Member descriptor of a plain (single-instance) solve.
template <typename T> static MemberDev<T> plain_member(const nls_problem *p, bool from = false) {
    MemberDev<T> d;
    memset(&d, 0, sizeof d);
    d.n = p->n;
    d.steps = 0x7fffffff;
    d.tab = -1;
    d.dt = (T)p->dt;
    d.c = make_coeffs<T>(p->coeffs);
    if (p->dim == 2) set_grid_coeffs(d, p->coeffs, p->order, p->dt, p->dx, from);
    T w[4] = {0, 0, 0, 0};
    for (int q = 0; q <= (p->order - 1) / 2; ++q) w[q] = (T)stencil_s2(p->order, q, p->dx);
    d.w0 = w[0]; d.w1 = w[1]; d.w2 = w[2]; d.w3 = w[3];
    return d;
}

// Steps a launch of a plain fused solve makes: several on a small grid, unless
// a tile form is asked for (tiles step once) or the arithmetic is
// NLS_FLAG_F64_ARITH's.
int fused_steps_per_launch(const nls_problem *p) {
    const bool from = p->engine == NLS_ENGINE_AUTO && p->dtype == NLS_F32 && p->n <= 64;
    if ((!from && get_fused_form(p->dtype) >= 0) || (p->flags & NLS_FLAG_F64_ARITH)) return 1;
    return std::max(1, multi_steps(p->n, p->order, device_cus()));
}

template <typename T>
static int fused_grid_run(const nls_problem *p, int iters, const T *P, cplx_t<T> *psi, T *nres, char *ws,
                          hipStream_t s) {
    using C = cplx_t<T>;
    const size_t N = (size_t)p->n * p->n;
    const bool dyn = p->coeffs[10] != 0.0;
    const int form = fused_form(p->dtype, p->order, p->bc, tiles_of(p->n, p->n));
    const int ty = fused_ty(p->order, form);
    FusedArgs<T> f;
    memset(&f, 0, sizeof f);
    f.grid_ntx = (p->n + 63) / 64;
    f.ntiles = f.grid_ntx * ((p->n + ty - 1) / ty);
    f.chunk = (f.ntiles + 7) / 8;
    // a small grid: its own tiles, several steps a launch
    // (of up to 64 points a side, in single precision: AUTO's choice instead of
    // the resident engine, with its bits)
    const int steps = multi_steps(p->n, p->order, device_cus());
    const bool from = steps > 0 && p->engine == NLS_ENGINE_AUTO && p->dtype == NLS_F32 && p->n <= 64;
    const int many = !from && get_fused_form(p->dtype) >= 0 ? 0 : steps;
    f.grid = plain_member<T>(p, from);
    f.P = P;
    const MarchGrid mg = march_grid(p);
    MarchArgs<T> a;
    memset(&a, 0, sizeof a);
    a.groups = mg.groups;
    a.chunk = (mg.groups + 7) / 8;
    a.grid_nx = mg.nx; a.grid_wd = mg.wd; a.grid_L = mg.rows;
    a.grid = f.grid;
    a.P = P;
    MultiArgs<T> b;
    memset(&b, 0, sizeof b);
    b.grid = f.grid;
    b.P = P;
    C *cur = psi, *alt = (C *)ws;
    T *curn = nres, *altn = dyn ? (T *)(ws + align256b(N * sizeof(C))) : nullptr;
    for (int it = 0, done; it < iters; it += done) {
        done = 1;
        if (many && (from || iters - it >= many)) {
            if (from) b.steps = std::min(many, iters - it);
            b.u = cur; b.un = curn; b.uo = alt; b.uno = altn;
            launch_multi<T>(p->order, p->bc, dyn, b, device_cus(), s);
            done = from ? b.steps : many;
        } else if (mg.groups) {
            a.it = it;
            a.u = cur; a.un = curn; a.uo = alt; a.uno = altn;
            launch_march<T>(dyn, false, mg.percu, a, s);
        } else {
            f.it = it;
            f.u = cur; f.un = curn; f.uo = alt; f.uno = altn;
            launch_fused<T>(p->order, p->bc, dyn, form, f, s);
        }
        std::swap(cur, alt);
        std::swap(curn, altn);
    }
    int rc = hip_check(hipGetLastError(), "fused step launch");
    if (rc) return rc;
    return cur == psi ? rc : copy_state<T>(N, cur, psi, dyn ? curn : nullptr, dyn ? nres : nullptr, s);
}

// One RK4 step of one row slab of a grid periodic along its rows (BC_SLAB):
// buffers of (rows + 8R) x n points, the slab's rows preceded and followed by
// 4R ghost rows; the step writes rows 4R .. 4R + rows - 1 of the output.
// The 4R-deep halo is exactly what the fused kernel recomputes on chip, so
// one exchange of ghost rows per step suffices.
template <typename T>
static int fused_slab_run(const nls_problem *p, int rows, const T *P, const cplx_t<T> *psi_in, const T *nres_in,
                          cplx_t<T> *psi_out, T *nres_out, hipStream_t s) {
    const int H = 2 * (p->order - 1);
    const int form = fused_form(p->dtype, p->order, BC_SLAB, tiles_of(p->n, rows));
    const int ty = fused_ty(p->order, form);
    FusedArgs<T> f;
    memset(&f, 0, sizeof f);
    f.grid_ntx = (p->n + 63) / 64;
    f.ntiles = f.grid_ntx * ((rows + ty - 1) / ty);
    f.chunk = (f.ntiles + 7) / 8;
    f.grid = plain_member<T>(p);
    f.slab_end = H + rows;
    f.P = P;
    f.u = psi_in; f.un = nres_in; f.uo = psi_out; f.uno = nres_out;
    launch_fused<T>(p->order, BC_SLAB, p->coeffs[10] != 0.0, form, f, s);
    return hip_check(hipGetLastError(), "slab step launch");
}

int fused_slab_step(const nls_problem *p, int rows, const void *P, const void *psi_in, const void *nres_in,
                    void *psi_out, void *nres_out, hipStream_t s) {
    if (!fused_holds((long long)(rows + 4 * (p->order - 1)) * p->n, p->dtype))
        return fail(NLS_EUNSUPPORTED, "a slab of %d rows x %d points is too large for the fused kernel (single "
                    "precision: complex array of 4 GiB or more; double: 2^32 points or more)", rows, p->n);
    if (p->dtype == NLS_F64)
        return fused_slab_run<double>(p, rows, (const double *)P, (const cplx_t<double> *)psi_in,
                                      (const double *)nres_in, (cplx_t<double> *)psi_out, (double *)nres_out, s);
    return fused_slab_run<float>(p, rows, (const float *)P, (const cplx_t<float> *)psi_in, (const float *)nres_in,
                                 (cplx_t<float> *)psi_out, (float *)nres_out, s);
}

// Plain solve of one line (n <= 4096) or small grid (n <= 64) on the
// resident kernel: one workgroup holds the instance on chip and runs a block
// of steps per launch.  Workspace: the radial row table of a 1-D ref solve.
bool resident_fits(const nls_problem *p) {
    if (p->scheme != NLS_SCHEME_RK4) return false;
    if (p->dim == 1) return p->n <= RES_MAXP;
    return (size_t)p->n * p->n <= (size_t)RES_MAXP && !(p->dtype == NLS_F64 && p->order == 7);
}

size_t resident_workspace_bytes(const nls_problem *p) {
    const size_t rs = p->dtype == NLS_F64 ? 8 : 4;
    return 256 + (p->dim == 1 && p->bc == NLS_BC_REF ? align256b((size_t)p->n * p->order * rs) : 0);
}

// Writes a by-value member descriptor into device memory (the one-entry
// member table of a plain resident solve), so no host-to-device copy is needed.
template <typename T> __global__ void k_put_member(MemberDev<T> *dst, const MemberDev<T> v) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *dst = v;
}

template <typename T>
static int resident_run(const nls_problem *p, int iters, const T *P, cplx_t<T> *psi, T *nres, char *ws,
                        hipStream_t s) {
    static_assert(sizeof(MemberDev<T>) <= 256, "member descriptor fits its workspace slot");
    MemberDev<T> one = plain_member<T>(p, true);
    ResidentArgs<T> r;
    memset(&r, 0, sizeof r);
    r.psi = psi;
    r.nres = nres;
    r.P = P;
    if (p->dim == 1 && p->bc == NLS_BC_REF) {
        launch_radial_table<T>(p->n, p->order, p->dx, (T *)(ws + 256), s);
        r.wtab = (const T *)(ws + 256);
        one.tab = 0;
    }
    hipLaunchKernelGGL((k_put_member<T>), dim3(1), dim3(64), 0, s, (MemberDev<T> *)ws, one);
    r.mem = (const MemberDev<T> *)ws;
    // bounded launches: each runs at most 4096 steps
    for (int done = 0; done < iters;) {
        r.iters = iters - done < 4096 ? iters - done : 4096;
        launch_resident<T>(p->dim, p->order, p->bc, p->coeffs[10] != 0.0, 1, p->n, r, s);
        done += r.iters;
    }
    return hip_check(hipGetLastError(), "resident launch");
}

int resident_advance(const nls_problem *p, int iters, const void *pumping, void *psi, void *nres, void *ws,
                     hipStream_t s) {
    if (p->dtype == NLS_F64)
        return resident_run<double>(p, iters, (const double *)pumping, (double2 *)psi, (double *)nres, (char *)ws, s);
    return resident_run<float>(p, iters, (const float *)pumping, (float2 *)psi, (float *)nres, (char *)ws, s);
}

// NLS_FLAG_F64_ARITH: the double-precision step (forms, member descriptor,
// arithmetic) on single-precision arrays.  The FusedArgs pointers carry the
// float arrays; the kernel (S32) reads and writes them as such.
static int fused_grid_run_s32(const nls_problem *p, int iters, const float *P, float2 *psi, float *nres, char *ws,
                              hipStream_t s) {
    const size_t N = (size_t)p->n * p->n;
    const bool dyn = p->coeffs[10] != 0.0;
    const int form = fused_form(NLS_F64, p->order, p->bc, tiles_of(p->n, p->n));
    const int ty = fused_ty(p->order, form);
    FusedArgs<double> f;
    memset(&f, 0, sizeof f);
    f.grid_ntx = (p->n + 63) / 64;
    f.ntiles = f.grid_ntx * ((p->n + ty - 1) / ty);
    f.chunk = (f.ntiles + 7) / 8;
    f.grid = plain_member<double>(p);
    f.P = (const double *)P;
    float2 *cur = psi, *alt = (float2 *)ws;
    float *curn = nres, *altn = dyn ? (float *)(ws + align256b(N * sizeof(float2))) : nullptr;
    for (int it = 0; it < iters; ++it) {
        f.it = it;
        f.u = (const double2 *)cur; f.un = (const double *)curn; f.uo = (double2 *)alt; f.uno = (double *)altn;
        launch_fused_s32(p->order, dyn, form, f, s);
        std::swap(cur, alt);
        std::swap(curn, altn);
    }
    int rc = hip_check(hipGetLastError(), "fused step launch");
    if (rc) return rc;
    if (cur != psi) {
        rc = hip_check(hipMemcpyAsync(psi, cur, N * sizeof(float2), hipMemcpyDeviceToDevice, s), "copy state");
        if (rc) return rc;
        if (dyn) rc = hip_check(hipMemcpyAsync(nres, curn, N * sizeof(float), hipMemcpyDeviceToDevice, s), "copy reservoir");
    }
    return rc;
}

int fused_grid_advance(const nls_problem *p, int iters, const void *pumping, void *psi, void *nres, void *ws,
                       hipStream_t s) {
    if (p->flags & NLS_FLAG_F64_ARITH) {
        // double-precision addressing: grids of fewer than 2^32 points
        if (!fused_holds((long long)p->n * p->n, NLS_F64))
            return fail(NLS_EUNSUPPORTED, "an %d x %d grid is too large for the fused kernel", p->n, p->n);
        return fused_grid_run_s32(p, iters, (const float *)pumping, (float2 *)psi, (float *)nres, (char *)ws, s);
    }
    if (!fused_holds((long long)p->n * p->n, p->dtype))
        return fail(NLS_EUNSUPPORTED, "an %d x %d grid is too large for the fused kernel (single precision: "
                    "complex array of 4 GiB or more; double: 2^32 points or more); the per-stage engine holds it",
                    p->n, p->n);
    if (p->dtype == NLS_F64)
        return fused_grid_run<double>(p, iters, (const double *)pumping, (double2 *)psi, (double *)nres, (char *)ws, s);
    return fused_grid_run<float>(p, iters, (const float *)pumping, (float2 *)psi, (float *)nres, (char *)ws, s);
}

}  // namespace nls

using namespace nls;

struct nls_batch {
    int dim, order, bc, dtype, engine;
    bool dyn;
    int count;
    size_t points;                 // length of the packed arrays
    int ntiles, chunk;
    // device tables (member table, tile list, member spacings, radial
    // tables) and their capacities in bytes; they grow when an update needs
    // more and are otherwise reused
    void *d_mem = nullptr, *d_tiles = nullptr, *d_dx = nullptr, *d_wtab = nullptr;
    size_t cap_mem = 0, cap_tiles = 0, cap_dx = 0, cap_wtab = 0;
    void *d_obs = nullptr;              // observables of every member (4 doubles each)
    size_t cap_obs = 0;
    // pinned host staging for the asynchronous table uploads: two slots used
    // in turn, each free again once its copy has run (event)
    struct Stage {
        void *host = nullptr;
        size_t cap = 0;
        hipEvent_t done = nullptr;
    } stage[2];
    int stage_next = 0;
    std::vector<unsigned char> h_mem;   // host image of the member table
    std::vector<TileDesc> h_tiles;      // host image of the tile list
    std::vector<double> h_dx;           // grid spacing of each member
    size_t mem_stride = 0;
    long long tab_total = 0;            // radial table entries (1-D reference grids)
    int min_steps = 0x7fffffff;         // smallest member step budget
    int fform = FORM_TALL;              // fused engine: tile form (fused_form)
    int nmax = 0;                       // points per axis of the largest member
    // fused engine, marching: the pieces of the members of up to 256 points a
    // side and of the others, on the device one behind the other (strips,
    // then the workgroups' first pieces, for each)
    MarchCut cuts[2];
    bool march = false;
    void *d_strips = nullptr;
    size_t cap_strips = 0;
    int flags = 0;                      // NLS_FLAG_EAGER: no step-block graphs
    // the captured step block and the buffers it was captured on
    hipGraphExec_t graph = nullptr;
    const void *g_P = nullptr, *g_psi = nullptr, *g_nres = nullptr, *g_ws = nullptr;
    hipStream_t capture = nullptr;
    // NLS_ENGINE_HYBRID: the members the resident engine holds (part 0) and
    // the others (part 1: fused in 2-D, per-stage in 1-D), each a batch of
    // its own over the same packed arrays (member offsets unchanged); ids[k]
    // lists part k's members by index in this batch, which is also the id in
    // the part's member table.  Part 0 runs on `side`, forked from the
    // caller's stream and joined back to it.
    nls_batch *part[2] = {nullptr, nullptr};
    std::vector<int> ids[2];
    hipStream_t side = nullptr;
    hipEvent_t fork_ev = nullptr, join_ev = nullptr;
};
static bool is_hybrid(const nls_batch *b) { return b->part[1] != nullptr; }

// Step-block graphs of a batch (fused and per-stage engines): a block of
// BATCH_GRAPH_BLOCK steps (even: the state ping-pong ends in the caller's
// buffers) is captured once per set of buffers and replayed as one graph
// launch.  A captured block bakes in the step index of each launch, which
// decides where a member whose budget ends inside the call starts passing
// its state through; blocks are therefore replayed only when every member's
// budget covers the whole call, and other calls issue their launches
// directly.
constexpr int BATCH_GRAPH_BLOCK = 64;

// Host image of the member table.  ids: each member's index in the caller's
// batch (NULL: its position here).
template <typename T>
static void fill_members(nls_batch *b, const nls_member *ms, const int *ids) {
    b->mem_stride = sizeof(MemberDev<T>);
    b->h_mem.assign(sizeof(MemberDev<T>) * b->count, 0);
    MemberDev<T> *md = (MemberDev<T> *)b->h_mem.data();
    const bool radial = b->dim == 1 && b->bc == NLS_BC_REF;
    long long tab = 0;
    for (int i = 0; i < b->count; ++i) {
        const nls_member &m = ms[i];
        MemberDev<T> d;
        memset(&d, 0, sizeof d);
        d.n = m.n;
        d.steps = 0x7fffffff;
        d.off = m.offset;
        d.id = ids ? ids[i] : i;
        // volume element of the observables: 2 pi r dr on the radial grid
        // (the sums carry the weight i, r = i dx), dx on a line, dx^2 on a square
        d.dV = radial ? 2.0 * M_PI * m.dx * m.dx : (b->dim == 1 ? m.dx : m.dx * m.dx);
        d.dt = (T)m.dt;
        d.c = make_coeffs<T>(m.coeffs);
        if (b->dim == 2) set_grid_coeffs(d, m.coeffs, b->order, m.dt, m.dx, b->engine == NLS_ENGINE_RESIDENT);
        const int R = (b->order - 1) / 2;
        T w[4] = {0, 0, 0, 0};
        for (int q = 0; q <= R; ++q) w[q] = (T)stencil_s2(b->order, q, m.dx);
        d.w0 = w[0]; d.w1 = w[1]; d.w2 = w[2]; d.w3 = w[3];
        d.tab = -1;
        if (radial) { d.tab = tab; tab += (long long)m.n * b->order; }
        md[i] = d;
    }
    b->tab_total = tab;
}

template <typename T>
static void set_member_steps(nls_batch *b, int i, int steps) {
    ((MemberDev<T> *)b->h_mem.data())[i].steps = steps;
}

// Copies the points of the batch's members from src to dst, a workgroup per
// entry of the tile list (tiles of tx x ty points): a call whose state ends in
// the workspace moves it back into the caller's buffers without touching the
// gaps between members, which in a hybrid batch hold the resident part's
// members (stepped concurrently on another stream).
template <typename T>
__global__ void __launch_bounds__(256) k_batch_carry(const MemberDev<T> *mem, const TileDesc *tiles, int ntiles,
                                                     int dim, int tx, int ty, const cplx_t<T> *src, const T *srcn,
                                                     cplx_t<T> *dst, T *dstn) {
    const int t = blockIdx.x;
    if (t >= ntiles) return;
    const TileDesc td = tiles[t];
    const MemberDev<T> m = mem[td.m];
    const int n = m.n;
    const long long o = m.off;
    for (int k = threadIdx.x; k < tx * ty; k += 256) {
        const int gx = td.x0 + k % tx, gy = td.y0 + k / tx;
        if (gx >= n || gy >= (dim == 2 ? n : 1)) continue;
        const size_t gi = (size_t)o + (dim == 2 ? (size_t)gy * n + gx : (size_t)gx);
        dst[gi] = src[gi];
        if (dstn) dstn[gi] = srcn[gi];
    }
}

// Steps it0 .. it0 + iters - 1 of the fused or per-stage engine, each
// launch issued on s.
template <typename T>
static int batch_steps(nls_batch *b, int it0, int iters, const T *P, cplx_t<T> *psi, T *nres, char *ws,
                       hipStream_t s) {
    using C = cplx_t<T>;
    const size_t cb = align256b(b->points * sizeof(C)), rb = align256b(b->points * sizeof(T));
    const bool dyn = b->dyn;
    C *cur = psi;
    T *curn = nres;
    if (b->engine == NLS_ENGINE_FUSED) {
        C *alt = (C *)ws;
        T *altn = dyn ? (T *)(ws + cb) : nullptr;
        FusedArgs<T> f;
        memset(&f, 0, sizeof f);
        f.mem = (const MemberDev<T> *)b->d_mem;
        f.tiles = (const TileDesc *)b->d_tiles;
        f.ntiles = b->ntiles;
        f.chunk = b->chunk;
        f.P = P;
        MarchArgs<T> a[2];
        const char *at = (const char *)b->d_strips;
        for (int w = 0; w < 2; ++w) {
            const MarchCut &cut = b->cuts[w];
            memset(&a[w], 0, sizeof a[w]);
            a[w].mem = f.mem;
            a[w].strips = (const StripDesc *)at;
            at += cut.strips.size() * sizeof(StripDesc);
            a[w].first = (const int *)at;
            at += cut.first.size() * sizeof(int);
            a[w].groups = cut.first.empty() ? 0 : (int)cut.first.size() - 1;
            a[w].chunk = (a[w].groups + 7) / 8;
            a[w].P = P;
        }
        for (int it = 0; it < iters; ++it) {
            f.it = it0 + it;
            f.u = cur; f.un = curn; f.uo = alt; f.uno = altn;
            if (!b->march) launch_fused<T>(b->order, b->bc, dyn, b->fform, f, s);
            else
                for (int w = 0; w < 2; ++w) {
                    a[w].it = it0 + it;
                    a[w].u = cur; a[w].un = curn; a[w].uo = alt; a[w].uno = altn;
                    if (a[w].groups) launch_march<T>(dyn, w == 0, b->cuts[w].percu, a[w], s);
                }
            std::swap(cur, alt);
            std::swap(curn, altn);
        }
    } else {
        C *kA = (C *)ws, *kB = (C *)(ws + cb), *acc = (C *)(ws + 2 * cb);
        T *kAn = nullptr, *kBn = nullptr, *accn = nullptr;
        if (dyn) { kAn = (T *)(ws + 3 * cb); kBn = (T *)(ws + 3 * cb + rb); accn = (T *)(ws + 3 * cb + 2 * rb); }
        C *alt = acc;
        T *altn = accn;
        BatchArgs<T> a;
        memset(&a, 0, sizeof a);
        a.mem = (const MemberDev<T> *)b->d_mem;
        a.tiles = (const TileDesc *)b->d_tiles;
        a.ntiles = b->ntiles;
        a.chunk = b->chunk;
        a.wtab = (const T *)b->d_wtab;
        a.P = P;
        for (int it = 0; it < iters; ++it) {
            a.it = it0 + it;
            a.u = cur; a.un = curn; a.acc = alt; a.acc_n = altn;
            a.stage = 1; a.scale = 0; a.kin = nullptr; a.kin_n = nullptr; a.kout = kA; a.kout_n = kAn;
            launch_batch_stage<T>(b->dim, b->order, b->bc, dyn, a, s);
            a.stage = 2; a.scale = (T)0.5; a.kin = kA; a.kin_n = kAn; a.kout = kB; a.kout_n = kBn;
            launch_batch_stage<T>(b->dim, b->order, b->bc, dyn, a, s);
            a.stage = 3; a.scale = (T)0.5; a.kin = kB; a.kin_n = kBn; a.kout = kA; a.kout_n = kAn;
            launch_batch_stage<T>(b->dim, b->order, b->bc, dyn, a, s);
            a.stage = 4; a.scale = (T)1; a.kin = kA; a.kin_n = kAn; a.kout = nullptr; a.kout_n = nullptr;
            launch_batch_stage<T>(b->dim, b->order, b->bc, dyn, a, s);
            std::swap(cur, alt);
            std::swap(curn, altn);
        }
    }
    int rc = hip_check(hipGetLastError(), "batch launch");
    if (rc) return rc;
    if (cur != psi) {
        // an odd step count ends in the workspace: carry the members' points
        // (only theirs) back
        const int tx = b->dim == 1 ? TILE1 : 64;
        const int ty = b->dim == 1 ? 1 : b->engine == NLS_ENGINE_FUSED ? fused_ty(b->order, b->fform) : BATCH_STAGE_TY;
        hipLaunchKernelGGL((k_batch_carry<T>), dim3(b->ntiles), dim3(256), 0, s, (const MemberDev<T> *)b->d_mem,
                           (const TileDesc *)b->d_tiles, b->ntiles, b->dim, tx, ty, (const C *)cur,
                           dyn ? (const T *)curn : nullptr, psi, dyn ? nres : nullptr);
        rc = hip_check(hipGetLastError(), "carry launch");
    }
    return rc;
}

// Per-member observables: one workgroup per member sums |psi|^2 (times the
// point index on the 1-D radial grid, whose weight is r = i dx) and the
// reservoir, takes the peak density and counts non-finite points, in double
// precision.  Each thread accumulates a fixed strided slice; the wavefront
// reduces with lane shuffles (xor 32 .. 1) and the four wavefronts' sums are
// added in order, so a member's values do not depend on the rest of the batch.
// Member i's values go to out[4 id ..], the norm and population times its
// volume element dV.
template <typename T>
__global__ void __launch_bounds__(256) k_batch_obs(const MemberDev<T> *mem, int dim, int radial,
                                                   const cplx_t<T> *psi, const T *nres, double *out) {
    __shared__ double part[4][4];
    const MemberDev<T> m = mem[blockIdx.x];
    const long long N = dim == 1 ? (long long)m.n : (long long)m.n * m.n;
    const cplx_t<T> *u = psi + m.off;
    const T *nn = nres ? nres + m.off : nullptr;
    double v[4] = {0, 0, 0, 0};
    for (long long i = threadIdx.x; i < N; i += 256) {
        const double w = radial ? (double)i : 1.0;
        const double pr = u[i].x, pi = u[i].y;
        const double sq = pr * pr + pi * pi;
        const double r = nn ? (double)nn[i] : 0.0;
        if (!isfinite(sq) || !isfinite(r)) { v[3] += 1.0; continue; }
        v[0] += sq * w;
        v[1] += r * w;
        v[2] = sq > v[2] ? sq : v[2];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        v[0] += __shfl_xor(v[0], off, 64);
        v[1] += __shfl_xor(v[1], off, 64);
        v[2] = fmax(v[2], __shfl_xor(v[2], off, 64));
        v[3] += __shfl_xor(v[3], off, 64);
    }
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0)
        for (int q = 0; q < 4; ++q) part[wave][q] = v[q];
    __syncthreads();
    if (threadIdx.x == 0) {
        double o[4] = {part[0][0], part[0][1], part[0][2], part[0][3]};
        for (int w = 1; w < 4; ++w) {
            o[0] += part[w][0]; o[1] += part[w][1]; o[2] = fmax(o[2], part[w][2]); o[3] += part[w][3];
        }
        double *dst = out + (size_t)m.id * 4;
        dst[0] = __dmul_rn(o[0], m.dV);
        dst[1] = __dmul_rn(o[1], m.dV);
        dst[2] = o[2];
        dst[3] = o[3];
    }
}

// Energy terms of every member (nls_energy per member): a workgroup per
// member, the Laplacian of each point from its neighbours in the packed
// array (the resident kernel's stencil: the member's weights, its radial
// table on the 1-D reference grid), FP64 accumulators, wavefront shuffles and
// the four wavefronts added in order.  out[4 i + 1..3] = kinetic
// -Re(conj psi L psi) w, (c5/2) |psi|^4 w, c6 r |psi|^2 w summed (w = i on the
// radial grid, else 1), each times the volume element dV, and out[4 id] their
// sum (products and sums rounded one by one, no fused multiply-add).
template <typename T, int ORDER, int BC, int DIM>
__global__ void __launch_bounds__(256) k_batch_energy(const MemberDev<T> *mem, const T *wtab,
                                                      const cplx_t<T> *psi, const T *P, const T *nres,
                                                      double *out) {
    __shared__ double part[4][3];
    const MemberDev<T> m = mem[blockIdx.x];
    const int n = m.n;
    const long long N = DIM == 1 ? (long long)n : (long long)n * n;
    const cplx_t<T> *u = psi + m.off;
    const T *pp = P + m.off;
    const T *nn = nres ? nres + m.off : nullptr;
    const T *wt = (DIM == 1 && BC == BC_REF) ? wtab + m.tab : nullptr;
    const T w[4] = {m.w0, m.w1, m.w2, m.w3};
    const double c12 = m.c.c12, c13 = m.c.c13, c14 = m.c.c14;
    double v[3] = {0, 0, 0};
    for (long long i = threadIdx.x; i < N; i += 256) {
        const double wi = (DIM == 1 && BC == BC_REF) ? (double)i : 1.0;
        cplx_t<T> lap;
        if constexpr (DIM == 1) lap = lap_line<T, ORDER, BC>(u, (int)i, n, w, wt ? wt + (size_t)i * ORDER : nullptr);
        else lap = lap_grid<T, ORDER, BC>(u, (int)i, n, w);
        const double pr = u[i].x, pi = u[i].y;
        const double sq = pr * pr + pi * pi;
        const double r = nn ? (double)nn[i] : c12 * (double)pp[i] / (c13 + c14 * sq);
        v[0] -= (pr * (double)lap.x + pi * (double)lap.y) * wi;
        v[1] += sq * sq * wi;
        v[2] += r * sq * wi;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        for (int q = 0; q < 3; ++q) v[q] += __shfl_xor(v[q], off, 64);
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0)
        for (int q = 0; q < 3; ++q) part[wave][q] = v[q];
    __syncthreads();
    if (threadIdx.x == 0) {
        double o[3] = {part[0][0], part[0][1], part[0][2]};
        for (int k = 1; k < 4; ++k)
            for (int q = 0; q < 3; ++q) o[q] += part[k][q];
        double *dst = out + (size_t)m.id * 4;
        const double e1 = __dmul_rn(o[0], m.dV);
        const double e2 = __dmul_rn(__dmul_rn(__dmul_rn(0.5, (double)m.c.c5), o[1]), m.dV);
        const double e3 = __dmul_rn(__dmul_rn((double)m.c.c6, o[2]), m.dV);
        dst[0] = __dadd_rn(__dadd_rn(e1, e2), e3);
        dst[1] = e1;
        dst[2] = e2;
        dst[3] = e3;
    }
}

template <typename T>
static void launch_batch_energy(const nls_batch *b, const T *P, const cplx_t<T> *psi, const T *nres, double *out,
                                hipStream_t s) {
    const MemberDev<T> *mem = (const MemberDev<T> *)b->d_mem;
    const T *wt = (const T *)b->d_wtab;
    const dim3 grid(b->count), blk(256);
#define NLS_CASE(O, B, D)                                                                                     \
    if (b->order == O && b->bc == B && b->dim == D) {                                                          \
        hipLaunchKernelGGL((k_batch_energy<T, O, B, D>), grid, blk, 0, s, mem, wt, psi, P, nres, out);         \
        return;                                                                                               \
    }
    NLS_CASE(3, 0, 1) NLS_CASE(3, 1, 1) NLS_CASE(3, 0, 2) NLS_CASE(3, 1, 2)
    NLS_CASE(5, 0, 1) NLS_CASE(5, 1, 1) NLS_CASE(5, 0, 2) NLS_CASE(5, 1, 2)
    NLS_CASE(7, 0, 1) NLS_CASE(7, 1, 1) NLS_CASE(7, 0, 2) NLS_CASE(7, 1, 2)
#undef NLS_CASE
}

static int drop_graph(nls_batch *b) {
    if (!b->graph) return NLS_OK;
    // an earlier launch of it may still be in flight on any stream
    int rc = hip_check(hipDeviceSynchronize(), "release batch graph");
    (void)hipGraphExecDestroy(b->graph);
    b->graph = nullptr;
    return rc;
}

// The batch's captured block of BATCH_GRAPH_BLOCK steps on these buffers,
// captured on the batch's private stream at first use.
template <typename T>
static int batch_graph(nls_batch *b, const T *P, cplx_t<T> *psi, T *nres, char *ws) {
    if (b->graph && b->g_P == P && b->g_psi == psi && b->g_nres == nres && b->g_ws == ws) return NLS_OK;
    int rc = drop_graph(b);
    if (rc) return rc;
    if (!b->capture && (rc = hip_check(hipStreamCreateWithFlags(&b->capture, hipStreamNonBlocking), "capture stream")))
        return rc;
    rc = hip_check(hipStreamBeginCapture(b->capture, hipStreamCaptureModeThreadLocal), "begin capture");
    if (rc) return rc;
    rc = batch_steps<T>(b, 0, BATCH_GRAPH_BLOCK, P, psi, nres, ws, b->capture);
    hipGraph_t g = nullptr;
    const int rc_end = hip_check(hipStreamEndCapture(b->capture, &g), "end capture");
    if (rc || rc_end) {
        if (g) (void)hipGraphDestroy(g);
        return rc ? rc : rc_end;
    }
    rc = hip_check(hipGraphInstantiate(&b->graph, g, nullptr, nullptr, 0), "instantiate graph");
    (void)hipGraphDestroy(g);
    if (rc) {
        b->graph = nullptr;
        return rc;
    }
    b->g_P = P; b->g_psi = psi; b->g_nres = nres; b->g_ws = ws;
    return NLS_OK;
}

static bool batch_graphs_apply(const nls_batch *b, int iters) {
    return b->engine != NLS_ENGINE_RESIDENT && !(b->flags & NLS_FLAG_EAGER) && iters >= 2 * BATCH_GRAPH_BLOCK &&
           b->min_steps >= iters;
}

template <typename T>
static int batch_advance(nls_batch *b, int iters, const T *P, cplx_t<T> *psi, T *nres, char *ws, hipStream_t s) {
    if (b->engine == NLS_ENGINE_RESIDENT) {
        // a persistent launch per block of steps already
        ResidentArgs<T> r;
        memset(&r, 0, sizeof r);
        r.mem = (const MemberDev<T> *)b->d_mem;
        r.iters = iters;
        r.wtab = (const T *)b->d_wtab;
        r.psi = psi;
        r.nres = nres;
        r.P = P;
        launch_resident<T>(b->dim, b->order, b->bc, b->dyn, b->count, b->nmax, r, s);
        return hip_check(hipGetLastError(), "resident launch");
    }
    if (!batch_graphs_apply(b, iters)) return batch_steps<T>(b, 0, iters, P, psi, nres, ws, s);
    int rc = batch_graph<T>(b, P, psi, nres, ws);
    if (rc) return rc;
    const int blocks = iters / BATCH_GRAPH_BLOCK, rest = iters % BATCH_GRAPH_BLOCK;
    for (int k = 0; k < blocks; ++k)
        if ((rc = hip_check(hipGraphLaunch(b->graph, s), "graph launch"))) return rc;
    return rest ? batch_steps<T>(b, iters - rest, rest, P, psi, nres, ws, s) : NLS_OK;
}

// ---- batch tables: planning and asynchronous upload -----------------------

// Member checks shared by create and update: sizes, spacings, offsets, one
// reservoir mode, no overlap in the packed arrays; *points = the packed
// length the members need.
static int check_members(int dim, int order, bool dyn, const nls_member *members, int count, size_t *points) {
    size_t pts = 0;
    std::vector<std::pair<long long, long long>> iv;
    for (int i = 0; i < count; ++i) {
        const nls_member &m = members[i];
        if (m.n < order) return fail(NLS_EINVAL, "member %d: n=%d smaller than the stencil width", i, m.n);
        if (dim == 2 && m.n > 46340) return fail(NLS_EINVAL, "member %d: n too large", i);
        if (!(m.dx > 0.0)) return fail(NLS_EINVAL, "member %d: dx must be positive", i);
        if (m.offset < 0) return fail(NLS_EINVAL, "member %d: negative offset", i);
        if ((m.coeffs[10] != 0.0) != dyn) return fail(NLS_EINVAL, "members mix reservoir modes");
        const long long np = dim == 1 ? (long long)m.n : (long long)m.n * m.n;
        pts = std::max(pts, (size_t)(m.offset + np));
        iv.push_back({m.offset, m.offset + np});
    }
    std::sort(iv.begin(), iv.end());
    for (size_t i = 1; i < iv.size(); ++i)
        if (iv[i].first < iv[i - 1].second) return fail(NLS_EINVAL, "members overlap in the packed arrays");
    *points = pts;
    return NLS_OK;
}

// Host images of the member table, the tile list and the spacings of
// `members` (ids: their indices in the caller's batch, NULL for 0..count-1).
// alone: the batch has the device to itself while it runs.  One whose members are
// exchanged (nls_batch_update) is a request loop's, beside the loop's other
// batches, and stays on tiles: marching workgroups, a few a CU of equal length,
// wait whole rounds for CUs that resident grids hold (400 requests at once: 99.8 G
// grid-point-steps/s marching, 109.9 on tiles; alone the same grids 125 and 110).
static void plan(nls_batch *b, const nls_member *members, int count, const int *ids, size_t points, bool alone) {
    b->count = count;
    b->points = points;
    b->h_dx.assign(count, 0.0);
    for (int i = 0; i < count; ++i) b->h_dx[i] = members[i].dx;
    b->nmax = 0;
    for (int i = 0; i < count; ++i) b->nmax = std::max(b->nmax, (int)members[i].n);
    if (b->dtype == NLS_F64) fill_members<double>(b, members, ids);
    else fill_members<float>(b, members, ids);
    b->min_steps = 0x7fffffff;
    // tiles, member by member, row-major inside a member
    int tx = 64, ty = BATCH_STAGE_TY;
    if (b->engine == NLS_ENGINE_FUSED) {
        TileCounts counts;
        for (int i = 0; i < count; ++i) {
            counts.add(members[i].n, members[i].n);
        }
        b->fform = fused_form(b->dtype, b->order, b->bc, counts);
        ty = fused_ty(b->order, b->fform);
        const int cus = device_cus();
        b->march = alone && cus > 0 && count > 0 && march_applies(b->dtype, b->order, b->bc);
        for (int i = 0; i < count; ++i) b->march = b->march && march_holds(members[i].n, b->dtype);
        b->cuts[0] = b->cuts[1] = MarchCut();
        if (b->march) {
            const double tiles = tiles_us(b->dtype, b->dyn, counts, cus);
            // (nothing marches faster than a few rows of every CU)
            b->march = tiles > MARCH_LAUNCH + march_us(b->dtype, b->dyn, 1, 12 + MARCH_PIECE);
            if (b->march)
                for (int w = 0; w < 2; ++w) b->cuts[w] = march_cut(b->dtype, b->dyn, members, count, w == 0, cus);
            b->march = b->march && b->cuts[0].us + b->cuts[1].us < tiles;
        }
    }
    if (b->dim == 1) { tx = TILE1; ty = 1; }
    b->h_tiles.clear();
    if (b->engine != NLS_ENGINE_RESIDENT)
        for (int i = 0; i < count; ++i) {
            const int n = members[i].n;
            const int nyt = b->dim == 1 ? 1 : (n + ty - 1) / ty, nxt = (n + tx - 1) / tx;
            for (int y = 0; y < nyt; ++y)
                for (int x = 0; x < nxt; ++x) b->h_tiles.push_back({i, x * tx, b->dim == 1 ? 0 : y * ty, 0});
        }
    b->ntiles = (int)b->h_tiles.size();
    b->chunk = (b->ntiles + 7) / 8;
}

// Device buffer of at least `need` bytes; a larger one replaces it after the
// work queued on s (the only stream that reads it) has run.
static int grow(void **p, size_t *cap, size_t need, hipStream_t s, const char *what) {
    if (need <= *cap) return NLS_OK;
    int rc = NLS_OK;
    if (*p) {
        rc = hip_check(hipStreamSynchronize(s), what);
        (void)hipFree(*p);
        *p = nullptr;
    }
    const size_t c = std::max(need, 2 * *cap);
    *cap = 0;
    if (!rc) rc = hip_check(hipMalloc(p, c), what);
    if (!rc) *cap = c;
    return rc;
}

// Copies the member table -- and with `tables` the tile list and spacings,
// then rebuilds the radial tables -- to the device, enqueued on s through the
// next pinned staging slot (the host waits only if that slot's previous copy
// has not run yet).
static int upload(nls_batch *b, hipStream_t s, bool tables) {
    const size_t nm = b->h_mem.size();
    if (nm == 0) return NLS_OK;
    const size_t nt = tables ? b->h_tiles.size() * sizeof(TileDesc) : 0;
    const size_t nd = tables ? b->h_dx.size() * sizeof(double) : 0;
    size_t ns = 0;
    if (tables && b->march)
        for (const MarchCut &c : b->cuts) ns += c.strips.size() * sizeof(StripDesc) + c.first.size() * sizeof(int);
    const size_t rs = b->dtype == NLS_F64 ? 8 : 4;
    int rc = grow(&b->d_mem, &b->cap_mem, nm, s, "batch members");
    if (!rc && nt) rc = grow(&b->d_tiles, &b->cap_tiles, nt, s, "batch tiles");
    if (!rc && nd) rc = grow(&b->d_dx, &b->cap_dx, nd, s, "batch spacings");
    if (!rc && ns) rc = grow(&b->d_strips, &b->cap_strips, ns, s, "batch strips");
    if (!rc && tables && b->tab_total > 0) rc = grow(&b->d_wtab, &b->cap_wtab, b->tab_total * rs, s, "radial tables");
    if (rc) return rc;
    nls_batch::Stage &st = b->stage[b->stage_next];
    b->stage_next ^= 1;
    if (!st.done) rc = hip_check(hipEventCreateWithFlags(&st.done, hipEventDisableTiming), "staging event");
    else rc = hip_check(hipEventSynchronize(st.done), "staging slot");
    if (rc) return rc;
    const size_t om = 0, ot = align256b(nm), od = ot + align256b(nt), os = od + align256b(nd), need = os + ns;
    if (need > st.cap) {
        if (st.host) (void)hipHostFree(st.host);
        st.host = nullptr;
        st.cap = 0;
        const size_t c = std::max(need, 2 * st.cap);
        if ((rc = hip_check(hipHostMalloc(&st.host, c, hipHostMallocDefault), "staging buffer"))) return rc;
        st.cap = c;
    }
    char *h = (char *)st.host;
    memcpy(h + om, b->h_mem.data(), nm);
    if (nt) memcpy(h + ot, b->h_tiles.data(), nt);
    if (nd) memcpy(h + od, b->h_dx.data(), nd);
    if (ns) {
        char *to = h + os;
        for (const MarchCut &c : b->cuts) {
            memcpy(to, c.strips.data(), c.strips.size() * sizeof(StripDesc));
            to += c.strips.size() * sizeof(StripDesc);
            memcpy(to, c.first.data(), c.first.size() * sizeof(int));
            to += c.first.size() * sizeof(int);
        }
    }
    rc = hip_check(hipMemcpyAsync(b->d_mem, h + om, nm, hipMemcpyHostToDevice, s), "upload members");
    if (!rc && nt) rc = hip_check(hipMemcpyAsync(b->d_tiles, h + ot, nt, hipMemcpyHostToDevice, s), "upload tiles");
    if (!rc && nd) rc = hip_check(hipMemcpyAsync(b->d_dx, h + od, nd, hipMemcpyHostToDevice, s), "upload spacings");
    if (!rc && ns)
        rc = hip_check(hipMemcpyAsync(b->d_strips, h + os, ns, hipMemcpyHostToDevice, s), "upload strips");
    if (!rc) rc = hip_check(hipEventRecord(st.done, s), "staging event");
    if (!rc && tables && b->tab_total > 0) {
        if (b->dtype == NLS_F64)
            hipLaunchKernelGGL(k_batch_radial_tables<double>, dim3(b->count), dim3(256), 0, s,
                               (const MemberDev<double> *)b->d_mem, b->count, b->order, (const double *)b->d_dx,
                               (double *)b->d_wtab);
        else
            hipLaunchKernelGGL(k_batch_radial_tables<float>, dim3(b->count), dim3(256), 0, s,
                               (const MemberDev<float> *)b->d_mem, b->count, b->order, (const double *)b->d_dx,
                               (float *)b->d_wtab);
        rc = hip_check(hipGetLastError(), "radial tables");
    }
    return rc;
}

// Budgets into the host image of the member table.
static int set_budgets(nls_batch *b, const int32_t *steps) {
    for (int i = 0; i < b->count; ++i)
        if (steps[i] < 0) return fail(NLS_EINVAL, "member %d: negative step budget", i);
    b->min_steps = 0x7fffffff;
    for (int i = 0; i < b->count; ++i) {
        if (b->dtype == NLS_F64) set_member_steps<double>(b, i, steps[i]);
        else set_member_steps<float>(b, i, steps[i]);
        b->min_steps = std::min(b->min_steps, (int)steps[i]);
    }
    return NLS_OK;
}

// A batch of one engine (not hybrid) over checked members; ids as plan().
static int create_single(int dim, int order, int bc, int dtype, int engine, bool dyn, const nls_member *members,
                         int count, const int *ids, size_t points, nls_batch **out) {
    nls_batch *b = new nls_batch();
    b->dim = dim; b->order = order; b->bc = bc; b->dtype = dtype; b->engine = engine; b->dyn = dyn;
    plan(b, members, count, ids, points, true);
    int rc = upload(b, nullptr, true);
    if (!rc) rc = hip_check(hipStreamSynchronize(nullptr), "batch tables");
    if (rc) { nls_batch_destroy(b); return rc; }
    *out = b;
    return NLS_OK;
}

// Observables / energy of every member into device memory out (4 doubles a
// member at 4 id), enqueued on s.
template <typename T>
static void launch_obs_t(nls_batch *b, const void *psi, const void *nres, double *out, hipStream_t s) {
    const int radial = (b->dim == 1 && b->bc == NLS_BC_REF) ? 1 : 0;
    hipLaunchKernelGGL((k_batch_obs<T>), dim3(b->count), dim3(256), 0, s, (const MemberDev<T> *)b->d_mem, b->dim,
                       radial, (const cplx_t<T> *)psi, b->dyn ? (const T *)nres : nullptr, out);
}

static int launch_obs(nls_batch *b, const void *psi, const void *nres, double *out, hipStream_t s) {
    if (is_hybrid(b)) {
        for (nls_batch *q : b->part) {
            const int rc = launch_obs(q, psi, nres, out, s);
            if (rc) return rc;
        }
        return NLS_OK;
    }
    if (b->count == 0) return NLS_OK;
    if (b->dtype == NLS_F64) launch_obs_t<double>(b, psi, nres, out, s);
    else launch_obs_t<float>(b, psi, nres, out, s);
    return hip_check(hipGetLastError(), "observables launch");
}

static int launch_energy(nls_batch *b, const void *P, const void *psi, const void *nres, double *out, hipStream_t s) {
    if (is_hybrid(b)) {
        for (nls_batch *q : b->part) {
            const int rc = launch_energy(q, P, psi, nres, out, s);
            if (rc) return rc;
        }
        return NLS_OK;
    }
    if (b->count == 0) return NLS_OK;
    if (b->dtype == NLS_F64)
        launch_batch_energy<double>(b, (const double *)P, (const double2 *)psi, b->dyn ? (const double *)nres : nullptr,
                                    out, s);
    else
        launch_batch_energy<float>(b, (const float *)P, (const float2 *)psi, b->dyn ? (const float *)nres : nullptr,
                                   out, s);
    return hip_check(hipGetLastError(), "energy launch");
}

// Runs launch (into the batch's device buffer) and downloads the 4 count
// doubles to the host array out; blocks until done.
template <typename F> static int obs_blocking(nls_batch *b, double *out, hipStream_t s, F launch) {
    const size_t bytes = (size_t)b->count * 4 * sizeof(double);
    if (bytes == 0) return NLS_OK;
    int rc = grow(&b->d_obs, &b->cap_obs, bytes, s, "observables buffer");
    if (!rc) rc = launch((double *)b->d_obs);
    if (!rc) rc = hip_check(hipMemcpyAsync(out, b->d_obs, bytes, hipMemcpyDeviceToHost, s), "observables download");
    if (!rc) rc = hip_check(hipStreamSynchronize(s), "observables sync");
    return rc;
}

extern "C" {

int nls_batch_create(int dim, int order, int bc, int dtype, int engine, const nls_member *members, int count,
                     nls_batch **out) {
    if (!out || !members || count <= 0) return fail(NLS_EINVAL, "batch needs members and an output handle");
    *out = nullptr;
    if (dim != 1 && dim != 2) return fail(NLS_EINVAL, "dim must be 1 or 2");
    if (order != 3 && order != 5 && order != 7) return fail(NLS_EINVAL, "order must be 3, 5 or 7");
    if (bc != NLS_BC_REF && bc != NLS_BC_PERIODIC) return fail(NLS_EINVAL, "bad bc");
    if (dtype != NLS_F32 && dtype != NLS_F64) return fail(NLS_EINVAL, "bad dtype");
    const int res_max = dim == 1 ? 4096 : 64;
    const bool res_built = !(dim == 2 && dtype == NLS_F64 && order == 7);
    int fit = 0;
    for (int i = 0; i < count; ++i) fit += res_built && members[i].n <= res_max;
    bool holds = true;                 // every member fits the fused kernel's 32-bit offsets
    for (int i = 0; i < count; ++i) holds = holds && fused_holds((long long)members[i].n * members[i].n, dtype);
    const int rest_engine = dim == 2 && holds ? NLS_ENGINE_FUSED : NLS_ENGINE_STAGE;
    if (engine == NLS_ENGINE_AUTO) engine = fit == count ? NLS_ENGINE_RESIDENT : fit > 0 ? NLS_ENGINE_HYBRID : rest_engine;
    if (engine == NLS_ENGINE_HYBRID && (fit == 0 || fit == count))      // one part only
        engine = fit == count ? NLS_ENGINE_RESIDENT : rest_engine;
    if (engine != NLS_ENGINE_STAGE && engine != NLS_ENGINE_FUSED && engine != NLS_ENGINE_RESIDENT &&
        engine != NLS_ENGINE_HYBRID)
        return fail(NLS_EINVAL, "bad engine");
    if (engine == NLS_ENGINE_RESIDENT && !res_built)
        return fail(NLS_EUNSUPPORTED, "the resident engine has no 2-D order-7 double-precision variant");
    if (engine == NLS_ENGINE_RESIDENT)
        for (int i = 0; i < count; ++i)
            if (members[i].n > res_max)
                return fail(NLS_EUNSUPPORTED, "member %d: n=%d does not fit one workgroup (resident engine: n <= %d)",
                            i, members[i].n, res_max);
    if (engine == NLS_ENGINE_FUSED && dim != 2) return fail(NLS_EUNSUPPORTED, "the fused engine is 2-D only");
    if (engine == NLS_ENGINE_FUSED && !holds)
        return fail(NLS_EUNSUPPORTED, "the fused engine holds members whose complex array is under 4 GiB");
    const bool dyn = members[0].coeffs[10] != 0.0;
    size_t points = 0;
    int rc = check_members(dim, order, dyn, members, count, &points);
    if (rc) return rc;
    if (engine != NLS_ENGINE_HYBRID)
        return create_single(dim, order, bc, dtype, engine, dyn, members, count, nullptr, points, out);
    nls_batch *b = new nls_batch();
    b->dim = dim; b->order = order; b->bc = bc; b->dtype = dtype; b->engine = engine; b->dyn = dyn;
    b->count = count; b->points = points;
    std::vector<nls_member> ms[2];
    for (int i = 0; i < count; ++i) {
        b->h_dx.push_back(members[i].dx);
        const int k = res_built && members[i].n <= res_max ? 0 : 1;
        b->ids[k].push_back(i);
        ms[k].push_back(members[i]);
    }
    size_t pts[2] = {0, 0};
    for (int k = 0; k < 2 && !rc; ++k) rc = check_members(dim, order, dyn, ms[k].data(), (int)ms[k].size(), &pts[k]);
    if (!rc)
        rc = create_single(dim, order, bc, dtype, NLS_ENGINE_RESIDENT, dyn, ms[0].data(), (int)ms[0].size(),
                           b->ids[0].data(), pts[0], &b->part[0]);
    if (!rc)
        rc = create_single(dim, order, bc, dtype, rest_engine, dyn, ms[1].data(), (int)ms[1].size(), b->ids[1].data(),
                           pts[1], &b->part[1]);
    if (!rc) rc = hip_check(hipStreamCreateWithFlags(&b->side, hipStreamNonBlocking), "hybrid stream");
    if (!rc) rc = hip_check(hipEventCreateWithFlags(&b->fork_ev, hipEventDisableTiming), "hybrid event");
    if (!rc) rc = hip_check(hipEventCreateWithFlags(&b->join_ev, hipEventDisableTiming), "hybrid event");
    if (rc) { nls_batch_destroy(b); return rc; }
    b->ntiles = b->part[1]->ntiles;
    *out = b;
    return NLS_OK;
}

int nls_batch_destroy(nls_batch *b) {
    if (!b) return NLS_OK;
    for (nls_batch *q : b->part) nls_batch_destroy(q);
    if (b->side) (void)hipStreamDestroy(b->side);
    if (b->fork_ev) (void)hipEventDestroy(b->fork_ev);
    if (b->join_ev) (void)hipEventDestroy(b->join_ev);
    (void)drop_graph(b);
    if (b->capture) (void)hipStreamDestroy(b->capture);
    for (nls_batch::Stage &st : b->stage) {
        if (st.done) {
            (void)hipEventSynchronize(st.done);
            (void)hipEventDestroy(st.done);
        }
        if (st.host) (void)hipHostFree(st.host);
    }
    for (void *p : {b->d_mem, b->d_tiles, b->d_dx, b->d_wtab, b->d_obs, b->d_strips})
        if (p) (void)hipFree(p);
    delete b;
    return NLS_OK;
}

size_t nls_batch_points(const nls_batch *b) { return b ? b->points : 0; }

int nls_batch_tiles(const nls_batch *b) { return b ? b->ntiles : 0; }

size_t nls_batch_workspace_bytes(const nls_batch *b) {
    if (!b) return 0;
    if (is_hybrid(b)) return nls_batch_workspace_bytes(b->part[1]);     // the resident part needs none
    const size_t rs = b->dtype == NLS_F64 ? 8 : 4;
    const size_t cb = align256b(b->points * 2 * rs), rb = align256b(b->points * rs);
    if (b->engine == NLS_ENGINE_RESIDENT) return 0;
    if (b->engine == NLS_ENGINE_FUSED) return cb + (b->dyn ? rb : 0);
    return 3 * cb + (b->dyn ? 3 * rb : 0);
}

int nls_batch_update(nls_batch *b, const nls_member *members, int count, const int32_t *steps, void *stream) {
    if (!b) return fail(NLS_EINVAL, "NULL batch");
    if (count < 0 || (count > 0 && !members)) return fail(NLS_EINVAL, "bad member list");
    if (is_hybrid(b))
        return fail(NLS_EUNSUPPORTED, "a hybrid batch splits its members between engines at creation; update "
                    "batches of one engine");
    if (b->engine == NLS_ENGINE_RESIDENT)
        for (int i = 0; i < count; ++i)
            if (members[i].n > (b->dim == 1 ? 4096 : 64))
                return fail(NLS_EUNSUPPORTED, "member %d: n=%d does not fit one workgroup", i, members[i].n);
    if (b->engine == NLS_ENGINE_FUSED)
        for (int i = 0; i < count; ++i)
            if (!fused_holds((long long)members[i].n * members[i].n, b->dtype))
                return fail(NLS_EUNSUPPORTED, "member %d is too large for the fused engine", i);
    size_t points = 0;
    int rc = check_members(b->dim, b->order, b->dyn, members, count, &points);
    if (rc) return rc;
    if (steps)
        for (int i = 0; i < count; ++i)
            if (steps[i] < 0) return fail(NLS_EINVAL, "member %d: negative step budget", i);
    hipStream_t s = (hipStream_t)stream;
    if (b->graph) {
        // a captured block holds the old launch shapes; it may be in flight on s
        if ((rc = hip_check(hipStreamSynchronize(s), "update"))) return rc;
        (void)hipGraphExecDestroy(b->graph);
        b->graph = nullptr;
    }
    plan(b, members, count, nullptr, points, false);
    if (steps && (rc = set_budgets(b, steps))) return rc;
    return upload(b, s, true);
}

int nls_batch_set_steps(nls_batch *b, const int32_t *steps, void *stream) {
    if (!b || !steps) return fail(NLS_EINVAL, "NULL argument");
    for (int i = 0; i < b->count; ++i)
        if (steps[i] < 0) return fail(NLS_EINVAL, "member %d: negative step budget", i);
    if (is_hybrid(b)) {
        // uploads on the caller's stream, which the side stream follows
        for (int k = 0; k < 2; ++k) {
            std::vector<int32_t> st;
            for (int i : b->ids[k]) st.push_back(steps[i]);
            const int rc = nls_batch_set_steps(b->part[k], st.data(), stream);
            if (rc) return rc;
        }
        return NLS_OK;
    }
    const int rc = set_budgets(b, steps);
    return rc ? rc : upload(b, (hipStream_t)stream, false);
}

int nls_batch_observables(nls_batch *b, const void *psi, const void *nres, double *out, void *stream) {
    if (!b || !psi || !out) return fail(NLS_EINVAL, "NULL argument");
    if (b->dyn && !nres) return fail(NLS_EINVAL, "NULL reservoir buffer");
    hipStream_t s = (hipStream_t)stream;
    return obs_blocking(b, out, s, [&](double *d) { return launch_obs(b, psi, nres, d, s); });
}

int nls_batch_observables_async(nls_batch *b, const void *psi, const void *nres, double *out, void *stream) {
    if (!b || !psi || !out) return fail(NLS_EINVAL, "NULL argument");
    if (b->dyn && !nres) return fail(NLS_EINVAL, "NULL reservoir buffer");
    return launch_obs(b, psi, nres, out, (hipStream_t)stream);
}

int nls_batch_energy(nls_batch *b, const void *pumping, const void *psi, const void *nres, double *out,
                     void *stream) {
    if (!b || !pumping || !psi || !out) return fail(NLS_EINVAL, "NULL argument");
    if (b->dyn && !nres) return fail(NLS_EINVAL, "NULL reservoir buffer");
    hipStream_t s = (hipStream_t)stream;
    return obs_blocking(b, out, s, [&](double *d) { return launch_energy(b, pumping, psi, nres, d, s); });
}

int nls_batch_energy_async(nls_batch *b, const void *pumping, const void *psi, const void *nres, double *out,
                           void *stream) {
    if (!b || !pumping || !psi || !out) return fail(NLS_EINVAL, "NULL argument");
    if (b->dyn && !nres) return fail(NLS_EINVAL, "NULL reservoir buffer");
    return launch_energy(b, pumping, psi, nres, out, (hipStream_t)stream);
}

int nls_batch_prepare(nls_batch *b, int iters, const void *pumping, void *psi, void *nres, void *workspace,
                      size_t workspace_bytes) {
    if (!b) return fail(NLS_EINVAL, "NULL batch");
    if (!pumping || !psi || (b->dyn && !nres)) return fail(NLS_EINVAL, "NULL device buffer");
    const size_t need = nls_batch_workspace_bytes(b);
    if (workspace_bytes < need || (need && !workspace))
        return fail(NLS_EINVAL, "workspace of %zu bytes is smaller than the %zu required", workspace_bytes, need);
    if (is_hybrid(b)) return nls_batch_prepare(b->part[1], iters, pumping, psi, nres, workspace, workspace_bytes);
    if (b->count == 0 || !batch_graphs_apply(b, iters)) return NLS_OK;
    if (b->dtype == NLS_F64)
        return batch_graph<double>(b, (const double *)pumping, (double2 *)psi, (double *)nres, (char *)workspace);
    return batch_graph<float>(b, (const float *)pumping, (float2 *)psi, (float *)nres, (char *)workspace);
}

int nls_batch_set_flags(nls_batch *b, int flags) {
    if (!b) return fail(NLS_EINVAL, "NULL batch");
    if (flags & ~NLS_FLAG_EAGER) return fail(NLS_EINVAL, "unknown flags 0x%x", flags);
    b->flags = flags;
    for (nls_batch *q : b->part)
        if (q) q->flags = flags;
    return NLS_OK;
}

int nls_batch_advance(nls_batch *b, int iters, const void *pumping, void *psi, void *nres, void *workspace,
                      size_t workspace_bytes, void *stream) {
    if (!b) return fail(NLS_EINVAL, "NULL batch");
    if (iters < 0) return fail(NLS_EINVAL, "iters must be >= 0");
    if (!pumping || !psi || (b->dyn && !nres)) return fail(NLS_EINVAL, "NULL device buffer");
    const size_t need = nls_batch_workspace_bytes(b);
    if (workspace_bytes < need || (need && !workspace))
        return fail(NLS_EINVAL, "workspace of %zu bytes is smaller than the %zu required", workspace_bytes, need);
    if (iters == 0 || b->count == 0) return NLS_OK;
    hipStream_t s = (hipStream_t)stream;
    if (is_hybrid(b)) {
        // resident part on the side stream, the rest on the caller's, joined
        int rc = hip_check(hipEventRecord(b->fork_ev, s), "hybrid fork");
        if (!rc) rc = hip_check(hipStreamWaitEvent(b->side, b->fork_ev, 0), "hybrid fork");
        if (!rc) rc = nls_batch_advance(b->part[0], iters, pumping, psi, nres, workspace, workspace_bytes, b->side);
        const int rc1 = rc ? rc : nls_batch_advance(b->part[1], iters, pumping, psi, nres, workspace, workspace_bytes, s);
        // join even after a failed launch, so the caller's stream never runs ahead of the side stream
        int rj = hip_check(hipEventRecord(b->join_ev, b->side), "hybrid join");
        if (!rj) rj = hip_check(hipStreamWaitEvent(s, b->join_ev, 0), "hybrid join");
        return rc1 ? rc1 : rj;
    }
    if (b->dtype == NLS_F64)
        return batch_advance<double>(b, iters, (const double *)pumping, (double2 *)psi, (double *)nres,
                                     (char *)workspace, s);
    return batch_advance<float>(b, iters, (const float *)pumping, (float2 *)psi, (float *)nres, (char *)workspace, s);
}

}  // extern "C"
