// nls_ssf.hip -- split-step Fourier scheme on periodic grids (no counterpart
// in the reference, which only has RK4 over finite differences).
//
// One step (Strang splitting):  N(dt/2) -> L(dt) -> N(dt/2)
//   L(dt): psi_hat(k) *= exp(-i |k|^2 dt), the exact flow of psi_t = i lap psi
//          on the spectral wavenumbers of the grid;
//   N(t):  one classical RK4 step of size t of the pointwise part of the
//          reference's right-hand side (nls/nls.f90:570-581, :637-644) plus
//          the reservoir equation when c11 != 0.
//
// 2-D: the state between passes is kept transformed along x ("row space"):
//   row pass  : inverse x-FFT -> N(dt/2) [end of step] -> N(dt/2) [start of
//               the next] -> forward x-FFT           (reads/writes psi, n, P)
//   column pass: forward y-FFT -> phase exp(-i (kx^2 + ky^2) dt)/n^2 ->
//               inverse y-FFT                          (reads/writes psi)
// so a step moves 4 c + 3 r bytes per point (c complex, r real).  The first
// row pass has no inverse transform and the last one no forward transform.
// 1-D: a workgroup holds a whole line (n <= 4096) in registers and runs all
// steps on chip.
//
// Precision: the fields sit in HBM in the problem's dtype; every kernel
// computes in double precision (FFT stages, pointwise RK4, twiddle and phase
// tables), with a single-precision state converted on load and rounded once
// on store.  On MI355X double-precision vector arithmetic issues at the
// single-precision rate (packed FP32 aside), so single precision only saves
// HBM bytes; rounding the state once per pass instead of at every FFT stage
// keeps its error far below that of single-precision transforms.
//
// FFTs: Stockham stages with a line's values in the registers of its threads,
// the stage-to-stage exchanges through LDS (fft_regs).  The kinetic energy keeps
// them in LDS and works in place: a stage stages its butterfly inputs and
// twiddles in registers, synchronises,
// then writes the outputs.  Twiddles exp(-2 pi i m / n) and the phase table are
// generated in double precision.
#include <cstring>
#include <type_traits>

#include "nls_core.h"
#include "nls_internal.h"

namespace nls {

// Row kernels with their values in LDS: one 2048-point line (or several
// shorter lines) per workgroup, 32 KB, so four workgroups share a CU.
constexpr int ROW_PTS = 2048, ROW_LOG_PTS = 11, ROW_NTH = 256;

// LDS layout of the transforms: element i at i + (i >> SHIFT), one complex of
// padding per 2^SHIFT, so that the strided writes of the first radix-8
// stages (stride 8, then groups of 8 at stride 64) spread over the LDS banks
// instead of piling on a few; SHIFT = 31 is the plain layout, 0 a swizzle without
// padding (each group of eight permuted by the number of its group).  Each kernel
// takes its own shift (the padding costs index arithmetic where the
// conflicts it removes are few).
#ifndef NLS_SSF_ROW_PAD
#define NLS_SSF_ROW_PAD 4
#endif
#ifndef NLS_SSF_COL_PAD
#define NLS_SSF_COL_PAD 4
#endif
#ifndef NLS_SSF_LINE_PAD
#define NLS_SSF_LINE_PAD 4
#endif
constexpr int lds_padded(int pts, int shift) { return pts + (shift < 31 ? pts >> shift : 0); }
template <typename T, int SHIFT> struct Lds {
    cplx_t<T> *p;
    __device__ __forceinline__ cplx_t<T> &operator[](int i) const {
        return p[SHIFT == 0 ? i ^ ((i >> 3) & 7) : SHIFT < 31 ? i + (i >> SHIFT) : i];
    }
};

template <typename T>
__device__ __forceinline__ cplx_t<T> cmul(cplx_t<T> a, cplx_t<T> b) {
    return mk<T>(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// Element m of line l lives at buf[l*lstride + m*estride].  LINE_FAST maps
// consecutive threads to consecutive lines (column pass: lines are adjacent
// in LDS) instead of consecutive elements (row pass).  A stage reads its
// butterfly inputs from LDS and its twiddles from the table (global memory,
// cached) before the barrier, so both are in flight together; after the
// barrier it computes and writes the outputs in place.
template <typename T, bool INV, bool LINE_FAST, int PTS, int NTH, typename LB>
__device__ __forceinline__ void fft_radix4_stage(LB buf, int logN, int logL, int lstride, int estride,
                                                 int logNs, const cplx_t<T> *tw) {
    using C = cplx_t<T>;
    constexpr int QB = (PTS / 4 + NTH - 1) / NTH;    // butterflies per thread
    const int lognb = logN - 2;
    const int total = 1 << (logL + lognb);           // butterflies in the workgroup
    const int Ns = 1 << logNs;
    const int sh = logN - logNs - 2;
    C v[QB][4], w[QB][3];
#pragma unroll
    for (int q = 0; q < QB; ++q) {
        const int b = threadIdx.x + NTH * q;
        if (b < total) {
            const int l = LINE_FAST ? (b & ((1 << logL) - 1)) : (b >> lognb);
            const int j = LINE_FAST ? (b >> logL) : (b & ((1 << lognb) - 1));
            const int k = j & (Ns - 1);
#pragma unroll
            for (int r = 1; r < 4; ++r) w[q][r - 1] = tw[(r * k) << sh];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[q][r] = buf[l * lstride + (j + (r << lognb)) * estride];
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < QB; ++q) {
        const int b = threadIdx.x + NTH * q;
        if (b < total) {
            const int l = LINE_FAST ? (b & ((1 << logL) - 1)) : (b >> lognb);
            const int j = LINE_FAST ? (b >> logL) : (b & ((1 << lognb) - 1));
            const int k = j & (Ns - 1);
#pragma unroll
            for (int r = 1; r < 4; ++r) {
                C wr = w[q][r - 1];
                if (INV) wr.y = -wr.y;
                v[q][r] = cmul<T>(v[q][r], wr);
            }
            const C t0 = mk<T>(v[q][0].x + v[q][2].x, v[q][0].y + v[q][2].y);
            const C t1 = mk<T>(v[q][0].x - v[q][2].x, v[q][0].y - v[q][2].y);
            const C t2 = mk<T>(v[q][1].x + v[q][3].x, v[q][1].y + v[q][3].y);
            const C d13 = mk<T>(v[q][1].x - v[q][3].x, v[q][1].y - v[q][3].y);
            // forward: (a1 - a3) * (-i); inverse: * (+i)
            const C t3 = INV ? mk<T>(-d13.y, d13.x) : mk<T>(d13.y, -d13.x);
            const int d = ((j >> logNs) << (logNs + 2)) + k;
            const int o = l * lstride;
            buf[o + (d) * estride] = mk<T>(t0.x + t2.x, t0.y + t2.y);
            buf[o + (d + Ns) * estride] = mk<T>(t1.x + t3.x, t1.y + t3.y);
            buf[o + (d + 2 * Ns) * estride] = mk<T>(t0.x - t2.x, t0.y - t2.y);
            buf[o + (d + 3 * Ns) * estride] = mk<T>(t1.x - t3.x, t1.y - t3.y);
        }
    }
    __syncthreads();
}

// Radix-8 stage: the 8-point DFT of each butterfly in registers, as two
// 4-point DFTs (even and odd inputs) joined by the eighth roots of unity.
template <typename T, bool INV>
__device__ __forceinline__ void dft4(cplx_t<T> &a0, cplx_t<T> &a1, cplx_t<T> &a2, cplx_t<T> &a3) {
    using C = cplx_t<T>;
    const C t0 = mk<T>(a0.x + a2.x, a0.y + a2.y);
    const C t1 = mk<T>(a0.x - a2.x, a0.y - a2.y);
    const C t2 = mk<T>(a1.x + a3.x, a1.y + a3.y);
    const C d13 = mk<T>(a1.x - a3.x, a1.y - a3.y);
    const C t3 = INV ? mk<T>(-d13.y, d13.x) : mk<T>(d13.y, -d13.x);
    a0 = mk<T>(t0.x + t2.x, t0.y + t2.y);
    a1 = mk<T>(t1.x + t3.x, t1.y + t3.y);
    a2 = mk<T>(t0.x - t2.x, t0.y - t2.y);
    a3 = mk<T>(t1.x - t3.x, t1.y - t3.y);
}

// w8 = exp(-2 pi i / 8), the twiddle table's entry N/8.
template <typename T, bool INV, bool LINE_FAST, int PTS, int NTH, typename LB>
__device__ __forceinline__ void fft_radix8_stage(LB buf, int logN, int logL, int lstride, int estride,
                                                 int logNs, const cplx_t<T> *tw, cplx_t<T> w8) {
    using C = cplx_t<T>;
    constexpr int QB = (PTS / 8 + NTH - 1) / NTH;
    const int lognb = logN - 3;
    const int total = 1 << (logL + lognb);
    const int Ns = 1 << logNs;
    const int sh = logN - logNs - 3;
    C v[QB][8], w[QB][7];
#pragma unroll
    for (int q = 0; q < QB; ++q) {
        const int b = threadIdx.x + NTH * q;
        if (b < total) {
            const int l = LINE_FAST ? (b & ((1 << logL) - 1)) : (b >> lognb);
            const int j = LINE_FAST ? (b >> logL) : (b & ((1 << lognb) - 1));
            const int k = j & (Ns - 1);
#pragma unroll
            for (int r = 1; r < 8; ++r) w[q][r - 1] = tw[(r * k) << sh];
#pragma unroll
            for (int r = 0; r < 8; ++r) v[q][r] = buf[l * lstride + (j + (r << lognb)) * estride];
        }
    }
    __syncthreads();
    if (INV) w8.y = -w8.y;
#pragma unroll
    for (int q = 0; q < QB; ++q) {
        const int b = threadIdx.x + NTH * q;
        if (b < total) {
            const int l = LINE_FAST ? (b & ((1 << logL) - 1)) : (b >> lognb);
            const int j = LINE_FAST ? (b >> logL) : (b & ((1 << lognb) - 1));
            const int k = j & (Ns - 1);
#pragma unroll
            for (int r = 1; r < 8; ++r) {
                C wr = w[q][r - 1];
                if (INV) wr.y = -wr.y;
                v[q][r] = cmul<T>(v[q][r], wr);
            }
            C e0 = v[q][0], e1 = v[q][2], e2 = v[q][4], e3 = v[q][6];
            C o0 = v[q][1], o1 = v[q][3], o2 = v[q][5], o3 = v[q][7];
            dft4<T, INV>(e0, e1, e2, e3);
            dft4<T, INV>(o0, o1, o2, o3);
            // o_r *= w8^r (inverse: conjugate), r = 1, 2, 3; w8^2 = -i, w8^3 = -i w8
            o1 = cmul<T>(o1, w8);
            o2 = INV ? mk<T>(-o2.y, o2.x) : mk<T>(o2.y, -o2.x);
            o3 = cmul<T>(o3, w8);
            o3 = INV ? mk<T>(-o3.y, o3.x) : mk<T>(o3.y, -o3.x);
            const int d = ((j >> logNs) << (logNs + 3)) + k;
            const int o = l * lstride;
            buf[o + d * estride] = mk<T>(e0.x + o0.x, e0.y + o0.y);
            buf[o + (d + Ns) * estride] = mk<T>(e1.x + o1.x, e1.y + o1.y);
            buf[o + (d + 2 * Ns) * estride] = mk<T>(e2.x + o2.x, e2.y + o2.y);
            buf[o + (d + 3 * Ns) * estride] = mk<T>(e3.x + o3.x, e3.y + o3.y);
            buf[o + (d + 4 * Ns) * estride] = mk<T>(e0.x - o0.x, e0.y - o0.y);
            buf[o + (d + 5 * Ns) * estride] = mk<T>(e1.x - o1.x, e1.y - o1.y);
            buf[o + (d + 6 * Ns) * estride] = mk<T>(e2.x - o2.x, e2.y - o2.y);
            buf[o + (d + 7 * Ns) * estride] = mk<T>(e3.x - o3.x, e3.y - o3.y);
        }
    }
    __syncthreads();
}

template <typename T, bool INV, bool LINE_FAST, int PTS, int NTH, typename LB>
__device__ __forceinline__ void fft_radix2_stage(LB buf, int logN, int logL, int lstride, int estride,
                                                 int logNs, const cplx_t<T> *tw) {
    using C = cplx_t<T>;
    constexpr int QB = (PTS / 2 + NTH - 1) / NTH;
    const int lognb = logN - 1;
    const int total = 1 << (logL + lognb);
    const int Ns = 1 << logNs;
    const int sh = logN - logNs - 1;
    C v[QB][2], w[QB];
#pragma unroll
    for (int q = 0; q < QB; ++q) {
        const int b = threadIdx.x + NTH * q;
        if (b < total) {
            const int l = LINE_FAST ? (b & ((1 << logL) - 1)) : (b >> lognb);
            const int j = LINE_FAST ? (b >> logL) : (b & ((1 << lognb) - 1));
            w[q] = tw[(j & (Ns - 1)) << sh];
            v[q][0] = buf[l * lstride + j * estride];
            v[q][1] = buf[l * lstride + (j + (1 << lognb)) * estride];
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < QB; ++q) {
        const int b = threadIdx.x + NTH * q;
        if (b < total) {
            const int l = LINE_FAST ? (b & ((1 << logL) - 1)) : (b >> lognb);
            const int j = LINE_FAST ? (b >> logL) : (b & ((1 << lognb) - 1));
            const int k = j & (Ns - 1);
            C wq = w[q];
            if (INV) wq.y = -wq.y;
            const C a1 = cmul<T>(v[q][1], wq);
            const int d = ((j >> logNs) << (logNs + 1)) + k;
            const int o = l * lstride;
            buf[o + d * estride] = mk<T>(v[q][0].x + a1.x, v[q][0].y + a1.y);
            buf[o + (d + Ns) * estride] = mk<T>(v[q][0].x - a1.x, v[q][0].y - a1.y);
        }
    }
    __syncthreads();
}

// In-place FFT of 2^logL lines of length 2^logN (2^(logL+logN) <= PTS) in LDS.
template <typename T, bool INV, bool LINE_FAST, int PTS, int NTH, typename LB>
__device__ __forceinline__ void lds_fft(LB buf, int logN, int logL, int lstride, int estride,
                                        const cplx_t<T> *tw) {
    int logNs = 0;
    if (sizeof(T) == 8 && logN >= 3) {
        // radix-8 stages (2048 = 8 8 8 4: four passes through LDS instead of six)
        const cplx_t<T> w8 = tw[(1 << logN) >> 3];
        do {
            fft_radix8_stage<T, INV, LINE_FAST, PTS, NTH>(buf, logN, logL, lstride, estride, logNs, tw, w8);
            logNs += 3;
        } while (logN - logNs >= 3);
    }
    while (logN - logNs >= 2) {
        fft_radix4_stage<T, INV, LINE_FAST, PTS, NTH>(buf, logN, logL, lstride, estride, logNs, tw);
        logNs += 2;
    }
    if (logN - logNs == 1) fft_radix2_stage<T, INV, LINE_FAST, PTS, NTH>(buf, logN, logL, lstride, estride, logNs, tw);
}

// One RK4 step of size tau of the pointwise system at one point.
template <typename T, bool DYN>
__device__ __forceinline__ void pointwise_rk4(const Coeffs<T> &c, T inv_c11, T P, T tau, cplx_t<T> &psi, T &n) {
    auto f = [&](cplx_t<T> y, T yn, cplx_t<T> &k, T &kn) {
        const T s = y.x * y.x + y.y * y.y;
        const T r = DYN ? yn : c.c12 * P / (c.c13 + c.c14 * s);
        const T g = c.c3 * r - c.c4, q = c.c5 * s + c.c6 * r;
        k = mk<T>(g * y.x + q * y.y, g * y.y - q * y.x);
        kn = DYN ? (c.c12 * P - (c.c13 + c.c14 * s) * yn) * inv_c11 : (T)0;
    };
    cplx_t<T> k1, k2, k3, k4;
    T m1, m2, m3, m4;
    const T h = tau * (T)0.5;
    f(psi, n, k1, m1);
    f(mk<T>(psi.x + k1.x * h, psi.y + k1.y * h), n + m1 * h, k2, m2);
    f(mk<T>(psi.x + k2.x * h, psi.y + k2.y * h), n + m2 * h, k3, m3);
    f(mk<T>(psi.x + k3.x * tau, psi.y + k3.y * tau), n + m3 * tau, k4, m4);
    const T t6 = tau / (T)6;
    psi = mk<T>(psi.x + (k1.x + (T)2 * k2.x + (T)2 * k3.x + k4.x) * t6,
                psi.y + (k1.y + (T)2 * k2.y + (T)2 * k3.y + k4.y) * t6);
    if (DYN) n = n + (m1 + (T)2 * m2 + (T)2 * m3 + m4) * t6;
}

// S: the precision of the fields in HBM (the problem's dtype); T: the
// arithmetic, LDS and tables, double in both cases -- on this GPU double
// precision vector arithmetic runs at the single-precision rate (no packed
// FP32), so a single-precision state only halves the HBM bytes and is
// rounded once per pass, not at every FFT stage.
template <typename S, typename T> struct SsfArgs {
    T half_dt, inv_c11;
    Coeffs<T> c;
    cplx_t<S> *psi;
    S *nres;
    const S *P;
    const cplx_t<T> *tw;      // exp(-2 pi i m / N)
    const cplx_t<T> *ph;      // exp(-i k_m^2 dt) / N
    int iters;                // 1-D kernel only
};

// A stored complex value in the arithmetic precision, and back.
template <typename T, typename S> __device__ __forceinline__ cplx_t<T> widen(cplx_t<S> v) {
    return mk<T>((T)v.x, (T)v.y);
}
template <typename S, typename T> __device__ __forceinline__ cplx_t<S> narrow(cplx_t<T> v) {
    return mk<S>((S)v.x, (S)v.y);
}

enum { ROWS_FIRST = 0, ROWS_MIDDLE = 1, ROWS_LAST = 2 };

// Lines of length 2^logN per workgroup of 2^logP points (at most n lines).
__host__ __device__ constexpr int lines_per_wg(int logN, int logP) {
    return logP - logN < logN ? logP - logN : logN;
}

// Radix-8 butterfly of Stockham stage logNs of a 2^LN-point transform on
// the inputs x[0..7] (elements j + r 2^(LN-3) of the line), in place: x[r]
// becomes the output element d + r Ns, d = ((j >> logNs) << (logNs + 3)) +
// (j & (Ns - 1)).  The arithmetic of fft_radix8_stage; TW = false skips the
// twiddles of the first stage, which are all 1.
template <typename T, bool INV, bool TW>
__device__ __forceinline__ void bfly8(cplx_t<T> x[8], int j, int logNs, int LN, const cplx_t<T> *tw, cplx_t<T> w8) {
    using C = cplx_t<T>;
    if (TW) {
        const int k = j & ((1 << logNs) - 1), sh = LN - logNs - 3;
#pragma unroll
        for (int r = 1; r < 8; ++r) {
            C wr = tw[(r * k) << sh];
            if (INV) wr.y = -wr.y;
            x[r] = cmul<T>(x[r], wr);
        }
    }
    if (INV) w8.y = -w8.y;
    C e0 = x[0], e1 = x[2], e2 = x[4], e3 = x[6];
    C o0 = x[1], o1 = x[3], o2 = x[5], o3 = x[7];
    dft4<T, INV>(e0, e1, e2, e3);
    dft4<T, INV>(o0, o1, o2, o3);
    o1 = cmul<T>(o1, w8);
    o2 = INV ? mk<T>(-o2.y, o2.x) : mk<T>(o2.y, -o2.x);
    o3 = cmul<T>(o3, w8);
    o3 = INV ? mk<T>(-o3.y, o3.x) : mk<T>(o3.y, -o3.x);
    x[0] = mk<T>(e0.x + o0.x, e0.y + o0.y);
    x[1] = mk<T>(e1.x + o1.x, e1.y + o1.y);
    x[2] = mk<T>(e2.x + o2.x, e2.y + o2.y);
    x[3] = mk<T>(e3.x + o3.x, e3.y + o3.y);
    x[4] = mk<T>(e0.x - o0.x, e0.y - o0.y);
    x[5] = mk<T>(e1.x - o1.x, e1.y - o1.y);
    x[6] = mk<T>(e2.x - o2.x, e2.y - o2.y);
    x[7] = mk<T>(e3.x - o3.x, e3.y - o3.y);
}

// Radix-4 butterfly of Stockham stage logNs on the inputs x[0..3] (elements
// j + r 2^(LN-2)), in place, as bfly8: x[r] becomes the output element d + r Ns,
// d = ((j >> logNs) << (logNs + 2)) + (j & (Ns - 1)).
template <typename T, bool INV, bool TW>
__device__ __forceinline__ void bfly4(cplx_t<T> &x0, cplx_t<T> &x1, cplx_t<T> &x2, cplx_t<T> &x3, int j, int logNs,
                                      int LN, const cplx_t<T> *tw) {
    using C = cplx_t<T>;
    if (TW) {
        const int k = j & ((1 << logNs) - 1), sh = LN - logNs - 2;
        C w1 = tw[k << sh], w2 = tw[(2 * k) << sh], w3 = tw[(3 * k) << sh];
        if (INV) { w1.y = -w1.y; w2.y = -w2.y; w3.y = -w3.y; }
        x1 = cmul<T>(x1, w1);
        x2 = cmul<T>(x2, w2);
        x3 = cmul<T>(x3, w3);
    }
    dft4<T, INV>(x0, x1, x2, x3);
}

// Radix-16 butterfly, as bfly8 (elements j + r 2^(LN-4), outputs d + r Ns, d =
// ((j >> logNs) << (logNs + 4)) + (j & (Ns - 1))): four 4-point DFTs over the
// inputs of equal remainder mod 4, the sixteenth roots of unity, four more.
template <typename T, bool INV, bool TW>
__device__ __forceinline__ void bfly16(cplx_t<T> x[16], int j, int logNs, int LN, const cplx_t<T> *tw) {
    using C = cplx_t<T>;
    if (TW) {
        const int k = j & ((1 << logNs) - 1), sh = LN - logNs - 4;
#pragma unroll
        for (int r = 1; r < 16; ++r) {
            C wr = tw[(r * k) << sh];
            if (INV) wr.y = -wr.y;
            x[r] = cmul<T>(x[r], wr);
        }
    }
    const T c1 = (T)0.92387953251128675613, s1 = (T)0.38268343236508977173, h = (T)0.70710678118654752440;
    const T wc[4] = {1, c1, h, s1}, ws[4] = {0, s1, h, c1};
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        dft4<T, INV>(x[m], x[4 + m], x[8 + m], x[12 + m]);
        // slot 4 k + m times exp(-+ 2 pi i k m / 16)
#pragma unroll
        for (int k = 1; k < 4; ++k) {
            const int e = k * m, f = e < 4 ? e : e == 4 ? 0 : e == 6 ? 2 : 1;      // quarter turns taken out below
            C v = x[4 * k + m];
            if (e != 0 && e != 4) v = cmul<T>(v, mk<T>(wc[f], INV ? ws[f] : -ws[f]));
            if (e == 4 || e == 6) v = INV ? mk<T>(-v.y, v.x) : mk<T>(v.y, -v.x);    // w16^4 = -i
            if (e == 9) v = mk<T>(-v.x, -v.y);                                      // w16^9 = -w16
            x[4 * k + m] = v;
        }
    }
    C y[16];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        dft4<T, INV>(x[4 * k], x[4 * k + 1], x[4 * k + 2], x[4 * k + 3]);
#pragma unroll
        for (int q = 0; q < 4; ++q) y[k + 4 * q] = x[4 * k + q];
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) x[r] = y[r];
}

// Transform of a 2^LN-point line (LN = 4 .. 12) whose values stay in
// registers: thread j of the line's 2^LN / PT holds the PT (4, 8 or 16)
// elements j + (2^LN / PT) s in x[s].  Those are the inputs of its radix-PT
// butterfly of every stage, and the inputs and outputs of its butterflies of
// the last one, whether that is radix 8, 4 (PT / 4 butterflies) or 2 (PT / 2).
// So a transform starts and ends in the thread's own elements, and only the
// exchanges between stages go through LDS: ex(logNs) writes the outputs of
// stage logNs (element d + r Ns from x[r]) and reads the thread's elements
// back.  Stages: radix PT, and one of a smaller radix for the bits left over.
__host__ __device__ constexpr int log2_pt(int PT) { return PT == 16 ? 4 : PT == 8 ? 3 : 2; }
template <typename T, bool INV, int LN, int PT, typename EX>
__device__ __forceinline__ void fft_regs(cplx_t<T> x[PT], int j, const cplx_t<T> *tw, EX ex) {
    using C = cplx_t<T>;
    static_assert(LN >= 4 && LN <= 12 && (PT == 4 || PT == 8 || PT == 16), "line length and points per thread");
    constexpr int LP = log2_pt(PT), Q = 1 << (LN - LP), REM = LN % LP, SP = LN / LP;
    C w8;
    if constexpr (PT >= 8) w8 = tw[(1 << LN) >> 3];
    auto stage = [&](auto first, int logNs) {
        if constexpr (PT == 16) bfly16<T, INV, !decltype(first)::value>(x, j, logNs, LN, tw);
        else if constexpr (PT == 8) bfly8<T, INV, !decltype(first)::value>(x, j, logNs, LN, tw, w8);
        else bfly4<T, INV, !decltype(first)::value>(x[0], x[1], x[2], x[3], j, logNs, LN, tw);
    };
    stage(std::true_type(), 0);
#pragma unroll
    for (int s = 1; s < SP; ++s) {
        ex(LP * (s - 1));
        stage(std::false_type(), LP * s);
    }
    if constexpr (REM > 0) ex(LP * (SP - 1));
    if constexpr (REM == 3) {
#pragma unroll
        for (int q = 0; q < PT / 8; ++q) {
            C y[8];
#pragma unroll
            for (int r = 0; r < 8; ++r) y[r] = x[q + PT / 8 * r];
            bfly8<T, INV, true>(y, j + Q * q, LN - 3, LN, tw, w8);
#pragma unroll
            for (int r = 0; r < 8; ++r) x[q + PT / 8 * r] = y[r];
        }
    } else if constexpr (REM == 2) {
        constexpr int M = PT / 4;
#pragma unroll
        for (int q = 0; q < M; ++q)
            bfly4<T, INV, true>(x[q], x[q + M], x[q + 2 * M], x[q + 3 * M], j + Q * q, LN - 2, LN, tw);
    } else if constexpr (REM == 1) {
        constexpr int M = PT / 2;
#pragma unroll
        for (int q = 0; q < M; ++q) {
            C w = tw[j + Q * q];
            if (INV) w.y = -w.y;
            const C v = cmul<T>(x[q + M], w), u = x[q];
            x[q] = mk<T>(u.x + v.x, u.y + v.y);
            x[q + M] = mk<T>(u.x - v.x, u.y - v.y);
        }
    }
}

// Order the wave's LDS accesses around this point for the compiler (the
// hardware runs one wave's LDS operations in order; no instruction).
__device__ __forceinline__ void wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Lines in registers, L of them in a workgroup of at least one wave: LDS for
// the exchanges of fft_regs.  One wave: its LDS operations run in order, one
// buffer and no barrier.  Several: two buffers in turn and one barrier each (a
// buffer is written again only after the next exchange's barrier, which every
// thread reaches after its reads); NBUF = 1: one buffer, two barriers, for half
// the LDS.  COLS: the lines interleaved (element e of line l at e L + l), else
// one behind the other.
template <typename T, int LN, int PT, int L, int PAD, bool COLS, int NBUF = 2> struct LineLds {
    static constexpr int LP = log2_pt(PT), Q = 1 << (LN - LP), NTH = L * Q;
    static constexpr bool WAVE = NTH <= 64;
    static constexpr int EX = (LN + LP - 1) / LP - 1;      // exchanges of a transform
    static constexpr int PTS = lds_padded(L << LN, PAD);
    static constexpr int MEM = WAVE ? PTS : NBUF * PTS;
    // the mth exchange since the start is at buffer (first + m) & 1
    static __device__ __forceinline__ auto exchange(cplx_t<T> *mem, cplx_t<T> x[PT], int j, int l, int first) {
        return [=](int logNs) {
            const int Ns = 1 << logNs, d = ((j >> logNs) << (logNs + LP)) + (j & (Ns - 1));
            const int es = COLS ? L : 1, l0 = COLS ? l : l << LN;
            const Lds<T, PAD> B{mem + (WAVE || NBUF == 1 ? 0 : ((first + logNs / LP) & 1) * PTS)};
            if (WAVE) wave_order();
            else if (NBUF == 1) __syncthreads();
#pragma unroll
            for (int r = 0; r < PT; ++r) B[l0 + (d + r * Ns) * es] = x[r];
            if (WAVE) wave_order();
            else __syncthreads();
#pragma unroll
            for (int r = 0; r < PT; ++r) x[r] = B[l0 + (j + Q * r) * es];
        };
    }
};

// Points per thread, lines per workgroup and LDS buffers of the passes in
// registers, by the line's length; double precision (f32: single-precision
// storage), us a step or a pass.  Few points a thread spread the pointwise part,
// which a small grid or a single line leaves to few waves, but cost more
// exchanges and narrower butterflies.
// - 1-D lines, 4 points against 8: n = 256 2.2 / 3.4 a step, 1024 4.3 / 6.2,
//   2048 8.3 / 7.5, 4096 18.0 / 14.6.
// - Rows, 4 against 8: a step of 64^2 6.9 / 9.2, 256^2 9.0 / 10.1; the pass at
//   512^2 7.2 / 6.6, without a reservoir (the stationary density divides) 8.4 /
//   9.6; at 1024^2 19.8 / 19.0.  2048-point rows take k_ssf_rows2048 between the
//   first and the last pass, which are in registers with one buffer, four
//   workgroups a CU.
// - Columns: a pass moves 32 bytes a point; the short ones are latency, one
//   column of 4 points a thread (a step of 64^2: 7.9, two columns 8.5, two of 8
//   points 8.7), 512^2 two of 8 points (5.3; of 4 points 5.8, of 16 6.5).
//   From 1024 on 16 points a thread, an exchange fewer a transform: the pass at 1024^2
//   four columns 17.6 against 19.1 of 8 points (f32 13.8 / 15.5), at 2048^2 two
//   columns 43.6, four 45.6 (f32, the same 32 bytes a row with four: 41.1 / 38.6),
//   four of 8 points in LDS 48.2 (43.9).
constexpr int line_pt(int LN) { return LN <= 10 ? 4 : 8; }
constexpr int row_pt(int LN, bool dyn) { return LN <= (dyn ? 8 : 9) ? 4 : 8; }
constexpr int row_bufs(int LN) { return LN <= 10 ? 2 : 1; }
constexpr int col_pt(int LN) { return LN <= 8 ? 4 : LN == 9 ? 8 : 16; }
constexpr int col_lines(int LN, bool f64) { return LN <= 8 ? 1 : LN == 9 || (LN == 11 && f64) ? 2 : 4; }
constexpr int col_bufs(int LN) { return LN <= 9 ? 2 : 1; }

// 1-D: one workgroup runs every step of a line in registers (fft_regs): the
// pointwise half steps and the phase act on the thread's own points.  The
// threads of a line shorter than a wave's points hold it several times over.
// Against the line in LDS, us a step: n = 16 2.3 -> 1.4, 256 3.6 -> 2.2, 1024
// 6.3 -> 4.2, 2048 10.0 -> 7.5 (4096 was in registers: 14.6).  One CU's VALU issue
// bounds the longest lines (8 us of 14.6), barriers and latency the rest.
template <int LN, int PT> constexpr int line_threads = (1 << LN) / PT < 64 ? 64 : (1 << LN) / PT;
template <typename S, typename T, bool DYN, int LN, int PT>
__global__ void __launch_bounds__((line_threads<LN, PT>)) k_ssf_line(const SsfArgs<S, T> a) {
    using C = cplx_t<T>;
    using LL = LineLds<T, LN, PT, 1, NLS_SSF_LINE_PAD, false>;
    constexpr int Q = LL::Q;
    __shared__ C mem[LL::MEM];
    const int j = threadIdx.x & (Q - 1);
    C x[PT], ph[PT];
    T pp[PT], nn[PT];
#pragma unroll
    for (int r = 0; r < PT; ++r) {
        const int e = j + Q * r;
        x[r] = widen<T, S>(a.psi[e]);
        ph[r] = a.ph[e];
        pp[r] = (T)a.P[e];
        nn[r] = DYN ? (T)a.nres[e] : (T)0;
    }
    for (int it = 0; it < a.iters; ++it) {
#pragma unroll
        for (int r = 0; r < PT; ++r) pointwise_rk4<T, DYN>(a.c, a.inv_c11, pp[r], a.half_dt, x[r], nn[r]);
        fft_regs<T, false, LN, PT>(x, j, a.tw, LL::exchange(mem, x, j, 0, 0));
#pragma unroll
        for (int r = 0; r < PT; ++r) x[r] = cmul<T>(x[r], ph[r]);
        fft_regs<T, true, LN, PT>(x, j, a.tw, LL::exchange(mem, x, j, 0, LL::EX));
#pragma unroll
        for (int r = 0; r < PT; ++r) pointwise_rk4<T, DYN>(a.c, a.inv_c11, pp[r], a.half_dt, x[r], nn[r]);
    }
    if (threadIdx.x >= Q) return;                    // a copy of a short line
#pragma unroll
    for (int r = 0; r < PT; ++r) {
        const int e = j + Q * r;
        a.psi[e] = narrow<S, T>(x[r]);
        if (DYN) a.nres[e] = (S)nn[r];
    }
}

// Middle row pass of a grid of 2048-point rows (8 x 8 x 8 x 4 points), one row a
// workgroup, in registers as k_ssf_row_regs but held to 128 registers and 40 KB of
// LDS, so that four workgroups share a CU: the exchanges go through one buffer,
// swizzled instead of padded, and the twiddles of the two middle stages, which
// are 448 entries of the table, come from LDS beside it (from the table, 28 of a
// thread's 40 loads of 16 bytes, each a miss of an L1 that the fields stream through).
// Per pass at 2048^2, against the row in LDS with all twiddles from the table:
// double precision 62.7 -> 57.4 us, without a reservoir 68.2 -> 65; single-precision
// storage 55.5 -> 50.8 and 62.0 -> 57.9; k_ssf_row_regs, two workgroups a CU, 66 and
// 60.  In a trace of 300 steps in turn a pass takes 46.9 us (40.7), of which VALU issue
// is 27, at 5.0 TB/s (2.9 in single): the transforms, the pointwise part and the
// memory phases overlap only across the four workgroups.
template <typename S, typename T, bool DYN>
__global__ void __launch_bounds__(ROW_NTH, 4) k_ssf_rows2048(const SsfArgs<S, T> a) {
    using C = cplx_t<T>;
    constexpr int LN = ROW_LOG_PTS, NN = 1 << LN, Q = NN / 8;
    static_assert(Q == ROW_NTH, "a thread holds eight points of the row");
    __shared__ C mem[NN];
    __shared__ C twt[7][72];                                    // w^(4 (r+1) k) at [r][k + k / 8], k < 64
    const int j = threadIdx.x;
    const size_t row = (size_t)blockIdx.x << LN;                // rows are contiguous
    cplx_t<S> *const psi = a.psi + row;
    S *const nres = DYN ? a.nres + row : nullptr;
    const S *const P = a.P + row;
    C x[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) x[r] = widen<T, S>(psi[(unsigned)(j + Q * r)]);
    // the fields stay in the storage precision until used (exact conversion;
    // single-precision storage then holds them in half the registers)
    S ps[8], ns[8];
    auto fields = [&] {
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            ps[r] = P[(unsigned)(j + Q * r)];
            ns[r] = DYN ? nres[(unsigned)(j + Q * r)] : (S)0;
        }
    };
    for (int e = j; e < 7 * 64; e += ROW_NTH) twt[e >> 6][(e & 63) + ((e & 63) >> 3)] = a.tw[(((e >> 6) + 1) * (e & 63)) << 2];
    const C w8 = a.tw[NN >> 3];
    const Lds<T, 0> B{mem};
    // the thread's index, opaque: the stages' addresses, equal in both
    // transforms, would otherwise stay in registers from one to the other
    auto fresh = [&] {
        int v = j;
        asm volatile("" : "+v"(v));
        return v;
    };
    auto ex = [&](int logNs) {
        const int j = fresh(), Ns = 1 << logNs, d = ((j >> logNs) << (logNs + 3)) + (j & (Ns - 1));
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 8; ++r) B[d + r * Ns] = x[r];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 8; ++r) x[r] = B[j + Q * r];
    };
    auto fft = [&](auto inv) {
        constexpr bool INV = decltype(inv)::value;
        const int j = fresh();
        auto turn = [&](int m) {
            const C *w0 = &twt[0][m];
#pragma unroll
            for (int r = 1; r < 8; ++r) {
                C w = w0[72 * (r - 1)];
                if (INV) w.y = -w.y;
                x[r] = cmul<T>(x[r], w);
                if (r == 4) __builtin_amdgcn_sched_barrier(0);      // half the twiddles in registers at once
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        bfly8<T, INV, false>(x, j, 0, LN, a.tw, w8);
        ex(0);
        turn(9 * (j & 7));
        bfly8<T, INV, false>(x, j, 3, LN, a.tw, w8);
        ex(3);
        if (INV) fields();               // in flight under the last two stages
        turn((j & 63) + ((j & 63) >> 3));
        bfly8<T, INV, false>(x, j, 6, LN, a.tw, w8);
        ex(6);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            bfly4<T, INV, true>(x[q], x[q + 2], x[q + 4], x[q + 6], j + Q * q, LN - 2, LN, a.tw);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    fft(std::true_type());
    const unsigned jn = (unsigned)fresh();
    // one point at a time (with their temporaries interleaved, a SIMD would
    // hold half the waves)
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        T nv = (T)ns[r];
        const T pv = (T)ps[r];
        pointwise_rk4<T, DYN>(a.c, a.inv_c11, pv, a.half_dt, x[r], nv);
        pointwise_rk4<T, DYN>(a.c, a.inv_c11, pv, a.half_dt, x[r], nv);
        // the reservoir is final here (the transforms act on psi only)
        if (DYN) nres[jn + Q * r] = (S)nv;
        __builtin_amdgcn_sched_barrier(0);
    }
    fft(std::false_type());
#pragma unroll
    for (int r = 0; r < 8; ++r) psi[(unsigned)(j + Q * r)] = narrow<S, T>(x[r]);
}

// Row pass: rows in registers (fft_regs), as many as fill a wave or one of
// several waves a workgroup; the points' pumping and reservoir are the thread's
// own.  Against whole rows in LDS, 2048 points a workgroup: a step of 64^2 16.6
// -> 6.6 us, 512^2 22.9 -> 13.2, 1024^2 42.0 -> 29.1 (single-precision storage,
// both passes), since 512 rows were 128 workgroups, half the CUs, and every
// stage cost two barriers.  Up to 512^2 a pass is latency: a wave or two a
// SIMD run six stages and 24 to 64 evaluations of the pointwise part.
template <typename S, typename T, bool DYN, int MODE, int LN, int PT>
__global__ void __launch_bounds__((line_threads<LN, PT>)) k_ssf_row_regs(const SsfArgs<S, T> a) {
    using C = cplx_t<T>;
    constexpr int Q = (1 << LN) / PT, L = line_threads<LN, PT> / Q;
    using LL = LineLds<T, LN, PT, L, NLS_SSF_ROW_PAD, false, row_bufs(LN)>;
    __shared__ C mem[LL::MEM];
    const int j = threadIdx.x & (Q - 1), l = threadIdx.x / Q;
    const size_t base = ((size_t)blockIdx.x * L + l) << LN;
    C x[PT];
    T pp[PT], nn[PT];
#pragma unroll
    for (int r = 0; r < PT; ++r) {
        const size_t e = base + j + Q * r;
        x[r] = widen<T, S>(a.psi[e]);
        pp[r] = (T)a.P[e];
        nn[r] = DYN ? (T)a.nres[e] : (T)0;
    }
    if (MODE != ROWS_FIRST) fft_regs<T, true, LN, PT>(x, j, a.tw, LL::exchange(mem, x, j, l, 0));
#pragma unroll
    for (int r = 0; r < PT; ++r) {
        pointwise_rk4<T, DYN>(a.c, a.inv_c11, pp[r], a.half_dt, x[r], nn[r]);
        if (MODE == ROWS_MIDDLE) pointwise_rk4<T, DYN>(a.c, a.inv_c11, pp[r], a.half_dt, x[r], nn[r]);
        if (DYN) a.nres[base + j + Q * r] = (S)nn[r];
    }
    if (MODE != ROWS_LAST) fft_regs<T, false, LN, PT>(x, j, a.tw, LL::exchange(mem, x, j, l, LL::EX));
#pragma unroll
    for (int r = 0; r < PT; ++r) a.psi[base + j + Q * r] = narrow<S, T>(x[r]);
}

// Column pass: L adjacent columns per workgroup, in registers.  Workgroups of
// one XCD take adjacent column blocks (round-robin dispatch), so the lines of
// memory that blocks share are in its L2.  At 2048^2 a pass of 300 in turn takes 38.7
// us (33.8 with single-precision storage), of which VALU issue is 10; its traffic, of
// which two columns write 1.39 times their bytes, is 155 MiB (65), 31 us (13) at the
// rate of a large copy.
template <typename S, typename T, int LN, int PT, int L>
__global__ void __launch_bounds__(((L << LN) / PT)) k_ssf_col_regs(const SsfArgs<S, T> a, int chunk) {
    using C = cplx_t<T>;
    using LL = LineLds<T, LN, PT, L, NLS_SSF_COL_PAD, true, col_bufs(LN)>;
    constexpr int NN = 1 << LN, Q = LL::Q;
    __shared__ C mem[LL::MEM];
    const int blk = (blockIdx.x & 7) * chunk + (blockIdx.x >> 3);
    if (blk >= NN / L) return;
    const int l = threadIdx.x % L, j = threadIdx.x / L, col = blk * L + l;
    C x[PT], ph[PT];
#pragma unroll
    for (int r = 0; r < PT; ++r) {
        x[r] = widen<T, S>(a.psi[(size_t)(j + Q * r) * NN + col]);
        ph[r] = a.ph[j + Q * r];
    }
    const C phc = a.ph[col];
    fft_regs<T, false, LN, PT>(x, j, a.tw, LL::exchange(mem, x, j, l, 0));
#pragma unroll
    for (int r = 0; r < PT; ++r) x[r] = cmul<T>(x[r], cmul<T>(ph[r], phc));
    fft_regs<T, true, LN, PT>(x, j, a.tw, LL::exchange(mem, x, j, l, LL::EX));
#pragma unroll
    for (int r = 0; r < PT; ++r) a.psi[(size_t)(j + Q * r) * NN + col] = narrow<S, T>(x[r]);
}

// The unit complex number (c, s) in T.  In single precision the rounded
// pair has |.|^2 = 1 + O(6e-8), a fixed gain or loss of the mode it
// multiplies on every use; of the pairs within one ulp of (c, s) the one
// closest to the unit circle is taken (|.|^2 - 1 ~ 1e-9), so thousands of
// transforms and phase steps do not drift the mode amplitudes.
template <typename T> __device__ __forceinline__ cplx_t<T> unit_round(double c, double s) {
    if (sizeof(T) == 8) return mk<T>((T)c, (T)s);
    const float c0 = (float)c, s0 = (float)s;
    float bc = c0, bs = s0;
    double best = fabs((double)c0 * c0 + (double)s0 * s0 - 1.0);
    const float cs[3] = {nextafterf(c0, -2.0f), c0, nextafterf(c0, 2.0f)};
    const float ss[3] = {nextafterf(s0, -2.0f), s0, nextafterf(s0, 2.0f)};
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const double e = fabs((double)cs[i] * cs[i] + (double)ss[j] * ss[j] - 1.0);
            if (e < best) { best = e; bc = cs[i]; bs = ss[j]; }
        }
    return mk<T>((T)bc, (T)bs);
}

// Twiddles and phase, double precision, rounded to T on the unit circle
// (unit_round); the phase carries the transform's 1/N (a power of two).
template <typename T>
__global__ void k_ssf_tables(int N, double dx, double dt, double scale, cplx_t<T> *tw, cplx_t<T> *ph) {
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= N) return;
    double s, c;
    sincospi(2.0 * (double)m / (double)N, &s, &c);
    tw[m] = unit_round<T>(c, -s);
    const int f = m < N / 2 ? m : m - N;                 // FFT frequency order
    const double k = 2.0 * M_PI * (double)f / ((double)N * dx);
    double ps, pc;
    sincos(k * k * dt, &ps, &pc);
    const cplx_t<T> u = unit_round<T>(pc, -ps);
    ph[m] = mk<T>(u.x * (T)scale, u.y * (T)scale);
}

static size_t align256s(size_t b) { return (b + 255) & ~(size_t)255; }

static int log2_exact(int n) {
    int l = 0;
    while ((1 << l) < n) ++l;
    return (1 << l) == n ? l : -1;
}

// A 2-D grid of 2^LN points a side.
template <typename S, typename T, bool DYN, int LN>
static int ssf_run_2d(const SsfArgs<S, T> &a, int iters, hipStream_t s) {
    constexpr int N = 1 << LN, RP = row_pt(LN, DYN), RT = line_threads<LN, RP>;
    constexpr int CP = col_pt(LN), L = col_lines(LN, sizeof(S) == 8), chunk = (N / L + 7) / 8;
    const dim3 rows(N / (RP * RT / N)), rth(RT), cols(8 * chunk), cth(L * N / CP);
    hipLaunchKernelGGL((k_ssf_row_regs<S, T, DYN, ROWS_FIRST, LN, RP>), rows, rth, 0, s, a);
    for (int it = 0; it < iters; ++it) {
        hipLaunchKernelGGL((k_ssf_col_regs<S, T, LN, CP, L>), cols, cth, 0, s, a, chunk);
        if (it + 1 == iters)
            hipLaunchKernelGGL((k_ssf_row_regs<S, T, DYN, ROWS_LAST, LN, RP>), rows, rth, 0, s, a);
        else if constexpr (LN == ROW_LOG_PTS)
            hipLaunchKernelGGL((k_ssf_rows2048<S, T, DYN>), dim3(N), dim3(ROW_NTH), 0, s, a);
        else
            hipLaunchKernelGGL((k_ssf_row_regs<S, T, DYN, ROWS_MIDDLE, LN, RP>), rows, rth, 0, s, a);
    }
    return hip_check(hipGetLastError(), "ssf launch");
}

template <typename S, bool DYN>
static int ssf_run(const nls_problem *p, int iters, const S *P, cplx_t<S> *psi, S *nres, char *ws, hipStream_t s) {
    using T = double;                 // arithmetic, LDS and tables
    using C = cplx_t<T>;
    const int N = p->n, logN = log2_exact(N);
    C *tw = (C *)ws, *ph = (C *)(ws + align256s(N * sizeof(C)));
    // 1/N per inverse transform: once in 1-D, once per axis (folded into the
    // product ph[ky] * ph[kx]) in 2-D
    hipLaunchKernelGGL(k_ssf_tables<T>, dim3((N + 255) / 256), dim3(256), 0, s, N, p->dx, p->dt, 1.0 / N, tw, ph);
    SsfArgs<S, T> a;
    memset(&a, 0, sizeof a);
    a.half_dt = (T)(0.5 * p->dt);
    a.c = make_coeffs<T>(p->coeffs);
    a.inv_c11 = DYN ? (T)(1.0 / p->coeffs[10]) : (T)0;
    a.psi = psi; a.nres = nres; a.P = P; a.tw = tw; a.ph = ph;
    if (p->dim == 1) {
        a.iters = iters;
        switch (logN) {
#define NLS_CASE(LN)                                                                                       \
    case LN:                                                                                               \
        hipLaunchKernelGGL((k_ssf_line<S, T, DYN, LN, line_pt(LN)>), dim3(1),                              \
                           dim3(line_threads<LN, line_pt(LN)>), 0, s, a);                                  \
        return hip_check(hipGetLastError(), "ssf line launch");
            NLS_CASE(4) NLS_CASE(5) NLS_CASE(6) NLS_CASE(7) NLS_CASE(8)
            NLS_CASE(9) NLS_CASE(10) NLS_CASE(11) NLS_CASE(12)
#undef NLS_CASE
        }
    } else {
        switch (logN) {
        case 4: return ssf_run_2d<S, T, DYN, 4>(a, iters, s);
        case 5: return ssf_run_2d<S, T, DYN, 5>(a, iters, s);
        case 6: return ssf_run_2d<S, T, DYN, 6>(a, iters, s);
        case 7: return ssf_run_2d<S, T, DYN, 7>(a, iters, s);
        case 8: return ssf_run_2d<S, T, DYN, 8>(a, iters, s);
        case 9: return ssf_run_2d<S, T, DYN, 9>(a, iters, s);
        case 10: return ssf_run_2d<S, T, DYN, 10>(a, iters, s);
        case 11: return ssf_run_2d<S, T, DYN, 11>(a, iters, s);
        }
    }
    return fail(NLS_EUNSUPPORTED, "no split-step kernel for %d points a side", N);
}

// ---------------------------------------------------------------------------
// Kinetic energy with the scheme's own (spectral) operator:
//   -Re<psi, L psi> = (1 / N^d) sum_k |k|^2 |psi_hat(k)|^2
// (psi_hat the unnormalised DFT, N^d grid points).  In 2-D it is taken from
// 1-D transforms only: by Parseval along the other axis,
//   sum_{kx,ky} kx^2 |psi_hat|^2 = N sum_rows sum_kx kx^2 |DFT_x(row)|^2
// and likewise for ky over the columns, so
//   -Re<psi, L psi> = (1/N) (sum over rows + sum over columns)
// with no 2-D transform and no intermediate field.  Each workgroup reduces
// its lines' sum of k^2 |DFT|^2 in a fixed tree into one partial; one
// workgroup adds the partials in order.  Double precision throughout.

// sum over the workgroup's threads of v, in a fixed order, into *out
// (thread 0); sh: NTH doubles of LDS, free on entry
template <int NTH> __device__ __forceinline__ void fixed_block_sum(double *sh, double v, double *out) {
    const int t = threadIdx.x;
    sh[t] = v;
    __syncthreads();
#pragma unroll
    for (int s = NTH / 2; s > 0; s >>= 1) {
        if (t < s) sh[t] += sh[t + s];
        __syncthreads();
    }
    if (t == 0) *out = sh[0];
}

// k_m^2 |v|^2 for FFT output index m of a length-N transform (frequency m,
// or m - N past N/2, as the phase table), k_m = k0 * frequency
__device__ __forceinline__ double k2_abs2(int m, int N, double k0, cplx_t<double> v) {
    const int f = m < N / 2 ? m : m - N;
    const double k = k0 * (double)f;
    return k * k * (v.x * v.x + v.y * v.y);
}

template <typename S>
__global__ void __launch_bounds__(ROW_NTH) k_ssf_kin_rows(const cplx_t<S> *psi, int logN, const cplx_t<double> *tw,
                                                          double k0, double *part) {
    using C = cplx_t<double>;
    constexpr int PPT = ROW_PTS / ROW_NTH;
    __shared__ C buf_mem[lds_padded(ROW_PTS, NLS_SSF_ROW_PAD)];
    const Lds<double, NLS_SSF_ROW_PAD> buf{buf_mem};
    const int N = 1 << logN;
    const int logL = lines_per_wg(logN, ROW_LOG_PTS);
    const int pts = 1 << (logL + logN);
    const size_t base = (size_t)blockIdx.x << (logL + logN);
#pragma unroll
    for (int q = 0; q < PPT; ++q) {
        const int idx = threadIdx.x + ROW_NTH * q;
        if (idx < pts) buf[idx] = widen<double, S>(psi[base + idx]);
    }
    __syncthreads();
    lds_fft<double, false, false, ROW_PTS, ROW_NTH>(buf, logN, logL, N, 1, tw);
    double v = 0.0;
#pragma unroll
    for (int q = 0; q < PPT; ++q) {
        const int idx = threadIdx.x + ROW_NTH * q;
        if (idx < pts) v += k2_abs2(idx & (N - 1), N, k0, buf[idx]);
    }
    __syncthreads();
    fixed_block_sum<ROW_NTH>((double *)buf_mem, v, part + blockIdx.x);
}

constexpr int COL_LOG_L = 1, COL_PTS = 4096, COL_NTH = 512;      // two columns per workgroup
template <typename S>
__global__ void __launch_bounds__(COL_NTH) k_ssf_kin_cols(const cplx_t<S> *psi, int logN,
                                                                         const cplx_t<double> *tw, double k0,
                                                                         double *part) {
    using C = cplx_t<double>;
    constexpr int PPT = COL_PTS / COL_NTH;
    __shared__ C buf_mem[lds_padded(COL_PTS, NLS_SSF_COL_PAD)];
    const Lds<double, NLS_SSF_COL_PAD> buf{buf_mem};
    const int N = 1 << logN;
    const int logL = COL_LOG_L < logN ? COL_LOG_L : logN;
    const int L = 1 << logL, pts = L << logN;
    const int col0 = blockIdx.x << logL;
#pragma unroll
    for (int q = 0; q < PPT; ++q) {
        const int idx = threadIdx.x + COL_NTH * q;
        if (idx < pts) buf[idx] = widen<double, S>(psi[(size_t)(idx >> logL) * N + col0 + (idx & (L - 1))]);
    }
    __syncthreads();
    lds_fft<double, false, true, COL_PTS, COL_NTH>(buf, logN, logL, 1, L, tw);
    double v = 0.0;
#pragma unroll
    for (int q = 0; q < PPT; ++q) {
        const int idx = threadIdx.x + COL_NTH * q;
        if (idx < pts) v += k2_abs2(idx >> logL, N, k0, buf[idx]);
    }
    __syncthreads();
    fixed_block_sum<COL_NTH>((double *)buf_mem, v, part + blockIdx.x);
}

// 1-D: one workgroup, the whole line (n <= 4096)
constexpr int LINE_PTS = 4096, LINE_NTH = 512;
template <typename S>
__global__ void __launch_bounds__(LINE_NTH) k_ssf_kin_line(const cplx_t<S> *psi, int logN,
                                                                          const cplx_t<double> *tw, double k0,
                                                                          double *part) {
    using C = cplx_t<double>;
    constexpr int PPT = LINE_PTS / LINE_NTH;
    __shared__ C buf_mem[lds_padded(LINE_PTS, NLS_SSF_LINE_PAD)];
    const Lds<double, NLS_SSF_LINE_PAD> buf{buf_mem};
    const int N = 1 << logN;
#pragma unroll
    for (int q = 0; q < PPT; ++q) {
        const int idx = threadIdx.x + LINE_NTH * q;
        if (idx < N) buf[idx] = widen<double, S>(psi[idx]);
    }
    __syncthreads();
    lds_fft<double, false, false, LINE_PTS, LINE_NTH>(buf, logN, 0, N, 1, tw);
    double v = 0.0;
#pragma unroll
    for (int q = 0; q < PPT; ++q) {
        const int idx = threadIdx.x + LINE_NTH * q;
        if (idx < N) v += k2_abs2(idx, N, k0, buf[idx]);
    }
    __syncthreads();
    fixed_block_sum<LINE_NTH>((double *)buf_mem, v, part);
}

// partials 0 .. nb-1 added in order by one workgroup of 256 threads: thread
// t adds t, t + 256, ...; then a fixed tree
__global__ void __launch_bounds__(256) k_ssf_kin_sum(int nb, const double *part, double *out) {
    __shared__ double sh[256];
    double v = 0.0;
    for (int b = threadIdx.x; b < nb; b += 256) v += part[b];
    fixed_block_sum<256>(sh, v, out);
}

size_t ssf_kinetic_scratch_bytes(const nls_problem *p) {
    // twiddles and phases (the table kernel writes both), the partials, the sum
    return 2 * align256s((size_t)p->n * 16) + align256s(((size_t)2 * p->n + 1) * sizeof(double));
}

int ssf_kinetic(const nls_problem *p, const void *psi, void *scratch, double *dev_sum, hipStream_t s) {
    int rc = ssf_check(p);
    if (rc) return rc;
    using C = cplx_t<double>;
    const int N = p->n, logN = log2_exact(N);
    char *ws = (char *)scratch;
    C *tw = (C *)ws, *ph = (C *)(ws + align256s((size_t)N * sizeof(C)));
    double *part = (double *)(ws + 2 * align256s((size_t)N * sizeof(C)));
    hipLaunchKernelGGL(k_ssf_tables<double>, dim3((N + 255) / 256), dim3(256), 0, s, N, p->dx, p->dt, 1.0, tw, ph);
    const double k0 = 2.0 * M_PI / ((double)N * p->dx);
    const bool f64 = p->dtype == NLS_F64;
    int nb;
    if (p->dim == 1) {
        nb = 1;
        if (f64) hipLaunchKernelGGL(k_ssf_kin_line<double>, dim3(1), dim3(LINE_NTH), 0, s,
                                    (const double2 *)psi, logN, tw, k0, part);
        else hipLaunchKernelGGL(k_ssf_kin_line<float>, dim3(1), dim3(LINE_NTH), 0, s,
                                (const float2 *)psi, logN, tw, k0, part);
    } else {
        const int rblocks = N >> lines_per_wg(logN, ROW_LOG_PTS);
        const int cblocks = N >> (COL_LOG_L < logN ? COL_LOG_L : logN);
        nb = rblocks + cblocks;
        if (f64) {
            hipLaunchKernelGGL(k_ssf_kin_rows<double>, dim3(rblocks), dim3(ROW_NTH), 0, s, (const double2 *)psi,
                               logN, tw, k0, part);
            hipLaunchKernelGGL(k_ssf_kin_cols<double>, dim3(cblocks), dim3(COL_NTH), 0, s,
                               (const double2 *)psi, logN, tw, k0, part + rblocks);
        } else {
            hipLaunchKernelGGL(k_ssf_kin_rows<float>, dim3(rblocks), dim3(ROW_NTH), 0, s, (const float2 *)psi,
                               logN, tw, k0, part);
            hipLaunchKernelGGL(k_ssf_kin_cols<float>, dim3(cblocks), dim3(COL_NTH), 0, s,
                               (const float2 *)psi, logN, tw, k0, part + rblocks);
        }
    }
    hipLaunchKernelGGL(k_ssf_kin_sum, dim3(1), dim3(256), 0, s, nb, part, dev_sum);
    return hip_check(hipGetLastError(), "ssf kinetic energy launch");
}

size_t ssf_workspace_bytes(const nls_problem *p) {
    return 2 * align256s((size_t)p->n * 16);          // twiddles and phases, double precision
}

int ssf_check(const nls_problem *p) {
    const int l = log2_exact(p->n);
    const int maxn = p->dim == 1 ? 4096 : 2048;
    if (l < 0 || p->n < 16 || p->n > maxn)
        return fail(NLS_EUNSUPPORTED, "split-step Fourier needs n a power of two in [16, %d] (got %d)", maxn, p->n);
    return NLS_OK;
}

int ssf_advance(const nls_problem *p, int iters, const void *pumping, void *psi, void *nres, void *ws,
                hipStream_t s) {
    int rc = ssf_check(p);
    if (rc) return rc;
    const bool dyn = p->coeffs[10] != 0.0;
    if (p->dtype == NLS_F64) {
        if (dyn) return ssf_run<double, true>(p, iters, (const double *)pumping, (double2 *)psi, (double *)nres, (char *)ws, s);
        return ssf_run<double, false>(p, iters, (const double *)pumping, (double2 *)psi, nullptr, (char *)ws, s);
    }
    if (dyn) return ssf_run<float, true>(p, iters, (const float *)pumping, (float2 *)psi, (float *)nres, (char *)ws, s);
    return ssf_run<float, false>(p, iters, (const float *)pumping, (float2 *)psi, nullptr, (char *)ws, s);
}

}  // namespace nls
