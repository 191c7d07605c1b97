// nls_march.h -- members of a launch (batches and plain grids) and the launch
// interfaces of the marching kernel (nls_march.hip) and of the small grids'
// kernels (nls_small.hip).
#pragma once
#include "nls_core.h"

namespace nls {

// What rounding leaves of GridCoeffs' dtw6 and dt6 (beside grid_ring1_from).
template <typename T> struct StepRest {};
template <> struct StepRest<float> {
    float lo[2];
};
template <typename T> struct MemberDev : StepRest<T> {
    int n, steps;
    long long off;          // first point of the member in the packed arrays
    long long tab;          // first entry of its radial table (1-D ref), else -1
    int id, pad;            // the member's index in the caller's batch (observables go to out[4 id ..])
    double dV;              // volume element of its observables
    T dt;
    T w0, w1, w2, w3;       // Cartesian second-derivative weights
    Coeffs<T> c;
    GridCoeffs<T> g;        // of the fused 2-D step
};

struct TileDesc {
    int m, x0, y0, pad;
};

// A piece of a member: columns x0 .. x0 + wd - 1, rows y0 .. y0 + L - 1 of each
// of `subs` row ranges of E rows side by side in the workgroup (range s starts
// at row s E; rows past the grid's end are dropped).
struct StripDesc {
    int m, x0, wd, y0, L, E, subs;
};

template <typename T> struct MarchArgs {
    const MemberDev<T> *mem;
    const StripDesc *strips;
    const int *first;                    // the workgroups' pieces
    int groups, chunk;                   // workgroups; an eighth of them, rounded up
    int it;
    const cplx_t<T> *u; const T *un;     // state at the start of the step
    cplx_t<T> *uo; T *uno;               // state at its end
    const T *P;
    // one grid (n > 256) instead of a member table: grid_nx > 0 strips of
    // grid_wd columns across, pieces of grid_L rows
    int grid_nx, grid_wd, grid_L;
    MemberDev<T> grid;
};

// full: every strip spans its member's whole rows (64 <= n <= 256 columns,
// up to 256 / n pieces side by side); else strips of at most 240 columns of
// members of n > 256.  percu: workgroups a CU is to hold at once, at most.
template <typename T> void launch_march(bool dyn, bool full, int percu, const MarchArgs<T> &a, hipStream_t s);

template <typename T> struct ResidentArgs {
    const MemberDev<T> *mem;
    int iters;
    const T *wtab;
    cplx_t<T> *psi;
    T *nres;
    const T *P;
};

// One workgroup per member of a batch of 2-D grids of up to 64 x 64, all steps
// of a call in one launch (nls_small.hip; not double precision of order 7).
// n: the largest grid's side.
template <typename T>
void launch_resident_2d(int order, int bc, bool dyn, int count, int n, const ResidentArgs<T> &r, hipStream_t s);

// Several steps of one small grid per launch (nls_small.hip).
template <typename T> struct MultiArgs {
    int ntx;                             // tiles across
    const cplx_t<T> *u; const T *un;
    cplx_t<T> *uo; T *uno;
    const T *P;
    int steps;                           // 0, or the steps of this launch, at most multi_steps, with
                                         // grid_ring1_from's sums (single precision, n <= 64)
    MemberDev<T> grid;
};
// Steps a launch makes on an n x n grid (0: not such a grid).
int multi_steps(int n, int order, int cus);
template <typename T>
void launch_multi(int order, int bc, bool dyn, MultiArgs<T> a, int cus, hipStream_t s);

}  // namespace nls
