// nls_rk4.h -- launch interface of the single-instance RK4 stage kernels.
#pragma once
#include "nls_stage.h"

namespace nls {

template <typename T>
void launch_rk4_stage(int dim, int order, int bc, bool dyn, const StageArgs<T> &a, hipStream_t s);

template <typename T>
void launch_radial_table(int n, int order, double h, T *wtab, hipStream_t s);

// A state of N points that ended in the workspace, back into the caller's arrays
// (srcn, dstn: reservoir, NULL without).  Up to COPY_POINTS one kernel moves both
// fields: behind one step of a 64^2 grid a call with a reservoir takes 9 us with it
// and 12.5 with two copies of the runtime's, whose rate larger states keep.
constexpr size_t COPY_POINTS = 65536;
template <typename T>
int copy_state(size_t N, const cplx_t<T> *src, cplx_t<T> *dst, const T *srcn, T *dstn, hipStream_t s);

// Tile height (4, 8, 16 or 32 rows) of the single-instance 2-D stage kernels, per
// dtype (0 = f32, 1 = f64).
int set_stage_tile(int dtype, int ty);
int get_stage_tile(int dtype);

}  // namespace nls
