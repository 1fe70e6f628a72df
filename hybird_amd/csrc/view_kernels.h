// Host-side launch interface of the view kernels (view.hip): device state packed into the layout of the host
// views (and back), so that a view is one kernel and one copy.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.h"
#include "lb_kernels.h"

namespace hyb {

// out[(i - i0) * W + k] = plane k of node i, NaN on inactive nodes, i0 <= i < i1; W = 1 or 3 (FP64 planes of
// stride `stride`).
void launch_view_planes(const double* planes, size_t stride, int W, const uint32_t* link, double* out, size_t i0,
                        size_t i1, hipStream_t s);
// The same with the 19 populations (FP32: the stored deviation plus the weight).
void launch_view_pops(Prec prec, const void* f, size_t PS, const uint32_t* link, double* out, size_t i0, size_t i1,
                      hipStream_t s);
// One scalar per node: interface nodes (split) take a[i] (nullptr: constA), the other active nodes b[i] (nullptr:
// constB; FP32 when bPrec says so), inactive nodes NaN.
void launch_view_scalar(bool split, const double* a, double constA, const void* b, Prec bPrec, double constB, const uint32_t* link,
                        double* out, size_t i0, size_t i1, hipStream_t s);
// Particle flag (bytes) or particle index of active nodes owned in coupling step ctag.
void launch_view_owner(const uint32_t* solid, const uint32_t* link, uint32_t ctag, bool index, void* out, size_t i0,
                       size_t i1, hipStream_t s);
// out[e * count + k] = el[(first + k) * E + e]
void launch_view_rows(const double* el, int E, int first, int count, double* out, hipStream_t s);
// Node-major host input to planes: populations (inactive nodes 0) and a force field.
void launch_fill_pops(Prec prec, const double* in, void* f, size_t PS, const uint32_t* link, size_t i0, size_t i1,
                      hipStream_t s);
void launch_fill_force(const float* in, float* planes, size_t N, size_t i0, size_t i1, hipStream_t s);

}  // namespace hyb
