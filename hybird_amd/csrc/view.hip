// Device side of the host views: the state packed into the views' node-major or element-major layout (and host
// inputs unpacked into planes). Bound by the copy to or from pageable host memory that follows (10 to 17 GB/s with
// the pages' first touch; the kernels move the same bytes at HBM rate). Packing on the host read every plane back
// and went through them with a stride per node. Before and after, 256^3 nodes: velocity 296 -> 38 ms, density
// 273 -> 13, types 38 -> 1.5, populations 522 -> 253 (velocity 25, with the
// pages of the caller's buffer made present meanwhile); 128^3 nodes: populations in 80 -> 12, a force field 3 to 7 -> 1.1;
// 7,728 elements: e_x 2 -> 0.1 ms.
//
// One thread per output value, so the wide side of every access is coalesced: consecutive threads write
// consecutive values and read 64 / W consecutive nodes of each plane.
#include <hip/hip_runtime.h>

#include "common.h"
#include "view_kernels.h"

namespace hyb {

namespace {

constexpr int VIEW_BLOCK = 256;
constexpr unsigned VIEW_GRID = 8192;

unsigned grid_for(size_t n) {
    const size_t g = (n + VIEW_BLOCK - 1) / VIEW_BLOCK;
    return (unsigned)(g < VIEW_GRID ? g : VIEW_GRID);
}

#define VIEW_FOR(t, n) \
    for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < (n); t += (size_t)gridDim.x * blockDim.x)

__device__ __forceinline__ bool active(const uint32_t* link, size_t i) { return (link[i] & LINK_ACTIVE) != 0u; }

template <int W>
__global__ void __launch_bounds__(VIEW_BLOCK) k_view_planes(const double* __restrict__ planes, size_t stride,
                                                            const uint32_t* __restrict__ link, double* __restrict__ out,
                                                            size_t i0, size_t n) {
    VIEW_FOR(t, n * W) {
        const size_t i = i0 + t / W, k = t % W;
        out[t] = active(link, i) ? planes[k * stride + i] : (double)NAN;
    }
}

template <typename T, bool SHIFT>
__global__ void __launch_bounds__(VIEW_BLOCK) k_view_pops(const T* __restrict__ f, size_t PS,
                                                          const uint32_t* __restrict__ link, double* __restrict__ out,
                                                          size_t i0, size_t n) {
#pragma clang fp contract(off)
    VIEW_FOR(t, n * 19) {
        const size_t i = i0 + t / 19;
        const int j = (int)(t % 19);
        double v = (double)NAN;
        if (active(link, i)) {
            v = (double)f[(size_t)j * PS + i];
            if (SHIFT) v = v + wgt(j);
        }
        out[t] = v;
    }
}

template <typename T>
__global__ void __launch_bounds__(VIEW_BLOCK) k_view_scalar(bool split, const double* __restrict__ a, double constA,
                                                            const T* __restrict__ b, double constB,
                                                            const uint32_t* __restrict__ link, double* __restrict__ out,
                                                            size_t i0, size_t n) {
    VIEW_FOR(t, n) {
        const size_t i = i0 + t;
        const uint32_t lw = link[i];
        double v = (double)NAN;
        if (lw & LINK_ACTIVE) {
            if (split && (lw & LINK_INTERFACE)) v = a ? a[i] : constA;
            else v = b ? (double)b[i] : constB;
        }
        out[t] = v;
    }
}

__global__ void __launch_bounds__(VIEW_BLOCK) k_view_owner(const uint32_t* __restrict__ solid,
                                                           const uint32_t* __restrict__ link, uint32_t ctag,
                                                           uint32_t* __restrict__ index, uint8_t* __restrict__ flag,
                                                           size_t i0, size_t n) {
    VIEW_FOR(t, n) {
        const size_t i = i0 + t;
        const uint32_t so = solid[i];
        const uint32_t s = active(link, i) && (so >> SOLID_SLOT_BITS) == ctag ? (so & SOLID_SLOT_MASK) : 0u;
        if (index) index[t] = s ? s - 1u : 0xFFFFFFFFu;
        else flag[t] = s ? 1 : 0;
    }
}

__global__ void __launch_bounds__(VIEW_BLOCK) k_view_rows(const double* __restrict__ el, int E, int first, int count,
                                                          double* __restrict__ out) {
    VIEW_FOR(t, (size_t)E * count) out[t] = el[(size_t)(first + (int)(t % count)) * E + t / count];
}

template <typename T, bool SHIFT>
__global__ void __launch_bounds__(VIEW_BLOCK) k_fill_pops(const double* __restrict__ in, T* __restrict__ f, size_t PS,
                                                          const uint32_t* __restrict__ link, size_t i0, size_t n) {
#pragma clang fp contract(off)
    VIEW_FOR(t, n * 19) {
        const size_t i = i0 + t / 19;
        const int j = (int)(t % 19);
        const double v = in[t];
        f[(size_t)j * PS + i] = active(link, i) ? (T)(SHIFT ? v - wgt(j) : v) : (T)0;
    }
}

__global__ void __launch_bounds__(VIEW_BLOCK) k_fill_force(const float* __restrict__ in, float* __restrict__ planes,
                                                           size_t N, size_t i0, size_t n) {
    VIEW_FOR(t, n * 3) planes[(t % 3) * N + i0 + t / 3] = in[t];
}

}  // namespace

void launch_view_planes(const double* planes, size_t stride, int W, const uint32_t* link, double* out, size_t i0,
                        size_t i1, hipStream_t s) {
    const unsigned g = grid_for((i1 - i0) * (size_t)W);
    if (W == 1) k_view_planes<1><<<g, VIEW_BLOCK, 0, s>>>(planes, stride, link, out, i0, i1 - i0);
    else k_view_planes<3><<<g, VIEW_BLOCK, 0, s>>>(planes, stride, link, out, i0, i1 - i0);
}

void launch_view_pops(Prec prec, const void* f, size_t PS, const uint32_t* link, double* out, size_t i0, size_t i1,
                      hipStream_t s) {
    const unsigned g = grid_for((i1 - i0) * 19);
    if (prec == Prec::F64) k_view_pops<double, false><<<g, VIEW_BLOCK, 0, s>>>((const double*)f, PS, link, out, i0, i1 - i0);
    else k_view_pops<float, true><<<g, VIEW_BLOCK, 0, s>>>((const float*)f, PS, link, out, i0, i1 - i0);
}

void launch_view_scalar(bool split, const double* a, double constA, const void* b, Prec bPrec, double constB,
                        const uint32_t* link, double* out, size_t i0, size_t i1, hipStream_t s) {
    const unsigned g = grid_for(i1 - i0);
    if (bPrec == Prec::F64)
        k_view_scalar<double><<<g, VIEW_BLOCK, 0, s>>>(split, a, constA, (const double*)b, constB, link, out, i0, i1 - i0);
    else
        k_view_scalar<float><<<g, VIEW_BLOCK, 0, s>>>(split, a, constA, (const float*)b, constB, link, out, i0, i1 - i0);
}

void launch_view_owner(const uint32_t* solid, const uint32_t* link, uint32_t ctag, bool index, void* out, size_t i0,
                       size_t i1, hipStream_t s) {
    k_view_owner<<<grid_for(i1 - i0), VIEW_BLOCK, 0, s>>>(solid, link, ctag, index ? (uint32_t*)out : nullptr,
                                                          (uint8_t*)out, i0, i1 - i0);
}

void launch_view_rows(const double* el, int E, int first, int count, double* out, hipStream_t s) {
    if (E > 0) k_view_rows<<<grid_for((size_t)E * count), VIEW_BLOCK, 0, s>>>(el, E, first, count, out);
}

void launch_fill_pops(Prec prec, const double* in, void* f, size_t PS, const uint32_t* link, size_t i0, size_t i1,
                      hipStream_t s) {
    const unsigned g = grid_for((i1 - i0) * 19);
    if (prec == Prec::F64) k_fill_pops<double, false><<<g, VIEW_BLOCK, 0, s>>>(in, (double*)f, PS, link, i0, i1 - i0);
    else k_fill_pops<float, true><<<g, VIEW_BLOCK, 0, s>>>(in, (float*)f, PS, link, i0, i1 - i0);
}

void launch_fill_force(const float* in, float* planes, size_t N, size_t i0, size_t i1, hipStream_t s) {
    k_fill_force<<<grid_for((i1 - i0) * 3), VIEW_BLOCK, 0, s>>>(in, planes, N, i0, i1 - i0);
}

}  // namespace hyb
