// Discrete-element kernels for gfx950.
//
// These kernels run beds with more elements than the whole-step kernel (dem_run.hip) can hold on the device at
// once, and steps that save MercuryDPM statistics. One DEM sub-step (DEM.cpp:331-376) is then three launches on the
// handle's stream (their device code is in dem_substep.h):
//  1. k_dem_rebuild (one workgroup): evalMaxDisp and, when the displacement
//     trigger fires, the whole neighbour rebuild of DEM.cpp:1369-1513 —
//     periodic shift, ghosts, linked-cell table, the 14-cell pair list and the
//     near-wall list — reproducing the reference's cell index (vector.cpp:147-149)
//     and unsigned stencil wrap, in the reference's pair order. It also builds a
//     per-particle list of the pairs each particle takes part in.
//  2. k_dem_pairs: one thread per pair evaluates the contact (DEM.cpp:1801-1900,
//     2138-2222) and writes each particle's signed increments into that
//     particle's slot of the pair (and, on saving sub-steps, its statistics).
//  3. k_dem_gather: per element, the increments in pair-list order (the same
//     order as the reference's sequential loop, so no atomics and bit-identical
//     sums; an element of several spheres merges its particles' lists by pair
//     index), the wall, object and cylinder contacts of its particles,
//     Newton-Euler (DEM.cpp:1149-1181), the Gear corrector (elmt.cpp:179-254),
//     the particle update (elmt.cpp:261-290) and the predictor (elmt.cpp:139-177)
//     of the next sub-step. An initial predictor runs once after initialisation.
// The corrector keeps the predicted copies it has just used until the new
// prediction overwrites them, so partner reads in k_dem_pairs always see the
// predicted state of the current sub-step.
//
// Single-sphere elements are their own particle (particle i = element i, the
// element arrays serve both). With multi-sphere elements (DEMParams::clumps)
// particles have their own state arrays, refreshed from their element after the
// corrector and after the predictor.
#include <hip/hip_runtime.h>

#include "common.h"
#include "dem_device.h"
#include "dem_kernels.h"
#include "dem_substep.h"
#include "hybird_amd.h"
#include "lattice.h"

namespace hyb {

namespace {

constexpr int RB = 1024;  // rebuild workgroup size

__global__ void __launch_bounds__(RB) k_dem_rebuild(DEMParams p, DEMBuffers b, int force) {
    rebuild_by_one<RB>(p, b, force);
}

// One thread per neighbour pair (grid-stride).
template <bool SP, bool CL>
__global__ void __launch_bounds__(256) k_dem_pairs(DEMParams p, DEMBuffers b) {
    const El E{b.el, p.E};
    if (b.st->error) return;
    const int T = b.st->nPairs;
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < T; k += gridDim.x * blockDim.x) eval_pair<SP, CL>(p, b, E, k);
}

__global__ void __launch_bounds__(64) k_dem_predict(DEMParams p, DEMBuffers b) {
#pragma clang fp contract(off)
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    const El E{b.el, p.E};
    double v2 = 0.0;
    if (e < p.E) {
        V3 x[6], w[6];
        Q4 q[6];
        for (int k = 0; k < 6; ++k) { x[k] = E.v3(EF_X + 3 * k, e); q[k] = E.q4(EF_Q + 4 * k, e); w[k] = E.v3(EF_W + 3 * k, e); }
        if (p.clumps) predict_elem<true>(E, p, b, e, x, q, w);
        else predict_elem<false>(E, p, b, e, x, q, w);
        v2 = x[1].norm2();
    }
    vmax_add(b, wave_max(v2));
}

template <bool SP, bool CL>
__global__ void __launch_bounds__(64) k_dem_gather(DEMParams p, DEMBuffers b) {
    if (b.st->error) return;
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    const double v2 = e < p.E ? gather_elem<SP, CL>(p, b, e) : 0.0;
    vmax_add(b, wave_max(v2));
}

// Element hydrodynamic force and torque (LB.cpp:1897-1918): the run sums the
// collision appended for the slots of the element's particles and their ghosts,
// added exactly (fixed point, so the result does not depend on the order of the
// appends), then scaled to physical units. One wavefront per element, one
// element per workgroup; lane l accumulates component l % 7 of every ninth
// entry (l / 7 < 9), so that each entry component is split once; the nine
// partial sums per component are then added through LDS. The lists are emptied
// for the next LB step. (Four elements per workgroup, each wavefront on its own
// LDS rows, gave results that varied from run to run for a few elements past
// the first 1024 on this hardware; one wavefront per workgroup does not.)
constexpr int COMBINE_BLOCK = 64;
constexpr int COMBINE_ROWS = 9;  // entries per pass (9 x 7 components = 63 lanes)
__global__ void __launch_bounds__(COMBINE_BLOCK) k_dem_hydro_combine(DEMParams p, DEMBuffers b, HydroSink hs, Units u) {
#pragma clang fp contract(off)
    __shared__ long long red[COMBINE_BLOCK / 64][64][4];
    __shared__ double val[COMBINE_BLOCK / 64][7];
    const int lane = (int)(threadIdx.x & 63);
    const int w = (int)(threadIdx.x >> 6);
    const int e = (int)((blockIdx.x * (unsigned)COMBINE_BLOCK + threadIdx.x) >> 6);
    if (e >= p.E) return;  // whole wavefronts
    const El E{b.el, p.E};
    const int ilo = p.clumps ? b.efirst[e] : e, ihi = p.clumps ? b.efirst[e + 1] : e + 1;
    const int q = lane % 7, j = lane / 7;
    long long acc[4] = {0, 0, 0, 0};
    for (int i = ilo; i < ihi; ++i)
    for (int k = -1, ng = b.ghostOfCount[i] < 8 ? b.ghostOfCount[i] : 8; k < ng; ++k) {
        const uint32_t slot = k < 0 ? (uint32_t)i : (uint32_t)b.ghostOf[i * 8 + k];
        const uint32_t cnt = hs.count[slot];
        const uint32_t n = cnt < hs.cap ? cnt : hs.cap;
        const HydroSeg* L = hs.segs + (size_t)slot * hs.cap;
        if (j < COMBINE_ROWS) {
            constexpr uint32_t AHEAD = 4;  // loads issued before the first split
            for (uint32_t i = (uint32_t)j; i < n; i += AHEAD * COMBINE_ROWS) {
                double v[AHEAD];
#pragma unroll
                for (uint32_t a = 0; a < AHEAD; ++a) {
                    const uint32_t ia = i + a * COMBINE_ROWS;
                    v[a] = ia < n ? L[ia].s[q] : 0.0;
                }
#pragma unroll
                for (uint32_t a = 0; a < AHEAD; ++a) exact_local(acc, v[a]);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) red[w][lane][i] = acc[i];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // every lane has read the counts above; empty the lists for the next step
    for (int i = ilo; i < ihi; ++i) {
        const int ng = b.ghostOfCount[i] < 8 ? b.ghostOfCount[i] : 8;
        if (lane <= ng) hs.count[lane == 0 ? (uint32_t)i : (uint32_t)b.ghostOf[i * 8 + lane - 1]] = 0u;
    }
    if (lane < 7) {
        long long t[4] = {0, 0, 0, 0};
        for (int r = 0; r < COMBINE_ROWS; ++r)
#pragma unroll
            for (int i = 0; i < 4; ++i) t[i] += red[w][lane + 7 * r][i];
        val[w][lane] = exact_value((const unsigned long long*)t);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (lane != 0) return;
    const double* v = val[w];
    E.set3(EF_FH, e, V3(v[0], v[1], v[2]) * u.Force);
    E.set3(EF_MH, e, V3(v[3], v[4], v[5]) * u.Torque);
    E.at(EF_FVOL, e) = v[6] * u.Volume;
}

}  // namespace

void launch_dem_rebuild(const DEMParams& p, const DEMBuffers& b, int force, hipStream_t s) {
    k_dem_rebuild<<<1, RB, 0, s>>>(p, b, force);
}

// particleEnergy after a sub-step (DEM.cpp:2226-2276, utils.cpp:324-327). The
// per-element terms of a chunk are computed in parallel; one lane then adds them
// in element order, so the sums are the reference's sequential sums.
constexpr int EN_BLOCK = 256;
__global__ void __launch_bounds__(EN_BLOCK) k_dem_energy(DEMParams p, DEMBuffers b, double sx, double sy, double sz,
                                                         double* __restrict__ out) {
#pragma clang fp contract(off)
    __shared__ double tk[EN_BLOCK], rk[EN_BLOCK], gp[EN_BLOCK];
    const El E{b.el, p.E};
    const V3 F(p.demF[0], p.demF[1], p.demF[2]);
    const double gn = sqrt(F.norm2());
    const bool grav = gn != 0.0;
    V3 n, c(0.0, 0.0, 0.0);
    if (grav) {
        n = V3(-1.0 * F.x / gn, -1.0 * F.y / gn, -1.0 * F.z / gn);
        // the plane through the box corner the gravity points to (n . X < 0 etc.)
        if (n.x * 1.0 + n.y * 0.0 + n.z * 0.0 < 0) c.x = c.x + sx;
        if (n.x * 0.0 + n.y * 1.0 + n.z * 0.0 < 0) c.y = c.y + sy;
        if (n.x * 0.0 + n.y * 0.0 + n.z * 1.0 < 0) c.z = c.z + sz;
    }
    double tKin = 0.0, rKin = 0.0, g = 0.0;
    for (int base = 0; base < p.E; base += EN_BLOCK) {
        const int e = base + threadIdx.x;
        if (e < p.E) {
            const double m = E.at(EF_M, e);
            const V3 v = E.v3(EF_X + 3, e);
            tk[threadIdx.x] = 0.5 * m * v.norm2();
            const V3 w = E.v3(EF_WL, e), I = E.v3(EF_I, e);
            rk[threadIdx.x] = I.dot(V3(w.x * w.x, w.y * w.y, w.z * w.z));
            if (grav) {
                const V3 x = E.v3(EF_X, e);
                const double h = n.dot(x - c);
                gp[threadIdx.x] = m * h * gn;
            }
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            const int cnt = min(EN_BLOCK, p.E - base);
            for (int i = 0; i < cnt; ++i) {
                tKin += tk[i];
                rKin += rk[i];
                if (grav) g += gp[i];
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double elastic = 0.0;  // not computed by the reference
        out[0] = rKin + tKin;
        out[1] = rKin;
        out[2] = tKin;
        out[3] = g;
        out[4] = elastic;
        out[5] = rKin + tKin + g + elastic;
    }
}

void launch_dem_energy(const DEMParams& p, const DEMBuffers& b, const double demSize[3], double* out, hipStream_t s) {
    k_dem_energy<<<1, EN_BLOCK, 0, s>>>(p, b, demSize[0], demSize[1], demSize[2], out);
}

namespace {
// Particle state of a saving sub-step, after the predictor (DEM.cpp:349-359:
// particles hold the predicted position and velocity; wGlobal is the element's
// last corrected angular velocity).
__global__ void k_dem_save_elements(DEMParams p, DEMBuffers b, double* __restrict__ out, double* __restrict__ info) {
    const El E{b.el, p.E};
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) info[0] = (double)b.st->nPairs;
    if (i >= p.P) return;
    const int e = part_elem(p, b, i);
    double* o = out + (size_t)i * 9;
    for (int k = 0; k < 3; ++k) {
        o[k] = p.clumps ? b.ppred[9 * (size_t)i + k] : E.at(EF_XP + k, e);
        o[3 + k] = p.clumps ? b.ppred[9 * (size_t)i + 3 + k] : E.at(EF_XP + 3 + k, e);
        o[6 + k] = E.at(EF_WG + k, e);
    }
}

// Both particle states of every element (set-up and state load).
__global__ void k_dem_particles(DEMParams p, DEMBuffers b) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= p.E) return;
    place_both(El{b.el, p.E}, b, e);
}
}  // namespace

void launch_dem_save_elements(const DEMParams& p, const DEMBuffers& b, double* out, double* info, hipStream_t s) {
    k_dem_save_elements<<<(p.P > 0 ? p.P + 63 : 64) / 64, 64, 0, s>>>(p, b, out, info);
}

void launch_dem_predict(const DEMParams& p, const DEMBuffers& b, hipStream_t s) {
    if (p.E <= 0) return;
    k_dem_predict<<<(p.E + 63) / 64, 64, 0, s>>>(p, b);
}

void launch_dem_particles(const DEMParams& p, const DEMBuffers& b, hipStream_t s) {
    if (p.E <= 0 || !p.clumps) return;
    k_dem_particles<<<(p.E + 63) / 64, 64, 0, s>>>(p, b);
}

void launch_dem_pairs(const DEMParams& p, const DEMBuffers& b, hipStream_t s) {
    if (p.P <= 0) return;
    int blocks = (p.pairCap + 255) / 256;
    if (blocks > 512) blocks = 512;
    if (p.spring) {
        if (p.clumps) k_dem_pairs<true, true><<<blocks, 256, 0, s>>>(p, b);
        else k_dem_pairs<true, false><<<blocks, 256, 0, s>>>(p, b);
    } else {
        if (p.clumps) k_dem_pairs<false, true><<<blocks, 256, 0, s>>>(p, b);
        else k_dem_pairs<false, false><<<blocks, 256, 0, s>>>(p, b);
    }
}

void launch_dem_gather(const DEMParams& p, const DEMBuffers& b, hipStream_t s) {
    if (p.E <= 0) return;
    const int g = (p.E + 63) / 64;
    if (p.spring) {
        if (p.clumps) k_dem_gather<true, true><<<g, 64, 0, s>>>(p, b);
        else k_dem_gather<true, false><<<g, 64, 0, s>>>(p, b);
    } else {
        if (p.clumps) k_dem_gather<false, true><<<g, 64, 0, s>>>(p, b);
        else k_dem_gather<false, false><<<g, 64, 0, s>>>(p, b);
    }
}



void launch_dem_hydro_combine(const DEMParams& p, const DEMBuffers& b, const HydroSink& hs, const Units& u,
                              hipStream_t s) {
    if (p.E <= 0) return;
    const int waves_per_block = COMBINE_BLOCK / 64;
    k_dem_hydro_combine<<<(p.E + waves_per_block - 1) / waves_per_block, COMBINE_BLOCK, 0, s>>>(p, b, hs, u);
}

}  // namespace hyb
