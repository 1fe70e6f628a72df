// All DEM sub-steps of one DEM step (DEM.cpp:331-376) in one launch.
//
// One launch per sub-step and phase leaves the device idle most of the time: 100 or 7,728 spheres need the
// same 17-22 us per sub-step (check 4.4, pairs 4-7, corrector 9-12 us), nearly all of it launch, first-touch
// memory latency and one lane's serial Gear update. Here the element state stays on chip over all sub-steps of
// the call, four lanes per element, and workgroups exchange only the predicted position, velocity and angular
// velocity (96 bytes per particle, two buffers) and one word each for the displacement maximum. What bounds a
// sub-step now is latency: in one workgroup (100 spheres) a wavefront lives about 15,000 cycles per sub-step, issues
// VALU instructions (the FP64 chain, with pow, square roots and divisions in a touching pair) in 26 % of them and
// waits at a counter or a barrier in 47 %. Over several workgroups, with two trips to memory per sub-step (the barrier's
// words, the partners' records), it lives 29,000 to 39,000 cycles, issues in 15 to 23 % and waits in 60 to 65 %.
// DEM step of ten sub-steps, before -> now, us: 6 spheres 140 -> 60, 100 spheres 171 -> 62, 561 (spring) 190 -> 131,
// 7,728 220 -> 122, 20,000 (two workgroups per CU) 330 -> 167; 600 clumps 440 -> 117.
//
//  * Lane c of an element's quad holds component c of position, angular velocity and orientation (lane 3: only
//    the quaternion's last component and the particle's radius and mass), so the Gear predictor and corrector
//    (elmt.cpp:139-254) run component-parallel; vectors are put together with quad broadcasts (DPP). Every
//    operation is the one the per-launch kernels (dem.hip) do, in the same order, so the results are
//    bit-identical.
//  * Each element evaluates its own pairs (both sides of a pair evaluate it; a pair test is cheaper than
//    passing its result through memory). The quad tests four pairs at once; the few that touch are evaluated
//    four at a time and added in pair-list order.
//  * Workgroups meet once per sub-step: each stores the bits of its max |x1|^2 into its own word, all poll all
//    words (that also gives everybody the displacement check's maximum). Three sets of words rotate, so that
//    a set is cleared again before it is polled next.
//  * A neighbour rebuild (DEM.cpp:1369-1513) runs in the same launch over all workgroups, phases separated by
//    the same barrier with device-scope release and acquire fences.
//
// Data that crosses workgroups between two fences (the exchange records, the barrier words) is read and written
// with device-scope atomics only. All workgroups must be on the device at once: dem_run_fits compares their number
// with what an otherwise idle device holds, and larger beds use the per-launch kernels. Two such launches of one
// process cannot wait for each other, since all handles use one stream; where another process or a mask of the CUs
// keeps some workgroups off the device, the roll call (dem_barrier.h) finds it out before anything is changed, and one
// workgroup does the step. After the roll call a barrier that does not complete within BARRIER_SECONDS ends the launch
// with DEM_ERR_BARRIER.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "common.h"
#include "dem_barrier.h"
#define HYB_DEM_POW_ATTR __attribute__((noinline))
#include "dem_device.h"
#include "dem_kernels.h"
#include "dem_substep.h"
#include "hybird_amd.h"

namespace hyb {

namespace {

constexpr u64 BITS_INF = 0x7FF0000000000000ull;
constexpr u64 TICKS_PER_SECOND = 100000000;  // wall_clock64
constexpr u64 BARRIER_SECONDS = 20;
constexpr int ALONE_LANES = 256;
constexpr int NOT_TOGETHER = -1;  // the roll call was refused
constexpr int ENT_LANE = 8;  // neighbours per lane kept in LDS (4 x 8 per element; more are read from memory)
constexpr uint32_t NO_GHOST = 0xFFFFFFFFu;

// ------------------------------------------------------------------ quads (four lanes per element)
template <int L>
__device__ __forceinline__ int quad(int v) {
    return __builtin_amdgcn_update_dpp(0, v, L * 0x55, 0xF, 0xF, true);
}
template <int L>
__device__ __forceinline__ double quad(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = quad<L>((int)b), hi = quad<L>((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}
template <int L>
__device__ __forceinline__ V3 quad(const V3& v) {
    return V3(quad<L>(v.x), quad<L>(v.y), quad<L>(v.z));
}
// the vector (quaternion) whose components the quad's lanes hold
__device__ __forceinline__ V3 full3(double v) { return V3(quad<0>(v), quad<1>(v), quad<2>(v)); }
__device__ __forceinline__ Q4 full4(double v) { return Q4(quad<0>(v), quad<1>(v), quad<2>(v), quad<3>(v)); }
// this lane's component (lane 3 of a vector: z)
__device__ __forceinline__ double comp(const V3& v, int c) { return c == 0 ? v.x : (c == 1 ? v.y : v.z); }
__device__ __forceinline__ double comp(const Q4& q, int c) { return c == 0 ? q.q0 : (c == 1 ? q.q1 : (c == 2 ? q.q2 : q.q3)); }
template <class F>
__device__ __forceinline__ void for_quad(F&& f) {
    f(std::integral_constant<int, 0>{});
    f(std::integral_constant<int, 1>{});
    f(std::integral_constant<int, 2>{});
    f(std::integral_constant<int, 3>{});
}

// ------------------------------------------------------------------ device-scope accesses and the barrier
// ONE: a single workgroup, whose records are in LDS.
typedef unsigned U4 __attribute__((ext_vector_type(4)));
struct Pair {
    double a, b;
};
constexpr int CACHE_SC1 = 16;  // cache policy bit of a device-scope access (what a relaxed agent-scope load carries)

// The exchange records of one sub-step: 16-byte reads of doubles 2k, 2k + 1 of a record.
template <bool ONE>
struct Records {
    double* base;                 // [particles][RUN_REC]
    __amdgpu_buffer_rsrc_t rsrc;  // both buffers
    unsigned offset;              // of base, in bytes
    __device__ __forceinline__ Pair get(uint32_t rec, int k) const {
        if constexpr (ONE) {
            const double* q = base + (size_t)rec * RUN_REC + 2 * k;
            return Pair{q[0], q[1]};
        } else {
            const U4 v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)(rec * (8u * RUN_REC) + 16u * (unsigned)k),
                                                               (int)offset, CACHE_SC1);
            return Pair{__longlong_as_double((long long)((u64)v.y << 32 | v.x)),
                        __longlong_as_double((long long)((u64)v.w << 32 | v.z))};
        }
    }
};
template <bool ONE>
__device__ __forceinline__ void xstore(double* a, double v) {
    if constexpr (ONE) *a = v;
    else __hip_atomic_store(a, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Maximum over the wavefront, valid in its last lane: DPP steps (within rows of 16 lanes, then across rows), a
// fifth of the latency of cross-lane reads through LDS. Lanes a step has no source for keep their value.
template <int CTRL, int ROWS>
__device__ __forceinline__ u64 dpp_max(u64 v) {
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp((int)(unsigned)v, (int)(unsigned)v, CTRL, ROWS, 0xF, false);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp((int)(v >> 32), (int)(v >> 32), CTRL, ROWS, 0xF, false);
    const u64 o = (u64)hi << 32 | lo;
    return o > v ? o : v;
}
__device__ __forceinline__ u64 wave_max_last(u64 v) {
    v = dpp_max<0x111, 0xF>(v);  // row_shr:1, 2, 4, 8
    v = dpp_max<0x112, 0xF>(v);
    v = dpp_max<0x114, 0xF>(v);
    v = dpp_max<0x118, 0xF>(v);
    v = dpp_max<0x142, 0xA>(v);  // row_bcast:15 into rows 1 and 3
    return dpp_max<0x143, 0xC>(v);  // row_bcast:31 into rows 2 and 3
}

struct DeviceWords {
    static __device__ __forceinline__ u64 load(u64* w) { return __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
    static __device__ __forceinline__ void store(u64* w, u64 v) {
        __hip_atomic_store(w, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    static __device__ __forceinline__ u64 swap(u64* w, u64 from, u64 to) {
        __hip_atomic_compare_exchange_strong(w, &from, to, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return from;
    }
    static __device__ __forceinline__ unsigned add(unsigned* w, unsigned v) {
        return __hip_atomic_fetch_add(w, v, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
    }
    static __device__ __forceinline__ u64 now() { return wall_clock64(); }
    static __device__ __forceinline__ void pause() { __builtin_amdgcn_s_sleep(1); }
};

template <bool ONE>
struct Grid : Meeting<DeviceWords> {
    int waves;

    // Maximum over the whole grid of `mine`; every store before it is visible to the exchange loads after it.
    // FULL: plain stores before it are visible to plain loads after it in every workgroup. Returns
    // SLOT_TIMEOUT when the other workgroups did not arrive. FIRST: the roll call after g launches, waiting `ticks` for
    // each workgroup; the verdict.
    template <bool FULL, bool FIRST = false>
    __device__ __forceinline__ u64 meet(u64 mine, u64 g = 0, u64 ticks = 0) {
        constexpr int W = ONE ? 8 : 4;  // wavefronts
        __shared__ u64 red[2][W], all[W];
        const int wave = (int)(threadIdx.x >> 6);
        mine = wave_max_last(mine);
        if ((threadIdx.x & 63) == 63) red[n & 1][wave] = mine;
        // exchange stores are complete at device scope once they no longer count here
        if constexpr (!ONE) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        u64 v = 0;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const u64 o = red[n & 1][w];
            v = o > v && w < waves ? o : v;
        }
        if constexpr (ONE) {
            ++n;
            return v;
        } else {
            if (threadIdx.x == 0) {
                if constexpr (FULL) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
                arrive((int)blockIdx.x, v);
            }
            constexpr u64 MOST = BARRIER_SECONDS * TICKS_PER_SECOND;
            u64 m;
            if constexpr (FIRST) m = call((int)threadIdx.x, (int)blockDim.x, g, ticks, MOST);
            else m = wait_all((int)threadIdx.x, (int)blockDim.x, MOST);
            m = wave_max_last(m);
            if ((threadIdx.x & 63) == 63) all[wave] = m;
            __syncthreads();
#pragma unroll
            for (int w = 0; w < W; ++w) v = all[w] > v ? all[w] : v;
            if (threadIdx.x == 0) free_last((int)blockIdx.x);
            ++n;
            if constexpr (FULL) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            return v;
        }
    }
    // The same without a value, with error codes: 0, or the largest code any workgroup gave.
    __device__ __forceinline__ int meet_full(int code) { return to_code(meet<true>((u64)code)); }
    __device__ static int to_code(u64 v) { return v == SLOT_TIMEOUT ? DEM_ERR_BARRIER : (int)v; }
};

// Exclusive scan over the workgroup's threads; total of the workgroup in tot.
__device__ __forceinline__ int wg_exscan(int v, int& tot) {
    __shared__ int part[16];
    const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6), waves = (int)(blockDim.x >> 6);
    int incl = v;
    for (int off = 1; off < 64; off <<= 1) {
        const int o = __shfl_up(incl, off, 64);
        if (lane >= off) incl += o;
    }
    __syncthreads();  // the previous call's readers are done
    if (lane == 63) part[wave] = incl;
    __syncthreads();
    int base = 0;
    tot = 0;
    for (int w = 0; w < waves; ++w) {
        if (w < wave) base += part[w];
        tot += part[w];
    }
    return base + incl - v;
}

// Sum over the workgroups before this one (before) and over all (total) of column col of the per-workgroup counts.
__device__ __forceinline__ void wg_offsets(const int* cnt, int nwg, int col, int& before, int& total) {
    __shared__ int acc[2];
    __syncthreads();
    if (threadIdx.x < 2) acc[threadIdx.x] = 0;
    __syncthreads();
    int a = 0, t = 0;
    for (int g = (int)threadIdx.x; g < nwg; g += (int)blockDim.x) {
        const int v = cnt[g * RUN_COUNTS + col];
        t += v;
        if (g < (int)blockIdx.x) a += v;
    }
    if (a) atomicAdd(&acc[0], a);
    if (t) atomicAdd(&acc[1], t);
    __syncthreads();
    before = acc[0];
    total = acc[1];
}

// Exclusive scan of a[0..n) over the grid, each workgroup on its own contiguous part; results to o1 and o2
// (may be a). col: a column of the per-workgroup counts, free again after the next barrier. Returns a barrier error or
// 0; readers of the result need a further barrier.
template <bool ONE>
__device__ __forceinline__ int grid_exscan(Grid<ONE>& grid, const DEMBuffers& b, const int* a, int n, int* o1, int* o2, int col, int& total) {
    const int len = (n + grid.nwg - 1) / grid.nwg;
    const int lo = min(n, len * (int)blockIdx.x), hi = min(n, lo + len);
    int s = 0, tot;
    for (int i = lo + (int)threadIdx.x; i < hi; i += (int)blockDim.x) s += a[i];
    wg_exscan(s, tot);
    if (threadIdx.x == 0) b.runCount[blockIdx.x * RUN_COUNTS + col] = tot;
    if (const int rc = grid.meet_full(0)) return rc;
    int base;
    wg_offsets(b.runCount, grid.nwg, col, base, total);
    for (int i0 = lo; i0 < hi; i0 += (int)blockDim.x) {
        const int i = i0 + (int)threadIdx.x;
        const int v = i < hi ? a[i] : 0;
        const int x = base + wg_exscan(v, tot);
        base += tot;
        if (i < hi) {
            o1[i] = x;
            if (o2) o2[i] = x;
        }
    }
    return 0;
}

// ------------------------------------------------------------------ element state of a quad
// The corrected state, the constants of the element and the lane's first neighbours are in LDS, one column per
// lane; of the predicted state only what contacts read is kept, the rest is predicted again from the corrected
// state where the corrector needs it (the same operations give the same bits; 90 more of them per sub-step).
// With all of it in registers the sub-step spilled to scratch memory and took twice as long.
struct State {
    double xp0, xp1, wp0, qp0;  // component c (of a vector, lane 3: z again): position, velocity, angular velocity,
                                // orientation
    double wpl;                 // component of wpLocal
    double r, m;
};

template <int LANES>
struct Cold {
    double x[6][LANES], w[6][LANES], q[6][LANES];  // corrected state
    double FH[LANES], MH[LANES];                   // hydrodynamic force and torque
    double I[LANES], dI[LANES];                    // I[c] and I[c+1] - I[c+2] (newtonAcc)
    uint2 nb[ENT_LANE][LANES];                     // partner and its ghost's period signs
    double c1[5], c2[5], co1[6], co2[6], demF[3];  // from DEMParams (as kernel arguments they are spilled)
    double period[3], wall[MAX_WALLS][6];          // periods along the axes (0: none); normal and point of each wall
};

template <int LANES>
__device__ __forceinline__ void load_state(const El& E, int e, int c, State& S, Cold<LANES>& K) {
    const int v = c < 3 ? c : 2, t = (int)threadIdx.x;
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        K.x[k][t] = E.at(EF_X + 3 * k + v, e);
        K.w[k][t] = E.at(EF_W + 3 * k + v, e);
        K.q[k][t] = E.at(EF_Q + 4 * k + c, e);
    }
    S.xp0 = E.at(EF_XP + v, e);
    S.xp1 = E.at(EF_XP + 3 + v, e);
    S.wp0 = E.at(EF_WP + v, e);
    S.qp0 = E.at(EF_QP + c, e);
    S.wpl = E.at(EF_WPL + v, e);
    K.FH[t] = E.at(EF_FH + v, e);
    K.MH[t] = E.at(EF_MH + v, e);
    const double Ic = E.at(EF_I + v, e);
    S.r = E.at(EF_RAD, e);
    S.m = E.at(EF_M, e);
    const V3 I = full3(Ic);
    K.I[t] = Ic;
    K.dI[t] = comp(V3(I.y - I.z, I.z - I.x, I.x - I.y), c);
}

// The predicted derivatives (elmt.cpp:139-177) of this lane's component; the orientation's first one is normalised.
template <int LANES>
__device__ __forceinline__ void predicted(const double (*a)[LANES], const double* coef, double o[6]) {
#pragma clang fp contract(off)
    const int t = (int)threadIdx.x;
    const double x[6] = {a[0][t], a[1][t], a[2][t], a[3][t], a[4][t], a[5][t]};
    gear_predict(x, coef, o);
}
__device__ __forceinline__ double normalised(double q) {
#pragma clang fp contract(off)
    return q / full4(q).norm();
}

// Position of the lane's own particle (proto: its prototype vector) from the element's centre and orientation.
__device__ __forceinline__ V3 placed(const V3& x0, double r, const V3& proto, const Q4& q, bool multi) {
#pragma clang fp contract(off)
    return multi ? x0 + r * project(proto, q) : x0;
}

// Exchange record of a particle: position, radius, velocity, mass, angular velocity.
template <bool CL, bool ONE>
__device__ __forceinline__ void publish(double* xch, int ilo, int size, int c, const State& S, const V3& proto) {
#pragma clang fp contract(off)
    if constexpr (CL) {
        const V3 x0 = full3(S.xp0), x1 = full3(S.xp1), w = full3(S.wp0);
        const Q4 q = full4(S.qp0);
        if (c >= size) return;
        double* o = xch + (size_t)(ilo + c) * RUN_REC;
        const V3 px = placed(x0, S.r, proto, q, size > 1);
        V3 pv = x1;
        if (size > 1) pv = pv + w.cross(px - x0);
        xstore<ONE>(o, px.x); xstore<ONE>(o + 1, px.y); xstore<ONE>(o + 2, px.z); xstore<ONE>(o + 3, S.r);
        xstore<ONE>(o + 4, pv.x); xstore<ONE>(o + 5, pv.y); xstore<ONE>(o + 6, pv.z); xstore<ONE>(o + 7, S.m);
        xstore<ONE>(o + 8, w.x); xstore<ONE>(o + 9, w.y); xstore<ONE>(o + 10, w.z);
    } else {
        if (size < 1) return;
        double* o = xch + (size_t)ilo * RUN_REC + c;
        xstore<ONE>(o, c < 3 ? S.xp0 : S.r);
        xstore<ONE>(o + 4, c < 3 ? S.xp1 : S.m);
        xstore<ONE>(o + 8, c < 3 ? S.wp0 : 0.0);
    }
}

__device__ __forceinline__ V3 ghost_vec(const DEMBuffers& b, uint32_t g) {
    return V3(b.ghostVec[3 * (size_t)g], b.ghostVec[3 * (size_t)g + 1], b.ghostVec[3 * (size_t)g + 2]);
}

// ------------------------------------------------------------------ neighbour entries
// DEMBuffers::ent: per element, its pairs in pair-list order.
//   x: origin particle of the partner | own particle within the element << 29 | (own is the pair's second) << 31
//   y: the partner's ghost index (NO_GHOST: a standard particle); z: pair; w: this element keeps the pair's spring
__device__ __forceinline__ uint4 make_entry(const DEMParams& p, const DEMBuffers& b, uint32_t k, int own, int nth) {
    const int n0 = (int)b.pairs[2 * (size_t)k], n1 = (int)b.pairs[2 * (size_t)k + 1];
    const bool second = n1 == own;
    const int o = second ? n0 : n1;
    uint4 r;
    r.x = (uint32_t)(o < p.P ? o : (int)b.ghostIndex[o - p.P]) | (uint32_t)nth << 29 | (second ? 0x80000000u : 0u);
    r.y = o < p.P ? NO_GHOST : (uint32_t)(o - p.P);
    r.z = k;
    r.w = !second || n0 >= p.P ? 1u : 0u;  // a pair whose first particle is a ghost has only its second
    return r;
}

// The entries of one element, its quad's lanes in turn, from the sorted per-particle lists. Pair indices of
// different particles of an element never coincide, so a pair's place is the number of smaller ones.
__device__ __forceinline__ void element_entries(const DEMParams& p, const DEMBuffers& b, int ilo, int size, int c) {
    const uint32_t elo = b.csrOff[ilo], ehi = b.csrOff[ilo + size];
    for (int n = 0; n < size; ++n) {
        const uint32_t lo = b.csrOff[ilo + n], hi = b.csrOff[ilo + n + 1];
        for (uint32_t i = lo + (uint32_t)c; i < hi; i += 4) {
            const uint32_t k = b.csr[i];
            uint32_t at = i;
            if (size > 1) {
                at = elo;
                for (uint32_t j = elo; j < ehi; ++j) at += b.csr[j] < k ? 1u : 0u;
            }
            b.ent[at] = make_entry(p, b, k, ilo + n, n);
        }
    }
}

__global__ void __launch_bounds__(256) k_dem_entries(DEMParams p, DEMBuffers b) {
    const int e = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 2), c = (int)(threadIdx.x & 3);
    if (e >= p.E || b.st->error) return;
    const int ilo = p.clumps ? b.efirst[e] : e, size = p.clumps ? b.efirst[e + 1] - ilo : 1;
    element_entries(p, b, ilo, size, c);
}

// ------------------------------------------------------------------ rebuild
// evalNeighborTable and its lists (DEM.cpp:1369-1635) by the whole grid: the counterpart of k_dem_rebuild, with
// the same lists in the same order. Ordered lists come from counts per workgroup, which owns consecutive
// elements (or cells, or cell pairs), and the sums over the workgroups before it. One workgroup alone needed
// 4.4 ms for 7,728 spheres at 256^3 and 22 ms for 20,000. px: the corrected position of the lane's particle,
// after the periodic shift. Not inlined, with its parameters in memory: its registers then cost the sub-steps
// nothing. Returns a DEM error code and the barriers passed.
struct RebuildResult {
    int code;
    unsigned n;
};
template <bool SP, bool ONE>
__device__ __forceinline__ int rebuild_body(const DEMParams& p, const DEMBuffers& b, Grid<ONE>& grid, int e, int c,
                                            int ilo, int size, const V3& px) {
#pragma clang fp contract(off)
    const El E{b.el, p.E};
    const int tid = (int)(blockIdx.x * blockDim.x + threadIdx.x), nth = (int)(gridDim.x * blockDim.x);
    const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6), waves = grid.waves;
    const bool mine = c < size;  // this lane stands for standard particle i (size 0: an element past the last)
    const int i = ilo + c;
    __shared__ int sums[16][6];
    int rc;
    // tangential springs: back to their pairs, then copies of the old lists, from which the new pairs take over
    if constexpr (SP) {
        const int oldT = b.st->nPairs, oldG = b.st->nGhost;
        if (size) {
            const uint32_t lo = b.csrOff[ilo], hi = b.csrOff[ilo + size];
            for (uint32_t j = lo + (uint32_t)c; j < hi; j += 4) {
                const uint4 en = b.ent[j];
                if (en.w)
                    for (int q = 0; q < 3; ++q) b.hist[3 * (size_t)en.z + q] = b.entHist[3 * (size_t)j + q];
            }
        }
        if ((rc = grid.meet_full(0))) return rc;
        for (int j = tid; j < 2 * oldT; j += nth) b.pairsOld[j] = b.pairs[j];
        for (int j = tid; j < 3 * oldT; j += nth) b.histOld[j] = b.hist[j];
        for (int j = tid; j <= p.P; j += nth) b.csrOffOld[j] = b.csrOff[j];
        const int nc = (int)b.csrOff[p.P];
        for (int j = tid; j < nc; j += nth) b.csrOld[j] = b.csr[j];
        for (int j = tid; j < oldG; j += nth) b.ghostIndexOld[j] = b.ghostIndex[j];
    }
    // ---- side ghosts in (periodic pair, particle) order and their corner ghosts (DEM.cpp:1590-1635): flags and counts
    int flag[3] = {0, 0, 0}, corner[3] = {0, 0, 0};
    for (int k = 0; k < 3; ++k) {
        if (k >= p.npbc || !mine) continue;
        const PbcDev& pb = p.pbc[k];
        const double left = pb.n1.dot(px - pb.p1);
        const double right = pb.n2.dot(px - pb.p2);
        flag[k] = left < p.nebrRange ? 1 : (right < p.nebrRange ? 2 : 0);
    }
    for (int k = 0; k < 3; ++k)
        for (int k2 = k + 1; k2 < 3; ++k2) corner[k] += flag[k] && flag[k2] ? 1 : 0;
    int rank[6];
    for (int k = 0; k < 3; ++k) {
        const u64 below = (1ull << lane) - 1ull;
        const u64 bs = __ballot(flag[k] != 0), b1 = __ballot(corner[k] >= 1), b2 = __ballot(corner[k] >= 2);
        rank[k] = __popcll(bs & below);
        rank[3 + k] = __popcll(b1 & below) + __popcll(b2 & below);
        if (lane == 0) {
            sums[wave][k] = __popcll(bs);
            sums[wave][3 + k] = __popcll(b1) + __popcll(b2);
        }
    }
    for (int j = tid; j <= b.ncells; j += nth) b.cellCount[j] = 0;
    for (int j = tid; j < p.P; j += nth) b.pairCount[j] = 0;
    if (tid == 0) b.st->nNearWall = 0;
    __syncthreads();
    for (int q = 0; q < 6; ++q)
        for (int w = 0; w < wave; ++w) rank[q] += sums[w][q];
    if (threadIdx.x < 6) {
        int t = 0;
        for (int w = 0; w < waves; ++w) t += sums[w][threadIdx.x];
        b.runCount[blockIdx.x * RUN_COUNTS + threadIdx.x] = t;
    }
    if ((rc = grid.meet_full(0))) return rc;
    int nSide = 0, G = 0;
    for (int q = 0; q < 6; ++q) {
        int before, total;
        wg_offsets(b.runCount, grid.nwg, q, before, total);
        rank[q] += before + G;  // G: ghosts of the kinds before this one
        G += total;
        if (q == 2) nSide = G;
    }
    if (nSide > p.Gcap || G > p.Gcap) return 1;
    const int S0 = p.P + G;
    // ---- ghosts, packed slot records (position, cluster) and cells
    int code = 0;
    const auto put_slot = [&](int s, const V3& x) {
        double* r = b.spos + 4 * (size_t)s;
        r[0] = x.x; r[1] = x.y; r[2] = x.z;
        r[3] = (double)e;
        const int cell = linearize(x, p.cellWidth, p.nCells) + S0;
        if (cell < S0 || cell >= S0 + b.ncells) {
            code = 2;
            b.cellOf[s] = 0;
        } else {
            b.cellOf[s] = cell - S0;
            atomicAdd(&b.cellCount[cell - S0], 1);
        }
    };
    if (mine) {
        put_slot(i, px);
        int ng = 0;
        const auto put_ghost = [&](int g, const V3& v) {
            b.ghostIndex[g] = (uint32_t)i;
            b.ghostVec[3 * (size_t)g] = v.x; b.ghostVec[3 * (size_t)g + 1] = v.y; b.ghostVec[3 * (size_t)g + 2] = v.z;
            b.ghostOf[(size_t)i * 8 + ng++] = p.P + g;
            put_slot(p.P + g, px + v);
        };
        for (int k = 0; k < 3; ++k) {
            if (k >= p.npbc) continue;
            b.side[(size_t)i * 3 + k] = flag[k] ? rank[k] : -1;
            if (!flag[k]) continue;
            b.ghostB[rank[k]] = k;
            put_ghost(rank[k], flag[k] == 1 ? p.pbc[k].v : -1.0 * p.pbc[k].v);
        }
        for (int k = 0; k < 3; ++k) {
            int g = rank[3 + k];
            for (int k2 = k + 1; k2 < 3; ++k2) {
                if (!flag[k] || !flag[k2]) continue;
                const V3 v1 = flag[k] == 1 ? p.pbc[k].v : -1.0 * p.pbc[k].v;
                const V3 v2 = flag[k2] == 1 ? p.pbc[k2].v : -1.0 * p.pbc[k2].v;
                put_ghost(g++, v1 + v2);
            }
        }
        b.ghostOfCount[i] = ng;
    }
    if ((rc = grid.meet_full(code))) return rc;
    // ---- linked-cell table (DEM.cpp:1326-1367): chains in descending slot order
    int total;
    if ((rc = grid_exscan(grid, b, b.cellCount, b.ncells + 1, b.cellCount, b.work, 6, total))) return rc;
    if ((rc = grid.meet_full(0))) return rc;
    for (int s = tid; s < S0; s += nth) b.cursor[atomicAdd(&b.work[b.cellOf[s]], 1)] = s;
    if ((rc = grid.meet_full(0))) return rc;
    for (int cell = tid; cell < b.ncells; cell += nth) {
        const int lo = b.cellCount[cell], hi = b.cellCount[cell + 1];
        for (int j0 = lo + 1; j0 < hi; ++j0) {  // insertion sort, descending
            const int v = b.cursor[j0];
            int j = j0 - 1;
            while (j >= lo && b.cursor[j] < v) { b.cursor[j + 1] = b.cursor[j]; --j; }
            b.cursor[j + 1] = v;
        }
        b.cellTable[S0 + cell] = hi > lo ? b.cursor[lo] : -1;
        for (int j = lo; j < hi; ++j) b.cellTable[b.cursor[j]] = (j + 1 < hi) ? b.cursor[j + 1] : -1;
    }
    if ((rc = grid.meet_full(0))) return rc;
    // ---- pair list in the reference's order (DEM.cpp:1425-1484): count, scan, fill; each workgroup takes
    // consecutive cell pairs, and the thread that counts one also fills it
    const int len = (b.W + grid.nwg - 1) / grid.nwg;
    const int wlo = min(b.W, len * (int)blockIdx.x), whi = min(b.W, wlo + len);
    int sum = 0;
    for (int w = wlo + (int)threadIdx.x; w < whi; w += (int)blockDim.x) {
        const int n = walk_pairs(p, b, E, S0, (unsigned)w, nullptr);
        if (n < 0) code = 3;
        b.work[w] = n < 0 ? 0 : n;
        sum += n < 0 ? 0 : n;
    }
    int tot;
    wg_exscan(sum, tot);
    if (threadIdx.x == 0) b.runCount[blockIdx.x * RUN_COUNTS + 7] = tot;
    if ((rc = grid.meet_full(code))) return rc;
    int base, T;
    wg_offsets(b.runCount, grid.nwg, 7, base, T);
    if (T > p.pairCap) return 4;
    for (int w0 = wlo; w0 < whi; w0 += (int)blockDim.x) {
        const int w = w0 + (int)threadIdx.x;
        const int n = w < whi ? b.work[w] : 0;
        const int at = base + wg_exscan(n, tot);
        base += tot;
        if (!n) continue;
        walk_pairs(p, b, E, S0, (unsigned)w, b.pairs + 2 * (size_t)at);
        for (int k = at; k < at + n; ++k) {
            const int n0 = (int)b.pairs[2 * (size_t)k], n1 = (int)b.pairs[2 * (size_t)k + 1];
            b.posI[k] = b.posJ[k] = 0xFFFFFFFFu;
            if (n0 < p.P) atomicAdd(&b.pairCount[n0], 1);
            if (n1 < p.P) atomicAdd(&b.pairCount[n1], 1);
        }
    }
    if ((rc = grid.meet_full(0))) return rc;
    // ---- per-particle pair lists, ascending pair index
    if ((rc = grid_exscan(grid, b, b.pairCount, p.P, (int*)b.csrOff, b.pairCount, 6, total))) return rc;
    if (tid == 0) {
        b.csrOff[p.P] = (uint32_t)total;
        b.st->nPairs = T;
        b.st->nGhost = G;
        b.st->nSlots = S0;
        b.st->rebuilds += 1;
        if (p.npbc) b.st->newNeighborList = 1;
    }
    if ((rc = grid.meet_full(0))) return rc;
    for (int k = tid; k < T; k += nth) {
        const int n0 = (int)b.pairs[2 * (size_t)k], n1 = (int)b.pairs[2 * (size_t)k + 1];
        if (n0 < p.P) b.csrTmp[atomicAdd(&b.pairCount[n0], 1)] = (uint32_t)k;
        if (n1 < p.P) b.csrTmp[atomicAdd(&b.pairCount[n1], 1)] = (uint32_t)k;
    }
    if ((rc = grid.meet_full(0))) return rc;
    // each quad puts its particles' lists in order and makes its element's entries
    for (int n = 0; n < size; ++n) {
        const uint32_t lo = b.csrOff[ilo + n], hi = b.csrOff[ilo + n + 1];
        for (uint32_t j = lo + (uint32_t)c; j < hi; j += 4) {
            const uint32_t k = b.csrTmp[j];
            uint32_t at = lo;
            for (uint32_t j2 = lo; j2 < hi; ++j2) at += b.csrTmp[j2] < k ? 1u : 0u;
            b.csr[at] = k;
            if ((int)b.pairs[2 * (size_t)k] == ilo + n) b.posI[k] = at;
            else b.posJ[k] = at;
        }
    }
    // ---- near walls, cylinders and objects of each particle (DEM.cpp:1496-1550)
    bool near = false;
    if (mine) {
        uint32_t wi = 0xFFFFFFFFu, mask = 0u;
        for (int k = 0; k < p.nwalls; ++k)
            if (p.walls[k].dist(px) < p.nebrRange) {
                if (wi == 0xFFFFFFFFu) wi = (uint32_t)k;
                mask |= 1u << k;
                if (!p.allWalls) break;
            }
        b.nearWall[i] = wi;
        if (p.allWalls) b.nearWallMask[i] = mask;
        near = wi != 0xFFFFFFFFu;
        if (p.ncyl) {
            uint32_t ci = 0xFFFFFFFFu;
            for (int k = 0; k < p.ncyl; ++k)
                if (p.cyl[k].dist(px) < p.nebrRange) { ci = (uint32_t)k; break; }
            b.nearCyl[i] = ci;
        }
        if (p.nobj) {
            int cnt = 0;
            for (int o = 0; o < p.nobj; ++o) {
                const V3 d = px - b.objs[o].x0;
                if (d.norm2() < p.nebrRange * p.nebrRange) {
                    if (cnt < NEAR_OBJ) b.nearObj[(size_t)i * NEAR_OBJ + cnt] = (uint32_t)o;
                    ++cnt;
                }
            }
            if (cnt > NEAR_OBJ) { code = 5; cnt = NEAR_OBJ; }
            b.nearObjCount[i] = cnt;
        }
    }
    const u64 nw = __ballot(near);
    if (lane == 0 && nw) atomicAdd(&b.st->nNearWall, (int)__popcll(nw));
    if ((rc = grid.meet_full(code))) return rc;
    if (size) element_entries(p, b, ilo, size, c);
    __threadfence_block();
    __syncthreads();  // a quad's entries are read by all of its lanes
    if constexpr (SP) {
        // a new pair takes the spring of the old pair of the same two standard particles (ghosts count as
        // their origin), turned to the new pair's orientation; pairs without one start with a released spring
        const auto origin = [&](int s, const uint32_t* gi) { return s < p.P ? s : (int)gi[s - p.P]; };
        if (size) {
            const uint32_t lo = b.csrOff[ilo], hi = b.csrOff[ilo + size];
            for (uint32_t j = lo + (uint32_t)c; j < hi; j += 4) {
                const uint4 en = b.ent[j];
                const int e0 = origin((int)b.pairs[2 * (size_t)en.z], b.ghostIndex);
                const int e1 = origin((int)b.pairs[2 * (size_t)en.z + 1], b.ghostIndex);
                double xi[3] = {0.0, 0.0, 0.0};
                bool found = false;
                for (int side = 0; side < 2 && !found; ++side) {
                    const int ei = side == 0 ? e0 : e1;
                    for (uint32_t o = b.csrOffOld[ei]; o < b.csrOffOld[ei + 1]; ++o) {
                        const uint32_t kk = b.csrOld[o];
                        const int f0 = origin((int)b.pairsOld[2 * (size_t)kk], b.ghostIndexOld);
                        const int f1 = origin((int)b.pairsOld[2 * (size_t)kk + 1], b.ghostIndexOld);
                        double sgn = 0.0;
                        if (f0 == e0 && f1 == e1) sgn = 1.0;
                        else if (f0 == e1 && f1 == e0) sgn = -1.0;
                        if (sgn == 0.0) continue;
                        for (int q = 0; q < 3; ++q) xi[q] = sgn * b.histOld[3 * (size_t)kk + q];
                        found = true;
                        break;
                    }
                }
                for (int q = 0; q < 3; ++q) {
                    b.entHist[3 * (size_t)j + q] = xi[q];
                    if (en.w) b.hist[3 * (size_t)en.z + q] = xi[q];
                }
            }
        }
        __threadfence_block();
        __syncthreads();
    }
    return 0;
}

template <bool SP, bool ONE>
__device__ __attribute__((noinline)) RebuildResult rebuild_lists(const DEMRunArgs* a, unsigned n, int e, int c, int ilo,
                                                                 int size, double x, double y, double z) {
    Grid<ONE> grid{{a->b.runSlots, n, (int)gridDim.x}, (int)(blockDim.x >> 6)};
    RebuildResult r;
    r.code = rebuild_body<SP, ONE>(a->p, a->b, grid, e, c, ilo, size, V3(x, y, z));
    r.n = grid.n;
    return r;
}

// pbcShift (DEM.cpp:1554-1584) of the quad's element; its prediction is made again from the shifted position.
template <int LANES>
__device__ __forceinline__ void pbc_shift(const DEMParams& p, const El& E, int e, int c, int size, State& S, Cold<LANES>& K) {
#pragma clang fp contract(off)
    const int t = (int)threadIdx.x;
    V3 x0 = full3(K.x[0][t]);
    bool moved = false;
    for (int k = 0; k < p.npbc; ++k) {
        const PbcDev& pb = p.pbc[k];
        const double left = pb.n1.dot(x0 - pb.p1);
        const double right = pb.n2.dot(x0 - pb.p2);
        if (left < 0.0) { x0 += pb.v; moved = true; }
        if (right < 0.0) { const V3 m = -1.0 * pb.v; x0 += m; moved = true; }
    }
    if (!moved) return;
    const double* c2 = p.c2;
    const double x = comp(x0, c);
    K.x[0][t] = x;
    S.xp0 = x + K.x[1][t] * c2[0] + K.x[2][t] * c2[1] + K.x[3][t] * c2[2] + K.x[4][t] * c2[3] + K.x[5][t] * c2[4];
    if (size && c < 3) {
        E.at(EF_X + c, e) = x;
        E.at(EF_XP + c, e) = S.xp0;
    }
}

// ------------------------------------------------------------------ contacts
// What one touching pair adds to this element (the increments of pair_contact in dem.hip for its side).
struct Touch {
    V3 fn, ft, m, mn;
    int flag;
};

template <bool SP, bool CL, bool ONE>
__device__ __forceinline__ void touch(const DEMParams& p, const DEMBuffers& b, const Records<ONE>& recs, uint32_t at, const V3& xe,
                                      const V3& ve, const V3& wO, double rO, double mO, int ilo, bool multi, Touch& o) {
#pragma clang fp contract(off)
    const uint4 en = b.ent[at];
    const bool second = (en.x >> 31) != 0u;
    const uint32_t part = en.x & 0x1FFFFFFFu;
    const Pair r0 = recs.get(part, 0), r1 = recs.get(part, 1), r2 = recs.get(part, 2), r3 = recs.get(part, 3);
    const Pair r4 = recs.get(part, 4), r5 = recs.get(part, 5);
    V3 xP(r0.a, r0.b, r1.a);
    const double rP = r1.b, mP = r3.b;
    const V3 vP(r2.a, r2.b, r3.a), wP(r4.a, r4.b, r5.a);
    if (en.y != NO_GHOST) xP = xP + ghost_vec(b, en.y);
    V3 xO = xe, vO = ve, rvO(0.0, 0.0, 0.0);
    if constexpr (CL) {
        const uint32_t own = (uint32_t)ilo + ((en.x >> 29) & 3u);
        const Pair q0 = recs.get(own, 0), q1 = recs.get(own, 1), q2 = recs.get(own, 2), q3 = recs.get(own, 3);
        xO = V3(q0.a, q0.b, q1.a);
        vO = V3(q2.a, q2.b, q3.a);
        if (multi) rvO = xO - xe;
    }
    const V3 xI = second ? xP : xO, xJ = second ? xO : xP, vI = second ? vP : vO, vJ = second ? vO : vP;
    const V3 wI = second ? wP : wO, wJ = second ? wO : wP;
    const double rI = second ? rP : rO, rJ = second ? rO : rP, mI = second ? mP : mO, mJ = second ? mO : mP;
    const V3 vd = xJ - xI;
    const double distance = vd.norm();
    const double overlap = rI + rJ - distance;
    const V3 relVel = vJ - vI;
    const V3 n = vd / distance;
    const double normRelVel = relVel.dot(n);
    const V3 normalRelVel = n * normRelVel;
    const double effMass = mI * mJ / (mI + mJ);
    const double effRad = rI * rJ / (rI + rJ);
    const double fn = normal_contact(p, overlap, normRelVel, effRad, effMass);
    const V3 normalForce = n * fn;
    const V3 vecRadI = rI * n, vecRadJ = -rJ * n;
    const V3 centerDist = (second ? vecRadJ : vecRadI) + rvO;
    o.fn = second ? normalForce : -1.0 * normalForce;
    o.flag = 1;
    if constexpr (CL) {
        if (multi) {
            const V3 mn = centerDist.cross(normalForce);
            o.mn = second ? mn : -1.0 * mn;
            o.flag = 5;
        }
    }
    const V3 relVelContact = relVel - wI.cross(vecRadI) + wJ.cross(vecRadJ);
    const V3 tangRelVelContact = relVelContact - normalRelVel;
    V3 tangForce;
    double nt;
    if constexpr (SP) {
        double* h = b.entHist + 3 * (size_t)at;
        double xi[3] = {h[0], h[1], h[2]};
        tangForce = spring_force(p, fn, effRad, effMass, p.fricPart, n, tangRelVelContact, xi);
        h[0] = xi[0]; h[1] = xi[1]; h[2] = xi[2];
        nt = tangForce.norm();
    } else {
        nt = tangRelVelContact.norm();
        if (nt != 0.0) {
            const double ft = tangential_contact(p, nt, fn, effRad, effMass, p.fricPart);
            tangForce = ft * (tangRelVelContact / nt);
        }
    }
    if (nt != 0.0) {
        const V3 m = centerDist.cross(tangForce);
        o.m = second ? -1.0 * m : m;
        o.ft = second ? -1.0 * tangForce : tangForce;
        o.flag |= 2;
    }
}

// ------------------------------------------------------------------ a step by one workgroup
// After a refused roll call: the whole step by the last workgroup to leave, on the state in memory, with the sub-steps
// of dem_substep.h (the same operations: the same results). Slow (ten sub-steps, one with a rebuild, 2.7 ms at 1,000
// spheres and 40 at 20,000, against 0.06 and 0.7 by all), so the host, told by the word after the handle's error word,
// then takes the launches of dem.hip for a while.
__device__ __forceinline__ void alone_sync() {
    __threadfence();  // also what the atomics of the part before left in memory
    __syncthreads();
}
template <bool SP, bool CL>
__device__ __attribute__((noinline)) void not_together(const DEMRunArgs* a, int nsub, int force) {
    __shared__ int last;
    const DEMParams& p = a->p;
    const DEMBuffers& b = a->b;
    const int t = (int)threadIdx.x, lanes = (int)blockDim.x;
    const Meeting<DeviceWords> m{b.runSlots, 0u, (int)gridDim.x};
    const u64 g = b.st2->launches;
    if (t == 0) last = m.last_out(&b.st2->left) ? 1 : 0;
    __syncthreads();
    if (!last) return;
    const El E{b.el, p.E};
    for (int sub = 0; sub < (force ? 1 : nsub); ++sub) {
        alone_sync();
        rebuild_by_one<ALONE_LANES>(p, b, force);
        if (force) break;
        alone_sync();
        if (b.st->error) return;
        const int T = b.st->nPairs;
        for (int k = t; k < T; k += lanes) eval_pair<SP, CL>(p, b, E, k);
        alone_sync();
        u64 vm = 0;
        for (int e = t; e < p.E; e += lanes) {
            const double v2 = gather_elem<SP, CL>(p, b, e);
            const u64 bits = v2 <= 1.79769313486231570e308 ? (u64)__double_as_longlong(v2) : BITS_INF;
            vm = bits > vm ? bits : vm;
        }
        vm = wave_max_last(vm);
        if ((t & 63) == 63) atomicMax(reinterpret_cast<u64*>(b.vmax), vm);
    }
    alone_sync();
    if (b.st->error) return;
    for (int q = t >> 2; q < p.E; q += lanes >> 2) {
        const int ilo = CL ? b.efirst[q] : q;
        element_entries(p, b, ilo, CL ? b.efirst[q + 1] - ilo : 1, t & 3);
    }
    m.clear_all(t, lanes, g);
    __syncthreads();
    if (t == 0) {
        b.st2->left = 0;
        b.st2->launches += 1;
        if (!force) b.st2->alone += 1;
        if (p.herr) __hip_atomic_store(p.herr + 1, (int)b.st2->alone, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// ------------------------------------------------------------------ the kernel
// ONE: the grid is one workgroup (up to 512 lanes, 128 elements; with multi-sphere elements 256 and 64);
// otherwise 256 lanes, 64 elements each.
template <bool SP, bool CL, bool ONE>
__global__ void __launch_bounds__(ONE && !CL ? 512 : 256, ONE && CL ? 1 : 2) k_dem_run(DEMParams p, DEMBuffers b, int nsub, int force) {
#pragma clang fp contract(off)
    if (b.st->error) return;
    const El E{b.el, p.E};
    const int c = (int)(threadIdx.x & 3);
    const int e0 = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 2);
    const int e = e0 < p.E ? e0 : p.E - 1;
    const int ilo = CL ? b.efirst[e] : e;
    // quads past the last element repeat it without particles (size 0): they store nothing
    const int size = e0 < p.E ? (CL ? b.efirst[e + 1] - ilo : 1) : 0;
    const bool multi = CL && size > 1;
    Grid<ONE> grid{{b.runSlots, b.st2->barriers, (int)gridDim.x}, (int)(blockDim.x >> 6)};
    u64 vm = *reinterpret_cast<const u64*>(b.vmax);
    double maxDisp = b.st->maxDisp;
    V3 proto;
    if (CL && c < size) proto = V3(b.pproto[3 * (size_t)(ilo + c)], b.pproto[3 * (size_t)(ilo + c) + 1], b.pproto[3 * (size_t)(ilo + c) + 2]);
    State S;
    constexpr int LANES = ONE && !CL ? 512 : 256;
    __shared__ Cold<LANES> K;
    // exchange records, two buffers: one workgroup's are in LDS
    constexpr int RECS = CL ? LANES : LANES / 4;
    __shared__ double own_recs[ONE ? 2 * RECS * RUN_REC : 1];
    double* const xbase = ONE ? own_recs : b.xch;
    const uint32_t xhalf = (ONE ? (uint32_t)RECS : (uint32_t)p.P) * RUN_REC;
    Records<ONE> recs{xbase, __builtin_amdgcn_make_buffer_rsrc(b.xch, 0, (int)(2u * (uint32_t)p.P * (8u * RUN_REC)), 0x00027000),
                      0u};
    const int t = (int)threadIdx.x;
    load_state(E, e, c, S, K);
    if (t == 0) {
        for (int k = 0; k < 6; ++k) { K.co1[k] = p.co1[k]; K.co2[k] = p.co2[k]; }
        for (int k = 0; k < 5; ++k) { K.c1[k] = p.c1[k]; K.c2[k] = p.c2[k]; }
        for (int k = 0; k < 3; ++k) {
            K.demF[k] = p.demF[k];
            K.period[k] = 0.0;
        }
        const DEMParams& g = b.runArgs->p;
        for (int k = 0; k < p.npbc; ++k) {  // period vectors lie along the axes
            if (g.pbc[k].v.x != 0.0) K.period[0] = g.pbc[k].v.x;
            if (g.pbc[k].v.y != 0.0) K.period[1] = g.pbc[k].v.y;
            if (g.pbc[k].v.z != 0.0) K.period[2] = g.pbc[k].v.z;
        }
        for (int k = 0; k < p.nwalls; ++k) {
            const WallDev& w = g.walls[k];
            K.wall[k][0] = w.n.x; K.wall[k][1] = w.n.y; K.wall[k][2] = w.n.z;
            K.wall[k][3] = w.p.x; K.wall[k][4] = w.p.y; K.wall[k][5] = w.p.z;
        }
    }

    uint32_t lo = 0, hi = 0, held = 0, nearW = 0xFFFFFFFFu, nearC = 0xFFFFFFFFu;
    int nObj = 0;
    // the partner of entry `at` (past the end: the element's own record) and, two bits per axis, the sign of its
    // ghost's period vector
    const auto neighbour = [&](uint32_t at) {
        uint2 nb{(uint32_t)ilo, 0u};
        if (at < hi) {
            const uint4 en = b.ent[at];
            nb.x = en.x;
            if (en.y != NO_GHOST) {
                const V3 v = ghost_vec(b, en.y);
                nb.y = (v.x > 0.0 ? 1u : (v.x < 0.0 ? 2u : 0u)) | (v.y > 0.0 ? 4u : (v.y < 0.0 ? 8u : 0u)) |
                       (v.z > 0.0 ? 16u : (v.z < 0.0 ? 32u : 0u));
            }
        }
        return nb;
    };
    const auto period = [&](int k, uint32_t code) {
        const uint32_t s = (code >> (2 * k)) & 3u;
        return s == 0u ? 0.0 : (s == 1u ? K.period[k] : -K.period[k]);
    };
    // the quad's lists: the first ENT_LANE entries per lane in LDS (bit m of `held`: spring m may be stretched)
    const auto load_lists = [&]() {
        lo = size ? b.csrOff[ilo] : 0u;
        hi = size ? b.csrOff[ilo + size] : 0u;
#pragma unroll
        for (int m = 0; m < ENT_LANE; ++m) {
            const uint32_t at = lo + 4u * (uint32_t)m + (uint32_t)c;
            K.nb[m][t] = neighbour(at);
        }
        held = 0xFFFFFFFFu;
        if (c < size) {
            nearW = p.allWalls ? b.nearWallMask[ilo + c] : b.nearWall[ilo + c];
            if (p.ncyl) nearC = b.nearCyl[ilo + c];
            if (p.nobj) nObj = b.nearObjCount[ilo + c];
        }
    };
    int err = 0, buf = 0;
    u64 checked = SLOT_PRESENT;
    const auto check_in = [&]() {
        if (!ONE && threadIdx.x == 0) checked = grid.check_in((int)blockIdx.x, b.st2->launches, b.runArgs->p.waitTicks);
    };
    if (force) check_in();
    if (!force) {
        load_lists();
        if constexpr (SP) {
            if (size)
                for (uint32_t j = lo + (uint32_t)c; j < hi; j += 4) {
                    const uint32_t k = b.ent[j].z;
                    for (int q = 0; q < 3; ++q) b.entHist[3 * (size_t)j + q] = b.hist[3 * (size_t)k + q];
                }
            __threadfence_block();
        }
        check_in();  // before the stores, whose completion is waited for anyway; loads after it would wait for it
        publish<CL, ONE>(recs.base, ilo, size, c, S, proto);
        if constexpr (ONE) (void)grid.template meet<false>(0);
    }
    if constexpr (!ONE) {  // up to here nothing that outlives the launch has been changed
        const u64 verdict = grid.template meet<false, true>(checked, b.st2->launches, b.runArgs->p.waitTicks);
        if (verdict != SLOT_PRESENT) err = verdict == SLOT_REFUSED ? NOT_TOGETHER : DEM_ERR_BARRIER;
    }
    V3 FP, MP, FW, MW;
    int done = 0;
    for (int sub = 0; (sub < nsub || force) && !err; ++sub) {
        // ---- displacement check (DEM.cpp:1314-1324, 342-347)
        if (!force) {
            const double vmax2 = __longlong_as_double((long long)vm);
            if (!(vmax2 <= 1.79769313486231570e308)) { err = DEM_ERR_NUMERIC; break; }
            maxDisp += sqrt(vmax2) * p.deltat;
        }
        if (__builtin_expect(force || maxDisp > p.trigger, 0)) {
            pbc_shift(b.runArgs->p, E, e, c, size, S, K);
            publish<CL, ONE>(recs.base, ilo, size, c, S, proto);
            V3 px = full3(K.x[0][t]);
            if constexpr (CL) px = placed(px, S.r, proto, full4(K.q[0][t]), size > 1);
            const RebuildResult rr = rebuild_lists<SP, ONE>(b.runArgs, grid.n, e, c, ilo, size, px.x, px.y, px.z);
            grid.n = rr.n;
            err = rr.code;
            if (err || force) break;
            maxDisp = 0.0;
            load_lists();
        }
        const bool last = sub == nsub - 1;
        const V3 xpe = full3(S.xp0), vpe = full3(S.xp1), wpg = full3(S.wp0);
        const double re = S.r, me = S.m;
        FP = V3(); MP = V3(); FW = V3(); MW = V3();
        // ---- particle pairs, 32 entries of the element's list at a time
        for (int block = 0; __any(lo + 4u * ENT_LANE * (uint32_t)block < hi); ++block) {
            const uint32_t base = lo + 4u * ENT_LANE * (uint32_t)block;
            uint32_t hit = 0;  // bit j: entry base + j touches
#pragma unroll
            for (int g = 0; g < ENT_LANE; g += 4) {
                if (g && !__any(base + 4u * (uint32_t)g < hi)) continue;
                // four entries per lane, all their loads before the first use (an entry past the end reads the
                // element's own record)
                uint32_t gm[4];
                Pair x[4][2], o[4][2];
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const uint32_t at = base + 4u * (uint32_t)(g + m) + (uint32_t)c;
                    uint2 nb = K.nb[g + m][t];
                    if (block) nb = neighbour(at);
                    gm[m] = nb.y;
                    x[m][0] = recs.get(nb.x & 0x1FFFFFFFu, 0);
                    x[m][1] = recs.get(nb.x & 0x1FFFFFFFu, 1);
                    if constexpr (CL) {
                        const uint32_t own = (uint32_t)ilo + ((nb.x >> 29) & 3u);
                        o[m][0] = recs.get(own, 0);
                        o[m][1] = recs.get(own, 1);
                    }
                }
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const uint32_t at = base + 4u * (uint32_t)(g + m) + (uint32_t)c;
                    // a ghost is its origin moved by whole periods (adding zero changes nothing)
                    const V3 xq(x[m][0].a + period(0, gm[m]), x[m][0].b + period(1, gm[m]), x[m][1].a + period(2, gm[m]));
                    const V3 own = CL ? V3(o[m][0].a, o[m][0].b, o[m][1].a) : xpe;
                    const double sig = re + x[m][1].b;
                    const bool in = at < hi && (xq - own).norm2() < sig * sig;
                    if (in) hit |= 1u << (4 * (g + m) + c);
                    if constexpr (SP) {  // out of contact: the spring is released
                        if (!in && at < hi && (block || (held >> (g + m) & 1u)))
                            for (int q = 0; q < 3; ++q) b.entHist[3 * (size_t)at + q] = 0.0;
                        if (!block) held = in ? held | 1u << (g + m) : held & ~(1u << (g + m));
                    }
                }
            }
            hit |= (uint32_t)__shfl_xor((int)hit, 1, 64);
            hit |= (uint32_t)__shfl_xor((int)hit, 2, 64);
            // the touching pairs in list order, one per lane
            while (__any(hit != 0u)) {
                uint32_t h = hit;
                for (int j = 0; j < c; ++j) h &= h - 1u;
                Touch o;
                o.flag = 0;
                if (h) touch<SP, CL, ONE>(p, b, recs, base + (uint32_t)__ffs((int)h) - 1u, xpe, vpe, wpg, re, me, ilo, multi, o);
                for_quad([&](auto L) {
                    const int f = quad<L>(o.flag);
                    const V3 fn = quad<L>(o.fn), ft = quad<L>(o.ft), m = quad<L>(o.m);
                    if (f & 1) FP = FP + fn;
                    if constexpr (CL) {
                        const V3 mn = quad<L>(o.mn);
                        if (f & 4) MP = MP + mn;
                    }
                    if (f & 2) {
                        MP = MP + m;
                        FP = FP + ft;
                    }
                });
                hit &= hit - 1u; hit &= hit - 1u; hit &= hit - 1u; hit &= hit - 1u;
            }
        }
        // ---- walls, objects, cylinders of the element's particles, in this order (dem.hip: k_dem_gather); every
        // lane of the quad does the same, lane 0 writes the records of the call's last sub-step
        V3 pxo = xpe, pvo = vpe;  // the lane's own particle
        if constexpr (CL) {
            if (multi) {
                pxo = placed(xpe, re, proto, full4(S.qp0), true);
                pvo = vpe + wpg.cross(pxo - xpe);
            }
        }
        const bool rec = last && c == 0;
        for_quad([&](auto L) {
            if constexpr (!CL && L > 0) return;
            const V3 px = CL ? quad<L>(pxo) : xpe, pv = CL ? quad<L>(pvo) : vpe;
            const uint32_t nw = (uint32_t)quad<L>((int)nearW);
            if (L >= size) return;
            const int i = ilo + L;
            const int ws = p.allWalls ? p.nwalls : 1;
            for (int s = 0; s < ws; ++s) {
                const int wi = p.allWalls ? s : (int)nw;
                const bool listed = p.allWalls ? (nw >> s & 1u) != 0u : nw != 0xFFFFFFFFu;
                const size_t slot = (size_t)i * ws + s;
                double wxi[3] = {0.0, 0.0, 0.0};
                ContactForce wcf{{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, 0.0, 0.0};
                bool contact = false;
                if (listed) {
                    const double* f = K.wall[wi];
                    const V3 wn(f[0], f[1], f[2]);
                    const double overlap = re - wn.dot(px - V3(f[3], f[4], f[5]));
                    contact = overlap > 0.0;
                    if (contact) {
                        const WallDev& w = b.runArgs->p.walls[wi];
                        if (SP && b.whist[4 * slot + 3] == (double)wi) {
                            wxi[0] = b.whist[4 * slot]; wxi[1] = b.whist[4 * slot + 1]; wxi[2] = b.whist[4 * slot + 2];
                        }
                        surface_contact<SP>(p, re, me, overlap, wn, pv - w.getSpeed(px), wpg, multi, px - xpe, p.fricWall,
                                            wxi, FW, MW, &wcf, nullptr);
                    }
                }
                if (rec && (listed || p.allWalls)) b.wcf[slot] = wcf;
                if constexpr (SP) {  // a contact that ends releases its spring
                    const double v = c < 3 ? (contact ? (c == 0 ? wxi[0] : (c == 1 ? wxi[1] : wxi[2])) : 0.0)
                                           : (contact ? (double)wi : -1.0);
                    b.whist[4 * slot + c] = v;
                }
            }
        });
        if (p.nobj) {
            for_quad([&](auto L) {
                if constexpr (!CL && L > 0) return;
                const V3 px = CL ? quad<L>(pxo) : xpe, pv = CL ? quad<L>(pvo) : vpe;
                const int no = quad<L>(nObj);
                if (L >= size) return;
                const int i = ilo + L;
                for (int k = 0; k < no; ++k) {
                    const ObjDev& ob = b.objs[b.nearObj[(size_t)i * NEAR_OBJ + k]];
                    const V3 d = px - ob.x0;
                    const double distance = d.norm();
                    const double overlap = re + ob.r - distance;
                    ContactForce ocf{{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, 0.0, 0.0};
                    if (overlap > 0.0)
                        surface_contact<false>(p, re, me, overlap, (1.0 / distance) * d, pv - ob.x1, wpg, multi, px - xpe,
                                               p.fricPart, nullptr, FW, MW, &ocf, nullptr);
                    if (rec) b.ocf[(size_t)i * NEAR_OBJ + k] = ocf;
                }
            });
        }
        if (p.ncyl) {
            for_quad([&](auto L) {
                if constexpr (!CL && L > 0) return;
                const V3 px = CL ? quad<L>(pxo) : xpe, pv = CL ? quad<L>(pvo) : vpe;
                const uint32_t ci = (uint32_t)quad<L>((int)nearC);
                if (L >= size || ci == 0xFFFFFFFFu) return;
                const CylDev& cyl = b.runArgs->p.cyl[ci];
                const double overlap = re - cyl.dist(px);
                if (!(overlap > 0.0)) return;
                const V3 d = cyl.vecDist(px);
                surface_contact<false>(p, re, me, overlap, d / (re - overlap), pv - cyl.getSpeed(px - d), wpg, multi,
                                       px - xpe, p.fricWall, nullptr, FW, MW, nullptr, nullptr);
            });
        }
        // ---- Newton-Euler (DEM.cpp:1149-1181), one component per lane
        const Q4 qp0 = full4(S.qp0);
        const double FVisc = -6.0 * M_PI * p.numVisc * re * S.xp1;
        const double MVisc = -8.0 * M_PI * p.numVisc * re * re * re * S.wp0;
        const double x2 = (FVisc + K.FH[t] + comp(FP, c) + comp(FW, c)) / me + K.demF[c < 3 ? c : 2];
        const double mom = MVisc + K.MH[t] + comp(MP, c) + comp(MW, c);
        const V3 mBf = project(full3(mom), qp0.adjoint());
        const V3 wpl = full3(S.wpl);
        const double wa = c == 0 ? wpl.y : (c == 1 ? wpl.z : wpl.x), wb = c == 0 ? wpl.z : (c == 1 ? wpl.x : wpl.y);
        const double acc = (comp(mBf, c) + K.dI[t] * wa * wb) / K.I[t];  // newtonAcc (vector.cpp:493-498)
        const V3 waBf = full3(acc);
        const double w1 = comp(project(waBf, qp0), c);
        double q2 = K.q[2][t];
        // ---- corrector (elmt.cpp:179-254), then the predictor of the next sub-step
        {
            double o[6];
            predicted(K.x, K.c2, o);
            const double d = x2 - o[2];
#pragma unroll
            for (int k = 0; k < 6; ++k) o[k] = k == 2 ? x2 : o[k] + d * K.co2[k];
#pragma unroll
            for (int k = 0; k < 6; ++k) K.x[k][t] = o[k];
            double n[6];
            gear_predict(o, K.c2, n);
            S.xp0 = n[0];
            S.xp1 = n[1];
        }
        {
            double o[6];
            predicted(K.q, K.c2, o);
            o[0] = S.qp0;
            if constexpr (CL) {
                const Q4 qp1 = full4(o[1]);
                if (multi) q2 = comp(0.5 * qp0.multiply(quatAcc(waBf, qp1)), c);
            }
            const double d = q2 - o[2];
#pragma unroll
            for (int k = 0; k < 6; ++k) o[k] = k == 2 ? q2 : o[k] + d * K.co2[k];
            o[0] = normalised(o[0]);
#pragma unroll
            for (int k = 0; k < 6; ++k) K.q[k][t] = o[k];
            double n[6];
            gear_predict(o, K.c2, n);
            S.qp0 = normalised(n[0]);
        }
        {
            double o[6];
            predicted(K.w, K.c1, o);
            const double d = w1 - o[1];
#pragma unroll
            for (int k = 0; k < 6; ++k) o[k] = k == 1 ? w1 : o[k] + d * K.co1[k];
#pragma unroll
            for (int k = 0; k < 6; ++k) K.w[k][t] = o[k];
            double n[6];
            gear_predict(o, K.c1, n);
            S.wp0 = n[0];
        }
        S.wpl = comp(project(full3(S.wp0), full4(S.qp0).adjoint()), c);
        buf ^= 1;
        recs.base = xbase + (size_t)buf * xhalf;
        recs.offset = (unsigned)buf * xhalf * 8u;
        if (!last) publish<CL, ONE>(recs.base, ilo, size, c, S, proto);
        const double v2 = full3(K.x[1][t]).norm2();
        const u64 bits = v2 <= 1.79769313486231570e308 ? (u64)__double_as_longlong(v2) : BITS_INF;
        vm = grid.template meet<false>(size ? bits : 0ull);
        done = sub + 1;
        if (vm == SLOT_TIMEOUT) err = DEM_ERR_BARRIER;
    }
    if constexpr (!ONE) {
        if (err == NOT_TOGETHER) {
            not_together<SP, CL>(b.runArgs, nsub, force);
            return;
        }
    }
    // ---- state of the last completed sub-step
    if (done && size) {
        double xp[6], qp[6], wp[6];
        predicted(K.x, K.c2, xp);
        predicted(K.q, K.c2, qp);
        predicted(K.w, K.c1, wp);
        qp[0] = S.qp0;
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            if (c < 3) {
                E.at(EF_X + 3 * k + c, e) = K.x[k][t];
                E.at(EF_XP + 3 * k + c, e) = xp[k];
                E.at(EF_W + 3 * k + c, e) = K.w[k][t];
                E.at(EF_WP + 3 * k + c, e) = wp[k];
            }
            if (k != 2 || multi) E.at(EF_Q + 4 * k + c, e) = K.q[k][t];
            E.at(EF_QP + 4 * k + c, e) = qp[k];
        }
        const Q4 q0 = full4(K.q[0][t]);
        const V3 w0 = full3(K.w[0][t]);
        const double wl = comp(project(w0, q0.adjoint()), c);
        if (c < 3) {
            E.at(EF_FP + c, e) = comp(FP, c);
            E.at(EF_MP + c, e) = comp(MP, c);
            E.at(EF_FW + c, e) = comp(FW, c);
            E.at(EF_MW + c, e) = comp(MW, c);
            E.at(EF_WG + c, e) = K.w[0][t];
            E.at(EF_WL + c, e) = wl;
            E.at(EF_WPG + c, e) = S.wp0;
            E.at(EF_WPL + c, e) = S.wpl;
        }
    }
    if constexpr (CL) {  // particles of the corrected and the predicted element (DEM.cpp:1184-1227)
        const V3 x0 = full3(K.x[0][t]), x1 = full3(K.x[1][t]), w0 = full3(K.w[0][t]);
        const V3 xp0 = full3(S.xp0), xp1 = full3(S.xp1), wp0 = full3(S.wp0);
        const Q4 q0 = full4(K.q[0][t]), qp0 = full4(S.qp0);
        if (c < size) {
            const auto place = [&](double* o, const V3& a0, const V3& a1, const Q4& q, const V3& w) {
                V3 x = a0, rv, v = a1;
                if (multi) {
                    x = placed(a0, S.r, proto, q, true);
                    rv = x - a0;
                    v = v + w.cross(rv);
                }
                o[0] = x.x; o[1] = x.y; o[2] = x.z;
                o[3] = v.x; o[4] = v.y; o[5] = v.z;
                o[6] = rv.x; o[7] = rv.y; o[8] = rv.z;
            };
            place(b.pcor + 9 * (size_t)(ilo + c), x0, x1, q0, w0);
            place(b.ppred + 9 * (size_t)(ilo + c), xp0, xp1, qp0, wp0);
        }
    }
    if constexpr (SP) {
        if (!force && !err && size)
            for (uint32_t j = lo + (uint32_t)c; j < hi; j += 4) {
                const uint4 en = b.ent[j];
                if (en.w)
                    for (int q = 0; q < 3; ++q) b.hist[3 * (size_t)en.z + q] = b.entHist[3 * (size_t)j + q];
            }
    }
    if (threadIdx.x == 0) {
        const Leaving end = leaving((int)blockIdx.x, err);
        if (end == LEAVE_ERROR) {
            dem_error(p, b, err);
        } else if (end == LEAVE_STATE) {
            if (!force) {
                *reinterpret_cast<u64*>(b.vmax) = vm;
                b.st->maxDisp = maxDisp;
            }
            if (!ONE) b.st2->launches += 1;
            b.st2->barriers = grid.n % 3u + 3u;  // only the set that comes next and the parity of the LDS words matter
        }
    }
}

}  // namespace

int dem_run_workgroups(const DEMParams& p) {
    return p.E <= (p.clumps ? 64 : 128) ? 1 : (p.E + 63) / 64;
}

bool dem_run_fits(const DEMParams& p) {
    const int g = dem_run_workgroups(p);
    if (p.E <= 0) return false;
    if (g == 1) return true;
    int dev = 0, cus = 0, per = 0;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return false;
    const auto ask = [&](auto k) { return hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k, 256, 0) == hipSuccess; };
    const bool ok = p.spring ? (p.clumps ? ask(k_dem_run<true, true, false>) : ask(k_dem_run<true, false, false>))
                             : (p.clumps ? ask(k_dem_run<false, true, false>) : ask(k_dem_run<false, false, false>));
    return ok && g <= cus * per;
}

void launch_dem_run(const DEMParams& p, const DEMBuffers& b, int nsub, int force, hipStream_t s) {
    const int g = dem_run_workgroups(p);
    const int lanes = g == 1 ? (p.E <= 64 ? 256 : 512) : 256;
    const auto go = [&](auto one) {
        constexpr bool ONE = decltype(one)::value;
        if (p.spring) {
            if (p.clumps) k_dem_run<true, true, ONE><<<g, lanes, 0, s>>>(p, b, nsub, force);
            else k_dem_run<true, false, ONE><<<g, lanes, 0, s>>>(p, b, nsub, force);
        } else {
            if (p.clumps) k_dem_run<false, true, ONE><<<g, lanes, 0, s>>>(p, b, nsub, force);
            else k_dem_run<false, false, ONE><<<g, lanes, 0, s>>>(p, b, nsub, force);
        }
    };
    if (g == 1) go(std::true_type{});
    else go(std::false_type{});
}

void launch_dem_entries(const DEMParams& p, const DEMBuffers& b, hipStream_t s) {
    if (p.E <= 0) return;
    k_dem_entries<<<(p.E + 63) / 64, 256, 0, s>>>(p, b);
}

}  // namespace hyb
