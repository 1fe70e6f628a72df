// Free-surface mass tracking and interface reclassification for gfx950.
//
// The reference walks its interface list serially (updateMass LB.cpp:1492-1590,
// updateInterface 1592-1618 -> findInterfaceMutants 1620-1650,
// smoothenInterface 1652-1701, updateMutants 1703-1742, removeIsolated
// 1744-1794, redistributeMass 1796-1804). Here every phase is one grid-stride
// kernel over a compacted node list; the phases are split where one reads
// what another writes, so that the outcome does not depend on thread order:
//
//   mass      interface nodes: stream their populations (gas links rebuilt
//             from the stored velocity), exchange mass with the neighbours,
//             mark filled (m > rho) / emptied (m < 0)
//   apply     new masses and types of the mutants
//   spread    gas neighbours of filled nodes are claimed by the filled node of
//             highest index (the reference visits filled nodes in descending
//             index order and the first visitor initialises the node); fluid
//             neighbours of emptied nodes become interface
//   mutate    claimed gas nodes get their equilibrium populations; unclaimed
//             mutants give their surplus
//   isolated  interface nodes without gas neighbours become fluid, then those
//             without fluid neighbours become gas; the survivors form the next list
//   spread    the surplus divided by the number of interface nodes
//
// The surplus terms are summed exactly in a fixed-point accumulator
// (integer atomics), so the sum does not depend on the order of the terms.
// Node ownership and list membership live in one tagged word per node,
// (tag << 32) | value, where the tag changes every step: nothing is cleared.
#include <hip/hip_runtime.h>

#include "common.h"
#include "fs_kernels.h"
#include "hybird_amd.h"
#include "lattice.h"
#include "lb_kernels.h"

namespace hyb {

namespace {

constexpr int FS_BLOCK = 256;
constexpr int FS_GRID = 1024;
// k_fs_mass: one wavefront per workgroup, so that a short list reaches more CUs (3,600 nodes 27 -> 12 us, 31,000
// nodes 43 -> 33, 262,144 nodes 31 -> 33)
constexpr int MASS_BLOCK = 64, MASS_GRID = FS_GRID * FS_BLOCK / MASS_BLOCK;
// Passes between two orderings of the interface list (k_fs_build_list). us a cycle after some 1,000 cycles, every pass / 8 /
// 16 / 32 / never: 262,144 interface nodes of 512 x 512 x 256 1670 / 1664 / 1667 / 1675 / 1896, 31,000 of 384 x 128 x 192 445
// / 426 / 428 / 430 / 443, 3,600 of 101 x 47 x 66 159 / 155 / 156 / 155 / 157. 8 and 16 are within the runs of one side.
constexpr uint32_t SORT_STEPS = 16;
enum : uint8_t { FS_STAY = 0, FS_FILLED = 1, FS_EMPTIED = 2 };

// Adds the lanes' sums to the accumulator: most wavefronts have none, the others one atomic per limb instead of one
// per node (atomics on one address take about 10 ns each, over all XCDs).
__device__ __forceinline__ void flush_acc(unsigned long long* acc, long long s[4]) {
    if (__any((s[0] | s[1] | s[2] | s[3]) != 0)) exact_flush(acc, s);
}

#define FS_FOR(i, n) \
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < (n); i += gridDim.x * blockDim.x)

template <typename T>
__device__ __forceinline__ double to_d(T v) {
    return (double)v;
}

// ---- 1. streaming of the interface nodes + updateMass (LB.cpp:1492-1590)
// SHIFT: populations are stored as f - w (rho0 = 1); f_opp - fs_j is the same in
// both forms because w_opp(j) = w_j.
//
// What link j of a node brings: the population v streamed in against j and the share a of the mass exchange. tl, vn
// and mL: the neighbour's type, its population opp(j) (only used with pull) and its mass.
struct MassNode {
    size_t idx;
    Coord c;
    V3 u;
    double usq, mi;
};
// Links to anything but slip walls and cylinders, after a collision.
__device__ __forceinline__ bool plain_link(uint8_t tl) { return !is_slip_wall(tl) && tl != T_CURVED; }
template <typename T, bool SHIFT>
__device__ __forceinline__ T link_in(int j, uint8_t tl, T fsj, T vn, double mL, const MassNode& nd, double rho0, double& a) {
#pragma clang fp contract(off)
    a = 0.0;
    if (tl == T_FLUID || tl == T_INTERFACE) {
        a = (tl == T_INTERFACE) ? 0.5 * (mL + nd.mi) : 1.0;
        return vn;  // fpost[opp][L], LB.cpp:1234
    }
    if (tl == T_GAS) {
        // LB.cpp:1237-1246 with the shifted velocity of the last collision
        const double vu = nd.u.dot(V3((double)cx(j), (double)cy(j), (double)cz(j)));
        const double g = wgt(j) * rho0 * (2.0 + 9.0 * (vu * vu) - 3.0 * nd.usq);
        return SHIFT ? (T)(-to_d(fsj) + (g - 2.0 * wgt(j))) : (T)(-to_d(fsj) + g);
    }
    if (tl == T_WALL_MOVING) a = 1.0 * nd.mi;  // zero velocity, so half-way bounce-back as at a static wall
    return fsj;
}
// The other links (slip walls, cylinders), and any link before the first collision (f = fs).
template <typename T, bool SHIFT>
__device__ __forceinline__ T wall_in(int j, bool pull, uint8_t tl, T fsj, const T* __restrict__ fpost,
                                     const uint8_t* __restrict__ type, const double* __restrict__ mass, const MassNode& nd,
                                     const LBKParams& p, double& a) {
#pragma clang fp contract(off)
    const double mi = nd.mi;
    const auto active = [&](size_t n) { const uint8_t t = type[n]; return t == T_FLUID || t == T_INTERFACE; };
    // moving walls have zero velocity. Mass exchange: a = m for a moving wall, the slip rule for a moving slip wall
    // (LB.cpp:1531-1575), else 0.
    a = 0.0;
    if (tl == T_WALL_MOVING || tl == T_CURVED) {  // LB.cpp:1539-1545
        a = 1.0 * mi;
    } else if (tl == T_SLIP_MOVING) {
        bool half = false;
        if (j > 6) {
            const bool a1 = active(nb_index(p, nd.c, slip1check(j))), a2 = active(nb_index(p, nd.c, slip2check(j)));
            half = (a1 && !a2) || (!a1 && a2);
        }
        a = half ? 0.0 + 1.0 * p.slipS2 * mi : 0.0 + 1.0 * mi;
    }
    if (!pull) {
        if (tl == T_INTERFACE) a = 0.5 * (mass[nb_index(p, nd.c, j)] + mi);
        else if (tl == T_FLUID) a = 1.0;
        return fpost[(size_t)opp(j) * p.PS + nd.idx];
    }
    // plane wall: bounce-back, slip reflection (LB.cpp:1321-1456); cylinder: Mei-Luo-Shyy (LB.cpp:1278-1319)
    if (tl == T_CURVED) return curved_link<T, SHIFT>(p, nd.c, j, fsj);
    if (is_slip_wall(tl)) return wall_link<T>(fpost, p.PS, p, nd.c, true, j, fsj, active);
    return fsj;
}

// Bound by memory latency and by the lines it touches: about 400 bytes a node where neighbouring lanes hold
// neighbouring nodes (FP32: 262,144 nodes of one z plane 147 us with the list as the atomics left it and one
// wavefront per SIMD, 33 now). PLAIN: after a collision, in a lattice without slip walls and cylinders. Otherwise the
// links to those are taken one at a time before the plain ones, whose loads still go together; their exchange waits in
// LDS, so that a node's exchange is added in the order of its links. us, all links one at a time / with every rule in
// the unrolled loop / so: slip walls, 256 x 128 x 128 nodes FP64 52.7 / 45.5 / 35.0, FP32 51.6 / 44.4 / 34.8, 101 x 47 x 66
// FP64 40.7 / 39.9 / 26.3, a cylinder in 56 x 40 x 40 49.2 / 43.0 / 30.6. Bounded to three wavefronts per SIMD, as the
// plain form is, it spills (49.4 and 42.6).
template <typename T, bool SHIFT, bool PLAIN>
__global__ void __launch_bounds__(MASS_BLOCK, PLAIN ? (sizeof(T) == 4 ? 4 : 3) : 1)
    k_fs_mass(const T* __restrict__ fpost, T* __restrict__ fout, const uint8_t* __restrict__ type,
              const double* __restrict__ mass, const T* __restrict__ rho, const double* __restrict__ uS,
              const uint32_t* __restrict__ list, FSCounters* __restrict__ ctr, int cur, double* __restrict__ mnew,
              uint8_t* __restrict__ state, LBKParams p, int pull) {
#pragma clang fp contract(off)
    __shared__ double otherDm[PLAIN ? 1 : 18][MASS_BLOCK];
    const size_t N = (size_t)p.X * p.Y * p.Z;
    const uint32_t nI = ctr->n[cur];
    if (blockIdx.x == 0 && threadIdx.x == 0) {  // counters of this step's later phases
        ctr->n[cur ^ 1] = 0;
        ctr->nA = 0;
        ctr->nB = 0;
        for (int i = 0; i < 4; ++i) ctr->acc[i] = 0ull;
        for (int i = 0; i < 4; ++i) ctr->tot[i] = 0ull;
    }
    const uint32_t sX = (uint32_t)p.X, sXY = (uint32_t)p.X * (uint32_t)p.Y;
    FS_FOR(pos, nI) {
        MassNode nd;
        nd.idx = list[pos];
        nd.c = coord_of(p, nd.idx);
        const size_t idx = nd.idx;
        const Nb3 nx = nb3(nd.c.x, p.X, p.per[0]), ny = nb3(nd.c.y, p.Y, p.per[1]), nz = nb3(nd.c.z, p.Z, p.per[2]);
        const auto nb = [&](int j) {
            return (uint32_t)pick(nx, cx(j)) + sX * (uint32_t)pick(ny, cy(j)) + sXY * (uint32_t)pick(nz, cz(j));
        };
        if (p.actPrev) {  // type class before this pass of the nodes it may change
            uint32_t* ap = const_cast<uint32_t*>(p.actPrev);
            ap[idx] = (p.actTag << 2) | 2u;
            for (int j = 1; j < 19; ++j) {
                const size_t L = nb_index(p, nd.c, j);
                if (type[L] == T_GAS) ap[L] = p.actTag << 2;
            }
        }
        nd.mi = mass[idx];
        nd.u = V3(uS[idx], uS[N + idx], uS[2 * N + idx]);
        nd.usq = nd.u.norm2();
        // every neighbour's type and mass and its opposite population, loaded together before any is used (a
        // neighbour index is always a node of the lattice, so the loads a neighbour's type makes unnecessary
        // stay in bounds): one round trip instead of one per link
        T fs[19], vn[19];
        uint8_t tn[19];
        double mL[19];
#pragma unroll
        for (int j = 0; j < 19; ++j) fs[j] = fpost[(size_t)j * p.PS + idx];
#pragma unroll
        for (int j = 1; j < 19; ++j) {
            const uint32_t L = nb(j);
            tn[j] = type[L];
            vn[j] = fpost[(size_t)opp(j) * p.PS + L];
            mL[j] = mass[L];
        }
        fout[idx] = fs[0];
        uint32_t other = 0;  // links that are not plain
        if constexpr (!PLAIN) {
#pragma unroll
            for (int j = 1; j < 19; ++j)
                if (!pull || !plain_link(tn[j])) other |= 1u << j;
            for (uint32_t rest = other; rest; rest &= rest - 1u) {
                const int j = __ffs((int)rest) - 1;
                double a;
                const T fsj = fpost[(size_t)j * p.PS + idx];
                const T v = wall_in<T, SHIFT>(j, pull != 0, type[nb_index(p, nd.c, j)], fsj, fpost, type, mass, nd, p, a);
                fout[(size_t)opp(j) * p.PS + idx] = v;
                otherDm[j - 1][threadIdx.x] = 1.0 * a * (to_d(v) - to_d(fsj));
            }
        }
        double dm = 0.0;
#pragma unroll
        for (int j = 1; j < 19; ++j) {
            if (!PLAIN && (other >> j & 1u)) {
                dm += otherDm[PLAIN ? 0 : j - 1][threadIdx.x];
                continue;
            }
            double a;
            const T v = link_in<T, SHIFT>(j, tn[j], fs[j], vn[j], mL[j], nd, p.initDensity, a);
            fout[(size_t)opp(j) * p.PS + idx] = v;
            dm += 1.0 * a * (to_d(v) - to_d(fs[j]));
        }
        const double mn = nd.mi + dm;
        const double n = to_d(rho[idx]);
        state[pos] = mn > n ? FS_FILLED : (mn < 0.0 ? FS_EMPTIED : FS_STAY);
        mnew[pos] = mn;
    }
}

// ---- 2. findInterfaceMutants (LB.cpp:1620-1650): new masses and types
__global__ void __launch_bounds__(FS_BLOCK)
    k_fs_apply(const uint32_t* __restrict__ list, const FSCounters* __restrict__ ctr, int cur,
               const double* __restrict__ mnew, const uint8_t* __restrict__ state, double* __restrict__ mass,
               uint8_t* __restrict__ type, uint32_t* __restrict__ link) {
    const uint32_t nI = ctr->n[cur];
    FS_FOR(pos, nI) {
        const size_t idx = list[pos];
        mass[idx] = mnew[pos];
        uint32_t lw = link[idx] | LINK_PRESTREAMED;
        const uint8_t s = state[pos];
        if (s == FS_FILLED) {
            type[idx] = T_FLUID;
            lw &= ~LINK_INTERFACE;
        } else if (s == FS_EMPTIED) {
            type[idx] = T_GAS;
            lw &= ~(LINK_ACTIVE | LINK_INTERFACE);
        }
        link[idx] = lw;
    }
}

// ---- 3. smoothenInterface (LB.cpp:1652-1701)
// Filled nodes claim their gas neighbours (highest filled index wins); emptied
// nodes turn their fluid neighbours (the node itself included, j = 0) into
// interface nodes with 99 % of their density as mass. Phase A reads only gas
// types and phase B changes only fluid types, so both run in one kernel.
template <typename T>
__global__ void __launch_bounds__(FS_BLOCK)
    k_fs_spread(const uint32_t* __restrict__ list, FSCounters* __restrict__ ctr, int cur,
                const uint8_t* __restrict__ state, uint8_t* __restrict__ type, uint32_t* __restrict__ link,
                unsigned long long* __restrict__ claim, uint32_t* __restrict__ listA, uint32_t* __restrict__ listB,
                double* __restrict__ mass, const T* __restrict__ rho, uint32_t tag, LBKParams p) {
#pragma clang fp contract(off)
    const uint32_t nI = ctr->n[cur];
    const unsigned long long tagv = (unsigned long long)tag << 32;
    long long acc[4] = {0, 0, 0, 0};
    FS_FOR(pos, nI) {
        const uint8_t s = state[pos];
        if (s == FS_STAY) continue;
        const size_t idx = list[pos];
        const Coord c = coord_of(p, idx);
        // the neighbours' types, then the claims, each loaded together: three round trips instead of one per link.
        // (A fluid neighbour that another node has turned meanwhile is found by its claim.)
        const uint8_t want = s == FS_FILLED ? T_GAS : T_FLUID;
        const unsigned long long mine = tagv | (s == FS_FILLED ? (unsigned long long)(idx + 1) : 1ull);
        uint8_t tn[19];
        unsigned long long old[19];
#pragma unroll
        for (int j = 0; j < 19; ++j) tn[j] = type[j == 0 ? idx : nb_index(p, c, j)];
#pragma unroll
        for (int j = 0; j < 19; ++j) {
            old[j] = ~0ull;
            if (tn[j] == want && !(s == FS_FILLED && j == 0)) old[j] = atomicMax(&claim[j == 0 ? idx : nb_index(p, c, j)], mine);
        }
        uint32_t first = 0;  // nodes nobody had claimed this step
#pragma unroll
        for (int j = 0; j < 19; ++j)
            if (old[j] < tagv) first |= 1u << j;
        if (!first) continue;
        uint32_t at = atomicAdd(s == FS_FILLED ? &ctr->nA : &ctr->nB, (uint32_t)__popc(first));
        uint32_t* out = s == FS_FILLED ? listA : listB;
        for (; first; first &= first - 1u) {
            const int j = __ffs((int)first) - 1;
            const size_t L = j == 0 ? idx : nb_index(p, c, j);
            out[at++] = (uint32_t)L;
            if (s == FS_FILLED) continue;
            if (p.actPrev) const_cast<uint32_t*>(p.actPrev)[L] = (p.actTag << 2) | 1u;  // was fluid
            type[L] = T_INTERFACE;
            link[L] |= LINK_INTERFACE;
            const double n = to_d(rho[L]);
            mass[L] = 0.99 * n;
            exact_local(acc, 0.01 * n);
        }
    }
    flush_acc(ctr->acc, acc);
}

// ---- 4. new interface nodes from gas (LB.cpp:1668-1682, node.cpp:26-61) and
// updateMutants (LB.cpp:1703-1742)
template <typename T, bool SHIFT>
__global__ void __launch_bounds__(FS_BLOCK)
    k_fs_mutate(const uint32_t* __restrict__ list, FSCounters* __restrict__ ctr, int cur,
                const uint8_t* __restrict__ state, uint8_t* __restrict__ type, uint32_t* __restrict__ link,
                const unsigned long long* __restrict__ claim, const uint32_t* __restrict__ listA,
                double* __restrict__ mass, T* __restrict__ rho, double* __restrict__ uS, double* __restrict__ hFi,
                double* __restrict__ visc, T* __restrict__ fout, uint32_t* __restrict__ slipw, uint32_t tag, double Fx,
                double Fy, double Fz, LBKParams p) {
#pragma clang fp contract(off)
    const size_t N = (size_t)p.X * p.Y * p.Z;
    const uint32_t nI = ctr->n[cur], nA = ctr->nA;
    const uint32_t n = nI > nA ? nI : nA;
    const double rho0 = p.initDensity;
    long long acc[4] = {0, 0, 0, 0};
    FS_FOR(pos, n) {
        if (pos < nA) {
            const size_t L = listA[pos];
            const size_t f = (size_t)(uint32_t)(claim[L] & 0xFFFFFFFFull) - 1;
            // nodeInitialize(rho0, u_f, 0.01 rho0, visc_f, hydroForce_f + lbF)
            const V3 F = V3(hFi[f], hFi[N + f], hFi[2 * N + f]) + V3(Fx, Fy, Fz);
            const V3 uf(uS[f], uS[N + f], uS[2 * N + f]);
            const V3 u = (1.0 * F) / 2.0 / rho0 + uf;
            const double usq = u.norm2();
#pragma unroll
            for (int j = 0; j < 19; ++j) {
                const double vu = u.dot(V3((double)cx(j), (double)cy(j), (double)cz(j)));
                const double feq = wgt(j) * rho0 * (1.0 + 3.0 * vu + 4.5 * vu * vu - 1.5 * usq);
                fout[(size_t)j * p.PS + L] = SHIFT ? (T)(feq - wgt(j)) : (T)feq;
            }
            const Coord c = coord_of(p, L);
            uint32_t lw = LINK_ACTIVE | LINK_INTERFACE | LINK_PRESTREAMED, sw = 0, cw = 0;
            for (int j = 1; j < 19; ++j) {
                const uint8_t tl = type[nb_index(p, c, j)];
                if (is_plane_wall(tl) || tl == T_CURVED) lw |= 1u << j;
                if (is_slip_wall(tl)) sw |= 1u << j;
                if (tl == T_CURVED) cw |= 1u << j;
            }
            if (sw) lw |= LINK_SLIP;
            if (cw) lw |= LINK_CURVED;
            if (slipw) slipw[L] = sw;
            if (p.curvw) const_cast<uint32_t*>(p.curvw)[L] = cw;
            link[L] = lw;
            type[L] = T_INTERFACE;
            mass[L] = 0.01 * rho0;
            rho[L] = (T)rho0;
            uS[L] = u.x; uS[N + L] = u.y; uS[2 * N + L] = u.z;
            hFi[L] = 0.0; hFi[N + L] = 0.0; hFi[2 * N + L] = 0.0;
            if (visc) visc[L] = visc[f];
            exact_local(acc, -(0.01 * rho0));
        }
        if (pos < nI) {
            const uint8_t s = state[pos];
            if (s == FS_STAY) continue;
            const size_t idx = list[pos];
            if ((claim[idx] >> 32) == tag) continue;  // became interface again this step
            if (s == FS_EMPTIED) {
                exact_local(acc, mass[idx]);
            } else {
                const double nn = to_d(rho[idx]);
                exact_local(acc, mass[idx] - nn);
                mass[idx] = nn;
            }
        }
    }
    flush_acc(ctr->acc, acc);
}

// Interface candidates after smoothenInterface: unchanged list entries, then the
// gas -> interface list, then the fluid -> interface list.
__device__ __forceinline__ bool fs_candidate(uint32_t q, uint32_t nI, uint32_t nA, const uint32_t* list,
                                             const uint8_t* state, const uint32_t* listA, const uint32_t* listB,
                                             size_t& idx) {
    if (q < nI) {
        if (state[q] != FS_STAY) return false;
        idx = list[q];
    } else if (q < nI + nA) {
        idx = listA[q - nI];
    } else {
        idx = listB[q - nI - nA];
    }
    return true;
}

// ---- 5. removeIsolated, first loop (LB.cpp:1744-1770): no gas neighbour -> fluid
template <typename T>
__global__ void __launch_bounds__(FS_BLOCK)
    k_fs_iso_fluid(const uint32_t* __restrict__ list, FSCounters* __restrict__ ctr, int cur,
                   const uint8_t* __restrict__ state, const uint32_t* __restrict__ listA,
                   const uint32_t* __restrict__ listB, uint8_t* __restrict__ type, uint32_t* __restrict__ link,
                   double* __restrict__ mass, const T* __restrict__ rho, LBKParams p) {
#pragma clang fp contract(off)
    const uint32_t nI = ctr->n[cur], nA = ctr->nA, nB = ctr->nB;
    long long acc[4] = {0, 0, 0, 0};
    FS_FOR(q, nI + nA + nB) {
        size_t idx;
        if (!fs_candidate(q, nI, nA, list, state, listA, listB, idx)) continue;
        const Coord c = coord_of(p, idx);
        uint8_t tn[19];  // all loaded before the test: one round trip
#pragma unroll
        for (int j = 1; j < 19; ++j) tn[j] = type[nb_index(p, c, j)];
        bool gasNb = false;
#pragma unroll
        for (int j = 1; j < 19; ++j) gasNb = gasNb || tn[j] == T_GAS;
        if (gasNb) continue;
        const double n = to_d(rho[idx]);
        exact_local(acc, mass[idx] - n);
        mass[idx] = n;
        type[idx] = T_FLUID;
        link[idx] &= ~LINK_INTERFACE;
    }
    flush_acc(ctr->acc, acc);
}

// Position of each lane that keeps a value in a list of `count` entries: the workgroup's values stay together and in
// order, one atomic for all of them. Every lane of the workgroup calls it; n values of this lane.
__device__ __forceinline__ uint32_t append_at(uint32_t n, uint32_t* count) {
    __shared__ uint32_t sum[FS_BLOCK / 64], base;
    const int lane = (int)(threadIdx.x & 63u), wave = (int)(threadIdx.x >> 6);
    uint32_t incl = n;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t v = __shfl_up(incl, off, 64);
        if (lane >= off) incl += v;
    }
    __syncthreads();  // the call before has read sum and base
    if (lane == 63) sum[wave] = incl;
    __syncthreads();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < FS_BLOCK / 64; ++w) {
        before += w < wave ? sum[w] : 0u;
        all += sum[w];
    }
    if (threadIdx.x == 0) base = all ? atomicAdd(count, all) : 0u;
    __syncthreads();
    return base + before + incl - n;
}

// ---- 6. removeIsolated, second loop (LB.cpp:1771-1792): no fluid neighbour ->
// gas; the remaining interface nodes form the next list. One atomic per workgroup for their places: one per
// wavefront bound the kernel (262,144 nodes 52 us, now 16) and scattered neighbouring nodes over the list.
__global__ void __launch_bounds__(FS_BLOCK)
    k_fs_iso_gas(const uint32_t* __restrict__ list, FSCounters* __restrict__ ctr, int cur,
                 const uint8_t* __restrict__ state, const uint32_t* __restrict__ listA,
                 const uint32_t* __restrict__ listB, uint8_t* __restrict__ type, uint32_t* __restrict__ link,
                 const double* __restrict__ mass, uint32_t* __restrict__ next, LBKParams p) {
    const uint32_t nI = ctr->n[cur], nA = ctr->nA, nB = ctr->nB, n = nI + nA + nB;
    long long acc[4] = {0, 0, 0, 0};
    for (uint32_t q0 = blockIdx.x * blockDim.x; q0 < n; q0 += gridDim.x * blockDim.x) {
        const uint32_t q = q0 + threadIdx.x;
        size_t idx = 0;
        bool keep = false;
        if (q < n && fs_candidate(q, nI, nA, list, state, listA, listB, idx) && type[idx] == T_INTERFACE) {
            const Coord c = coord_of(p, idx);
            uint8_t tn[19];  // all loaded before the test: one round trip
#pragma unroll
            for (int j = 1; j < 19; ++j) tn[j] = type[nb_index(p, c, j)];
#pragma unroll
            for (int j = 1; j < 19; ++j) keep = keep || tn[j] == T_FLUID;
            if (!keep) {
                exact_local(acc, mass[idx]);
                type[idx] = T_GAS;
                link[idx] = 0u;
            }
        }
        const uint32_t at = append_at(keep ? 1u : 0u, &ctr->n[cur ^ 1]);
        if (keep) next[at] = (uint32_t)idx;
    }
    flush_acc(ctr->acc, acc);
}

// ---- 7. redistributeMass (LB.cpp:1796-1804)
__global__ void __launch_bounds__(FS_BLOCK)
    k_fs_redistribute(const uint32_t* __restrict__ next, FSCounters* __restrict__ ctr, int cur,
                      double* __restrict__ mass) {
#pragma clang fp contract(off)
    const uint32_t n = ctr->n[cur ^ 1];
    if (blockIdx.x == 0 && threadIdx.x == 0) ctr->nA = 0;  // k_fs_build_list may count with it
    if (n == 0) return;
    const double add = exact_value(ctr->acc) / (double)n;
    FS_FOR(q, n) mass[next[q]] += add;
}

// ---- interface list in lattice order (4,096 nodes of a workgroup stay together): at the start, and every
// SORT_STEPS passes, since the passes append new nodes and deal the workgroups' parts out in any order, after which
// neighbouring lanes of k_fs_mass read lines far apart. 16 node types per lane; read-bound. `count` starts at zero
// and ends as the list's length.
constexpr int BUILD_NODES = 16;
__global__ void __launch_bounds__(FS_BLOCK) k_fs_build_list(const uint8_t* __restrict__ type, uint32_t* __restrict__ list,
                                                            uint32_t* __restrict__ count, size_t N) {
    const size_t per = (size_t)FS_BLOCK * BUILD_NODES;
    for (size_t i0 = blockIdx.x * per; i0 < N; i0 += gridDim.x * per) {
        const size_t i = i0 + threadIdx.x * (size_t)BUILD_NODES;
        uint32_t itf = 0;  // bit k: node i + k
        if (i + BUILD_NODES <= N) {
            const uint4 t = *reinterpret_cast<const uint4*>(type + i);  // type is aligned, i a multiple of 16
            const uint32_t w[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
            for (int k = 0; k < BUILD_NODES; ++k)
                if (((w[k / 4] >> (8 * (k % 4))) & 0xFFu) == (uint32_t)T_INTERFACE) itf |= 1u << k;
        } else {
            for (size_t k = i; k < N; ++k)
                if (type[k] == T_INTERFACE) itf |= 1u << (k - i);
        }
        if (!__syncthreads_or(itf != 0u)) continue;
        uint32_t at = append_at((uint32_t)__popc(itf), count);
        for (; itf; itf &= itf - 1u) list[at++] = (uint32_t)(i + (size_t)(__ffs((int)itf) - 1));
    }
}

// ---- post-stream populations for the host view (LB.cpp:1144-1488)
template <typename T, bool SHIFT>
__global__ void k_fs_stream_view(const T* __restrict__ fin, T* __restrict__ fout, const uint8_t* __restrict__ type,
                                 const uint32_t* __restrict__ link, const double* __restrict__ uS, LBKParams p) {
#pragma clang fp contract(off)
    const size_t N = (size_t)p.X * p.Y * p.Z;
    for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < N; idx += (size_t)gridDim.x * blockDim.x) {
        if (!(link[idx] & LINK_ACTIVE)) continue;
        const Coord c = coord_of(p, idx);
        const bool itf = (link[idx] & LINK_INTERFACE) != 0;
        V3 u;
        if (itf) u = V3(uS[idx], uS[N + idx], uS[2 * N + idx]);
        const double usq = u.norm2();
        fout[idx] = fin[idx];
        for (int j = 1; j < 19; ++j) {
            const int o = opp(j);
            const size_t L = nb_index(p, c, j);
            const uint8_t tl = type[L];
            T v;
            if (tl == T_FLUID || tl == T_INTERFACE) {
                v = fin[(size_t)o * p.PS + L];
            } else if (tl == T_GAS) {
                const double vu = u.dot(V3((double)cx(j), (double)cy(j), (double)cz(j)));
                const double g = wgt(j) * p.initDensity * (2.0 + 9.0 * (vu * vu) - 3.0 * usq);
                const double fsj = (double)fin[(size_t)j * p.PS + idx];
                v = SHIFT ? (T)(-fsj + (g - 2.0 * wgt(j))) : (T)(-fsj + g);
            } else {
                v = fin[(size_t)j * p.PS + idx];
                if (tl == T_CURVED)
                    v = curved_link<T, SHIFT>(p, c, j, v);
                else if (is_slip_wall(tl))
                    v = wall_link<T>(fin, p.PS, p, c, true, j, v,
                                     [&](size_t n) { const uint8_t t = type[n]; return t == T_FLUID || t == T_INTERFACE; });
            }
            fout[(size_t)o * p.PS + idx] = v;
        }
    }
}

}  // namespace

// Extra mass of the curved-wall rule in the streaming of the last LB step
// (LB.cpp:1315-1317): every active node adds m (chi fs_j - chi fStar + BBi) per
// curved link, m its mass (interface mass, or the fluid node's last density).
// Summed exactly into ctr->extra.
template <typename T, bool SHIFT>
__global__ void __launch_bounds__(FS_BLOCK) k_fs_curved_extra(const T* __restrict__ fpost,
                                                              const uint32_t* __restrict__ link,
                                                              const double* __restrict__ mass,
                                                              const T* __restrict__ rhoFluid, FSCounters* __restrict__ ctr,
                                                              double rho0, int massKnown, LBKParams p) {
#pragma clang fp contract(off)
    const size_t N = (size_t)p.X * p.Y * p.Z;
    FS_FOR(i, (uint32_t)N) {
        const uint32_t lw = link[i];
        if (!(lw & LINK_ACTIVE) || !(lw & LINK_CURVED)) continue;
        const uint32_t cw = p.curvw[i];
        const Coord c = coord_of(p, i);
        double m;
        if (lw & LINK_INTERFACE) m = mass[i];
        else m = massKnown ? to_d(rhoFluid[i]) : rho0;
        for (int j = 1; j < 19; ++j) {
            if (!(cw & (1u << j))) continue;
            const CurvedParts q = curved_parts(p, c, j);
            const double fs = SHIFT ? to_d(fpost[(size_t)j * p.PS + i]) + wgt(j) : to_d(fpost[(size_t)j * p.PS + i]);
            exact_add(ctr->extra, m * (q.chi * fs - q.chi * q.fStar + q.BBi));
        }
    }
}

// redistributeMass(extraMass) at the end of the streaming (LB.cpp:1477,
// 1796-1804): every interface node of the current list gains extra / count.
// One workgroup; the accumulator is cleared for the next step.
__global__ void __launch_bounds__(FS_BLOCK) k_fs_add_extra(const uint32_t* __restrict__ list,
                                                           FSCounters* __restrict__ ctr, int cur,
                                                           double* __restrict__ mass) {
#pragma clang fp contract(off)
    const uint32_t nI = ctr->n[cur];
    const double add = exact_value(ctr->extra) / (double)nI;
    for (uint32_t pos = threadIdx.x; pos < nI; pos += blockDim.x) mass[list[pos]] += add;
    __syncthreads();
    if (threadIdx.x == 0)
        for (int i = 0; i < 4; ++i) ctr->extra[i] = 0ull;
}

// Mass of the active nodes outside particles after the pass (LB.cpp:1807-1813):
// interface nodes their mass, fluid nodes their last density; summed exactly.
template <typename T>
__global__ void __launch_bounds__(FS_BLOCK) k_fs_total_mass(const uint8_t* __restrict__ type,
                                                            const uint32_t* __restrict__ solid, uint32_t ctag,
                                                            const double* __restrict__ mass, const T* __restrict__ rho,
                                                            FSCounters* __restrict__ ctr, size_t N) {
    long long acc[4] = {0, 0, 0, 0};
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += (size_t)gridDim.x * blockDim.x) {
        const uint8_t t = type[i];
        if (t != T_FLUID && t != T_INTERFACE) continue;
        if (solid && owner_slot(solid[i], ctag)) continue;
        exact_local(acc, t == T_INTERFACE ? mass[i] : to_d(rho[i]));
    }
    exact_flush(ctr->tot, acc);
}

// redistributeMass(-0.01 * (mass - totalMass)) over the new interface list
// (LB.cpp:1815-1821, 1796-1804), grid-stride; the next pass's first kernel
// clears the sum.
__global__ void __launch_bounds__(FS_BLOCK) k_fs_mass_fix(const uint32_t* __restrict__ next,
                                                          const FSCounters* __restrict__ ctr, int cur,
                                                          double* __restrict__ mass, double totalMass) {
#pragma clang fp contract(off)
    const uint32_t n = ctr->n[cur ^ 1];
    if (!n) return;
    const double massDeficit = exact_value(ctr->tot) - totalMass;
    const double massSurplus = -0.01 * massDeficit;
    const double add = massSurplus / (double)n;
    FS_FOR(q, n) mass[next[q]] += add;
}

void launch_fs_mass_fix(Prec prec, const uint8_t* type, const uint32_t* solid, uint32_t ctag, FSBuffers& b, int cur,
                        int rcur, double totalMass, const LBKParams& p, hipStream_t s) {
    const size_t N = (size_t)p.X * p.Y * p.Z;
    size_t g = (N + FS_BLOCK - 1) / FS_BLOCK;
    if (g > FS_GRID) g = FS_GRID;
    if (prec == Prec::F64)
        k_fs_total_mass<double><<<(unsigned)g, FS_BLOCK, 0, s>>>(type, solid, ctag, b.mass,
                                                                 (const double*)b.rho[rcur], b.ctr, N);
    else
        k_fs_total_mass<float><<<(unsigned)g, FS_BLOCK, 0, s>>>(type, solid, ctag, b.mass, (const float*)b.rho[rcur],
                                                                b.ctr, N);
    k_fs_mass_fix<<<FS_GRID, FS_BLOCK, 0, s>>>(b.list[cur ^ 1], b.ctr, cur, b.mass, totalMass);
}

void launch_fs_curved_extra(Prec prec, const void* fpost, const uint32_t* link, FSBuffers& b, int cur,
                            const void* rhoFluid, bool massKnown, const LBKParams& p, hipStream_t s) {
    if (prec == Prec::F64)
        k_fs_curved_extra<double, false><<<FS_GRID, FS_BLOCK, 0, s>>>((const double*)fpost, link, b.mass,
                                                                      (const double*)rhoFluid, b.ctr, p.initDensity,
                                                                      massKnown ? 1 : 0, p);
    else
        k_fs_curved_extra<float, true><<<FS_GRID, FS_BLOCK, 0, s>>>((const float*)fpost, link, b.mass,
                                                                    (const float*)rhoFluid, b.ctr, p.initDensity,
                                                                    massKnown ? 1 : 0, p);
    k_fs_add_extra<<<1, FS_BLOCK, 0, s>>>(b.list[cur], b.ctr, cur, b.mass);
}

static void build_list(const uint8_t* type, uint32_t* list, uint32_t* count, const LBKParams& p, hipStream_t s) {
    const size_t N = (size_t)p.X * p.Y * p.Z, per = (size_t)FS_BLOCK * BUILD_NODES;
    size_t g = (N + per - 1) / per;
    if (g > 4096) g = 4096;
    k_fs_build_list<<<(unsigned)g, FS_BLOCK, 0, s>>>(type, list, count, N);
}

void launch_fs_build_list(const uint8_t* type, FSBuffers& b, int cur, const LBKParams& p, hipStream_t s) {
    build_list(type, b.list[cur], &b.ctr->n[cur], p, s);
}

template <typename T, bool SHIFT>
static void fs_step_t(const T* fpost, T* fout, uint8_t* type, uint32_t* link, uint32_t* slipw, double* visc, FSBuffers& b,
                      int cur, int rcur, uint32_t tag, const double* Fnew, bool pull, const LBKParams& p, hipStream_t s) {
    const T* rho = (const T*)b.rho[rcur];
    if (pull && !p.slipw && !p.curvw)
        k_fs_mass<T, SHIFT, true><<<MASS_GRID, MASS_BLOCK, 0, s>>>(fpost, fout, type, b.mass, rho, b.uS, b.list[cur], b.ctr,
                                                               cur, b.mnew, b.state, p, 1);
    else
        k_fs_mass<T, SHIFT, false><<<MASS_GRID, MASS_BLOCK, 0, s>>>(fpost, fout, type, b.mass, rho, b.uS, b.list[cur], b.ctr,
                                                                cur, b.mnew, b.state, p, pull ? 1 : 0);
    k_fs_apply<<<FS_GRID, FS_BLOCK, 0, s>>>(b.list[cur], b.ctr, cur, b.mnew, b.state, b.mass, type, link);
    k_fs_spread<T><<<FS_GRID, FS_BLOCK, 0, s>>>(b.list[cur], b.ctr, cur, b.state, type, link, b.claim, b.listA, b.listB,
                                               b.mass, rho, tag, p);
    k_fs_mutate<T, SHIFT><<<FS_GRID, FS_BLOCK, 0, s>>>(b.list[cur], b.ctr, cur, b.state, type, link, b.claim, b.listA,
                                                      b.mass, (T*)b.rho[rcur], b.uS, b.hFi, visc, fout, slipw, tag,
                                                      Fnew[0], Fnew[1], Fnew[2], p);
    k_fs_iso_fluid<T><<<FS_GRID, FS_BLOCK, 0, s>>>(b.list[cur], b.ctr, cur, b.state, b.listA, b.listB, type, link,
                                                  b.mass, rho, p);
    k_fs_iso_gas<<<FS_GRID, FS_BLOCK, 0, s>>>(b.list[cur], b.ctr, cur, b.state, b.listA, b.listB, type, link, b.mass,
                                             b.list[cur ^ 1], p);
    k_fs_redistribute<<<FS_GRID, FS_BLOCK, 0, s>>>(b.list[cur ^ 1], b.ctr, cur, b.mass);
    if (tag % SORT_STEPS == 0) build_list(type, b.list[cur ^ 1], &b.ctr->nA, p, s);
}

void launch_fs_step(Prec prec, const void* fpost, void* fout, uint8_t* type, uint32_t* link, uint32_t* slipw,
                    double* visc, FSBuffers& b, int cur, int rcur, uint32_t tag, const double* Fnew, bool pull,
                    const LBKParams& p, hipStream_t s) {
    if (prec == Prec::F64)
        fs_step_t<double, false>((const double*)fpost, (double*)fout, type, link, slipw, visc, b, cur, rcur, tag, Fnew,
                                 pull, p, s);
    else
        fs_step_t<float, true>((const float*)fpost, (float*)fout, type, link, slipw, visc, b, cur, rcur, tag, Fnew, pull,
                               p, s);
}

void launch_fs_stream_view(Prec prec, const void* fin, void* fout, const uint8_t* type, const uint32_t* link,
                           const double* uS, const LBKParams& p, hipStream_t s) {
    const size_t N = (size_t)p.X * p.Y * p.Z;
    size_t g = (N + 255) / 256;
    if (g > 8192) g = 8192;
    if (prec == Prec::F64)
        k_fs_stream_view<double, false><<<(unsigned)g, 256, 0, s>>>((const double*)fin, (double*)fout, type, link, uS, p);
    else
        k_fs_stream_view<float, true><<<(unsigned)g, 256, 0, s>>>((const float*)fin, (float*)fout, type, link, uS, p);
}

}  // namespace hyb
