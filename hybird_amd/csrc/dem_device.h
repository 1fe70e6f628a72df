// Device code shared by the discrete-element kernels (dem.hip, dem_run.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"
#include "dem_kernels.h"

namespace hyb {

namespace {

struct El {
    double* el;
    int E;
    __device__ double& at(int f, int e) const { return el[(size_t)f * E + e]; }
    __device__ V3 v3(int f, int e) const { return V3(at(f, e), at(f + 1, e), at(f + 2, e)); }
    __device__ void set3(int f, int e, const V3& v) const { at(f, e) = v.x; at(f + 1, e) = v.y; at(f + 2, e) = v.z; }
    __device__ Q4 q4(int f, int e) const { return Q4(at(f, e), at(f + 1, e), at(f + 2, e), at(f + 3, e)); }
    __device__ void set4(int f, int e, const Q4& q) const {
        at(f, e) = q.q0; at(f + 1, e) = q.q1; at(f + 2, e) = q.q2; at(f + 3, e) = q.q3;
    }
};

// Records a device error: the sticky DEMState word (which stops every later DEM
// kernel) and the handle's host-visible error word.
__device__ __forceinline__ void dem_error(const DEMParams& p, const DEMBuffers& b, int code) {
    b.st->error = code;
    if (p.herr) *p.herr = code;
}

// vector.cpp:147-149 (offsets +1, +2, 0 through the parenthesisation).
__device__ __forceinline__ int linearize(const V3& x, const double cw[3], const unsigned nC[3]) {
    return (int)(floor(x.x / cw[0]) + 1 +
                 (double)nC[0] * (floor(x.y / cw[1]) + 1 + ((double)nC[1] * (floor(x.z / cw[2])) + 1)));
}

// Element (clusterIndex) of standard particle i.
__device__ __forceinline__ int part_elem(const DEMParams& p, const DEMBuffers& b, int i) {
    return p.clumps ? b.pelem[i] : i;
}

// Corrected position of standard particle i (particle::updateCorrected, elmt.cpp:277-290).
__device__ __forceinline__ V3 part_x(const El& E, const DEMParams& p, const DEMBuffers& b, int i) {
    if (p.clumps) {
        const double* c = b.pcor + 9 * (size_t)i;
        return V3(c[0], c[1], c[2]);
    }
    return E.v3(EF_X, i);
}

// Position of a particle slot: standard particles, then ghosts = origin + period vector (elmt.cpp:292-298).
__device__ __forceinline__ V3 slot_pos(const El& E, const DEMParams& p, const DEMBuffers& b, int s) {
    if (s < p.P) return part_x(E, p, b, s);
    const int g = s - p.P;
    const int o = (int)b.ghostIndex[g];
    return part_x(E, p, b, o) + V3(b.ghostVec[3 * g], b.ghostVec[3 * g + 1], b.ghostVec[3 * g + 2]);
}

__device__ __forceinline__ int slot_cluster(const DEMParams& p, const DEMBuffers& b, int s) {
    return part_elem(p, b, s < p.P ? s : (int)b.ghostIndex[s - p.P]);
}

// particle::updateCorrected / updatePredicted (elmt.cpp:261-290) for the
// particles of element e, from the element's position x0, velocity x1,
// orientation q and angular velocity w (the corrected or the predicted set):
// position x0 + r project(prototype, q), radiusVec = position - x0, velocity
// x1 + w x radiusVec; the particle of a size-1 element sits at its centre.
// out: DEMBuffers::pcor or ppred.
__device__ __forceinline__ void place_particles(const DEMBuffers& b, double* out, int e, double r, const V3& x0,
                                                const V3& x1, const Q4& q, const V3& w) {
#pragma clang fp contract(off)
    const int lo = b.efirst[e], hi = b.efirst[e + 1];
    for (int i = lo; i < hi; ++i) {
        V3 px = x0, rv(0.0, 0.0, 0.0), pv = x1;
        if (hi - lo > 1) {
            const V3 proto(b.pproto[3 * (size_t)i], b.pproto[3 * (size_t)i + 1], b.pproto[3 * (size_t)i + 2]);
            px = px + r * project(proto, q);
            rv = px - x0;
            pv = pv + w.cross(rv);
        }
        double* o = out + 9 * (size_t)i;
        o[0] = px.x; o[1] = px.y; o[2] = px.z;
        o[3] = pv.x; o[4] = pv.y; o[5] = pv.z;
        o[6] = rv.x; o[7] = rv.y; o[8] = rv.z;
    }
}

// Both particle states of element e from the element arrays.
__device__ __forceinline__ void place_both(const El& E, const DEMBuffers& b, int e) {
    const double r = E.at(EF_RAD, e);
    place_particles(b, b.pcor, e, r, E.v3(EF_X, e), E.v3(EF_X + 3, e), E.q4(EF_Q, e), E.v3(EF_WG, e));
    place_particles(b, b.ppred, e, r, E.v3(EF_XP, e), E.v3(EF_XP + 3, e), E.q4(EF_QP, e), E.v3(EF_WPG, e));
}

// Walks the chains of the cell pair (cell0, cell1) exactly as DEM.cpp:1455-1481.
// A chain is the cell's run of the slot array sorted by cell with slots
// descending (the order of the linked list), so its loads do not wait on each
// other; positions and clusters come from the packed slot records (spos).
// With out == nullptr only counts. Returns -1 when the stencil leaves the table.
__device__ __forceinline__ int walk_pairs(const DEMParams& p, const DEMBuffers& b, const El& E, int S, unsigned w, uint32_t* out) {
    static constexpr int sc[14][3] = {{0, 0, 0},  {1, 0, 0},  {1, 1, 0},  {0, 1, 0},  {-1, 1, 0},
                                      {0, 0, 1},  {1, 0, 1},  {1, 1, 1},  {0, 1, 1},  {-1, 1, 1},
                                      {-1, 0, 1}, {-1, -1, 1}, {0, -1, 1}, {1, -1, 1}};
    const unsigned sh = w % 14u;
    unsigned r = w / 14u;
    unsigned i0[3];
    i0[2] = r % p.nCells[2];
    r /= p.nCells[2];
    i0[1] = r % p.nCells[1];
    i0[0] = r / p.nCells[1];
    unsigned i1[3];
    for (int k = 0; k < 3; ++k) {
        i1[k] = i0[k] + (unsigned)sc[sh][k];
        if (i1[k] == p.nCells[k]) i1[k] = 0;
    }
    const uint32_t Su = (uint32_t)S;
    const uint32_t cell0 = (i0[2] * p.nCells[1] + i0[1]) * p.nCells[0] + i0[0] + Su;
    const uint32_t cell1 = (i1[2] * p.nCells[1] + i1[1]) * p.nCells[0] + i1[0] + Su;
    const uint32_t tsize = Su + (uint32_t)b.ncells;
    const double r2 = p.nebrRange * p.nebrRange;
    int cnt = 0;
    const int a0 = b.cellCount[cell0 - Su], e0 = b.cellCount[cell0 - Su + 1];  // cell0 - Su < ncells
    if (a0 >= e0) return 0;
    if (cell1 >= tsize) return -1;
    // A stencil step of -1 from index 0 wraps through unsigned arithmetic to the
    // previous linear cell, and from linear cell 0 below the cell heads: then
    // cellTable[cell1] is the link of slot cell1 and the reference walks the
    // rest of that slot's chain (DEM.cpp:1373-1390, 1455-1481). Only that case
    // follows the links.
    const bool linked = cell1 < Su;
    const int a1 = linked ? 0 : b.cellCount[cell1 - Su], e1 = linked ? 0 : b.cellCount[cell1 - Su + 1];
    const auto visit = [&](int n0, const V3& x0, int c0, int n1) {
        if (cell0 != cell1 || n1 < n0) {
            const double* s1 = b.spos + 4 * (size_t)n1;
            if (c0 != (int)s1[3]) {
                const V3 r10 = V3(s1[0], s1[1], s1[2]) - x0;
                if (r10.norm2() < r2) {
                    if (out) {
                        out[2 * cnt] = (uint32_t)n0;
                        out[2 * cnt + 1] = (uint32_t)n1;
                    }
                    ++cnt;
                }
            }
        }
    };
    // the same visit on a record already loaded (s1: position and cluster of n1)
    const auto visit_rec = [&](int n0, const V3& x0, int c0, int n1, const double s1[4]) {
        if (cell0 != cell1 || n1 < n0) {
            if (c0 != (int)s1[3]) {
                const V3 r10 = V3(s1[0], s1[1], s1[2]) - x0;
                if (r10.norm2() < r2) {
                    if (out) {
                        out[2 * cnt] = (uint32_t)n0;
                        out[2 * cnt + 1] = (uint32_t)n1;
                    }
                    ++cnt;
                }
            }
        }
    };
    for (int i0 = a0; i0 < e0; ++i0) {
        const int n0 = b.cursor[i0];
        const double* s0 = b.spos + 4 * (size_t)n0;
        const V3 x0(s0[0], s0[1], s0[2]);
        const int c0 = (int)s0[3];
        if (linked) {
            for (int n1 = b.cellTable[cell1]; n1 > -1; n1 = b.cellTable[n1]) visit(n0, x0, c0, n1);
        } else {
            // cell1's slots WB at a time: their slot numbers, then their records, are loaded together
            constexpr int WB = 8;
            for (int i1 = a1; i1 < e1; i1 += WB) {
                int n1[WB];
                double s1[WB][4];
#pragma unroll
                for (int k = 0; k < WB; ++k) n1[k] = i1 + k < e1 ? b.cursor[i1 + k] : -1;
#pragma unroll
                for (int k = 0; k < WB; ++k)
                    if (n1[k] >= 0) {
                        const double* q = b.spos + 4 * (size_t)n1[k];
                        s1[k][0] = q[0]; s1[k][1] = q[1]; s1[k][2] = q[2]; s1[k][3] = q[3];
                    }
#pragma unroll
                for (int k = 0; k < WB; ++k)
                    if (n1[k] >= 0) visit_rec(n0, x0, c0, n1[k], s1[k]);
            }
        }
    }
    return cnt;
}

// ------------------------------------------------------------------ contacts, Newton-Euler, Gear
__device__ __forceinline__ double normal_contact(const DEMParams& p, double overlap, double vrel, double effRad,
                                                 double effMass) {  // DEM.cpp:2138-2174
    if (p.hertzian) {
        const double sqrtEffRad = sqrt(effRad);
        const double sqrtOverlap = sqrt(overlap);
        const double kn = p.knConst * sqrtEffRad * sqrtOverlap;
        const double gamman = 2.0 * p.dampCoeff * sqrt(kn * effMass);
        const double dumpfn = -gamman * vrel;
        const double elasticfn = kn * overlap;
        const double fn = elasticfn + dumpfn;
        return (fn < 0.0) ? 0.0 : fn;  // std::max(fn, 0.0)
    }
    const double elasticfn = p.linearStiff * overlap;
    const double gamman = 2.0 * p.dampCoeff * sqrt(p.linearStiff * effMass);
    const double dumpfn = -gamman * vrel;
    const double fn = elasticfn + dumpfn;
    return (fn < 0.0) ? 0.0 : fn;
}

// pow(x, 1/3). HYB_DEM_POW_ATTR = noinline where the function's some forty constants would otherwise occupy
// registers over a whole loop.
#ifndef HYB_DEM_POW_ATTR
#define HYB_DEM_POW_ATTR __attribute__((always_inline))
#endif
__device__ HYB_DEM_POW_ATTR inline double pow_third(double x) { return pow(x, 1.0 / 3.0); }

// Tangential stiffness and damping coefficient of a contact (DEM.cpp:2176-2222).
__device__ __forceinline__ void tangential_coeffs(const DEMParams& p, double fn, double effRad, double effMass,
                                                  double& ks, double& gammas) {
    if (p.hertzian) ks = p.ksConst * sqrt(effRad) * pow_third(fabs(fn));
    else ks = p.linearStiff;
    gammas = 2.0 * p.viscTang * sqrt(effMass * ks);
}

__device__ __forceinline__ double tangential_contact(const DEMParams& p, double vrelt, double fn, double effRad,
                                                     double effMass, double friction) {  // DEM.cpp:2176-2222
    double ks, gammas;
    tangential_coeffs(p, fn, effRad, effMass, ks, gammas);
    const double fsMax = friction * fn;
    const double dumpfs = gammas * vrelt;
    return (fsMax < dumpfs) ? fsMax : dumpfs;  // std::min(dumpfs, fsMax)
}

// Tangential spring (extension, not in the reference): the spring xi of the
// contact is turned onto the current tangent plane (normal en), advanced by the
// tangential relative velocity vt over one sub-step, and gives F = k_s xi +
// gamma_s vt with the viscous law's k_s and gamma_s; above friction x fn the
// force is scaled to that limit and xi set to the spring length that gives it.
// Returns F (the force on the contact's first body, along vt while sticking).
__device__ __forceinline__ V3 spring_force(const DEMParams& p, double fn, double effRad, double effMass,
                                           double friction, const V3& en, const V3& vt, double xi[3]) {
#pragma clang fp contract(off)
    double ks, gammas;
    tangential_coeffs(p, fn, effRad, effMass, ks, gammas);
    V3 s(xi[0], xi[1], xi[2]);
    s = s - en * s.dot(en);
    s = s + vt * p.deltat;
    V3 F = s * ks + vt * gammas;
    const double fsMax = friction * fn;
    const double fm = F.norm();
    if (fm > fsMax) {
        F = fm > 0.0 ? F * (fsMax / fm) : V3(0.0, 0.0, 0.0);
        s = ks > 0.0 ? (F - vt * gammas) / ks : V3(0.0, 0.0, 0.0);
    }
    xi[0] = s.x; xi[1] = s.y; xi[2] = s.z;
    return F;
}

// Contact statistics and wall/object force records written by the contact code.
__device__ __forceinline__ void set_stat(StatRec& s, double ov, double fn, double ft, const V3& en, const V3& et) {
    s.ov = ov; s.fn = fn; s.ft = ft;
    s.en[0] = en.x; s.en[1] = en.y; s.en[2] = en.z;
    s.et[0] = et.x; s.et[1] = et.y; s.et[2] = et.z;
    s.flag = 1.0;
}

__device__ __forceinline__ void set_force(ContactForce& c, const V3& fn, double flag) {
    c.fn[0] = fn.x; c.fn[1] = fn.y; c.fn[2] = fn.z;
    c.flag = flag;
}

__device__ __forceinline__ void set_force_t(ContactForce& c, const V3& ft) {
    c.ft[0] = ft.x; c.ft[1] = ft.y; c.ft[2] = ft.z;
    c.flag = 3.0;
}

// The contact of a sphere (radius re, mass me) with a fixed surface: a wall (DEM.cpp:1902-1982), an object
// (DEM.cpp:2060-2136) or a cylinder (DEM.cpp:1984-2058). en: unit normal towards the sphere; relVel: the
// sphere's velocity relative to the surface; wpg: its element's angular velocity; offset: sphere centre minus
// element centre, used when the element has several spheres (multi). Adds the force and the moment to FW, MW;
// cf and st (nullptr: not wanted) get the force record and the contact statistics.
// SP: tangential spring xi instead of the viscous law.
template <bool SP>
__device__ __forceinline__ void surface_contact(const DEMParams& p, double re, double me, double overlap, const V3& en,
                                                const V3& relVel, const V3& wpg, bool multi, const V3& offset,
                                                double friction, double* xi, V3& FW, V3& MW, ContactForce* cf,
                                                StatRec* st) {
#pragma clang fp contract(off)
    const double normRelVel = relVel.dot(en);
    const V3 normalRelVel = en * normRelVel;
    const double fn = normal_contact(p, 2.0 * overlap, normRelVel, re, me);
    const V3 normalForce = en * fn;
    const V3 vecRadJ = -re * en;
    V3 centerDistJ = vecRadJ;
    if (multi) centerDistJ = centerDistJ + offset;
    FW = FW + normalForce;
    if (multi) MW = MW + centerDistJ.cross(normalForce);
    if (cf) set_force(*cf, normalForce, 1.0);
    const V3 relVelContact = relVel + wpg.cross(vecRadJ);
    const V3 tangRelVelContact = relVelContact - normalRelVel;
    double ft;
    V3 et, tangForce;
    if constexpr (SP) {
        tangForce = spring_force(p, fn, re, me, friction, en, tangRelVelContact, xi);
        ft = tangForce.norm();
        if (ft == 0.0) return;
        et = tangForce / ft;
    } else {
        const double nt = tangRelVelContact.norm();
        if (nt == 0.0) return;
        ft = tangential_contact(p, nt, fn, re, me, friction);
        et = tangRelVelContact / nt;
        tangForce = ft * et;
    }
    MW = MW - centerDistJ.cross(tangForce);
    FW = FW - tangForce;
    if (cf) set_force_t(*cf, tangForce);
    if (st) set_stat(*st, overlap, fn, ft, en, et);
}

// Maximum over the 64 lanes of a wavefront (order-free, so deterministic).
__device__ __forceinline__ double wave_max(double v) {
    for (int off = 32; off > 0; off >>= 1) {
        const double o = __shfl_xor(v, off, 64);
        v = o > v ? o : v;
    }
    return v;
}

// Folds a wavefront's max |x1|^2 (>= 0, or NaN) into DEMBuffers::vmax: the bit
// patterns of non-negative doubles order like the values, and NaN patterns lie
// above every finite value, so an integer atomic max keeps the maximum (order-free).
__device__ __forceinline__ void vmax_add(const DEMBuffers& b, double v2) {
    if ((threadIdx.x & 63) == 0)
        atomicMax(reinterpret_cast<unsigned long long*>(b.vmax), (unsigned long long)__double_as_longlong(v2));
}

// Gear predictor of one quantity's six derivatives (elmt.cpp:139-177), with the
// position (c2) or angular-velocity (c1) coefficients.
template <class T>
__device__ __forceinline__ void gear_predict(const T x[6], const double* c, T o[6]) {
    o[0] = x[0] + x[1] * c[0] + x[2] * c[1] + x[3] * c[2] + x[4] * c[3] + x[5] * c[4];
    o[1] = x[1] + x[2] * c[0] + x[3] * c[1] + x[4] * c[2] + x[5] * c[3];
    o[2] = x[2] + x[3] * c[0] + x[4] * c[1] + x[5] * c[2];
    o[3] = x[3] + x[4] * c[0] + x[5] * c[1];
    o[4] = x[4] + x[5] * c[0];
    o[5] = x[5];
}

}  // namespace

}  // namespace hyb
