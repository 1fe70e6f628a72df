// One DEM sub-step in three parts (DEM.cpp:331-376), each over any number of threads: the neighbour rebuild by one
// workgroup, a pair per thread, an element per thread. Launched one after the other over the whole device (dem.hip), or
// run by one workgroup where those of a whole-step launch are not resident together (dem_run.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"
#include "dem_device.h"
#include "dem_kernels.h"

namespace hyb {

namespace {

// In-place exclusive scan of a[0..n) by the whole (single) workgroup; returns the total.
template <int RB>
__device__ int block_exscan(int* a, int n) {
    __shared__ int sh[RB];
    __shared__ int carry;
    const int t = threadIdx.x;
    if (t == 0) carry = 0;
    __syncthreads();
    for (int base = 0; base < n; base += RB) {
        const int i = base + t;
        const int v = i < n ? a[i] : 0;
        sh[t] = v;
        __syncthreads();
        for (int off = 1; off < RB; off <<= 1) {
            const int add = t >= off ? sh[t - off] : 0;
            __syncthreads();
            sh[t] += add;
            __syncthreads();
        }
        const int incl = sh[t];
        const int c0 = carry;
        if (i < n) a[i] = c0 + incl - v;
        __syncthreads();
        if (t == RB - 1) carry = c0 + incl;
        __syncthreads();
    }
    const int total = carry;
    __syncthreads();
    return total;
}

// evalMaxDisp and, when the displacement trigger fires (or force), the neighbour rebuild of DEM.cpp:1369-1513, by one
// workgroup of RB lanes.
template <int RB>
__device__ __forceinline__ void rebuild_by_one(const DEMParams& p, const DEMBuffers& b, int force) {
#pragma clang fp contract(off)
    const El E{b.el, p.E};
    const int t = threadIdx.x;
    const int P = p.P;
    __shared__ double red[RB];
    __shared__ int doit;
    __shared__ int sh_err;
    if (b.st->error) return;
    if (t == 0) sh_err = 0;
    __syncthreads();
    // ---- evalMaxDisp (DEM.cpp:1314-1324) and the trigger (DEM.cpp:342-347)
    if (!force) {
        // max |x1|^2 over elements, left by the corrector (and cleared here for the
        // next one); a NaN or infinite maximum stops the DEM (error 6)
        if (t == 0) {
            unsigned long long* vb = reinterpret_cast<unsigned long long*>(b.vmax);
            const double m = __longlong_as_double((long long)*vb);
            *vb = 0ull;
            if (!(m <= 1.79769313486231570e308)) {
                sh_err = DEM_ERR_NUMERIC;
            } else {
                const double maxVel = sqrt(m);
                b.st->maxDisp += maxVel * p.deltat;
                doit = b.st->maxDisp > p.trigger;
                if (doit) b.st->maxDisp = 0.0;
            }
        }
        __syncthreads();
        if (sh_err) { if (t == 0) dem_error(p, b, DEM_ERR_NUMERIC); return; }
    } else if (t == 0) {
        doit = 1;
    }
    __syncthreads();
    if (!doit || P == 0) return;
    if (t == 0) b.st->rebuilds += 1;
    // tangential springs: keep the old pair list, springs, per-particle lists and
    // ghosts; the new pairs take over the springs of the same element pairs below
    __shared__ int oldT, oldG;
    if (p.spring) {
        if (t == 0) { oldT = b.st->nPairs; oldG = b.st->nGhost; }
        __syncthreads();
        for (int i = t; i < 2 * oldT; i += RB) b.pairsOld[i] = b.pairs[i];
        for (int i = t; i < 3 * oldT; i += RB) b.histOld[i] = b.hist[i];
        for (int i = t; i <= P; i += RB) b.csrOffOld[i] = b.csrOff[i];
        const int nc = (int)b.csrOff[P];
        for (int i = t; i < nc; i += RB) b.csrOld[i] = b.csr[i];
        for (int i = t; i < oldG; i += RB) b.ghostIndexOld[i] = b.ghostIndex[i];
        __syncthreads();
    }
    int G = 0;
    if (p.npbc) {
        // ---- pbcShift (DEM.cpp:1554-1584)
        // The predictor of this sub-step already ran (fused into the previous
        // corrector), so a shifted element gets its predicted position
        // recomputed from the shifted x0 exactly as the predictor would, and
        // its particles are placed again (updateParticlesCorrected, DEM.cpp:1398).
        for (int e = t; e < p.E; e += RB) {
            V3 x0 = E.v3(EF_X, e);
            bool moved = false;
            for (int k = 0; k < p.npbc; ++k) {
                const PbcDev& pb = p.pbc[k];
                const double left = pb.n1.dot(x0 - pb.p1);
                const double right = pb.n2.dot(x0 - pb.p2);
                if (left < 0.0) { x0 += pb.v; moved = true; }
                if (right < 0.0) { const V3 m = -1.0 * pb.v; x0 += m; moved = true; }
            }
            if (moved) {
                E.set3(EF_X, e, x0);
                const double* c2 = p.c2;
                const V3 xp0 = x0 + E.v3(EF_X + 3, e) * c2[0] + E.v3(EF_X + 6, e) * c2[1] + E.v3(EF_X + 9, e) * c2[2] +
                               E.v3(EF_X + 12, e) * c2[3] + E.v3(EF_X + 15, e) * c2[4];
                E.set3(EF_XP, e, xp0);
                if (p.clumps) place_both(E, b, e);
            }
        }
        __syncthreads();
        // ---- side ghosts in (pbc, element) order (DEM.cpp:1590-1618)
        int nSide = 0;
        for (int k = 0; k < p.npbc; ++k) {
            const PbcDev& pb = p.pbc[k];
            for (int e = t; e < P; e += RB) {  // e: standard particle
                const V3 x0 = part_x(E, p, b, e);
                const double left = pb.n1.dot(x0 - pb.p1);
                const double right = pb.n2.dot(x0 - pb.p2);
                const int flag = left < p.nebrRange ? 1 : (right < p.nebrRange ? 2 : 0);
                b.work[e] = flag ? 1 : 0;
                b.side[e * 3 + k] = flag;  // temporarily the flag
            }
            __syncthreads();
            const int tot = block_exscan<RB>(b.work, P);
            for (int e = t; e < P; e += RB) {
                const int flag = b.side[e * 3 + k];
                if (flag) {
                    const int g = nSide + b.work[e];
                    if (g < p.Gcap) {
                        b.ghostIndex[g] = (uint32_t)e;
                        const V3 v = flag == 1 ? pb.v : -1.0 * pb.v;
                        b.ghostVec[3 * g] = v.x;
                        b.ghostVec[3 * g + 1] = v.y;
                        b.ghostVec[3 * g + 2] = v.z;
                        b.ghostB[g] = k;
                    }
                    b.side[e * 3 + k] = g;
                } else {
                    b.side[e * 3 + k] = -1;
                }
            }
            nSide += tot;
            __syncthreads();
        }
        if (nSide > p.Gcap) { if (t == 0) sh_err = 1; }
        __syncthreads();
        if (sh_err) { if (t == 0) dem_error(p, b, 1); return; }
        // ---- corner ghosts: every pair g1 < g2 of side ghosts of one particle (DEM.cpp:1620-1635)
        for (int g = t; g < nSide; g += RB) {
            const int e = (int)b.ghostIndex[g];
            int c = 0;
            for (int k2 = b.ghostB[g] + 1; k2 < p.npbc; ++k2) c += b.side[e * 3 + k2] >= 0 ? 1 : 0;
            b.work[g] = c;
        }
        __syncthreads();
        const int nCorner = block_exscan<RB>(b.work, nSide);
        G = nSide + nCorner;
        if (G > p.Gcap) { if (t == 0) dem_error(p, b, 1); return; }
        for (int g = t; g < nSide; g += RB) {
            const int e = (int)b.ghostIndex[g];
            int slot = nSide + b.work[g];
            const V3 v1(b.ghostVec[3 * g], b.ghostVec[3 * g + 1], b.ghostVec[3 * g + 2]);
            for (int k2 = b.ghostB[g] + 1; k2 < p.npbc; ++k2) {
                const int g2 = b.side[e * 3 + k2];
                if (g2 < 0) continue;
                const V3 v2(b.ghostVec[3 * g2], b.ghostVec[3 * g2 + 1], b.ghostVec[3 * g2 + 2]);
                const V3 v = v1 + v2;
                b.ghostIndex[slot] = (uint32_t)e;
                b.ghostVec[3 * slot] = v.x;
                b.ghostVec[3 * slot + 1] = v.y;
                b.ghostVec[3 * slot + 2] = v.z;
                ++slot;
            }
        }
        if (t == 0) b.st->newNeighborList = 1;
        __syncthreads();
    }
    const int S = P + G;
    if (t == 0) { b.st->nGhost = G; b.st->nSlots = S; }
    // ---- linked-cell table (DEM.cpp:1326-1367): chains in descending slot order
    const int nc = b.ncells;
    for (int c = t; c <= nc; c += RB) b.cellCount[c] = 0;
    __syncthreads();
    for (int s = t; s < S; s += RB) {
        const int c = linearize(slot_pos(E, p, b, s), p.cellWidth, p.nCells) + S;
        if (c < S || c >= S + nc) {  // below S: a slot, not a cell
            sh_err = 2;
            b.cellOf[s] = 0;
        } else {
            b.cellOf[s] = c - S;
            atomicAdd(&b.cellCount[c - S], 1);
        }
    }
    __syncthreads();
    if (sh_err) { if (t == 0) dem_error(p, b, 2); return; }
    block_exscan<RB>(b.cellCount, nc + 1);
    for (int c = t; c < nc; c += RB) b.work[c] = b.cellCount[c];
    __syncthreads();
    for (int s = t; s < S; s += RB) {
        const int pos = atomicAdd(&b.work[b.cellOf[s]], 1);
        b.cursor[pos] = s;  // cursor holds the slots sorted by cell (order within a cell fixed below)
    }
    __syncthreads();
    for (int c = t; c < nc; c += RB) {
        const int lo = b.cellCount[c], hi = b.cellCount[c + 1];
        for (int i = lo + 1; i < hi; ++i) {  // insertion sort, descending
            const int v = b.cursor[i];
            int j = i - 1;
            while (j >= lo && b.cursor[j] < v) { b.cursor[j + 1] = b.cursor[j]; --j; }
            b.cursor[j + 1] = v;
        }
        b.cellTable[S + c] = hi > lo ? b.cursor[lo] : -1;
        for (int i = lo; i < hi; ++i) b.cellTable[b.cursor[i]] = (i + 1 < hi) ? b.cursor[i + 1] : -1;
    }
    __syncthreads();
    // ---- pair list in the reference's order (DEM.cpp:1425-1484): count, scan, fill
    for (int s = t; s < S; s += RB) {  // packed slot records: position, cluster
        const V3 x = slot_pos(E, p, b, s);
        double* r = b.spos + 4 * (size_t)s;
        r[0] = x.x;
        r[1] = x.y;
        r[2] = x.z;
        r[3] = (double)slot_cluster(p, b, s);
    }
    __syncthreads();
    const int W = b.W;
    for (int w = t; w < W; w += RB) {
        const int c = walk_pairs(p, b, E, S, (unsigned)w, nullptr);
        if (c < 0) { sh_err = 3; b.work[w] = 0; }
        else b.work[w] = c;
    }
    __syncthreads();
    if (sh_err) { if (t == 0) dem_error(p, b, 3); return; }
    const int T = block_exscan<RB>(b.work, W);
    if (T > p.pairCap) { if (t == 0) dem_error(p, b, 4); return; }
    for (int w = t; w < W; w += RB) walk_pairs(p, b, E, S, (unsigned)w, b.pairs + 2 * (size_t)b.work[w]);
    if (t == 0) b.st->nPairs = T;
    // ---- near-wall list (DEM.cpp:1496-1513): the first wall within range of each standard particle
    // (all walls within range as a bit mask with DEMParams::allWalls)
    int nw = 0;
    for (int e = t; e < P; e += RB) {
        const V3 x0 = part_x(E, p, b, e);
        uint32_t wi = 0xFFFFFFFFu, mask = 0u;
        for (int k = 0; k < p.nwalls; ++k)
            if (p.walls[k].dist(x0) < p.nebrRange) {
                if (wi == 0xFFFFFFFFu) wi = (uint32_t)k;
                mask |= 1u << k;
                if (!p.allWalls) break;
            }
        b.nearWall[e] = wi;
        if (p.allWalls) b.nearWallMask[e] = mask;
        nw += wi != 0xFFFFFFFFu;
        // near-cylinder list (DEM.cpp:1535-1550): the first cylinder within range
        if (p.ncyl) {
            uint32_t ci = 0xFFFFFFFFu;
            for (int k = 0; k < p.ncyl; ++k)
                if (p.cyl[k].dist(x0) < p.nebrRange) { ci = (uint32_t)k; break; }
            b.nearCyl[e] = ci;
        }
    }
    red[t] = (double)nw;
    // ---- near-object lists (DEM.cpp:1515-1532): every object within range, in list order
    if (p.nobj) {
        const double nebrRange2 = p.nebrRange * p.nebrRange;
        for (int e = t; e < P; e += RB) {
            const V3 x0 = part_x(E, p, b, e);
            int c = 0;
            for (int o = 0; o < p.nobj; ++o) {
                const V3 x0ij = x0 - b.objs[o].x0;
                if (x0ij.norm2() < nebrRange2) {
                    if (c < NEAR_OBJ) b.nearObj[(size_t)e * NEAR_OBJ + c] = (uint32_t)o;
                    ++c;
                }
            }
            if (c > NEAR_OBJ) { sh_err = 5; c = NEAR_OBJ; }
            b.nearObjCount[e] = c;
        }
    }
    __syncthreads();
    if (sh_err) { if (t == 0) dem_error(p, b, 5); return; }
    // ---- per-particle pair lists, ascending pair index
    for (int e = t; e < P; e += RB) b.cursor[e] = 0;
    __syncthreads();
    for (int k = t; k < T; k += RB) {
        const uint32_t n0 = b.pairs[2 * k], n1 = b.pairs[2 * k + 1];
        if ((int)n0 < P) atomicAdd(&b.cursor[n0], 1);
        if ((int)n1 < P) atomicAdd(&b.cursor[n1], 1);
    }
    __syncthreads();
    for (int e = t; e < P; e += RB) b.work[e] = b.cursor[e];
    __syncthreads();
    const int tot2 = block_exscan<RB>(b.work, P);
    for (int e = t; e < P; e += RB) { b.csrOff[e] = (uint32_t)b.work[e]; b.cursor[e] = b.work[e]; }
    if (t == 0) b.csrOff[P] = (uint32_t)tot2;
    __syncthreads();
    for (int k = t; k < T; k += RB) {
        const uint32_t n0 = b.pairs[2 * k], n1 = b.pairs[2 * k + 1];
        if ((int)n0 < P) b.csr[atomicAdd(&b.cursor[n0], 1)] = (uint32_t)k;
        if ((int)n1 < P) b.csr[atomicAdd(&b.cursor[n1], 1)] = (uint32_t)k;
    }
    __syncthreads();
    for (int e = t; e < P; e += RB) {
        const int lo = (int)b.csrOff[e], hi = (int)b.csrOff[e + 1];
        for (int i = lo + 1; i < hi; ++i) {
            const uint32_t v = b.csr[i];
            int j = i - 1;
            while (j >= lo && b.csr[j] > v) { b.csr[j + 1] = b.csr[j]; --j; }
            b.csr[j + 1] = v;
        }
    }
    // ---- slot of each pair in its particles' lists
    for (int k = t; k < T; k += RB) { b.posI[k] = 0xFFFFFFFFu; b.posJ[k] = 0xFFFFFFFFu; }
    __syncthreads();
    for (int e = t; e < P; e += RB) {
        const int lo = (int)b.csrOff[e], hi = (int)b.csrOff[e + 1];
        for (int i = lo; i < hi; ++i) {
            const uint32_t k = b.csr[i];
            if ((int)b.pairs[2 * k] == e) b.posI[k] = (uint32_t)i;
            else b.posJ[k] = (uint32_t)i;
        }
    }
    // ---- ghost slots of each particle, ascending (for the hydrodynamic sums)
    for (int e = t; e < P; e += RB) b.ghostOfCount[e] = 0;
    __syncthreads();
    for (int g = t; g < G; g += RB) {
        const int e = (int)b.ghostIndex[g];
        const int k = atomicAdd(&b.ghostOfCount[e], 1);
        if (k < 8) b.ghostOf[e * 8 + k] = P + g;
    }
    __syncthreads();
    for (int e = t; e < P; e += RB) {
        const int n = b.ghostOfCount[e] < 8 ? b.ghostOfCount[e] : 8;
        int* l = b.ghostOf + e * 8;
        for (int i = 1; i < n; ++i) {
            const int v = l[i];
            int j = i - 1;
            while (j >= 0 && l[j] > v) { l[j + 1] = l[j]; --j; }
            l[j + 1] = v;
        }
    }
    // near-wall count
    for (int w = RB / 2; w > 0; w >>= 1) {
        if (t < w) red[t] += red[t + w];
        __syncthreads();
    }
    if (t == 0) b.st->nNearWall = (int)red[0];
    if (p.spring) {
        // a new pair takes the spring of the old pair of the same two standard
        // particles (ghosts count as their origin; found in the old lists of
        // either particle), turned to the new pair's orientation; pairs without
        // one start with a released spring
        for (int k = t; k < T; k += RB) {
            const int n0 = (int)b.pairs[2 * k], n1 = (int)b.pairs[2 * k + 1];
            const int e0 = n0 < P ? n0 : (int)b.ghostIndex[n0 - P];
            const int e1 = n1 < P ? n1 : (int)b.ghostIndex[n1 - P];
            double xi[3] = {0.0, 0.0, 0.0};
            bool found = false;
            for (int side = 0; side < 2 && !found; ++side) {
                const int e = side == 0 ? e0 : e1;
                for (uint32_t i = b.csrOffOld[e]; i < b.csrOffOld[e + 1]; ++i) {
                    const uint32_t kk = b.csrOld[i];
                    const int m0 = (int)b.pairsOld[2 * kk], m1 = (int)b.pairsOld[2 * kk + 1];
                    const int f0 = m0 < P ? m0 : (int)b.ghostIndexOld[m0 - P];
                    const int f1 = m1 < P ? m1 : (int)b.ghostIndexOld[m1 - P];
                    double sgn = 0.0;
                    if (f0 == e0 && f1 == e1) sgn = 1.0;
                    else if (f0 == e1 && f1 == e0) sgn = -1.0;
                    if (sgn == 0.0) continue;
                    for (int c = 0; c < 3; ++c) xi[c] = sgn * b.histOld[3 * (size_t)kk + c];
                    found = true;
                    break;
                }
            }
            for (int c = 0; c < 3; ++c) b.hist[3 * (size_t)k + c] = xi[c];
        }
    }
}

// Predicted position, velocity and radiusVec of a particle slot and its element
// (updateParticlesPredicted, DEM.cpp:1184-1204; a ghost is its origin moved by
// the period vector, with the origin's velocity and radiusVec, elmt.cpp:292-298).
template <bool CL>
__device__ __forceinline__ void slot_pred(const El& E, const DEMParams& p, const DEMBuffers& b, int s, V3& x, V3& v,
                                          V3& rv, int& elem) {
    const int o = s < p.P ? s : (int)b.ghostIndex[s - p.P];
    if constexpr (CL) {
        const double* c = b.ppred + 9 * (size_t)o;
        x = V3(c[0], c[1], c[2]);
        v = V3(c[3], c[4], c[5]);
        rv = V3(c[6], c[7], c[8]);
        elem = b.pelem[o];
    } else {
        x = E.v3(EF_XP, o);
        v = E.v3(EF_XP + 3, o);
        rv = V3(0.0, 0.0, 0.0);
        elem = o;
    }
    if (s >= p.P) {
        const int g = s - p.P;
        x = x + V3(b.ghostVec[3 * g], b.ghostVec[3 * g + 1], b.ghostVec[3 * g + 2]);
    }
}

// Number of spheres of element e.
template <bool CL>
__device__ __forceinline__ int elem_size(const DEMBuffers& b, int e) {
    if constexpr (CL) return b.efirst[e + 1] - b.efirst[e];
    return 1;
}

// The contact of neighbour pair k (DEM.cpp:1801-1900) at the predicted state:
// the signed increments for the pair's first (ri) and second (rj) particle's
// element, the normal-force moments of elements of size > 1 (mnI, mnJ; flag
// bit 2), and its statistics record st.
// SP: tangential spring (xi: the pair's spring); CL: multi-sphere elements present.
template <bool SP, bool CL>
__device__ __forceinline__ void pair_contact(const DEMParams& p, const DEMBuffers& b, const El& E, int k, PairRec& ri,
                                             PairRec& rj, StatRec& st, double* xi, V3& mnI, V3& mnJ) {
#pragma clang fp contract(off)
    const int n0 = (int)b.pairs[2 * k], n1 = (int)b.pairs[2 * k + 1];
    V3 xI, vI, rvI, xJ, vJ, rvJ;
    int eI, eJ;
    slot_pred<CL>(E, p, b, n0, xI, vI, rvI, eI);
    slot_pred<CL>(E, p, b, n1, xJ, vJ, rvJ, eJ);
    const double rI = E.at(EF_RAD, eI), rJ = E.at(EF_RAD, eJ);
    const double sigij = rI + rJ;
    const double sigij2 = sigij * sigij;
    const V3 vd = xJ - xI;
    ri.flag = rj.flag = 0;
    ri.pad = rj.pad = 0;
    st = StatRec{(double)n0, (double)n1, 0.0, 0.0, 0.0, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, 0.0};
    if (!(vd.norm2() < sigij2)) {
        if constexpr (SP) xi[0] = xi[1] = xi[2] = 0.0;  // out of contact: the spring is released
        return;
    }
    const double distance = vd.norm();
    const double overlap = rI + rJ - distance;
    const V3 relVel = vJ - vI;
    const V3 en = vd / distance;
    const double normRelVel = relVel.dot(en);
    const V3 normalRelVel = en * normRelVel;
    const double mI = E.at(EF_M, eI), mJ = E.at(EF_M, eJ);
    const double effMass = mI * mJ / (mI + mJ);
    const double effRad = rI * rJ / (rI + rJ);
    const double fn = normal_contact(p, overlap, normRelVel, effRad, effMass);
    const V3 normalForce = en * fn;
    const V3 vecRadI = rI * en;
    const V3 vecRadJ = -rJ * en;
    // radiusVec is zero for single-sphere elements
    const V3 centerDistI = vecRadI + rvI;
    const V3 centerDistJ = vecRadJ + rvJ;
    const V3 mn = -1.0 * normalForce;
    ri.fn[0] = mn.x; ri.fn[1] = mn.y; ri.fn[2] = mn.z;  // F - n == F + (-n)
    rj.fn[0] = normalForce.x; rj.fn[1] = normalForce.y; rj.fn[2] = normalForce.z;
    ri.flag = rj.flag = 1;
    if constexpr (CL) {  // only elements of size > 1 take the normal force's moment (DEM.cpp:1862-1867)
        if (elem_size<CL>(b, eI) > 1) {
            mnI = -1.0 * centerDistI.cross(normalForce);  // M - c x F == M + (-(c x F))
            ri.flag = 5;
        }
        if (elem_size<CL>(b, eJ) > 1) {
            mnJ = centerDistJ.cross(normalForce);
            rj.flag = 5;
        }
    }
    const V3 wI = E.v3(EF_WPG, eI), wJ = E.v3(EF_WPG, eJ);
    const V3 relVelContact = relVel - wI.cross(vecRadI) + wJ.cross(vecRadJ);
    const V3 tangRelVelContact = relVelContact - normalRelVel;
    double nt, ft;
    V3 et, tangForce;
    if constexpr (SP) {
        tangForce = spring_force(p, fn, effRad, effMass, p.fricPart, en, tangRelVelContact, xi);
        nt = tangForce.norm();
        ft = nt;
        if (nt != 0.0) et = tangForce / nt;
    } else {
        nt = tangRelVelContact.norm();
        if (nt != 0.0) {
            ft = tangential_contact(p, nt, fn, effRad, effMass, p.fricPart);
            et = tangRelVelContact / nt;
            tangForce = ft * et;
        }
    }
    if (nt != 0.0) {
        const V3 mI3 = centerDistI.cross(tangForce);
        const V3 mJ3 = -1.0 * centerDistJ.cross(tangForce);
        const V3 mt = -1.0 * tangForce;
        ri.ft[0] = tangForce.x; ri.ft[1] = tangForce.y; ri.ft[2] = tangForce.z;
        ri.m[0] = mI3.x; ri.m[1] = mI3.y; ri.m[2] = mI3.z;
        rj.ft[0] = mt.x; rj.ft[1] = mt.y; rj.ft[2] = mt.z;
        rj.m[0] = mJ3.x; rj.m[1] = mJ3.y; rj.m[2] = mJ3.z;
        ri.flag |= 2;
        rj.flag |= 2;
        set_stat(st, overlap, fn, ft, en, et);
    }
}

// Pair k at the predicted state; the signed increments for each of its two elements go into that element's slot of the
// pair in its csr list, so that gather_elem adds them in pair-list order.
template <bool SP, bool CL>
__device__ __forceinline__ void eval_pair(const DEMParams& p, const DEMBuffers& b, const El& E, int k) {
    const uint32_t si = b.posI[k], sj = b.posJ[k];
    PairRec ri, rj;
    StatRec st;
    double xi[3];
    if constexpr (SP) {
        xi[0] = b.hist[3 * (size_t)k]; xi[1] = b.hist[3 * (size_t)k + 1]; xi[2] = b.hist[3 * (size_t)k + 2];
    }
    V3 mnI, mnJ;
    pair_contact<SP, CL>(p, b, E, k, ri, rj, st, xi, mnI, mnJ);
    if constexpr (SP) {
        b.hist[3 * (size_t)k] = xi[0]; b.hist[3 * (size_t)k + 1] = xi[1]; b.hist[3 * (size_t)k + 2] = xi[2];
    }
    if (b.pstat) b.pstat[k] = st;
    // a record without contact is read only for its flag: the other fields are not rewritten
    if (si != 0xFFFFFFFFu) {
        if (ri.flag) b.prec[si] = ri;
        else b.prec[si].flag = 0;
    }
    if (sj != 0xFFFFFFFFu) {
        if (rj.flag) b.prec[sj] = rj;
        else b.prec[sj].flag = 0;
    }
    if constexpr (CL) {
        if (si != 0xFFFFFFFFu && (ri.flag & 4)) {
            b.pmn[3 * (size_t)si] = mnI.x; b.pmn[3 * (size_t)si + 1] = mnI.y; b.pmn[3 * (size_t)si + 2] = mnI.z;
        }
        if (sj != 0xFFFFFFFFu && (rj.flag & 4)) {
            b.pmn[3 * (size_t)sj] = mnJ.x; b.pmn[3 * (size_t)sj + 1] = mnJ.y; b.pmn[3 * (size_t)sj + 2] = mnJ.z;
        }
    }
}

// Gear predictor of one element from its corrected state (elmt.cpp:139-177).
template <bool CL>
__device__ __forceinline__ void predict_elem(const El& E, const DEMParams& p, const DEMBuffers& b, int e, const V3 x[6],
                                             const Q4 q[6], const V3 w[6]) {
    V3 xp[6], wp[6];
    Q4 qp[6];
    gear_predict(x, p.c2, xp);
    gear_predict(q, p.c2, qp);
    qp[0].normalize();
    gear_predict(w, p.c1, wp);
    for (int k = 0; k < 6; ++k) {
        E.set3(EF_XP + 3 * k, e, xp[k]);
        E.set4(EF_QP + 4 * k, e, qp[k]);
        E.set3(EF_WP + 3 * k, e, wp[k]);
    }
    E.set3(EF_WPG, e, wp[0]);
    E.set3(EF_WPL, e, project(wp[0], qp[0].adjoint()));
    // particles from the predicted element (updateParticlesPredicted, DEM.cpp:1184-1204)
    if constexpr (CL) place_particles(b, b.ppred, e, E.at(EF_RAD, e), xp[0], xp[1], qp[0], wp[0]);
}

// Per element: particle-contact increments in pair-list order, the wall contact
// (DEM.cpp:1692-1717, 1902-1982), Newton-Euler (DEM.cpp:1149-1181), the Gear
// corrector (elmt.cpp:179-254) and the predictor of the next sub-step.
// Returns |x1|^2 of the corrected element for the next displacement check.
// SP: tangential spring; CL: multi-sphere elements present.
template <bool SP, bool CL>
__device__ __forceinline__ double gather_elem(const DEMParams& p, const DEMBuffers& b, int e) {
#pragma clang fp contract(off)
    const El E{b.el, p.E};
    V3 FP(0.0, 0.0, 0.0), MP(0.0, 0.0, 0.0), FW(0.0, 0.0, 0.0), MW(0.0, 0.0, 0.0);
    // the element's standard particles (consecutive; a single sphere is its own particle)
    const int ilo = CL ? b.efirst[e] : e, ihi = CL ? b.efirst[e + 1] : e + 1;
    const bool multi = CL && ihi - ilo > 1;
    // the state the contacts and Newton-Euler need; it does not depend on the
    // contact records, so its loads are issued first (the rest of the Gear state is
    // loaded group by group in the corrector, which keeps the registers in use low)
    const V3 xpe = E.v3(EF_XP, e);
    const V3 vpe = E.v3(EF_XP + 3, e);
    const double re = E.at(EF_RAD, e), me = E.at(EF_M, e);
    const V3 wpg = E.v3(EF_WPG, e);
    const V3 FH = E.v3(EF_FH, e), MH = E.v3(EF_MH, e);
    const V3 Ie = E.v3(EF_I, e), wpl = E.v3(EF_WPL, e);
    Q4 q2 = E.q4(EF_Q + 8, e);  // single spheres: q2 is never set by the force routine
    const Q4 qp0 = E.q4(EF_QP, e), qp1 = E.q4(EF_QP + 4, e);
    // contact increments in pair-list order
    const auto add = [&](const PairRec& r) {
        const int flag = r.flag;
        if (flag & 1) FP = FP + V3(r.fn[0], r.fn[1], r.fn[2]);
        if (flag & 2) {
            MP = MP + V3(r.m[0], r.m[1], r.m[2]);
            FP = FP + V3(r.ft[0], r.ft[1], r.ft[2]);
        }
    };
    if (!multi) {  // one list; records are loaded GU at a time
        const uint32_t lo = b.csrOff[ilo], hi = b.csrOff[ilo + 1];
        constexpr uint32_t GU = 4;
        uint32_t i = lo;
        for (; i + GU <= hi; i += GU) {
            PairRec r[GU];
#pragma unroll
            for (uint32_t k = 0; k < GU; ++k) r[k] = b.prec[i + k];
#pragma unroll
            for (uint32_t k = 0; k < GU; ++k) add(r[k]);
        }
        for (; i < hi; ++i) add(b.prec[i]);
    } else {
        // the lists of the element's particles merged by pair index: every pair
        // of the element appears in exactly one of them (pairs within one
        // element are never listed), so this is the reference's pair order
        constexpr int MAXS = 4;
        uint32_t cur[MAXS], end[MAXS];
        const int nl = ihi - ilo;
        for (int l = 0; l < MAXS; ++l) {
            cur[l] = l < nl ? b.csrOff[ilo + l] : 0u;
            end[l] = l < nl ? b.csrOff[ilo + l + 1] : 0u;
        }
        for (;;) {
            int best = -1;
            uint32_t bk = 0xFFFFFFFFu;
            for (int l = 0; l < nl; ++l)
                if (cur[l] < end[l]) {
                    const uint32_t k = b.csr[cur[l]];
                    if (k < bk) { bk = k; best = l; }
                }
            if (best < 0) break;
            const uint32_t i = cur[best]++;
            const PairRec r = b.prec[i];
            if (r.flag & 1) FP = FP + V3(r.fn[0], r.fn[1], r.fn[2]);
            if (r.flag & 4) MP = MP + V3(b.pmn[3 * (size_t)i], b.pmn[3 * (size_t)i + 1], b.pmn[3 * (size_t)i + 2]);
            if (r.flag & 2) {
                MP = MP + V3(r.m[0], r.m[1], r.m[2]);
                FP = FP + V3(r.ft[0], r.ft[1], r.ft[2]);
            }
        }
    }
    // predicted position and velocity of standard particle i of this element
    const auto part_pred = [&](int i, V3& px, V3& pv) {
        if constexpr (CL) {
            const double* c = b.ppred + 9 * (size_t)i;
            px = V3(c[0], c[1], c[2]);
            pv = V3(c[3], c[4], c[5]);
        } else {
            px = xpe;
            pv = vpe;
        }
    };
    // the contact of standard particle i (predicted px, pv) with wall wi (DEM.cpp:1902-1982): adds to FW, MW
    // and fills its force record and statistics; wxi: the spring (spring model)
    const auto wall_contact = [&](int i, uint32_t wi, const V3& px, const V3& pv, ContactForce& wcf, StatRec& wst,
                                  double wxi[3]) -> bool {
        const WallDev& w = p.walls[wi];
        const double distance = w.dist(px);
        const double overlap = re - distance;
        if (!(overlap > 0.0)) return false;
        surface_contact<SP>(p, re, me, overlap, w.n, pv - w.getSpeed(px), wpg, multi, px - xpe, p.fricWall, wxi, FW, MW,
                            &wcf, b.wstat ? &wst : nullptr);
        return true;
    };
    // wall contacts of the element's particles (DEM.cpp:1692-1717): the first wall within range of each
    // particle, or every wall within range in wall order (DEMParams::allWalls; record i * nwalls + w)
    for (int i = ilo; i < ihi; ++i) {
        V3 px, pv;
        part_pred(i, px, pv);
        if (p.allWalls) {
            const uint32_t mask = b.nearWallMask[i];
            const int ws = p.nwalls;
            for (int wi = 0; wi < ws; ++wi) {
                const size_t slot = (size_t)i * ws + wi;
                StatRec wst{(mask >> wi & 1u) ? (double)wi : -1.0, (double)i, 0.0, 0.0, 0.0, {0.0, 0.0, 0.0},
                            {0.0, 0.0, 0.0}, 0.0};
                ContactForce wcf{{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, 0.0, 0.0};
                // spring model: one spring per (particle, wall), kept while that wall stays in contact
                double wxi[3] = {0.0, 0.0, 0.0};
                bool wcontact = false;
                if (mask >> wi & 1u) {
                    if (SP && b.whist[4 * slot + 3] == (double)wi) {
                        wxi[0] = b.whist[4 * slot]; wxi[1] = b.whist[4 * slot + 1]; wxi[2] = b.whist[4 * slot + 2];
                    }
                    wcontact = wall_contact(i, (uint32_t)wi, px, pv, wcf, wst, wxi);
                }
                b.wcf[slot] = wcf;
                if (b.wstat) b.wstat[slot] = wst;
                if constexpr (SP) {
                    double* wh = b.whist + 4 * slot;
                    wh[0] = wcontact ? wxi[0] : 0.0;
                    wh[1] = wcontact ? wxi[1] : 0.0;
                    wh[2] = wcontact ? wxi[2] : 0.0;
                    wh[3] = wcontact ? (double)wi : -1.0;
                }
            }
            continue;
        }
        const uint32_t wi = b.nearWall[i];
        StatRec wst{wi == 0xFFFFFFFFu ? -1.0 : (double)wi, (double)i, 0.0, 0.0, 0.0, {0.0, 0.0, 0.0},
                    {0.0, 0.0, 0.0}, 0.0};
        ContactForce wcf{{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, 0.0, 0.0};
        // spring against the near wall (spring model): kept while the same wall stays in contact
        double wxi[3] = {0.0, 0.0, 0.0};
        bool wcontact = false;
        if (SP && wi != 0xFFFFFFFFu && b.whist[4 * (size_t)i + 3] == (double)wi) {
            wxi[0] = b.whist[4 * (size_t)i]; wxi[1] = b.whist[4 * (size_t)i + 1]; wxi[2] = b.whist[4 * (size_t)i + 2];
        }
        if (wi != 0xFFFFFFFFu) {
            wcontact = wall_contact(i, wi, px, pv, wcf, wst, wxi);
            b.wcf[i] = wcf;
        }
        if constexpr (SP) {
            double* wh = b.whist + 4 * (size_t)i;
            wh[0] = wcontact ? wxi[0] : 0.0;
            wh[1] = wcontact ? wxi[1] : 0.0;
            wh[2] = wcontact ? wxi[2] : 0.0;
            wh[3] = wcontact ? (double)wi : -1.0;
        }
        if (b.wstat) b.wstat[i] = wst;
    }
    // object contacts (DEM.cpp:1747-1770, 2060-2136), in list order after the walls
    if (p.nobj) {
        for (int i = ilo; i < ihi; ++i) {
            V3 px, pv;
            part_pred(i, px, pv);
            const int no = b.nearObjCount[i];
            if (b.ostat)
                for (int k = no; k < NEAR_OBJ; ++k)
                    b.ostat[(size_t)i * NEAR_OBJ + k] = StatRec{-1.0, (double)i, 0.0, 0.0, 0.0, {0.0, 0.0, 0.0},
                                                                {0.0, 0.0, 0.0}, 0.0};
            for (int k = 0; k < no; ++k) {
                const uint32_t oslot = b.nearObj[(size_t)i * NEAR_OBJ + k];
                const ObjDev& ob = b.objs[oslot];
                const V3 vectorDistance = px - ob.x0;
                const double distance = vectorDistance.norm();
                const double overlap = re + ob.r - distance;
                StatRec ost{(double)oslot, (double)i, 0.0, 0.0, 0.0, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, 0.0};
                ContactForce ocf{{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, 0.0, 0.0};
                if (!(overlap > 0.0)) {
                    if (b.ostat) b.ostat[(size_t)i * NEAR_OBJ + k] = ost;
                    b.ocf[(size_t)i * NEAR_OBJ + k] = ocf;
                    continue;
                }
                const V3 en = (1.0 / distance) * vectorDistance;
                surface_contact<false>(p, re, me, overlap, en, pv - ob.x1, wpg, multi, px - xpe, p.fricPart, nullptr, FW,
                                       MW, &ocf, b.ostat ? &ost : nullptr);
                if (b.ostat) b.ostat[(size_t)i * NEAR_OBJ + k] = ost;
                b.ocf[(size_t)i * NEAR_OBJ + k] = ocf;
            }
        }
    }
    // cylinder contacts (DEM.cpp:1719-1744, 1984-2058), after the objects
    if (p.ncyl) {
        for (int i = ilo; i < ihi; ++i) {
            const uint32_t ci = b.nearCyl[i];
            if (ci == 0xFFFFFFFFu) continue;
            V3 px, pv;
            part_pred(i, px, pv);
            const CylDev& cyl = p.cyl[ci];
            const double distance = cyl.dist(px);
            const double overlap = re - distance;
            if (!(overlap > 0.0)) continue;
            const V3 vecDistance = cyl.vecDist(px);
            const V3 contactPoint = px - vecDistance;
            const V3 en = vecDistance / (re - overlap);
            surface_contact<false>(p, re, me, overlap, en, pv - cyl.getSpeed(contactPoint), wpg, multi, px - xpe,
                                   p.fricWall, nullptr, FW, MW, nullptr, nullptr);
        }
    }
    // Newton-Euler
    const V3 xp1 = vpe;
    const double rad = re;
    const V3 FVisc = -6.0 * M_PI * p.numVisc * rad * xp1;
    const V3 MVisc = -8.0 * M_PI * p.numVisc * rad * rad * rad * wpg;
    const V3 demF(p.demF[0], p.demF[1], p.demF[2]);
    const V3 x2 = (FVisc + FH + FP + FW) / me + demF;
    const V3 moment = MVisc + MH + MP + MW;
    const V3 momentBf = project(moment, qp0.adjoint());
    const V3 waBf = newtonAcc(momentBf, Ie, wpl);
    const V3 w1 = project(waBf, qp0);
    if (multi) {  // rotational acceleration as a quaternion (DEM.cpp:1176-1179)
        const Q4 waQuat = quatAcc(waBf, qp1);
        q2 = 0.5 * qp0.multiply(waQuat);
    }
    E.set3(EF_FP, e, FP); E.set3(EF_MP, e, MP); E.set3(EF_FW, e, FW); E.set3(EF_MW, e, MW);
    // corrector (elmt.cpp:179-254) and the next sub-step's predictor, one quantity at a time
    const double* co1 = p.co1;
    const double* co2 = p.co2;
    V3 xc[2], xn[2];  // corrected and predicted position and velocity
    {
        const V3 xp[6] = {xpe, vpe, E.v3(EF_XP + 6, e), E.v3(EF_XP + 9, e), E.v3(EF_XP + 12, e), E.v3(EF_XP + 15, e)};
        const V3 x2Corr = x2 - xp[2];
        V3 x[6], o[6];
        x[0] = xp[0] + x2Corr * co2[0];
        x[1] = xp[1] + x2Corr * co2[1];
        x[2] = x2;
        x[3] = xp[3] + x2Corr * co2[3];
        x[4] = xp[4] + x2Corr * co2[4];
        x[5] = xp[5] + x2Corr * co2[5];
        gear_predict(x, p.c2, o);
        for (int k = 0; k < 6; ++k) {
            E.set3(EF_X + 3 * k, e, x[k]);
            E.set3(EF_XP + 3 * k, e, o[k]);
        }
        xc[0] = x[0]; xc[1] = x[1];
        xn[0] = o[0]; xn[1] = o[1];
    }
    Q4 qc0, qn0;  // corrected and predicted orientation
    {
        const Q4 qp[6] = {qp0, qp1, E.q4(EF_QP + 8, e), E.q4(EF_QP + 12, e), E.q4(EF_QP + 16, e), E.q4(EF_QP + 20, e)};
        const Q4 q2Corr = q2 - qp[2];
        Q4 q[6], o[6];
        q[0] = qp[0] + q2Corr * co2[0];
        q[1] = qp[1] + q2Corr * co2[1];
        q[2] = q2;
        q[3] = qp[3] + q2Corr * co2[3];
        q[4] = qp[4] + q2Corr * co2[4];
        q[5] = qp[5] + q2Corr * co2[5];
        q[0].normalize();
        gear_predict(q, p.c2, o);
        o[0].normalize();
        for (int k = 0; k < 6; ++k) {
            if (k != 2 || multi) E.set4(EF_Q + 4 * k, e, q[k]);
            E.set4(EF_QP + 4 * k, e, o[k]);
        }
        qc0 = q[0];
        qn0 = o[0];
    }
    V3 wc0, wn0;  // corrected and predicted angular velocity
    {
        const V3 wp[6] = {E.v3(EF_WP, e), E.v3(EF_WP + 3, e), E.v3(EF_WP + 6, e), E.v3(EF_WP + 9, e),
                          E.v3(EF_WP + 12, e), E.v3(EF_WP + 15, e)};
        const V3 w1Corr = w1 - wp[1];
        V3 w[6], o[6];
        w[0] = wp[0] + w1Corr * co1[0];
        w[1] = w1;
        w[2] = wp[2] + w1Corr * co1[2];
        w[3] = wp[3] + w1Corr * co1[3];
        w[4] = wp[4] + w1Corr * co1[4];
        w[5] = wp[5] + w1Corr * co1[5];
        gear_predict(w, p.c1, o);
        for (int k = 0; k < 6; ++k) {
            E.set3(EF_W + 3 * k, e, w[k]);
            E.set3(EF_WP + 3 * k, e, o[k]);
        }
        E.set3(EF_WG, e, w[0]);
        E.set3(EF_WL, e, project(w[0], qc0.adjoint()));
        E.set3(EF_WPG, e, o[0]);
        E.set3(EF_WPL, e, project(o[0], qn0.adjoint()));
        wc0 = w[0];
        wn0 = o[0];
    }
    // particles from the corrected and from the predicted element (updateParticlesCorrected and
    // updateParticlesPredicted, DEM.cpp:1184-1227)
    if constexpr (CL) {
        place_particles(b, b.pcor, e, re, xc[0], xc[1], qc0, wc0);
        place_particles(b, b.ppred, e, re, xn[0], xn[1], qn0, wn0);
    }
    return xc[1].norm2();
}

}  // namespace

}  // namespace hyb
