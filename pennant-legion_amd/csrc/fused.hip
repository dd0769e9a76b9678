// Fused PENNANT cycle for gfx950.
//
// The reference issues ~36 launches per cycle (src/Hydro.cc:342-983), each a
// streaming pass over sides, zones or points with intermediate arrays in
// memory.  Every task from advPosHalf to setVelDiff only couples a zone to
// its own sides and corners, so the whole predictor half of doCycle is one
// zone-local computation; the only cross-zone couplings are the two point
// sums (corner mass, corner force) and the corrector's point positions.  The
// fused cycle is therefore three streaming passes and a one-block finalize:
//
//   K1 zone pass   advPosHalf (per corner), calcCtrs, calcVols, calcSurfVecs,
//                  calcEdgeLen, calcCharLen, calcRho, calcCrnrMass (per-corner
//                  mass), calcStateHalf, calcForcePGas, calcForceTTS,
//                  setCornerDiv, setQCnForce, setForceQCS, setVelDiff, the
//                  corner force of sumCrnrForce, calcDtNew's per-zone dt
//   K2 point pass  corner-mass and corner-force sums (ascending side order;
//                  K1 stores each corner's values at its point's slot for
//                  that corner, corner-major so that neighbouring points'
//                  slots are adjacent), applyFixedBC, calcAccel, advPosFull
//   K3 zone pass   calcCtrs, calcVols (corrector), calcWork, calcWorkRate,
//                  calcEnergy, calcRho, calcDvol's per-zone ratio
//   K4 finalize    dt minimum, dvol maximum and bad-side counts over the
//                  block partials of K1 and K3, calcDt, checkBadSides, the
//                  time/cycle update and calcGlobalDt for the next cycle
//
// Every expression is evaluated exactly as in the task kernels (and the
// reference's serial bodies), so the end-of-cycle state is bit-identical to
// the task-by-task path.  Each kernel starts by reading the device `done`
// flag, which plays the role of the reference's cycle predicate
// (src/Driver.cc:140-144): launches after the stop condition do nothing, so
// the host can queue many cycles without reading anything back.
//
// K1 has two layouts, chosen per problem (pennant_set_tuning):
//   zone-per-thread  one thread holds a whole zone in registers: no
//                    redundant zone-level arithmetic (EOS, density, dt);
//   corner-per-lane  a zone with NS sides occupies NS adjacent lanes of a
//                    64-lane wave (16 quads or 21 triangles per wave); side
//                    arrays are read and written fully coalesced and zone
//                    sums read the group's values with cross-lane shuffles in
//                    ascending corner order, so every lane of the group forms
//                    the same sum in the reference's order.
// K1 and K3 are grid-stride kernels with a bounded grid, each block writing
// one partial per reduction (no same-address atomics on the hot path).  The
// host launches K1 and K3 once per run of consecutive zones with equal side
// count (rect: one run of quads; pie: triangles, then quads).
#include <algorithm>
#include <cstring>
#include <type_traits>

#include "closure.h"
#include "common.h"
#include "cycle_end.h"
#include "problem.h"

using namespace pn;

#define PN_FIN_BLOCK 256     // finalize block size

namespace {

struct FusedArgs {
    // mesh
    const int32_t* mapsp1;
    const int32_t* pcbeg;
    const int32_t* pcpos;      // side -> slot of its corner record (corner_slot)
    const double* smf;
    int nump;
    int npown;                 // K2 updates points [0, npown)
    int la_npred;              // pipelined cycle: K2's last block folds a redone predictor's partials
    // state (in place)
    double* pxx; double* pxy; double* pux; double* puy;
    double* oxx; double* oxy; double* oux; double* ouy;   // K2's new point state (the arrays above, or a tile cycle's others)
    double* zr; double* ze; double* zetot; double* zwrate; double* zvol; double* zp;
    const double* zm;
    double* zpn;               // pipelined mixed cycle: the look-ahead predictor's zp
    // per-side intermediates
    double* cfx; double* cfy; double* cmass; double* sfwx; double* sfwy;
    // the mixed-precision form's FP32 counterparts, and smf in FP32
    float* fcrn;               // per corner slot {fx, fy, mass} (corner_slot order)
    float* fsfw;               // per side {x, y}
    const float* fsmf;
    // per-point intermediates
    double* vs2; double* pxpx;   // vs2: per point {x, y} (see point_update)
    const unsigned char* pbc;
    const int* heavy;
    int nheavy;
    // block partials
    double* part_dt; double* part_dv; int* part_bp; int* part_bc;
    Ctl* ctl;
    // physics parameters
    double gamma, ssmin, alfa, qgamma, q1, q2, cfl;
    int nbcs;
    const double* bcv;         // BC plane normals: x components [0, 8), y components [8, 16)
    int xcd;   // XCD-aware unit mapping in the grid-stride kernels
    // learned closure and training-tuple capture
    const ClosurePack* pack;
    float* cap_buf;
    long long cap;
    unsigned long long* cap_count;
    unsigned long long* cl_stats;
    // structured rect mesh (rect_nzx > 0): points and corner slots of a zone
    // from its index instead of mapsp1 and pcpos (rect_zone)
    int rect_nzx;
    unsigned long long rect_m;  // z / nzx = (z * rect_m) >> rect_sh
    int rect_sh;
    int rect_so, rect_po;       // the mesh's first side and point in the arrays (a batch's arena)
    int* zlist;                // zones for the learned pass, run r at [zbeg_r, zend_r)
    unsigned* zcount;          // per run and list slice (list_count)
    int nzruns;
};

// Work units of a grid-stride launch.  MI355X dispatches workgroups to its 8
// XCDs round-robin by workgroup id, and each XCD has its own L2; with `xcd`
// set (and a grid that is a multiple of 8) XCD x's blocks take the x-th
// contiguous eighth of the units, so neighbouring zones -- which share points
// and write neighbouring point-corner slots -- meet in the same L2.
struct Units {
    int u, end, step;
    int band;   // the eighth of the units (x) with `xcd`, else 0
};
__device__ __forceinline__ Units block_units(int nunits, int xcd) {
    const int G = gridDim.x, b = blockIdx.x;
    Units r;
    if (xcd && G >= 8 && (G & 7) == 0) {
        const int x = b & 7, per = G >> 3;
        r.u = (int)((long long)nunits * x / 8) + (b >> 3);
        r.end = (int)((long long)nunits * (x + 1) / 8);
        r.step = per;
        r.band = x;
    } else {
        r.u = b;
        r.end = nunits;
        r.step = G;
        r.band = 0;
    }
    return r;
}

template <int NS>
__device__ __forceinline__ int nxt(int k) { return (k + 1 == NS) ? 0 : k + 1; }
template <int NS>
__device__ __forceinline__ int prv(int k) { return (k == 0) ? NS - 1 : k - 1; }

// Streaming accesses (each element touched once per kernel): nontemporal
// loads and stores, which a plain copy kernel measures 9% faster than
// ordinary ones on MI355X.
template <class T>
__device__ __forceinline__ T ld_nt(const T* p) { return __builtin_nontemporal_load(p); }
template <class T>
__device__ __forceinline__ void st_nt(T v, T* p) { __builtin_nontemporal_store(v, p); }

// A structured rect mesh, as the generator numbers it (the set-up checks
// every side against mapsp1 and pcpos before it sets a.rect_nzx): zone
// z = zy nzx + zx has sides 4z .. 4z + 3 from points p0, p0 + 1,
// p0 + 1 + npx, p0 + npx (npx = nzx + 1, p0 = zy npx + zx = z + zy), and the
// corner of side k is the rank-th corner of its point in ascending side
// order -- the number of the point's zones before z, of the four (zx-1,
// zy-1), (zx, zy-1), (zx-1, zy), (zx, zy) around it that exist. In a batch's
// arena z counts from the mesh's first side a.rect_so / 4 and p0 is offset
// by its first point a.rect_po (both 0 for a single problem).
struct RectZone {
    int p0, zx, zy;
};
__device__ __forceinline__ RectZone rect_zone(const FusedArgs& a, int z) {
    RectZone r;
    r.zy = (int)(((unsigned long long)(unsigned)z * a.rect_m) >> a.rect_sh);
    r.zx = z - r.zy * a.rect_nzx;
    r.p0 = z + r.zy + a.rect_po;
    return r;
}
__device__ __forceinline__ int rect_point(const FusedArgs& a, const RectZone& r, int k) {
    const int npx = a.rect_nzx + 1;
    return k == 0 ? r.p0 : (k == 1 ? r.p0 + 1 : (k == 2 ? r.p0 + 1 + npx : r.p0 + npx));
}
__device__ __forceinline__ int rect_rank(const FusedArgs& a, const RectZone& r, int k) {
    const int left = r.zx >= 1, below = r.zy >= 1;
    if (k == 0) return (left & below) + below + left;
    if (k == 1) return below + (below & (r.zx + 1 < a.rect_nzx));
    return k == 2 ? 0 : left;
}

// The points of a zone: mapsp1 of its sides sb..sb+NS-1.
template <int NS>
__device__ __forceinline__ void load_pp(const FusedArgs& a, int sb, int (&pp)[NS]) {
    if constexpr (NS == 4) {
        if (a.rect_nzx > 0) {
            const RectZone r = rect_zone(a, (sb - a.rect_so) >> 2);
#pragma unroll
            for (int k = 0; k < NS; ++k) pp[k] = rect_point(a, r, k);
            return;
        }
    }
#pragma unroll
    for (int k = 0; k < NS; ++k) pp[k] = ld_nt(a.mapsp1 + sb + k);
}

// The corner-record slots of a zone's corners: pcpos of its sides (the
// slot is corner_slot(p, rank, k); a rect mesh's ranks are below 4).
template <int NS>
__device__ __forceinline__ void load_slots(const FusedArgs& a, int sb, int (&slot)[NS]) {
    if constexpr (NS == 4) {
        if (a.rect_nzx > 0) {
            const RectZone r = rect_zone(a, (sb - a.rect_so) >> 2);
#pragma unroll
            for (int k = 0; k < NS; ++k) slot[k] = rect_rank(a, r, k) * a.nump + rect_point(a, r, k);
            return;
        }
    }
#pragma unroll
    for (int k = 0; k < NS; ++k) slot[k] = ld_nt(a.pcpos + sb + k);
}

// The learned pass's zone list of a run is kept in PN_LSLICES slices, one
// per band of block_units (all in slice 0 without the XCD mapping).  Slice s
// starts at its band's first zone, list_unit0 units into the run, so its
// entries fit in the band's own zone range; each slice has its own count on
// its own 128-byte line, so the flagging waves of the 8 XCDs add to 8
// counts instead of queueing on one.
#define PN_LSLICES 8
#define PN_LSTRIDE 32
__device__ __forceinline__ int list_unit0(int nunits, int s) {
    return (int)((long long)nunits * s / 8);
}
__device__ __forceinline__ unsigned* list_count(const FusedArgs& a, int run, int s) {
    return a.zcount + (run * PN_LSLICES + s) * PN_LSTRIDE;
}

// ---------------------------------------------------------------------------
// Side work forces (K1 writes them, K3 reads them) are stored pair-major
// within each unit of n <= PN_BLOCK zones of a run (sides u0 .. u0 + NS n - 1):
// sides 2j and 2j+1 of the unit's zone i sit together at u0 + 2 j n + 2 i
// (a lone last side of an odd NS at u0 + 2 j n + i), so that a wave's lanes
// (consecutive zones) cover one contiguous run per side pair and each lane
// moves a pair in one access.  SideW locates a zone in its unit.
struct SideW {
    int u0, i, n;
};
template <int NS>
__device__ __forceinline__ int sw_slot(const SideW& w, int k) {
    const int j = k >> 1;
    return w.u0 + 2 * j * w.n + (((k | 1) < NS) ? 2 * w.i + (k & 1) : w.i);
}
// A side pair's two values as one access (the types carry only the element
// alignment: gfx950 global memory takes dword-aligned multi-dword accesses).
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef double f64x2u __attribute__((ext_vector_type(2), aligned(8)));

__device__ __forceinline__ SideW side_w(int z, int zbeg, int zend, int sbeg, int ns) {
    const int zu = zbeg + ((z - zbeg) / PN_BLOCK) * PN_BLOCK;
    SideW w;
    w.u0 = sbeg + (zu - zbeg) * ns;
    w.i = z - zu;
    w.n = (zend - zu < PN_BLOCK) ? zend - zu : PN_BLOCK;
    return w;
}

// One corner's QCS results, as the two sides that meet at the corner use
// them: setCornerDiv, setQCnForce and setForceQCS's corner weight
// (src/QCS.cc:116-380) for corner k of a zone, whose point has velocity up0
// and half-step position xp0, neighbouring points' velocities u0p (previous)
// and u0n (next), edge centres xp1 = ex[k] and xp3 = ex[k-1], and edge
// lengths de1 = elen[k-1] (reciprocal r1) and de2 = elen[k] (reciprocal r2).
struct CrnQ {
    d2 q1, q2;      // cqe1, cqe2
    double w, c;    // cw and the clamped ccos
};
__device__ __forceinline__ CrnQ qcs_corner(d2 up0, d2 u0p, d2 u0n, d2 xp0, d2 xp1, d2 xp3, d2 zx, d2 zuc,
                                           double de1, double de2, double r1, double r2, double ztmp1,
                                           double g2, double zrp) {
    const d2 up1 = scl(0.5, add(up0, u0n));
    const d2 up2 = zuc;
    const d2 xp2 = zx;
    const d2 up3 = scl(0.5, add(u0p, up0));
    const double cvolume = 0.5 * cross(sub(xp2, xp0), sub(xp3, xp1));
    const d2 v1 = sub(xp3, xp0);
    const d2 v2 = sub(xp1, xp0);
    const double minelen = smin(de1, de2);
    const double cc = ((minelen < 1.e-12) ? 0. : 4. * dot(v1, v2) / (de1 * de2));
    const double div = (cross(sub(up2, up0), sub(xp3, xp1)) - cross(sub(up3, up1), sub(xp2, xp0))) /
                       (2.0 * cvolume);
    const d2 dxx1 = scl(0.5, sub(sub(add(xp1, xp2), xp0), xp3));
    const d2 dxx2 = scl(0.5, sub(sub(add(xp2, xp3), xp0), xp1));
    const double dx1 = len(dxx1);
    const double dx2 = len(dxx2);
    const d2 duav = scl(0.25, add(add(add(up0, up1), up2), up3));
    const double test1 = fabs(dot(dxx1, duav) * dx2);
    const double test2 = fabs(dot(dxx2, duav) * dx1);
    const double num = (test1 > test2 ? dx1 : dx2);
    const double den = (test1 > test2 ? dx2 : dx1);
    const double rr = num / den;
    double evol = __builtin_sqrt(4.0 * cvolume * rr);
    evol = smin(evol, 2.0 * minelen);
    const double dv1 = len2(sub(sub(add(up1, up2), up0), up3));
    const double dv2 = len2(sub(sub(add(up2, up3), up0), up1));
    const double du = __builtin_sqrt(smax(dv1, dv2));
    const double cevol = (div < 0.0 ? evol : 0.);
    const double cdu = (div < 0.0 ? du : 0.);
    // setQCnForce (g2 = q2 * 0.25 * (qgamma + 1), the reference's left-to-right product)
    const double ztmp2 = g2 * cdu;
    const double zkur = ztmp2 + __builtin_sqrt(ztmp2 * ztmp2 + ztmp1 * ztmp1);
    const double mu = zkur * zrp * cevol;
    const double cm = ((div > 0.0) ? 0. : mu);
    CrnQ r;
    const d2 d1 = scl(cm, sub(up0, u0p));
    const d2 d2_ = scl(cm, sub(u0n, up0));
    r.q1 = mk(d1.x * r1, d1.y * r1);     // Vec2 / double: times the reciprocal
    r.q2 = mk(d2_.x * r2, d2_.y * r2);
    // setForceQCS's corner weight and clamped cosine
    const double csin2 = 1.0 - cc * cc;
    r.w = ((csin2 < 1.e-4) ? 0. : cvolume / csin2);
    r.c = ((csin2 < 1.e-4) ? 0. : cc);
    return r;
}

// K1, zone-per-thread: the whole predictor half of doCycle for zone z, whose
// sides are sb..sb+NS-1 (side work force slots sw).  Returns the zone's
// calcDtNew candidate.
//
// Every value is the reference's expression, but the corners and sides are
// visited in a streaming order that keeps few of them live at once: corner
// k+1's QCS, then side k's forces (which need corners k and k+1), then
// corner k's force tot[k] - tot[k-1]; corner 0 is kept for the last side.
// Each side's 1/elen is formed once and used by both corners at the side and
// by its viscous force (the reference divides a Vec2 by elen through the
// same reciprocal, src/Vec2.hh:145-149).
// What the FP64 predictor of a zone reads: its points' positions and
// velocities, its state from the previous cycle, its side fractions and its
// corners' slots.
template <int NS>
struct ZoneIn {
    d2 x[NS], u[NS];
    double zm, zr, ze, zvol, zwr;
    double mf[NS];
};
template <int NS>
__device__ __forceinline__ void load_zone(const FusedArgs& a, int z, int sb, const int (&pp)[NS],
                                          ZoneIn<NS>& in) {
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        in.x[k] = mk(a.pxx[pp[k]], a.pxy[pp[k]]);
        in.u[k] = mk(a.pux[pp[k]], a.puy[pp[k]]);
    }
    in.zm = a.zm[z];
    in.zr = a.zr[z];
    in.ze = a.ze[z];
    in.zvol = a.zvol[z];
    in.zwr = a.zwrate[z];
#pragma unroll
    for (int k = 0; k < NS; ++k) in.mf[k] = a.smf[sb + k];
}

// Where a predictor puts its results: the arrays that K2 and K3 read (a
// corner's values at its slot, side work forces pair-major).
template <int NS>
struct ZoneToArrays {
    const FusedArgs& a;
    int z;
    SideW sw;
    int slot[NS];
    __device__ __forceinline__ void zp(double v) { a.zp[z] = v; }
    __device__ __forceinline__ void mass(int k, double v) { a.cmass[slot[k]] = v; }
    __device__ __forceinline__ void force(int k, d2 f) {
        a.cfx[slot[k]] = f.x;
        a.cfy[slot[k]] = f.y;
    }
    // the work forces of sides k and k + 1, and of a lone last side
    __device__ __forceinline__ void sides(int k, d2 f0, d2 f1) {
        const int sl = sw_slot<NS>(sw, k);
        const f64x2u vx = {f0.x, f1.x}, vy = {f0.y, f1.y};
        __builtin_nontemporal_store(vx, reinterpret_cast<f64x2u*>(a.sfwx + sl));
        __builtin_nontemporal_store(vy, reinterpret_cast<f64x2u*>(a.sfwy + sl));
    }
    __device__ __forceinline__ void side(int k, d2 f) {
        const int sl = sw_slot<NS>(sw, k);
        st_nt(f.x, a.sfwx + sl);
        st_nt(f.y, a.sfwy + sl);
    }
};

template <int NS, class Out>
__device__ __forceinline__ double zone_pred_core(const FusedArgs& a, const ZoneIn<NS>& in, double dt, int& bad,
                                                 Out& out) {
    const double dth = 0.5 * dt;
    const double n = (double)NS;
    d2 u0[NS], xp[NS];
    double mf[NS];
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        u0[k] = in.u[k];
        mf[k] = in.mf[k];
    }
    const double zm = in.zm;
    const double zr0 = in.zr;
    const double ze0 = in.ze;
    const double zvol0 = in.zvol;
    const double zwr = in.zwr;
#pragma unroll
    for (int k = 0; k < NS; ++k) xp[k] = add(in.x[k], scl(dth, u0[k]));   // advPosHalf
    // calcCtrs
    d2 ex[NS];
    d2 zx = mk(0., 0.);
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        ex[k] = scl(0.5, add(xp[k], xp[nxt<NS>(k)]));
        zx = add(zx, dvs(xp[k], n));
    }
    // calcVols, calcEdgeLen, calcCharLen
    const double third = 1. / 3.;
    double sa[NS], el[NS], rel[NS];
    double zarea = 0., zvolp = 0.;
    const double fac = (NS == 3 ? 3. : 4.);
    double zdl = 1.e99;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const d2 p1 = xp[k], p2 = xp[nxt<NS>(k)];
        sa[k] = 0.5 * cross(sub(p2, p1), sub(zx, p1));
        const double sv = third * sa[k] * (p1.x + p2.x + zx.x);
        zarea += sa[k];
        zvolp += sv;
        if (sv <= 0.) bad += 1;
        el[k] = len(sub(p2, p1));
    }
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        zdl = smin(zdl, fac * sa[k] / el[k]);
        rel[k] = 1. / el[k];
    }
    // calcRho (pred)
    const double zrp = zm / zvolp;
    // calcStateHalf (reads ZR, ZE, ZWRATE of the previous cycle, ZVOL0 = ZVOL)
    const double gm1 = a.gamma - 1.;
    const double ssmin2 = smax(a.ssmin * a.ssmin, 1.e-99);
    const double r = zr0;
    const double e = smax(ze0, 0.);
    const double p = gm1 * r * e;
    const double pre = gm1 * e;
    const double per = gm1 * r;
    const double csqd = smax(ssmin2, pre + per * p / (r * r));
    const double zss = __builtin_sqrt(csqd);
    const double minv = 1. / zm;
    const double dv = (zvolp - zvol0) * minv;
    const double bulk = r * csqd;
    const double denom = 1. + 0.5 * per * dv;
    const double src = zwr * dth * minv;
    const double zp = p + (per * src - r * bulk * dv) / denom;
    out.zp(zp);
    // calcCrnrMass's corner mass
    const double mzz = zrp * zarea;
#pragma unroll
    for (int k = 0; k < NS; ++k) out.mass(k, mzz * 0.5 * (mf[k] + mf[prv<NS>(k)]));
    // calcSurfVecs, calcForcePGas, calcForceTTS per side (below)
    double sstmp = smax(zss, a.ssmin);
    sstmp = a.alfa * sstmp * sstmp;
    // setCornerDiv's zone velocity
    d2 zuc = mk(0., 0.);
#pragma unroll
    for (int k = 0; k < NS; ++k) zuc = add(zuc, dvs(u0[k], n));
    const double g2 = a.q2 * 0.25 * (a.qgamma + 1.0);
    const double ztmp1 = a.q1 * zss;
    // corners, sides and corner forces in streaming order
    const CrnQ c0 = qcs_corner(u0[0], u0[NS - 1], u0[1], xp[0], ex[0], ex[NS - 1], zx, zuc, el[NS - 1], el[0],
                               rel[NS - 1], rel[0], ztmp1, g2, zrp);
    CrnQ ck = c0;
    d2 tot0 = mk(0., 0.), totk = mk(0., 0.), sfw_prev = mk(0., 0.);
    double ztmp = 0.;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const int kp = nxt<NS>(k);
        const CrnQ cn = (kp == 0) ? c0
                                  : qcs_corner(u0[kp], u0[k], u0[nxt<NS>(kp)], xp[kp], ex[kp], ex[k], zx, zuc,
                                               el[k], el[kp], rel[k], rel[kp], ztmp1, g2, zrp);
        // side k: pressure, TTS and viscous forces
        const d2 ss = rot_ccw(sub(ex[k], zx));
        const d2 sfp = scl(-zp, ss);
        const double vfacinv = zarea / sa[k];
        const double srho = zrp * mf[k] * vfacinv;
        const double sdp = sstmp * (srho - zrp);
        const d2 sft = scl(-sdp, ss);
        const d2 f = add(scl(ck.w, add(ck.q2, scl(ck.c, ck.q1))), scl(cn.w, add(cn.q1, scl(cn.c, cn.q2))));
        const d2 sfq = mk(f.x * rel[k], f.y * rel[k]);
        const d2 sfw = add(sfp, sfq);                    // calcWork's sf + sf2
        const d2 tot = add(add(sfp, sfq), sft);          // sumCrnrForce's sfp+sfq+sft
        // setVelDiff's side k, in ascending order from 0
        {
            const d2 dx = sub(xp[kp], xp[k]);
            const d2 du = sub(u0[kp], u0[k]);
            const double lenx = el[k];
            double dux = dot(du, dx);
            dux = (lenx > 0. ? fabs(dux) / lenx : 0.);
            ztmp = smax(ztmp, dux);
        }
        // corner k's force (point mapsp1[sb+k]) once sides k-1 and k are known
        if (k == 0) {
            tot0 = tot;
        } else {
            out.force(k, sub(tot, totk));
        }
        totk = tot;
        // the work forces of a side pair together
        if (k & 1) out.sides(k - 1, sfw_prev, sfw);
        else if (k + 1 == NS) out.side(k, sfw);
        sfw_prev = sfw;
        ck = cn;
    }
    out.force(0, sub(tot0, totk));
    const double zdu = a.q1 * zss + 2. * a.q2 * ztmp;
    // calcDtNew for this zone
    const double fuzz = 1.e-99;
    const double cdt = smax(zdu, smax(zss, fuzz));
    return zdl * a.cfl / cdt;
}

template <int NS>
__device__ __forceinline__ double zone_pred(const FusedArgs& a, int z, int sb, SideW sw,
                                            const int (&pp)[NS], double dt, int& bad) {
    ZoneIn<NS> in;
    load_zone<NS>(a, z, sb, pp, in);      // every load of the zone first
    ZoneToArrays<NS> out{a, z, sw, {}};
    load_slots<NS>(a, sb, out.slot);
    return zone_pred_core<NS>(a, in, dt, bad, out);
}

template <int NS>
__device__ __forceinline__ double zone_pred(const FusedArgs& a, int z, int sb, SideW sw, double dt,
                                            int& bad) {
    int pp[NS];
    load_pp<NS>(a, sb, pp);
    return zone_pred<NS>(a, z, sb, sw, pp, dt, bad);
}

template <int NS>
__global__ void __launch_bounds__(PN_BLOCK) k_pred_zone(FusedArgs a, int zbeg, int zend, int sbeg,
                                                        int poff) {
    if (a.ctl->done) return;
    const double dt = a.ctl->dt;
    double dtmin = 1.e99;
    int bad = 0;
    const int nunits = (zend - zbeg + PN_BLOCK - 1) / PN_BLOCK;
    Units w = block_units(nunits, a.xcd);
    int zn = zbeg + w.u * PN_BLOCK + threadIdx.x;
    int pn[NS];
    if (w.u < w.end && zn < zend) load_pp<NS>(a, sbeg + (zn - zbeg) * NS, pn);
    for (; w.u < w.end; w.u += w.step) {
        // this zone's points were loaded by the previous iteration; load the next zone's
        const int z = zn;
        int pp[NS];
#pragma unroll
        for (int k = 0; k < NS; ++k) pp[k] = pn[k];
        zn = zbeg + (w.u + w.step) * PN_BLOCK + threadIdx.x;
        if (w.u + w.step < w.end && zn < zend) load_pp<NS>(a, sbeg + (zn - zbeg) * NS, pn);
        if (z >= zend) continue;
        const double zdthyd = zone_pred<NS>(a, z, sbeg + (z - zbeg) * NS,
                                            side_w(z, zbeg, zend, sbeg, NS), pp, dt, bad);
        // the running minimum of src/Hydro.cc:1615 (a NaN never replaces it)
        dtmin = (zdthyd < dtmin) ? zdthyd : dtmin;
    }
    const double m = block_min(dtmin);
    const int b = block_sum(bad);
    if (threadIdx.x == 0) {
        a.part_dt[poff + blockIdx.x] = m;
        a.part_bp[poff + blockIdx.x] = b;
    }
}

// ---------------------------------------------------------------------------
// K1, mixed precision (zone per thread).
//
// FP64: positions and their midpoints, the zone centre, side and zone areas
// and volumes (cross products of nearly equal coordinates), the zone EOS with
// its (zvolp - zvol0) difference, the TTS density difference srho - r, the
// corner-force difference tot[k] - tot[k-1], the corner mass, and the dt
// candidate.  FP32: edge lengths, the per-side pressure/TTS force products
// and the whole QCS chain (corner divergence, evolution factor, Kurapatenko
// coefficient, corner weights, edge viscous force).  Coordinate and velocity
// differences are formed in FP64 and rounded once.  Like every kernel here it
// is compiled without contraction, so each operation rounds on its own and
// the results do not depend on how the function is inlined (a batched
// problem gives the same bits as its own run).

struct f2 {
    float x, y;
};
__device__ __forceinline__ f2 fmk(float x, float y) { f2 v; v.x = x; v.y = y; return v; }
__device__ __forceinline__ f2 tof(d2 v) { return fmk((float)v.x, (float)v.y); }
__device__ __forceinline__ f2 fadd(f2 a, f2 b) { return fmk(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ f2 fscl(float r, f2 v) { return fmk(v.x * r, v.y * r); }
// 1/x in FP64 from the hardware reciprocal and two Newton steps (within an
// ulp or two of the quotient; the mixed form's FP64 divisions use it)
__device__ __forceinline__ double drcp(double x) {
    double r = __builtin_amdgcn_rcp(x);
    double e = __builtin_fma(-x, r, 1.);
    r = __builtin_fma(r, e, r);
    e = __builtin_fma(-x, r, 1.);
    return __builtin_fma(r, e, r);
}

// The mixed form's FP32 products fold one multiply into a fused multiply-add
// (explicitly: the FP64 form is built without contraction, and explicit
// fmaf keeps every kernel that runs this code bit-identical).
__device__ __forceinline__ float fdot(f2 a, f2 b) { return __builtin_fmaf(a.x, b.x, a.y * b.y); }
__device__ __forceinline__ float fcross(f2 a, f2 b) { return __builtin_fmaf(a.x, b.y, -(a.y * b.x)); }
// a + r b
__device__ __forceinline__ f2 faxpy(float r, f2 b, f2 a) {
    return fmk(__builtin_fmaf(r, b.x, a.x), __builtin_fmaf(r, b.y, a.y));
}
// the hardware square root (1 ulp), without the correctly rounded expansion
__device__ __forceinline__ float fsqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
__device__ __forceinline__ float flen(f2 v) { return fsqrt(fdot(v, v)); }
__device__ __forceinline__ float frcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float fminr(float a, float b) { return (b < a) ? b : a; }
__device__ __forceinline__ float fmaxr(float a, float b) { return (a < b) ? b : a; }

// The work forces of a zone's sides, {x, y} per side slot (sw_slot).
template <int NS>
__device__ __forceinline__ void store_sides(float* w, const SideW& sw, const f2 (&v)[NS]) {
#pragma unroll
    for (int k = 0; k < NS; k += 2) {
        float* q = w + 2 * sw_slot<NS>(sw, k);
        if (k + 1 < NS) {
            const f32x4u t = {v[k].x, v[k].y, v[k + 1].x, v[k + 1].y};
            __builtin_nontemporal_store(t, reinterpret_cast<f32x4u*>(q));
        } else {
            st_nt(v[k].x, q);
            st_nt(v[k].y, q + 1);
        }
    }
}
template <int NS>
__device__ __forceinline__ void load_sides(const float* w, const SideW& sw, f2 (&v)[NS]) {
#pragma unroll
    for (int k = 0; k < NS; k += 2) {
        const float* q = w + 2 * sw_slot<NS>(sw, k);
        if (k + 1 < NS) {
            const f32x4u t = __builtin_nontemporal_load(reinterpret_cast<const f32x4u*>(q));
            v[k] = fmk(t[0], t[1]);
            v[k + 1] = fmk(t[2], t[3]);
        } else {
            v[k] = fmk(ld_nt(q), ld_nt(q + 1));
        }
    }
}

// Closure kinds of the mixed K1:
//   CL_EXACT    the exact QCS coefficient;
//   CL_FLAG     the exact coefficient, and the zone is reported (ClCount.flag)
//               when one of its corners passes the network's gate;
//   CL_LEARNED  the network's coefficient on the corners that pass the gate
//               (the exact one elsewhere, and on zones outside the envelope);
//   CL_RECOMP   CL_LEARNED for a zone that a CL_FLAG pass has already handled:
//               stores only what the coefficient changes (corner and work
//               forces);
//   CL_CAPTURE  the exact coefficient, recording training tuples;
//   CL_PACKED   CL_LEARNED with the wave's gated corners packed into as few
//               evaluations as possible, as CL_RECOMP does;
//   CL_LEAN     CL_PACKED in fewer registers: 32 corners at a time instead of
//               two groups in one stream, the weights read at each use.
// The gate: a compressing corner (cdiv < 0) whose quadratic term matters,
// G du > PN_GATE (q1 zss + G du), i.e. f9 > PN_GATE.  Below it the exact
// coefficient equals its acoustic limit q1 zss + G du to within 0.1%; the
// round-off velocities of a quiescent region stay far below it.
enum { CL_EXACT = 0, CL_LEARNED = 1, CL_CAPTURE = 2, CL_FLAG = 3, CL_RECOMP = 4, CL_PACKED = 5, CL_LEAN = 6 };
#define PN_GATE 1.e-3f

// Zone counters of the learned form, summed per thread.
struct ClCount {
    int learned = 0;    // zones with gated corners evaluated by the network
    int fallback = 0;   // such zones outside the envelope (exact coefficient)
    bool flag = false;  // CL_FLAG: this zone has a gated corner
};

// The zone state a predictor starts from (the previous cycle's results).
struct ZoneState {
    double zm, zr, ze, zvol, zwrate;
};

// The FP64 half of the mixed predictor of a zone: half-step positions,
// centre, areas and volumes, edge lengths and characteristic length, the
// zone EOS and the pressure and TTS side forces, with positions and
// velocities moved into the zone's FP32 frame for the QCS half.
template <int NS>
struct MixedFrame {
    float mf[NS];     // FP32 side mass fractions
    f2 ul[NS];        // point velocities relative to the zone-mean velocity zuc
    f2 xl[NS];        // half-step positions relative to the zone centre
    f2 exl[NS];       // edge midpoints, same frame
    float el[NS];     // edge lengths
    f2 sfp[NS];       // pressure side forces
    f2 sft[NS];       // TTS side forces
    d2 zuc;
    double zss, zrp, zarea, r, zp;
    float zdl;
};

// The frame of a zone from its points' positions x0 and velocities u0, its
// state st and its side fractions (F.mf, set by the caller).
template <int NS>
__device__ __forceinline__ void mixed_frame(MixedFrame<NS>& F, const FusedArgs& a, const d2 (&x0)[NS],
                                            const d2 (&u0)[NS], const ZoneState& st, double dt, int& bad,
                                            bool valid) {
    const double dth = 0.5 * dt;
    const double n = (double)NS;
    d2 xp[NS];
    const float (&mf)[NS] = F.mf;
    const double zm = st.zm;
    const double r = st.zr;
    const double ze0 = st.ze;
    const double zvol0 = st.zvol;
    const double zwr = st.zwrate;
    F.r = r;
#pragma unroll
    for (int k = 0; k < NS; ++k)
        xp[k] = mk(__builtin_fma(dth, u0[k].x, x0[k].x), __builtin_fma(dth, u0[k].y, x0[k].y));
    // zone-mean velocity; velocities from here on live in FP32 relative to it
    d2& zuc = F.zuc;
    zuc = mk(0., 0.);
#pragma unroll
    for (int k = 0; k < NS; ++k) zuc = add(zuc, dvs(u0[k], n));
    f2 (&ul)[NS] = F.ul;
#pragma unroll
    for (int k = 0; k < NS; ++k) ul[k] = tof(sub(u0[k], zuc));
    d2 zx = mk(0., 0.);
#pragma unroll
    for (int k = 0; k < NS; ++k) zx = add(zx, dvs(xp[k], n));
    const double third = 1. / 3.;
    double sa[NS];
    float (&el)[NS] = F.el;
    double zarea = 0., zvolp = 0.;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const d2 p1 = xp[k], p2 = xp[nxt<NS>(k)];
        const d2 e = sub(p2, p1);
        sa[k] = 0.5 * cross(e, sub(zx, p1));
        const double sv = third * sa[k] * (p1.x + p2.x + zx.x);
        zarea += sa[k];
        zvolp += sv;
        if (valid && sv <= 0.) bad += 1;
        el[k] = flen(tof(e));
    }
    F.zarea = zarea;
    // positions from here on live in FP32 relative to the zone centre (which
    // is the origin of this frame); edge midpoints follow from them
    f2 (&xl)[NS] = F.xl;
    f2 (&exl)[NS] = F.exl;
#pragma unroll
    for (int k = 0; k < NS; ++k) xl[k] = tof(sub(xp[k], zx));
#pragma unroll
    for (int k = 0; k < NS; ++k) exl[k] = fscl(0.5f, fadd(xl[k], xl[nxt<NS>(k)]));
    const float fac = (NS == 3 ? 3.f : 4.f);
    float zdl = 1.e30f;
#pragma unroll
    for (int k = 0; k < NS; ++k) zdl = fminr(zdl, fac * (float)sa[k] * frcp(el[k]));
    F.zdl = zdl;
    // zone EOS in FP64
    const double zrp = zm * drcp(zvolp);
    F.zrp = zrp;
    const double gm1 = a.gamma - 1.;
    const double ssmin2 = smax(a.ssmin * a.ssmin, 1.e-99);
    const double e = smax(ze0, 0.);
    const double pz = gm1 * r * e;
    const double per = gm1 * r;
    // pre + per pz / r^2 = (gamma - 1) e + (gamma - 1)^2 e = gamma (gamma - 1) e
    const double csqd = smax(ssmin2, a.gamma * gm1 * e);
    const double zss = __builtin_sqrt(csqd);
    F.zss = zss;
    const double minv = drcp(zm);
    const double dv = (zvolp - zvol0) * minv;
    const double bulk = r * csqd;
    const double denom = 1. + 0.5 * per * dv;
    const double src = zwr * dth * minv;
    const double zp = pz + (per * src - r * bulk * dv) * drcp(denom);
    F.zp = zp;
    // pressure and TTS side forces
    const float zpf = (float)zp;
    double sstmp = smax(zss, a.ssmin);
    sstmp = a.alfa * sstmp * sstmp;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const f2 ss = fmk(-exl[k].y, exl[k].x);                       // rotCCW(ex - zx)
        F.sfp[k] = fscl(-zpf, ss);
        // srho - r = zrp (mf zarea - sa) / sa: the difference in FP64, the
        // division in FP32 (relative to the difference itself)
        const float drho = (float)(zrp * ((double)mf[k] * zarea - sa[k])) * frcp((float)sa[k]);
        F.sft[k] = fscl(-(float)sstmp * drho, ss);
    }
}

// Corner k's QCS quantities in the frame F (setCornerDiv,
// src/QCS.cc:116-242; corner k: xp0 = x[k], xp1 = ex[k], xp2 = zx,
// xp3 = ex[k-1]; up2 = zuc is the frame's zero velocity).  evol and du are
// the values before the compression test.
struct MixedCrn {
    float area, ccos, div, evol, du, minelen;
    f2 duav;
};
template <int NS>
__device__ __forceinline__ MixedCrn mixed_corner(const MixedFrame<NS>& F, int k, f2 zucf) {
    const f2 (&ul)[NS] = F.ul;
    const f2 (&xl)[NS] = F.xl;
    const f2 (&exl)[NS] = F.exl;
    const float (&el)[NS] = F.el;
    const int km = prv<NS>(k), kp = nxt<NS>(k);
    MixedCrn c;
    const f2 u1 = fscl(0.5f, fadd(ul[k], ul[kp]));                 // up1 - zuc
    const f2 u3 = fscl(0.5f, fadd(ul[km], ul[k]));                 // up3 - zuc
    const f2 A = fmk(-xl[k].x, -xl[k].y);                           // xp2 - xp0
    const f2 B = fmk(exl[km].x - exl[k].x, exl[km].y - exl[k].y);   // xp3 - xp1
    const f2 v1 = fmk(exl[km].x - xl[k].x, exl[km].y - xl[k].y);    // xp3 - xp0
    const f2 v2 = fmk(exl[k].x - xl[k].x, exl[k].y - xl[k].y);      // xp1 - xp0
    const f2 dxx1 = fscl(0.5f, fmk(exl[k].x - xl[k].x - exl[km].x, exl[k].y - xl[k].y - exl[km].y));
    const f2 dxx2 = fscl(0.5f, fmk(exl[km].x - xl[k].x - exl[k].x, exl[km].y - xl[k].y - exl[k].y));
    const f2 du20 = fmk(-ul[k].x, -ul[k].y);                        // up2 - up0
    const f2 du31 = fmk(u3.x - u1.x, u3.y - u1.y);                  // up3 - up1
    const f2 dva = fmk(u1.x - ul[k].x - u3.x, u1.y - ul[k].y - u3.y);   // up1+up2-up0-up3
    const f2 dvb = fmk(u3.x - ul[k].x - u1.x, u3.y - ul[k].y - u1.y);   // up2+up3-up0-up1
    c.duav = faxpy(0.25f, fadd(fadd(ul[k], u1), u3), zucf);
    const float cvol = 0.5f * fcross(A, B);
    c.area = cvol;
    const float de1 = el[km], de2 = el[k];
    const float minelen = fminr(de1, de2);
    c.minelen = minelen;
    c.ccos = (minelen < 1.e-12f) ? 0.f : 4.f * fdot(v1, v2) * frcp(de1 * de2);
    c.div = (fcross(du20, B) - fcross(du31, A)) * frcp(2.f * cvol);
    const float dx1 = flen(dxx1), dx2 = flen(dxx2);
    const float t1 = fabsf(fdot(dxx1, c.duav) * dx2);
    const float t2 = fabsf(fdot(dxx2, c.duav) * dx1);
    const float num = (t1 > t2) ? dx1 : dx2;
    const float den = (t1 > t2) ? dx2 : dx1;
    float evol = fsqrt(4.f * cvol * num * frcp(den));
    c.evol = fminr(evol, 2.f * minelen);
    c.du = fsqrt(fmaxr(fdot(dva, dva), fdot(dvb, dvb)));
    return c;
}

// The network features of corner k (closure.h); the quotients are reciprocal
// products (within an ulp or two: the network reads them in BF16).
template <int NS>
__device__ __forceinline__ void corner_features(const MixedFrame<NS>& F, int k, const MixedCrn& c,
                                                float zssf, float zrpf, float q1f, float gq,
                                                float (&f)[PN_MLP_NF]) {
    const f2 (&ul)[NS] = F.ul;
    const int km = prv<NS>(k), kp = nxt<NS>(k);
    const float inv = frcp(zssf);
    f[0] = slog((ul[k].x - ul[km].x) * inv);
    f[1] = slog((ul[k].y - ul[km].y) * inv);
    f[2] = slog((ul[kp].x - ul[k].x) * inv);
    f[3] = slog((ul[kp].y - ul[k].y) * inv);
    f[4] = slog(c.div * c.evol * inv);
    f[5] = c.evol * frcp(c.minelen);
    f[6] = zssf * frcp(zssf + flen(c.duav));
    f[7] = zrpf * frcp((float)F.r);
    f[8] = slog(c.du * inv);
    const float tl = q1f * zssf, tq = gq * c.du;
    f[9] = (tl + tq > 0.f) ? tq * frcp(tl + tq) : 0.f;
}

// Where a mixed predictor puts its results: the arrays that K2 and K3 read.
template <int NS>
struct MixedToArrays {
    const FusedArgs& a;
    int z;
    SideW sw;
    int slot[NS];
    __device__ __forceinline__ void zp(double v) { a.zp[z] = v; }
    __device__ __forceinline__ void sides(const f2 (&f)[NS]) { store_sides<NS>(a.fsfw, sw, f); }
    __device__ __forceinline__ void force(int k, float fx, float fy) {
        a.fcrn[3 * slot[k]] = fx;
        a.fcrn[3 * slot[k] + 1] = fy;
    }
    __device__ __forceinline__ void mass(int k, float m) { a.fcrn[3 * slot[k] + 2] = m; }
};

// The mixed-precision predictor half of a zone, from its points' positions x0
// and velocities u0, its state st and its FP32 side fractions mf.  With CL !=
// CL_EXACT it must be called by all 64 lanes of a wave together (the network
// runs across the wave); `valid` false marks a lane that only takes part in
// the wave-wide steps and stores nothing.
template <int NS, int CL, class Out>
__device__ __forceinline__ double zone_pred_mixed_core(const FusedArgs& a, const d2 (&x0)[NS],
                                                       const d2 (&u0)[NS], const ZoneState& st,
                                                       const float (&mf0)[NS], double dt, int& bad,
                                                       bool valid, ClCount& cnt, Out& out) {
    constexpr bool PACK = CL == CL_RECOMP || CL == CL_PACKED || CL == CL_LEAN, NET = CL == CL_LEARNED || PACK;
    MixedFrame<NS> F;
#pragma unroll
    for (int k = 0; k < NS; ++k) F.mf[k] = mf0[k];
    mixed_frame<NS>(F, a, x0, u0, st, dt, bad, valid);
    if (CL != CL_RECOMP && valid) out.zp(F.zp);
    const float (&mf)[NS] = F.mf;
    const f2 (&ul)[NS] = F.ul;
    const f2 (&xl)[NS] = F.xl;
    const float (&el)[NS] = F.el;
    const f2 (&sfp)[NS] = F.sfp;
    const f2 (&sft)[NS] = F.sft;
    const d2 zuc = F.zuc;
    const double zss = F.zss, zrp = F.zrp, zarea = F.zarea;
    const float zdl = F.zdl;
    // QCS corner quantities (corner k: xp0 = x[k], xp1 = ex[k], xp2 = zx,
    // xp3 = ex[k-1]; up2 = zuc is the frame's zero velocity)
    const f2 zucf = tof(zuc);
    const float gq = (float)(a.q2 * 0.25 * (a.qgamma + 1.0));
    const float q1f = (float)a.q1;
    const float zssf = (float)zss;
    const float zt1 = (float)(a.q1 * zss);
    const float zrpf = (float)zrp;
    // gate threshold on du / zss (no corner passes when G = 0)
    const float gthr = (gq > 0.f) ? PN_GATE * q1f / ((1.f - PN_GATE) * gq) : 3.4e38f;
    float carea[NS], ccos[NS], cdiv[NS], cevol[NS], cdu[NS];
    u32x4 flo[NS];            // packed network inputs, slots 0-7
    unsigned fhi[NS];         // slots 8-9
    bool inenv = true;        // every gated corner inside the envelope
    bool comp = false;        // some corner passes the gate
    unsigned gated = 0;       // bit k: corner k passes the gate
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const MixedCrn c = mixed_corner<NS>(F, k, zucf);
        const float div = c.div, evol = c.evol, du = c.du;
        carea[k] = c.area;
        ccos[k] = c.ccos;
        cdiv[k] = div;
        cevol[k] = (div < 0.f) ? evol : 0.f;
        cdu[k] = (div < 0.f) ? du : 0.f;
        if constexpr (CL == CL_FLAG || NET) {
            // G du > PN_GATE (q1 zss + G du)  <=>  du > gthr zss
            if (div < 0.f && du > gthr * zssf) {
                gated |= 1u << k;
                comp = true;
            }
        }
        if constexpr (NET || CL == CL_CAPTURE) {
            float f[PN_MLP_NF];
            corner_features<NS>(F, k, c, zssf, zrpf, q1f, gq, f);
            if constexpr (NET) {
                if (gated & (1u << k)) {
#pragma unroll
                    for (int j = 0; j < PN_MLP_NF; ++j)
                        inenv = inenv && (f[j] >= a.pack->lo[j]) && (f[j] <= a.pack->hi[j]);
                }
            }
            if constexpr (NET) {
                u32x4 hi;
                pack_features(f, flo[k], hi);
                fhi[k] = hi[0];
            } else {
                // a training tuple: features and the exact coefficients
                const float tl = q1f * zssf, tq = gq * du;
                const uint64_t m = __ballot(valid && div < 0.f);
                if (m) {
                    unsigned long long base = 0;
                    if ((threadIdx.x & 63) == 0) base = atomicAdd(a.cap_count, (unsigned long long)__popcll(m));
                    base = __shfl(base, 0, 64);
                    const uint64_t below = m & ((1ull << (threadIdx.x & 63)) - 1ull);
                    const unsigned long long slot = base + (unsigned long long)__popcll(below);
                    if (valid && div < 0.f && slot < (unsigned long long)a.cap) {
                        const float s2 = fsqrt(tl * tl + tq * tq);
                        float* o = a.cap_buf + slot * PN_MLP_TUPLE;
#pragma unroll
                        for (int j = 0; j < PN_MLP_NF; ++j) o[j] = f[j];
                        o[PN_MLP_NF] = (s2 > 0.f) ? tl / s2 : 1.f;
                        o[PN_MLP_NF + 1] = (s2 > 0.f) ? 1.f + tq / s2 : 1.f;
                    }
                }
            }
        }
    }
    f2 cqe1[NS], cqe2[NS];
    float crmu[NS];
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const float zt2 = gq * cdu[k];
        const float zkur = zt2 + fsqrt(zt2 * zt2 + zt1 * zt1);
        crmu[k] = (cdiv[k] > 0.f) ? 0.f : zkur * zrpf * cevol[k];
    }
    if constexpr (CL == CL_FLAG) cnt.flag = comp;
    if constexpr (PACK) {
        // The wave's corners that need the network, packed into as few
        // evaluations as possible: corner k of a lane goes to slot off_k +
        // its rank among the lanes needing corner k, in an LDS row of the
        // wave's own; every evaluation takes 64 slots, and its results come
        // back through the same slots.  A corner's result does not depend on
        // the other corners of its evaluation (each is its own MFMA column),
        // so the bits are those of the corner-by-corner evaluation.
        __shared__ uint32_t xw_all[PN_BLOCK / 64][NS * 64][5];
        uint32_t (*xw)[5] = xw_all[threadIdx.x >> 6];
        const int lane = threadIdx.x & 63;
        const uint64_t below = (1ull << lane) - 1ull;
        const bool use = valid && comp && inenv;
        if (valid && comp) {
            if (inenv) cnt.learned += 1;
            else cnt.fallback += 1;
        }
        int dest[NS];
        int total = 0;
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            const bool need = use && ((gated >> k) & 1u);
            const uint64_t m = __ballot(need);
            dest[k] = need ? total + (int)__popcll(m & below) : -1;
            total += (int)__popcll(m);
            if (need) {
#pragma unroll
                for (int j = 0; j < 4; ++j) xw[dest[k]][j] = flo[k][j];
                xw[dest[k]][4] = fhi[k];
            }
        }
        // LDS accesses of one wave are performed in order; the fence keeps
        // the compiler from moving them across
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        // the lane's weight fragments, read once for all of the wave's
        // evaluations (CL_LEAN: at each use)
        typename std::conditional<CL == CL_LEAN, MlpPackSrc, MlpRegs>::type wr;
        if constexpr (CL == CL_LEAN) wr = {a.pack, lane};
        else if (total > 0) mlp_load_regs(a.pack, lane, wr);
        for (int e = 0; e < total; e += 64) {
            const int sl = e + lane;
            const bool act = sl < total;
            const uint64_t am = __ballot(act);
            u32x4 lo, hi;
#pragma unroll
            for (int j = 0; j < 4; ++j) lo[j] = act ? xw[sl][j] : 0u;
            hi[0] = act ? xw[sl][4] : 0u;
            hi[1] = pack_bf16(1.f, 0.f);
            hi[2] = 0u;
            hi[3] = 0u;
            float y0, y1;
            mlp_wave_w<decltype(wr), CL != CL_LEAN>(wr, lo, hi, (uint32_t)am != 0u, (am >> 32) != 0u, y0, y1);
            if (act) {
                xw[sl][0] = __float_as_uint(y0);
                xw[sl][1] = __float_as_uint(y1);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            if (dest[k] >= 0) {
                const float y0 = __uint_as_float(xw[dest[k]][0]);
                const float y1 = __uint_as_float(xw[dest[k]][1]);
                crmu[k] = (q1f * y0 * zssf + gq * y1 * cdu[k]) * zrpf * cevol[k];
            }
        }
    }
    if constexpr (CL == CL_LEARNED) {
        const bool use = valid && comp && inenv;
        if (valid && comp) {
            if (inenv) cnt.learned += 1;
            else cnt.fallback += 1;
        }
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            const bool need = use && ((gated >> k) & 1u);
            const uint64_t m = __ballot(need);
            if (m) {
                u32x4 hi;
                hi[0] = fhi[k];
                hi[1] = pack_bf16(1.f, 0.f);
                hi[2] = 0u;
                hi[3] = 0u;
                float y0, y1;
                mlp_wave_w<MlpPackSrc, true>(MlpPackSrc{a.pack, (int)(threadIdx.x & 63)}, flo[k], hi,
                                             (uint32_t)m != 0u, (m >> 32) != 0u, y0, y1);
                if (need) crmu[k] = (q1f * y0 * zssf + gq * y1 * cdu[k]) * zrpf * cevol[k];
            }
        }
    }
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const int km = prv<NS>(k), kp = nxt<NS>(k);
        cqe1[k] = fscl(crmu[k] * frcp(el[km]), fmk(ul[k].x - ul[km].x, ul[k].y - ul[km].y));
        cqe2[k] = fscl(crmu[k] * frcp(el[k]), fmk(ul[kp].x - ul[k].x, ul[kp].y - ul[k].y));
    }
    float cw[NS];
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const float csin2 = __builtin_fmaf(-ccos[k], ccos[k], 1.f);
        cw[k] = (csin2 < 1.e-4f) ? 0.f : carea[k] * frcp(csin2);
        ccos[k] = (csin2 < 1.e-4f) ? 0.f : ccos[k];
    }
    d2 tot[NS];
    f2 sfwk[NS];
    float dux_max = 0.f;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const int kp = nxt<NS>(k);
        const f2 fq = faxpy(cw[k], faxpy(ccos[k], cqe1[k], cqe2[k]),
                            fscl(cw[kp], faxpy(ccos[kp], cqe2[kp], cqe1[kp])));
        const f2 sfw = faxpy(frcp(el[k]), fq, sfp[k]);
        sfwk[k] = sfw;
        tot[k] = mk((double)sfw.x + (double)sft[k].x, (double)sfw.y + (double)sft[k].y);
        // setVelDiff
        const f2 du = fmk(ul[kp].x - ul[k].x, ul[kp].y - ul[k].y);
        const f2 dx = fmk(xl[kp].x - xl[k].x, xl[kp].y - xl[k].y);
        const float dux = fabsf(fdot(du, dx)) * frcp(el[k]);
        dux_max = fmaxr(dux_max, (el[k] > 0.f) ? dux : 0.f);
    }
    if (valid) out.sides(sfwk);
    const double zdu = a.q1 * zss + 2. * a.q2 * (double)dux_max;
    const double mzz = zrp * zarea;
    if (valid) {
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            const int km = prv<NS>(k);
            const d2 cf = sub(tot[k], tot[km]);
            out.force(k, (float)cf.x, (float)cf.y);
            if constexpr (CL != CL_RECOMP) out.mass(k, (float)(mzz * 0.5 * ((double)mf[k] + (double)mf[km])));
        }
    }
    const double cdt = smax(zdu, smax(zss, 1.e-99));
    return (double)zdl * a.cfl * drcp(cdt);
}

// zone_pred_mixed_core of zone z (sides sb..sb+NS-1), its results to the
// arrays that K2 and K3 read.
template <int NS, int CL>
__device__ __forceinline__ double zone_pred_mixed_arrays(const FusedArgs& a, int z, int sb, SideW sw,
                                                         const d2 (&x0)[NS], const d2 (&u0)[NS],
                                                         const ZoneState& st, double dt, int& bad,
                                                         bool valid, ClCount& cnt) {
    float mf[NS];
#pragma unroll
    for (int k = 0; k < NS; ++k) mf[k] = ld_nt(a.fsmf + sb + k);
    MixedToArrays<NS> out{a, z, sw, {}};
    load_slots<NS>(a, sb, out.slot);
    return zone_pred_mixed_core<NS, CL>(a, x0, u0, st, mf, dt, bad, valid, cnt, out);
}

// The predictor of zone z whose points are pp (mapsp1 of its sides); every
// load of the zone is issued before the first use of a loaded value.  zre:
// the control block's zre_valid, read once by the caller.
template <int NS>
__device__ __forceinline__ void load_zone_mixed(const FusedArgs& a, int z, const int (&pp)[NS], bool zre,
                                                d2 (&x0)[NS], d2 (&u0)[NS], ZoneState& st) {
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        x0[k] = mk(a.pxx[pp[k]], a.pxy[pp[k]]);
        u0[k] = mk(a.pux[pp[k]], a.puy[pp[k]]);
    }
    st.zm = a.zm[z];
    st.zvol = a.zvol[z];
    st.zwrate = a.zwrate[z];
    if (zre) {
        st.zr = a.zr[z];
        st.ze = a.ze[z];
    } else {
        // the mixed corrector stored neither; these are its quotients
        st.zr = st.zm / st.zvol;
        st.ze = a.zetot[z] / (st.zm + 1.e-99);
    }
}

template <int NS, int CL>
__device__ __forceinline__ double zone_pred_mixed(const FusedArgs& a, int z, int sb, SideW sw,
                                                  const int (&pp)[NS], double dt, int& bad,
                                                  bool valid, ClCount& cnt, bool zre) {
    d2 x0[NS], u0[NS];
    ZoneState st;
    load_zone_mixed<NS>(a, z, pp, zre, x0, u0, st);
    return zone_pred_mixed_arrays<NS, CL>(a, z, sb, sw, x0, u0, st, dt, bad, valid, cnt);
}

template <int NS, int CL>
__device__ __forceinline__ double zone_pred_mixed(const FusedArgs& a, int z, int sb, SideW sw,
                                                  double dt, int& bad, bool valid, ClCount& cnt,
                                                  bool zre) {
    int pp[NS];
    load_pp<NS>(a, sb, pp);
    return zone_pred_mixed<NS, CL>(a, z, sb, sw, pp, dt, bad, valid, cnt, zre);
}

// K1, mixed precision.  With FLAG, zones with a gated corner are appended to
// their block's band slice of the run's zone list (list_count) for the
// learned pass; their order in the list is not fixed, their results are.
// With REDO it runs only when the pipelined cycle's finalize asked for the
// predictor to be redone (Ctl::redo).
template <int NS, bool FLAG, bool REDO = false>
__global__ void __launch_bounds__(PN_BLOCK) __attribute__((amdgpu_waves_per_eu(4)))
k_pred_mixed(FusedArgs a, int zbeg, int zend, int sbeg, int poff, int run) {
    if (a.ctl->done) return;
    if (REDO && !a.ctl->redo) return;
    const double dt = a.ctl->dt;
    const bool zre = a.ctl->zre_valid != 0;   // read once: the loop stores
    double dtmin = 1.e99;
    int bad = 0;
    const int nunits = (zend - zbeg + PN_BLOCK - 1) / PN_BLOCK;
    Units w = block_units(nunits, a.xcd);
    int zn = zbeg + w.u * PN_BLOCK + threadIdx.x;
    int pn[NS];
    if (w.u < w.end && zn < zend) load_pp<NS>(a, sbeg + (zn - zbeg) * NS, pn);
    for (; w.u < w.end; w.u += w.step) {
        // this zone's points were loaded by the previous iteration; load the next zone's
        const int z = zn;
        int pp[NS];
#pragma unroll
        for (int k = 0; k < NS; ++k) pp[k] = pn[k];
        zn = zbeg + (w.u + w.step) * PN_BLOCK + threadIdx.x;
        if (w.u + w.step < w.end && zn < zend) load_pp<NS>(a, sbeg + (zn - zbeg) * NS, pn);
        ClCount cnt;
        if (z < zend) {
            const double zdthyd = zone_pred_mixed<NS, FLAG ? CL_FLAG : CL_EXACT>(
                a, z, sbeg + (z - zbeg) * NS, side_w(z, zbeg, zend, sbeg, NS), pp, dt, bad, true, cnt,
                zre);
            dtmin = (zdthyd < dtmin) ? zdthyd : dtmin;
        }
        if constexpr (FLAG) {
            const uint64_t m = __ballot(cnt.flag);
            if (m) {
                unsigned base = 0;
                if ((threadIdx.x & 63) == 0) base = atomicAdd(list_count(a, run, w.band), (unsigned)__popcll(m));
                base = __shfl(base, 0, 64);
                if (cnt.flag) {
                    const uint64_t below = m & ((1ull << (threadIdx.x & 63)) - 1ull);
                    a.zlist[zbeg + list_unit0(nunits, w.band) * PN_BLOCK + base + (unsigned)__popcll(below)] = z;
                }
            }
        }
    }
    const double m = block_min(dtmin);
    const int b = block_sum(bad);
    if (threadIdx.x == 0) {
        a.part_dt[poff + blockIdx.x] = m;
        a.part_bp[poff + blockIdx.x] = b;
    }
}

// Learned pass over the zones a flagging K1 listed for this run: recomputes
// each listed zone with the network's coefficient on its gated corners and
// rewrites its corner and work forces.  The packed weights are staged in LDS
// once per block.  Every lane takes part in every unit (the network runs
// across the wave); lanes past the list's end repeat its first zone and
// store nothing.
template <int NS>
__global__ void __launch_bounds__(PN_BLOCK) __attribute__((amdgpu_waves_per_eu(2)))
k_pred_list(FusedArgs a, int zbeg, int zend, int sbeg, int run) {
    // The pass is the latency of a few waves, so everything it starts from
    // (done flag, dt, the slices' counts, the weights) is loaded at once,
    // before the first wait; the weights go to LDS before the exit test.
    const int done = a.ctl->done;
    const double dt = a.ctl->dt;
    const bool zre = a.ctl->zre_valid != 0;   // read once: the loop stores
    int lcnt[PN_LSLICES];
#pragma unroll
    for (int s = 0; s < PN_LSLICES; ++s) lcnt[s] = (int)*list_count(a, run, s);
    constexpr int NQ = (int)(sizeof(ClosurePack) / 16);
    constexpr int NQT = (NQ + PN_BLOCK - 1) / PN_BLOCK;
    __shared__ ClosurePack wp;
    {
        const uint4* src = reinterpret_cast<const uint4*>(a.pack);
        uint4* dst = reinterpret_cast<uint4*>(&wp);
        // indices past the end repeat the last quad (the same value to the
        // same LDS address), so there is no branch between the loads
#pragma unroll
        for (int j = 0; j < NQT; ++j) {
            const int i = min((int)threadIdx.x + j * PN_BLOCK, NQ - 1);
            dst[i] = src[i];
        }
    }
    // the slices' units of listed zones (lu0[s] the first)
    const int runits = (zend - zbeg + PN_BLOCK - 1) / PN_BLOCK;
    int lu0[PN_LSLICES + 1];
    lu0[0] = 0;
#pragma unroll
    for (int s = 0; s < PN_LSLICES; ++s) lu0[s + 1] = lu0[s] + (lcnt[s] + PN_BLOCK - 1) / PN_BLOCK;
    const int nunits = lu0[PN_LSLICES];
    Units w = block_units(nunits, a.xcd);
    if (done || w.u >= w.end) return;     // nothing listed for this block
    __syncthreads();
    FusedArgs b = a;
    b.pack = &wp;
    int bad = 0;
    ClCount cnt;
    for (; w.u < w.end; w.u += w.step) {
        // the slice holding unit w.u (constant indices only: the arrays stay in registers)
        int s = 0, sc = lcnt[0], su0 = 0;
#pragma unroll
        for (int t = 1; t < PN_LSLICES; ++t)
            if (lu0[t] <= w.u) {
                s = t;
                sc = lcnt[t];
                su0 = lu0[t];
            }
        const int i = (w.u - su0) * PN_BLOCK + threadIdx.x;
        const bool valid = i < sc;
        const int z = a.zlist[zbeg + list_unit0(runits, s) * PN_BLOCK + (valid ? i : 0)];
        (void)zone_pred_mixed<NS, CL_RECOMP>(b, z, sbeg + (z - zbeg) * NS, side_w(z, zbeg, zend, sbeg, NS),
                                             dt, bad, valid, cnt, zre);
    }
    const int nl = block_sum(cnt.learned);
    const int nf = block_sum(cnt.fallback);
    if (threadIdx.x == 0 && (nl | nf)) {
        atomicAdd(a.cl_stats, (unsigned long long)nl);
        atomicAdd(a.cl_stats + 1, (unsigned long long)nf);
    }
}

// Mixed K1 with the learned closure or with tuple capture: every lane of a
// wave runs every unit (lanes past the run's end work on a copy of its last
// zone and store nothing), because the network and the capture slots are
// computed across the wave.
template <int NS, int CL>
__global__ void __launch_bounds__(PN_BLOCK) __attribute__((amdgpu_waves_per_eu(2)))
k_pred_cl(FusedArgs a, int zbeg, int zend, int sbeg, int poff) {
    if (a.ctl->done) return;
    const double dt = a.ctl->dt;
    const bool zre = a.ctl->zre_valid != 0;   // read once: the loop stores
    double dtmin = 1.e99;
    int bad = 0;
    ClCount cnt;
    const int nunits = (zend - zbeg + PN_BLOCK - 1) / PN_BLOCK;
    for (Units w = block_units(nunits, a.xcd); w.u < w.end; w.u += w.step) {
        const int z = zbeg + w.u * PN_BLOCK + threadIdx.x;
        const bool valid = z < zend;
        const int zc = valid ? z : zend - 1;
        const double zdthyd = zone_pred_mixed<NS, CL>(a, zc, sbeg + (zc - zbeg) * NS,
                                                      side_w(zc, zbeg, zend, sbeg, NS), dt, bad, valid,
                                                      cnt, zre);
        if (valid) dtmin = (zdthyd < dtmin) ? zdthyd : dtmin;
    }
    const double m = block_min(dtmin);
    const int b = block_sum(bad);
    if constexpr (CL == CL_LEARNED) {
        const int nl = block_sum(cnt.learned);
        const int nf = block_sum(cnt.fallback);
        if (threadIdx.x == 0 && (nl | nf)) {
            atomicAdd(a.cl_stats, (unsigned long long)nl);
            atomicAdd(a.cl_stats + 1, (unsigned long long)nf);
        }
    }
    if (threadIdx.x == 0) {
        a.part_dt[poff + blockIdx.x] = m;
        a.part_bp[poff + blockIdx.x] = b;
    }
}

// ---------------------------------------------------------------------------
// K1, corner-per-lane.

// Corner group of a lane: the NS lanes holding one zone's corners.
template <int NS>
struct Grp {
    int base;   // lane of corner 0
    int k;      // this lane's corner
    __device__ __forceinline__ double at(double v, int j) const { return __shfl(v, base + j, 64); }
    __device__ __forceinline__ double nx(double v) const {
        return __shfl(v, base + (k + 1 == NS ? 0 : k + 1), 64);
    }
    __device__ __forceinline__ double pv(double v) const {
        return __shfl(v, base + (k == 0 ? NS - 1 : k - 1), 64);
    }
    __device__ __forceinline__ d2 at(d2 v, int j) const { return mk(at(v.x, j), at(v.y, j)); }
    __device__ __forceinline__ d2 nx(d2 v) const { return mk(nx(v.x), nx(v.y)); }
    __device__ __forceinline__ d2 pv(d2 v) const { return mk(pv(v.x), pv(v.y)); }
    // sum over the group's corners in ascending order, starting from 0
    __device__ __forceinline__ double sum(double v) const {
        double acc = 0.;
#pragma unroll
        for (int j = 0; j < NS; ++j) acc += at(v, j);
        return acc;
    }
    __device__ __forceinline__ d2 sum(d2 v) const {
        d2 acc = mk(0., 0.);
#pragma unroll
        for (int j = 0; j < NS; ++j) acc = add(acc, at(v, j));
        return acc;
    }
};

// One corner of zone z (sides s - k .. s - k + NS - 1); returns the zone's
// calcDtNew candidate on the group's corner 0 and 1e99 elsewhere.
template <int NS>
__device__ __forceinline__ double corner_pred(const FusedArgs& a, const Grp<NS>& g, int z, int s,
                                              int sws, bool live, double dt, int& bad) {
    const double dth = 0.5 * dt;
    const double n = (double)NS;
    // advPosHalf at this corner's point
    const int p = a.mapsp1[s];
    const d2 x0 = mk(a.pxx[p], a.pxy[p]);
    const d2 u0 = mk(a.pux[p], a.puy[p]);
    const d2 xp = add(x0, scl(dth, u0));
    const double mf = a.smf[s];
    const d2 xpn = g.nx(xp), u0n = g.nx(u0), u0p = g.pv(u0);
    // calcCtrs
    const d2 ex = scl(0.5, add(xp, xpn));
    const d2 zx = g.sum(dvs(xp, n));
    const d2 exp_ = g.pv(ex);
    // calcVols, calcEdgeLen
    const double third = 1. / 3.;
    const double sa = 0.5 * cross(sub(xpn, xp), sub(zx, xp));
    const double sv = third * sa * (xp.x + xpn.x + zx.x);
    const double zarea = g.sum(sa);
    const double zvolp = g.sum(sv);
    if (live && sv <= 0.) bad += 1;
    const double el = len(sub(xpn, xp));
    const double elp = g.pv(el);
    // calcCharLen: min over the zone's sides in ascending order from 1e99
    const double fac = (NS == 3 ? 3. : 4.);
    const double sdl = fac * sa / el;
    double zdl = 1.e99;
#pragma unroll
    for (int j = 0; j < NS; ++j) zdl = smin(zdl, g.at(sdl, j));
    // calcRho (pred)
    const double zm = a.zm[z];
    const double zrp = zm / zvolp;
    // calcStateHalf (reads ZR, ZE, ZWRATE of the previous cycle, ZVOL0 = ZVOL)
    const double gm1 = a.gamma - 1.;
    const double ssmin2 = smax(a.ssmin * a.ssmin, 1.e-99);
    const double r = a.zr[z];
    const double e = smax(a.ze[z], 0.);
    const double pp = gm1 * r * e;
    const double pre = gm1 * e;
    const double per = gm1 * r;
    const double csqd = smax(ssmin2, pre + per * pp / (r * r));
    const double zss = __builtin_sqrt(csqd);
    const double minv = 1. / zm;
    const double dv = (zvolp - a.zvol[z]) * minv;
    const double bulk = r * csqd;
    const double denom = 1. + 0.5 * per * dv;
    const double src = a.zwrate[z] * dth * minv;
    const double zp = pp + (per * src - r * bulk * dv) / denom;
    // calcSurfVecs, calcForcePGas, calcForceTTS
    const d2 ssurf = rot_ccw(sub(ex, zx));
    const d2 sfp = scl(-zp, ssurf);
    double sstmp = smax(zss, a.ssmin);
    sstmp = a.alfa * sstmp * sstmp;
    const double vfacinv = zarea / sa;
    const double srho = zrp * mf * vfacinv;
    const double sdp = sstmp * (srho - zrp);
    const d2 sft = scl(-sdp, ssurf);
    // setCornerDiv for corner k (s = ss3[c] is side k-1, s2 = c is side k)
    const d2 zuc = g.sum(dvs(u0, n));
    const d2 up0 = u0;
    const d2 xp0 = xp;
    const d2 up1 = scl(0.5, add(up0, u0n));
    const d2 xp1 = ex;
    const d2 up2 = zuc;
    const d2 xp2 = zx;
    const d2 up3 = scl(0.5, add(u0p, up0));
    const d2 xp3 = exp_;
    const double cvolume = 0.5 * cross(sub(xp2, xp0), sub(xp3, xp1));
    const d2 v1 = sub(xp3, xp0);
    const d2 v2 = sub(xp1, xp0);
    const double de1 = elp;
    const double de2 = el;
    const double minelen = smin(de1, de2);
    double ccos = ((minelen < 1.e-12) ? 0. : 4. * dot(v1, v2) / (de1 * de2));
    const double cdiv = (cross(sub(up2, up0), sub(xp3, xp1)) - cross(sub(up3, up1), sub(xp2, xp0))) /
                        (2.0 * cvolume);
    const d2 dxx1 = scl(0.5, sub(sub(add(xp1, xp2), xp0), xp3));
    const d2 dxx2 = scl(0.5, sub(sub(add(xp2, xp3), xp0), xp1));
    const double dx1 = len(dxx1);
    const double dx2 = len(dxx2);
    const d2 duav = scl(0.25, add(add(add(up0, up1), up2), up3));
    const double test1 = fabs(dot(dxx1, duav) * dx2);
    const double test2 = fabs(dot(dxx2, duav) * dx1);
    const double num = (test1 > test2 ? dx1 : dx2);
    const double den = (test1 > test2 ? dx2 : dx1);
    const double rr = num / den;
    double evol = __builtin_sqrt(4.0 * cvolume * rr);
    evol = smin(evol, 2.0 * minelen);
    const double dv1 = len2(sub(sub(add(up1, up2), up0), up3));
    const double dv2 = len2(sub(sub(add(up2, up3), up0), up1));
    double du = __builtin_sqrt(smax(dv1, dv2));
    evol = (cdiv < 0.0 ? evol : 0.);
    du = (cdiv < 0.0 ? du : 0.);
    // setQCnForce
    const double gammap1 = a.qgamma + 1.0;
    const double ztmp2 = a.q2 * 0.25 * gammap1 * du;
    const double ztmp1 = a.q1 * zss;
    const double zkur = ztmp2 + __builtin_sqrt(ztmp2 * ztmp2 + ztmp1 * ztmp1);
    const double mu = zkur * zrp * evol;
    const double crmu = ((cdiv > 0.0) ? 0. : mu);
    const d2 cqe1 = dvs(scl(crmu, sub(u0, u0p)), elp);
    const d2 cqe2 = dvs(scl(crmu, sub(u0n, u0)), el);
    // setForceQCS: side k joins corner k (c1) and corner k+1 (c2)
    const double csin2 = 1.0 - ccos * ccos;
    const double cw = ((csin2 < 1.e-4) ? 0. : cvolume / csin2);
    ccos = ((csin2 < 1.e-4) ? 0. : ccos);
    const double cw2 = g.nx(cw), ccos2 = g.nx(ccos);
    const d2 cqe12 = g.nx(cqe1), cqe22 = g.nx(cqe2);
    const d2 fq = add(scl(cw, add(cqe2, scl(ccos, cqe1))), scl(cw2, add(cqe12, scl(ccos2, cqe22))));
    const d2 sfq = dvs(fq, el);
    // setVelDiff: max over the zone's sides from 0
    const d2 dxs = sub(xpn, xp);
    const d2 dus = sub(u0n, u0);
    double dux = dot(dus, dxs);
    dux = (el > 0. ? fabs(dux) / el : 0.);
    double ztmp = 0.;
#pragma unroll
    for (int j = 0; j < NS; ++j) ztmp = smax(ztmp, g.at(dux, j));
    const double zdu = a.q1 * zss + 2. * a.q2 * ztmp;
    // sumCrnrForce's corner force, calcCrnrMass's corner mass, calcWork's
    // side force
    const d2 tot = add(add(sfp, sfq), sft);
    const d2 cf = sub(tot, g.pv(tot));
    const double mfp = g.pv(mf);
    const double cmass = zrp * zarea * 0.5 * (mf + mfp);
    if (live) {
        const int slot = a.pcpos[s];
        a.cfx[slot] = cf.x;
        a.cfy[slot] = cf.y;
        a.cmass[slot] = cmass;
        const d2 sfw = add(sfp, sfq);
        a.sfwx[sws] = sfw.x;
        a.sfwy[sws] = sfw.y;
        if (g.k == 0) a.zp[z] = zp;
    }
    const double fuzz = 1.e-99;
    const double cdt = smax(zdu, smax(zss, fuzz));
    const double zdthyd = zdl * a.cfl / cdt;
    return (live && g.k == 0) ? zdthyd : 1.e99;
}

template <int NS>
__global__ void __launch_bounds__(PN_BLOCK) k_pred_corner(FusedArgs a, int zbeg, int zend, int sbeg,
                                                          int poff) {
    if (a.ctl->done) return;
    constexpr int ZPW = 64 / NS;                      // zones per wave
    constexpr int ZPB = ZPW * (PN_BLOCK / 64);        // zones per block tile
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    Grp<NS> g;
    const int gi = lane / NS;
    g.k = lane - gi * NS;
    g.base = gi * NS;
    const double dt = a.ctl->dt;
    double dtmin = 1.e99;
    int bad = 0;
    const int nunits = (zend - zbeg + ZPB - 1) / ZPB;
    for (Units w = block_units(nunits, a.xcd); w.u < w.end; w.u += w.step) {
        const int zw = zbeg + w.u * ZPB + wave * ZPW + gi;
        const bool live = (gi < ZPW) && (zw < zend);
        const int z = live ? zw : zbeg;               // idle lanes read a valid zone
        const SideW sw = side_w(z, zbeg, zend, sbeg, NS);
        const double zdthyd = corner_pred<NS>(a, g, z, sbeg + (z - zbeg) * NS + g.k,
                                              sw_slot<NS>(sw, g.k), live, dt, bad);
        dtmin = (zdthyd < dtmin) ? zdthyd : dtmin;
    }
    const double m = block_min(dtmin);
    const int b = block_sum(bad);
    if (threadIdx.x == 0) {
        a.part_dt[poff + blockIdx.x] = m;
        a.part_bp[poff + blockIdx.x] = b;
    }
}

// ---------------------------------------------------------------------------
// K2

// point update shared by the regular and the heavy-point paths
// A point's state as K2 reads it.
struct PointIn {
    d2 x0, u0;
    unsigned bits;
};
__device__ __forceinline__ PointIn load_point(const FusedArgs& a, int p) {
    PointIn q;
    q.x0 = mk(a.pxx[p], a.pxy[p]);
    q.u0 = mk(a.pux[p], a.puy[p]);
    q.bits = a.pbc[p];
    return q;
}

// A point's new state, and what calcWork reads at it: T = float (the mixed
// form) needs (pu0 + pu) only times pxp.x, so that product is vs and xpx is
// not used.
struct PointOut {
    d2 x, u, vs;
    double xpx;
};
template <typename T>
__device__ __forceinline__ PointOut point_new(const FusedArgs& a, const PointIn& q, double mass, d2 f, double dt) {
    const double dth = 0.5 * dt;
    const d2 x0 = q.x0;
    const d2 uin = q.u0;
    d2 u0 = uin;
    const unsigned bits = q.bits;
    if (bits) {
        for (int b = 0; b < a.nbcs; ++b) {
            if (bits & (1u << b)) {
                const d2 v = mk(a.bcv[b], a.bcv[8 + b]);
                u0 = project(u0, v);
                f = project(f, v);
            }
        }
    }
    const double fuzz = 1.e-99;
    const d2 acc = dvs(f, smax(mass, fuzz));
    PointOut r;
    r.u = add(u0, scl(dt, acc));
    r.x = add(x0, scl(dt * 0.5, add(u0, r.u)));
    r.xpx = x0.x + dth * uin.x;              // pxp.x for calcWork
    r.vs = add(u0, r.u);                     // pu0 + pu for calcWork
    if constexpr (sizeof(T) == 4) r.vs = mk(r.vs.x * r.xpx, r.vs.y * r.xpx);
    return r;
}

// calcWork's values of a point (vs2 holds the pair {x, y} together: K3
// gathers it as one 16-byte access).
template <typename T>
__device__ __forceinline__ void store_work_point(const FusedArgs& a, int p, const PointOut& r) {
    if constexpr (sizeof(T) == 8) a.pxpx[p] = r.xpx;
    const f64x2u v = {r.vs.x, r.vs.y};
    *reinterpret_cast<f64x2u*>(a.vs2 + 2 * (int64_t)p) = v;
}

template <typename T>
__device__ __forceinline__ void point_update(const FusedArgs& a, int p, const PointIn& q,
                                             double mass, d2 f, double dt) {
    const PointOut r = point_new<T>(a, q, mass, f, dt);
    store_work_point<T>(a, p, r);
    a.oxx[p] = r.x.x;
    a.oxy[p] = r.x.y;
    a.oux[p] = r.u.x;
    a.ouy[p] = r.u.y;
}

// Corner values by corner slot: FP64 arrays for the plain form, FP32 records
// for the mixed-precision form (summed in FP64 either way).
template <typename T> struct Corners;
template <> struct Corners<double> {
    __device__ static double mass(const FusedArgs& a, int k) { return a.cmass[k]; }
    __device__ static double fx(const FusedArgs& a, int k) { return a.cfx[k]; }
    __device__ static double fy(const FusedArgs& a, int k) { return a.cfy[k]; }
};
template <> struct Corners<float> {
    __device__ static double mass(const FusedArgs& a, int k) { return (double)a.fcrn[3 * k + 2]; }
    __device__ static double fx(const FusedArgs& a, int k) { return (double)a.fcrn[3 * k]; }
    __device__ static double fy(const FusedArgs& a, int k) { return (double)a.fcrn[3 * k + 1]; }
};

// The slot of position c (CSR index k) of point p's corner list (the host's
// corner_slot, with a.nump the mesh's or the batch arena's point count).
__device__ __forceinline__ int corner_slot(const FusedArgs& a, int p, int c, int k) {
    return (c < 4) ? c * a.nump + p : 4 * a.nump + k;
}

// Point gathers, fixed BCs, acceleration and position update.
//
// A high-valence point (the pie origin has one corner per centre triangle)
// takes a whole block: the block stages the corner values in LDS, a chunk
// ahead, and one lane per sum (mass, force x, force y) adds them in ascending
// order.  It is a serial chain of additions: with one lane for all three sums,
// waiting for LDS at every corner, the point pass of a pie with 640 corners at
// its origin took 18.7 us; now 11.5.  Called by every thread of the block.
template <typename T, class Update>
__device__ __forceinline__ void point_heavy(const FusedArgs& a, int p, const Update& update) {
    using C = Corners<T>;
    __shared__ double sv[3][PN_BLOCK];
    const int kb = a.pcbeg[p], ke = a.pcbeg[p + 1], t = threadIdx.x;
    double m = 0., acc = 0.;
    d2 f = mk(0., 0.);
    auto load = [&](int k) {
        if (k < ke) {
            const int sl = corner_slot(a, p, k - kb, k);
            m = C::mass(a, sl);
            f = mk(C::fx(a, sl), C::fy(a, sl));
        }
    };
    load(kb + t);
    for (int c0 = kb; c0 < ke; c0 += PN_BLOCK) {
        sv[0][t] = m;
        sv[1][t] = f.x;
        sv[2][t] = f.y;
        __syncthreads();
        load(c0 + PN_BLOCK + t);
        if (t < 3) {
            const int cnt = (ke - c0 < PN_BLOCK) ? ke - c0 : PN_BLOCK;
            int i = 0;
            for (; i + 16 <= cnt; i += 16) {
                double v[16];
#pragma unroll
                for (int j = 0; j < 16; ++j) v[j] = sv[t][i + j];
#pragma unroll
                for (int j = 0; j < 16; ++j) acc += v[j];
            }
            for (; i < cnt; ++i) acc += sv[t][i];
        }
        __syncthreads();
    }
    if (t < 3) sv[t][0] = acc;
    __syncthreads();
    if (t == 0) update(p, load_point(a, p), sv[0][0], mk(sv[1][0], sv[2][0]));
}
template <typename T>
__device__ __forceinline__ void point_heavy(const FusedArgs& a, int p, double dt) {
    point_heavy<T>(a, p, [&](int p, const PointIn& q, double mass, d2 f) { point_update<T>(a, p, q, mass, f, dt); });
}

// An ordinary point, one thread; points with more than PN_HEAVY corners are
// left to point_heavy.
//
// The point's state and its first four corners (most points have at most
// four) are loaded together, then summed in ascending order.
template <typename T, class Update>
__device__ __forceinline__ void point_light(const FusedArgs& a, int p, const Update& update) {
    using C = Corners<T>;
    const int kb = a.pcbeg[p], ke = a.pcbeg[p + 1];
    const int n = ke - kb;
    if (n > PN_HEAVY) return;
    const PointIn q = load_point(a, p);
    double m4[4];
    d2 f4[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        // every point has a corner: clamped to the last one, the load is in
        // range and unconditional (no branch between the loads)
        const int sl = ((j < n) ? j : n - 1) * a.nump + p;
        m4[j] = C::mass(a, sl);
        f4[j] = mk(C::fx(a, sl), C::fy(a, sl));
    }
    double mass = 0.;
    d2 f = mk(0., 0.);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if (kb + j < ke) {
            mass += m4[j];
            f = add(f, f4[j]);
        }
    }
    for (int k = kb + 4; k < ke; ++k) {
        const int sl = 4 * a.nump + k;
        mass += C::mass(a, sl);
        f = add(f, mk(C::fx(a, sl), C::fy(a, sl)));
    }
    update(p, q, mass, f);
}
template <typename T>
__device__ __forceinline__ void point_light(const FusedArgs& a, int p, double dt) {
    point_light<T>(a, p, [&](int p, const PointIn& q, double mass, d2 f) { point_update<T>(a, p, q, mass, f, dt); });
}

// The point pass of a task-mode cycle: the sums of k_point over the same
// corner slots, then the fields that the point tasks leave: copies and half
// step (advPosHalf), corner mass and force sums, the force and start velocity
// with the fixed velocities applied, calcAccel and advPosFull.
struct TaskPoints {
    pennant_vec px0, pu0, pxp, pf, pap;
    double* pmaswt;
};
__global__ void __launch_bounds__(PN_BLOCK) k_cycle_points(FusedArgs a, TaskPoints t) {
    if (a.ctl->done) return;
    const double dt = a.ctl->dt;
    auto update = [&](int p, const PointIn& q, double mass, d2 f) {
        st(t.px0, p, q.x0);
        st(t.pxp, p, add(q.x0, scl(0.5 * dt, q.u0)));
        d2 u0 = q.u0;
        if (q.bits)
            for (int b = 0; b < a.nbcs; ++b)
                if (q.bits & (1u << b)) {
                    const d2 v = mk(a.bcv[b], a.bcv[8 + b]);
                    u0 = project(u0, v);
                    f = project(f, v);
                }
        const d2 acc = dvs(f, smax(mass, 1.e-99));
        const d2 u = add(u0, scl(dt, acc)), x = add(q.x0, scl(dt * 0.5, add(u0, u)));
        t.pmaswt[p] = mass;
        st(t.pf, p, f);
        st(t.pu0, p, u0);
        st(t.pap, p, acc);
        a.pxx[p] = x.x;
        a.pxy[p] = x.y;
        a.pux[p] = u.x;
        a.puy[p] = u.y;
    };
    if ((int)blockIdx.x < a.nheavy) {
        point_heavy<double>(a, a.heavy[blockIdx.x], update);
        return;
    }
    const int p = (blockIdx.x - a.nheavy) * PN_BLOCK + threadIdx.x;
    if (p < a.npown) point_light<double>(a, p, update);
}

// K2: blocks [0, nheavy) take the heavy points, the rest one point per thread.
// Block 0 also clears the learned pass's zone counts: that pass has run
// before K2, and the next predictor appends to them.
template <bool REDO>
__device__ __forceinline__ void fold_lookahead(const FusedArgs& a, int npred);

template <typename T>
__global__ void __launch_bounds__(PN_BLOCK) k_point(FusedArgs a) {
    // The pipelined cycle's K2 has one block more: it folds the partials of
    // the previous cycle's redone predictor, if there was one, into the
    // look-ahead values -- the work of a separate one-block launch after the
    // redo, here before the zone pass overwrites the partials.
    if (a.la_npred > 0 && (int)blockIdx.x == (int)gridDim.x - 1) {
        fold_lookahead<true>(a, a.la_npred);
        return;
    }
    if (a.zcount && blockIdx.x == 0)
        for (int i = threadIdx.x; i < a.nzruns * PN_LSLICES; i += PN_BLOCK) a.zcount[i * PN_LSTRIDE] = 0u;
    if (a.ctl->done) return;
    const double dt = a.ctl->dt;
    if ((int)blockIdx.x < a.nheavy) {
        point_heavy<T>(a, a.heavy[blockIdx.x], dt);
        return;
    }
    const int p = (blockIdx.x - a.nheavy) * PN_BLOCK + threadIdx.x;
    if (p < a.npown) point_light<T>(a, p, dt);
}

// The corrector of a zone from its state before the cycle (et, zvol0, zm), its
// predictor's pressure and side work forces, and its points' new positions x
// and work values vs, xp; folds the bad-side count and the dvol ratio.
struct CorrOut {
    double zwrate, zetot, ze, zr, zvol;
};
template <int NS, typename T>
__device__ __forceinline__ CorrOut corr_core(double et, double zvol0, double zm, double zp, const d2 (&sfw)[NS],
                                             const d2 (&x)[NS], const d2 (&vs)[NS], const double (&xp)[NS],
                                             double dt, int& bad, double& dvov) {
    const double dth = 0.5 * dt;
    const double n = (double)NS;
    d2 zx = mk(0., 0.);
#pragma unroll
    for (int k = 0; k < NS; ++k) zx = add(zx, dvs(x[k], n));
    const double third = 1. / 3.;
    double zvol = 0.;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const d2 p1 = x[k], p2 = x[nxt<NS>(k)];
        const double sa = 0.5 * cross(sub(p2, p1), sub(zx, p1));
        const double sv = third * sa * (p1.x + p2.x + zx.x);
        zvol += sv;
        if (sv <= 0.) bad += 1;
    }
    // calcWork
    double w = 0.;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const int k2 = nxt<NS>(k);
        const d2 sftot = sfw[k];
        const double sd1 = dot(sftot, vs[k]);
        const double sd2 = dot(neg(sftot), vs[k2]);
        const double dwork = (sizeof(T) == 8) ? -dth * (sd1 * xp[k] + sd2 * xp[k2]) : -dth * (sd1 + sd2);
        et += dwork;
        w += dwork;
    }
    // calcWorkRate, calcEnergy, calcRho (corr), calcDvol
    const double dtinv = 1. / dt;
    const double dvol = zvol - zvol0;
    const double zwr = (w + zp * dvol) * dtinv;
    const double fuzz = 1.e-99;
    CorrOut r;
    r.zwrate = zwr;
    r.zetot = et;
    r.ze = et / (zm + fuzz);
    r.zr = zm / zvol;
    r.zvol = zvol;
    const double zdvov = fabs((zvol - zvol0) / zvol0);
    dvov = (zdvov > dvov) ? zdvov : dvov;
    return r;
}

// ---------------------------------------------------------------------------
// K3: corrector geometry, work, work rate, energy, density, dvol of zone z
// (sides sb..sb+NS-1, points pp); folds the bad-side count and the dvol
// ratio.  The zone's own loads are issued before the point gathers, which
// wait for the point indices.  Returns the points' positions x and the zone's
// new state st (the next cycle's predictor starts from them).  With PIPE the
// cycle's predictor pressure comes from a.zpn and is stored to a.zp.
template <int NS, typename T, bool PIPE>
__device__ __forceinline__ void corr_zone_core(const FusedArgs& a, int z, int sb, SideW sw,
                                               const int (&pp)[NS], double dt, int& bad,
                                               double& dvov, d2 (&x)[NS], ZoneState& st) {
    double et = a.zetot[z];
    const double zvol0 = a.zvol[z];
    const double zm = a.zm[z];
    const double zp = PIPE ? a.zpn[z] : a.zp[z];
    d2 sfw[NS];
    if constexpr (sizeof(T) == 4) {
        f2 v[NS];
        load_sides<NS>(a.fsfw, sw, v);
#pragma unroll
        for (int k = 0; k < NS; ++k) sfw[k] = mk((double)v[k].x, (double)v[k].y);
    } else {
#pragma unroll
        for (int k = 0; k < NS; k += 2) {
            const int sl = sw_slot<NS>(sw, k);
            if (k + 1 < NS) {
                const f64x2u vx = __builtin_nontemporal_load(reinterpret_cast<const f64x2u*>(a.sfwx + sl));
                const f64x2u vy = __builtin_nontemporal_load(reinterpret_cast<const f64x2u*>(a.sfwy + sl));
                sfw[k] = mk(vx[0], vy[0]);
                sfw[k + 1] = mk(vx[1], vy[1]);
            } else {
                sfw[k] = mk(ld_nt(a.sfwx + sl), ld_nt(a.sfwy + sl));
            }
        }
    }
    d2 vs[NS];                 // mixed form: (pu0 + pu) pxp.x
    double xp[NS];
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        x[k] = mk(a.pxx[pp[k]], a.pxy[pp[k]]);
        const f64x2u v = *reinterpret_cast<const f64x2u*>(a.vs2 + 2 * (int64_t)pp[k]);
        vs[k] = mk(v[0], v[1]);
        if constexpr (sizeof(T) == 8) xp[k] = a.pxpx[pp[k]];
    }
    const CorrOut r = corr_core<NS, T>(et, zvol0, zm, zp, sfw, x, vs, xp, dt, bad, dvov);
    a.zwrate[z] = r.zwrate;
    a.zetot[z] = r.zetot;
    if constexpr (sizeof(T) == 8) {
        // the mixed form's predictors derive zr and ze from zm, zvol, zetot
        a.ze[z] = r.ze;
        a.zr[z] = r.zr;
    }
    a.zvol[z] = r.zvol;
    if (PIPE) a.zp[z] = zp;
    st.zm = zm;
    st.zr = r.zr;
    st.ze = r.ze;
    st.zvol = r.zvol;
    st.zwrate = r.zwrate;
}

template <int NS, typename T>
__device__ __forceinline__ void corr_zone_pp(const FusedArgs& a, int z, int sb, SideW sw,
                                             const int (&pp)[NS], double dt, int& bad, double& dvov) {
    d2 x[NS];
    ZoneState st;
    corr_zone_core<NS, T, false>(a, z, sb, sw, pp, dt, bad, dvov, x, st);
}

template <int NS, typename T>
__device__ __forceinline__ void corr_zone(const FusedArgs& a, int z, int sb, SideW sw, double dt,
                                          int& bad, double& dvov) {
    int pp[NS];
    load_pp<NS>(a, sb, pp);
    corr_zone_pp<NS, T>(a, z, sb, sw, pp, dt, bad, dvov);
}

// The point indices of a thread's next zone are loaded while the current
// zone is processed.
template <int NS, typename T>
__global__ void __launch_bounds__(PN_BLOCK) k_corr(FusedArgs a, int zbeg, int zend, int sbeg,
                                                   int poff) {
    if (a.ctl->done) return;
    const double dt = a.ctl->dt;
    double dvov = 1.e-99;
    int bad = 0;
    const int nunits = (zend - zbeg + PN_BLOCK - 1) / PN_BLOCK;
    Units wu = block_units(nunits, a.xcd);
    int z = zbeg + wu.u * PN_BLOCK + threadIdx.x;
    int pp[NS];
    if (wu.u < wu.end && z < zend) load_pp<NS>(a, sbeg + (z - zbeg) * NS, pp);
    for (; wu.u < wu.end; wu.u += wu.step) {
        const int zc = z;
        int pc[NS];
#pragma unroll
        for (int k = 0; k < NS; ++k) pc[k] = pp[k];
        z = zbeg + (wu.u + wu.step) * PN_BLOCK + threadIdx.x;
        if (wu.u + wu.step < wu.end && z < zend) load_pp<NS>(a, sbeg + (z - zbeg) * NS, pp);
        if (zc < zend)
            corr_zone_pp<NS, T>(a, zc, sbeg + (zc - zbeg) * NS, side_w(zc, zbeg, zend, sbeg, NS), pc, dt,
                                bad, dvov);
    }
    const double m = block_max(dvov);
    const int b = block_sum(bad);
    if (threadIdx.x == 0) {
        a.part_dv[poff + blockIdx.x] = m;
        a.part_bc[poff + blockIdx.x] = b;
    }
}

// ---------------------------------------------------------------------------
// Pipelined mixed cycle.  The predictor of cycle n+1 needs dt(n+1), which the
// finalize of cycle n computes from this cycle's predictor dt limit (known
// before K2) and its corrector's volume-change limit (known after K3).  The
// zone pass of cycle n runs each zone's corrector and then, from the state it
// has just computed, the zone's predictor of cycle n+1 with the dt that the
// finalize gives when the volume-change limit does not bind.  The finalize
// checks that dt bit for bit; when it differs, the predictor is redone with
// the actual dt.  Either way cycle n+1 starts from the same bits as the
// unpipelined cycle.

// The control-block values the end of a cycle and the look-ahead dt start from.
// dt of the cycle after the current one as the finalize computes it
// (src/Hydro.cc:1647-1667, src/Driver.cc:213-245) when the volume-change
// limit does not bind; `last` when the current cycle ends the run.
__device__ __forceinline__ double lookahead_dt(const CtlSnap& c, const DtParams& q, bool& last) {
    const double t1 = c.time + c.dt;
    last = (c.cycle + 1 >= q.cstop || t1 >= q.tstop);
    double r = 1.e99;
    if (c.la_dtnew < r) r = c.la_dtnew;
    double dt = q.dtmax;
    const double dtrecover = q.dtfac * c.dt;
    if (dtrecover < dt) dt = dtrecover;
    if ((q.tstop - t1) < dt) dt = q.tstop - t1;
    if (r < dt) dt = r;
    return dt;
}

// Zone pass of the pipelined mixed cycle: the corrector of every zone, then
// (unless the cycle ends the run) its predictor of the next cycle, which
// writes zp to a.zpn and, with FLAG, lists zones for the learned pass.
// Partials: corrector at part_dv/part_bc, predictor at part_dt/part_bp.
template <int NS, bool FLAG>
__global__ void __launch_bounds__(PN_BLOCK) __attribute__((amdgpu_waves_per_eu(3)))
k_zone_pipe(FusedArgs a, int zbeg, int zend, int sbeg, int poff, int run, DtParams q) {
    const Ctl* c = a.ctl;
    if (c->done) return;
    const double dt = c->dt;
    CtlSnap v;                 // this kernel does not write the control block
    v.time = c->time;
    v.dt = dt;
    v.la_dtnew = c->la_dtnew;
    v.cycle = c->cycle;
    v.la_bp = 0;
    v.done = 0;
    bool last;
    const double dtn = lookahead_dt(v, q, last);
    FusedArgs b = a;
    b.zp = a.zpn;
    double dvov = 1.e-99, dtmin = 1.e99;
    int badc = 0, badp = 0;
    const int nunits = (zend - zbeg + PN_BLOCK - 1) / PN_BLOCK;
    Units w = block_units(nunits, a.xcd);
    int zn = zbeg + w.u * PN_BLOCK + threadIdx.x;
    int pn[NS];
    if (w.u < w.end && zn < zend) load_pp<NS>(a, sbeg + (zn - zbeg) * NS, pn);
    for (; w.u < w.end; w.u += w.step) {
        const int z = zn;
        int pp[NS];
#pragma unroll
        for (int k = 0; k < NS; ++k) pp[k] = pn[k];
        zn = zbeg + (w.u + w.step) * PN_BLOCK + threadIdx.x;
        if (w.u + w.step < w.end && zn < zend) load_pp<NS>(a, sbeg + (zn - zbeg) * NS, pn);
        ClCount cnt;
        if (z < zend) {
            const int sb = sbeg + (z - zbeg) * NS;
            const SideW sw = side_w(z, zbeg, zend, sbeg, NS);
            d2 u[NS];
            if (!last) {
#pragma unroll
                for (int k = 0; k < NS; ++k) u[k] = mk(a.pux[pp[k]], a.puy[pp[k]]);
            }
            d2 x[NS];
            ZoneState st;
            corr_zone_core<NS, float, true>(a, z, sb, sw, pp, dt, badc, dvov, x, st);
            if (!last) {
                const double zdthyd = zone_pred_mixed_arrays<NS, FLAG ? CL_FLAG : CL_EXACT>(
                    b, z, sb, sw, x, u, st, dtn, badp, true, cnt);
                dtmin = (zdthyd < dtmin) ? zdthyd : dtmin;
            }
        }
        if constexpr (FLAG) {
            const uint64_t m = __ballot(cnt.flag);
            if (m) {
                unsigned base = 0;
                if ((threadIdx.x & 63) == 0) base = atomicAdd(list_count(a, run, w.band), (unsigned)__popcll(m));
                base = __shfl(base, 0, 64);
                if (cnt.flag) {
                    const uint64_t below = m & ((1ull << (threadIdx.x & 63)) - 1ull);
                    a.zlist[zbeg + list_unit0(nunits, w.band) * PN_BLOCK + base + (unsigned)__popcll(below)] = z;
                }
            }
        }
    }
    const double mv = block_max(dvov);
    const int bc = block_sum(badc);
    const double mt = block_min(dtmin);
    const int bp = block_sum(badp);
    if (threadIdx.x == 0) {
        a.part_dv[poff + blockIdx.x] = mv;
        a.part_bc[poff + blockIdx.x] = bc;
        a.part_dt[poff + blockIdx.x] = mt;
        a.part_bp[poff + blockIdx.x] = bp;
    }
}

// ---------------------------------------------------------------------------
// K4: reductions over the block partials (min and max are exact in any
// order; NaN partials cannot occur, the per-zone folds skip NaN) and the end
// of the cycle: calcDt (src/Hydro.cc:1647-1667), checkBadSides
// (src/Mesh.cc:1531-1550), the time/cycle update (src/Driver.cc:266-295), the
// stop test and calcGlobalDt (src/Driver.cc:213-245) for the next cycle.
__device__ __forceinline__ double blk_min_fin(double v) {
    __shared__ double part[PN_FIN_BLOCK / 64];
    __syncthreads();   // a previous call's partials may still be read
    v = wave_min(v);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0)
        for (int i = 1; i < PN_FIN_BLOCK / 64; ++i) v = (part[i] < v) ? part[i] : v;
    return v;
}
__device__ __forceinline__ int blk_sum_fin(int v) {
    __shared__ int part[PN_FIN_BLOCK / 64];
    __syncthreads();   // a previous call's partials may still be read
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0)
        for (int i = 1; i < PN_FIN_BLOCK / 64; ++i) v += part[i];
    return v;
}

// The four folds of a finalize in one pass over the block: wave folds, one
// LDS row per wave, and thread 0 folds the rows in wave order (the result is
// thread 0's).
template <int BS>
__device__ __forceinline__ void blk_fold_fin(double& mn, double& mx, int& bp, int& bc) {
    __shared__ double pmn[BS / 64], pmx[BS / 64];
    __shared__ int pbp[BS / 64], pbc[BS / 64];
    mn = wave_min(mn);
    mx = wave_max(mx);
    bp = wave_sum(bp);
    bc = wave_sum(bc);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        pmn[w] = mn;
        pmx[w] = mx;
        pbp[w] = bp;
        pbc[w] = bc;
    }
    __syncthreads();
    if (threadIdx.x == 0)
        for (int i = 1; i < BS / 64; ++i) {
            mn = (pmn[i] < mn) ? pmn[i] : mn;
            mx = (pmx[i] > mx) ? pmx[i] : mx;
            bp += pbp[i];
            bc += pbc[i];
        }
}

// Each thread's share of the partials (thread t of BS folds t, t + BS, ...),
// loaded PN_FIN_PER per thread at a time with no branch between the
// loads.  Indices past the end read the last partial again: a repeat leaves a
// min or max unchanged and adds 0 to a count.  npred, ncorr >= 1 (every
// launch has at least one block, every problem at least one unit).
#define PN_FIN_PER 8
template <int BS>
__device__ __forceinline__ void fold_partials(const double* part_dt, const int* part_bp, int npred,
                                              const double* part_dv, const int* part_bc, int ncorr,
                                              double& mn, int& bp, double& mx, int& bc) {
    const int n = npred > ncorr ? npred : ncorr;
    for (int base = 0; base < n; base += PN_FIN_PER * BS) {
        double dv[PN_FIN_PER], dd[PN_FIN_PER];
        int ip[PN_FIN_PER], ic[PN_FIN_PER];
#pragma unroll
        for (int j = 0; j < PN_FIN_PER; ++j) {
            const int i = base + (int)threadIdx.x + j * BS;
            const int ipd = min(i, npred - 1), icr = min(i, ncorr - 1);
            dd[j] = part_dt[ipd];
            ip[j] = part_bp[ipd];
            dv[j] = part_dv[icr];
            ic[j] = part_bc[icr];
        }
#pragma unroll
        for (int j = 0; j < PN_FIN_PER; ++j) {
            const int i = base + (int)threadIdx.x + j * BS;
            mn = (dd[j] < mn) ? dd[j] : mn;
            bp += (i < npred) ? ip[j] : 0;
            mx = (dv[j] > mx) ? dv[j] : mx;
            bc += (i < ncorr) ? ic[j] : 0;
        }
    }
}

__device__ __forceinline__ void finalize_block(Ctl* c, const double* part_dt, const int* part_bp,
                                               int npred, const double* part_dv, const int* part_bc,
                                               int ncorr, double cflv, int cstop, double dtmax,
                                               double dtfac, double tstop, int zre) {
    // The control block and the partials are read at once, so the block
    // waits for memory once (the partials of a run that has stopped are read
    // but not used).
    const CtlSnap v = snap_ctl(c);
    double mn = 1.e99, mx = 1.e-99;
    int bp = 0, bc = 0;
    fold_partials<PN_FIN_BLOCK>(part_dt, part_bp, npred, part_dv, part_bc, ncorr, mn, bp, mx, bc);
    blk_fold_fin<PN_FIN_BLOCK>(mn, mx, bp, bc);
    if (threadIdx.x != 0 || v.done) return;
    c->zre_valid = zre;
    end_cycle(c, v, mn, mx, bp, bc, {cflv, dtmax, dtfac, tstop, cstop});
}

__global__ void __launch_bounds__(PN_FIN_BLOCK) k_finalize(FusedArgs a, int npred, int ncorr,
                                                           double cflv, int cstop, double dtmax,
                                                           double dtfac, double tstop, int zre) {
    // the learned pass of this cycle has consumed its zone lists
    if (a.zcount)
        for (int i = threadIdx.x; i < a.nzruns * PN_LSLICES; i += PN_FIN_BLOCK) a.zcount[i * PN_LSTRIDE] = 0u;
    finalize_block(a.ctl, a.part_dt, a.part_bp, npred, a.part_dv, a.part_bc, ncorr, cflv, cstop,
                   dtmax, dtfac, tstop, zre);
}

// K4 of the pipelined mixed cycle: ends cycle n from its predictor's results
// (carried in Ctl::la_*) and its corrector's partials, then accepts the
// look-ahead predictor of cycle n+1 when the dt it assumed is the dt just
// computed, or asks for it to be redone (clearing the learned pass's zone
// counts, which the redo fills again).  The learned pass's zone counts of
// cycle n move from the pending to the reported counters.
__global__ void __launch_bounds__(PN_FIN_BLOCK) k_finalize_pipe(FusedArgs a, int npred, int ncorr,
                                                                DtParams q) {
    Ctl* c = a.ctl;
    if (c->done) return;
    double mn = 1.e99, mx = 1.e-99;
    int bp = 0, bc = 0;
    fold_partials<PN_FIN_BLOCK>(a.part_dt, a.part_bp, npred, a.part_dv, a.part_bc, ncorr, mn, bp, mx, bc);
    blk_fold_fin<PN_FIN_BLOCK>(mn, mx, bp, bc);
    if (threadIdx.x != 0) return;
    if (a.cl_stats) {
        const unsigned long long nl = atomicExch(a.cl_stats + 2, 0ull);
        const unsigned long long nf = atomicExch(a.cl_stats + 3, 0ull);
        atomicAdd(a.cl_stats, nl);
        atomicAdd(a.cl_stats + 1, nf);
    }
    const CtlSnap v = snap_ctl(c);
    bool last;
    const double dtn = lookahead_dt(v, q, last);
    double dt1 = 0.;
    c->zre_valid = 0;
    if (end_cycle(c, v, v.la_dtnew, mx, v.la_bp, bc, q, &dt1)) return;
    if (!last && dt1 == dtn) {
        c->la_dtnew = mn;
        c->la_bp = bp;
        c->redo = 0;
    } else {
        c->redo = 1;
        c->la_redos += 1;
        if (a.zcount)
            for (int r = 0; r < a.nzruns * PN_LSLICES; ++r) a.zcount[r * PN_LSTRIDE] = 0u;
    }
}

// After a predictor of the pipelined cycle (the prologue's, or with REDO a
// redone one): its dt limit and bad-side count become the Ctl::la_* values
// the next finalize ends the cycle with.  One block of PN_FIN_BLOCK threads.
template <bool REDO>
__device__ __forceinline__ void fold_lookahead(const FusedArgs& a, int npred) {
    Ctl* c = a.ctl;
    if (c->done) return;
    if (REDO && !c->redo) return;
    double mn = 1.e99;
    int bp = 0;
    for (int i = threadIdx.x; i < npred; i += PN_FIN_BLOCK) {
        const double v = a.part_dt[i];
        mn = (v < mn) ? v : mn;
        bp += a.part_bp[i];
    }
    mn = blk_min_fin(mn);
    bp = blk_sum_fin(bp);
    if (threadIdx.x != 0) return;
    c->la_dtnew = mn;
    c->la_bp = bp;
    c->redo = 0;
}
template <bool REDO>
__global__ void __launch_bounds__(PN_FIN_BLOCK) k_finalize_la(FusedArgs a, int npred) {
    fold_lookahead<REDO>(a, npred);
}

// ---------------------------------------------------------------------------
// Tile cycle: the whole cycle of a structured mesh in one kernel.
//
// On a rect or pie mesh in the generator's numbering a block takes a tile of
// PN_TILE x PN_TILE quads, one per thread: its (PN_TILE - 2)^2 inner zones and
// a ring of neighbours.  It runs the predictor of all of them, hands the
// corner values to the points between them through LDS, and finishes its
// inner zones' corrector from registers and LDS.  Neither corner records, nor
// side work forces, nor the points' work values go through memory, and a zone
// and its points are read once per cycle instead of two or three times: about
// 190 bytes a zone instead of 690 (FP64) or 460 (mixed).  The ring costs
// (16 / 14)^2 = 1.31 times the predictor's arithmetic.
//
// A block reads its ring from zones that other blocks own, so a cycle never
// writes what it reads: odd cycles of a launch go from the problem's arrays
// to a second set, even ones back (Ctl::cur says where the state is, and the
// second cycle of a pair copies it back when the first ended the run), so the
// problem's own arrays hold the state after every pair.
//
// Tiles hand their dt limits and dvol ratios on in slots (cycle_end.h).  On a
// rect of few tiles, all of them at work together, each tile of the next cycle
// ends the cycle from them by itself while its loads are under way (linked
// cycles: no launch between two tile kernels).  With many tiles each would pay
// for that, and one wave ends the cycle between the two: 3.5 us, where folding
// an array of 10600 partials took 9.5.  On a pie the triangles' few blocks end
// the cycle, whatever the number of tiles.
//
// The triangles of a pie's first row and the origin are not part of a tile:
// their predictor and corrector run as in the separate passes, before and
// after, and the tiles of the first row of quads read the triangles' corner
// records.  Sums run in the order of the separate passes (a point's corners in
// ascending side order), so the results are the same bits.
//
// What bounds it: a tile's chain of loads, arithmetic and barriers, with few
// waves to hide it (Sedov 1440^2 FP64: 240 VGPRs, two waves per SIMD, vector unit
// 0.86 busy; mixed: 128 VGPRs, four, saturated).  Larger tiles have less ring but more
// waves in step: 32 x 16 zones took 258 us where 16 x 16 takes 212 (FP64), and
// 139 where it takes 117 (mixed).  FP64 square roots and quotients without the
// scaling of their operands (9% fewer instructions) gained 1 to 3%; blocks
// that loop over tiles, loading the next one early, spilled (265 us).  Corner
// sums without branches (zones outside the mesh give zeros), 32-bit byte
// offsets and one fold of both counts together took Sedov 1440^2 from 211 to
// 205 us (FP64), 108.5 to 106.6 (mixed) and 154 to 149 (learned).
// Per cycle, separate passes (for mixed and learned the pipelined ones) ->
// tiles: FP64 Sedov 1440^2 306 -> 201 us, Noh pie 1024^2 178 -> 115 us; mixed
// LeBlanc 4096 x 256 87 -> 55 us, 333 x 217 23 -> 10.1 us; learned Sedov
// 1440^2 176 -> 141 us early in its run, 182 -> 187 with a developed front (see
// k_tile_list; separate passes unpipelined 202); FP64 90^2 12.6 -> 10.1 us by the
// linking alone.  Faster at every size but for that front's last tenth of the
// run, by 4%, so structured meshes take it by default.
#define PN_TILE 16
#define PN_TIN (PN_TILE - 2)
// Most tiles of linked cycles (tile_cycles).  Linked and not, us a cycle, FP64
// and mixed: 90^2 (49 tiles) 10.1 and 12.7, 7.6 and 10.1; 333 x 217 (384) 14.9
// and 17.1, 10.1 and 12.4; 420^2 (900) 25.8 and 27.3, 16.1 and 17.8; 500^2
// (1296) 35.4 both, 21.4 and 21.3; 1440^2 (10609) 213 and 200, 120 and 102.
#define PN_LINK_TILES 1024

// A structured mesh in the arrays: zone (i, j) of nzx x nzy has its points
// (i, j), (i + 1, j), (i + 1, j + 1), (i, j + 1); row 0 of a pie is the
// triangles, whose first point is the origin.
struct TileMesh {
    int nzx, nzy, pie;
    int zo, so, po;              // first zone, side and point in the arrays
};
__device__ __forceinline__ int tile_zone(const TileMesh& g, int i, int j) { return g.zo + j * g.nzx + i; }
__device__ __forceinline__ int tile_side(const TileMesh& g, int i, int j) {
    return g.so + 4 * (j * g.nzx + i) - (g.pie ? g.nzx : 0);
}
__device__ __forceinline__ int tile_point(const TileMesh& g, int i, int j) {
    return g.po + j * (g.nzx + 1) + i - (g.pie ? g.nzx : 0);
}

// Where a tile cycle writes the state (the points' through FusedArgs::oxx..).
struct TileOut {
    double* zr; double* ze; double* zetot; double* zwrate; double* zvol;
};

// A predictor's results kept in the block: corner forces and masses in LDS,
// [3 k + {0, 1, 2}][thread], the rest in registers.
template <typename T> struct TileKeep;
template <> struct TileKeep<double> {
    double* c;
    d2 sfw[4];
    double p;
    __device__ __forceinline__ void zp(double v) { p = v; }
    __device__ __forceinline__ void mass(int k, double v) { c[(3 * k + 2) * PN_BLOCK] = v; }
    __device__ __forceinline__ void force(int k, d2 f) {
        c[(3 * k) * PN_BLOCK] = f.x;
        c[(3 * k + 1) * PN_BLOCK] = f.y;
    }
    __device__ __forceinline__ void sides(int k, d2 f0, d2 f1) {
        sfw[k] = f0;
        sfw[k + 1] = f1;
    }
    __device__ __forceinline__ void side(int k, d2 f) { sfw[k] = f; }
};
template <> struct TileKeep<float> {
    float* c;
    f2 sfw[4];
    double p;
    __device__ __forceinline__ void zp(double v) { p = v; }
    __device__ __forceinline__ void mass(int k, float v) { c[(3 * k + 2) * PN_BLOCK] = v; }
    __device__ __forceinline__ void force(int k, float fx, float fy) {
        c[(3 * k) * PN_BLOCK] = fx;
        c[(3 * k + 1) * PN_BLOCK] = fy;
    }
    __device__ __forceinline__ void sides(const f2 (&f)[4]) {
#pragma unroll
        for (int k = 0; k < 4; ++k) sfw[k] = f[k];
    }
};

// The element at a byte offset (and a constant) from an array's start.  A
// scalar base, a 32-bit offset and the constant are one access's address,
// where an index takes a 64-bit addition and two registers per access; the
// arrays of a structured mesh are below 4 GiB (corner_slots_fit).
template <typename E, int C = 0, typename A>
__device__ __forceinline__ E at_byte(const A* p, unsigned off) {
    return *reinterpret_cast<const E*>(reinterpret_cast<const char*>(p) + off + C);
}
__device__ __forceinline__ void put_byte(double* p, unsigned off, double v) {
    *reinterpret_cast<double*>(reinterpret_cast<char*>(p) + off) = v;
}

// What a thread reads of its tile, as loaded.
template <typename T> struct TileIn;
template <> struct TileIn<double> {
    ZoneIn<4> z;
    double et;
    unsigned bits;
};
template <> struct TileIn<float> {
    d2 x[4], u[4];
    double zm, zvol, zwrate, et;
    f32x4u mf;
    unsigned bits;
};

// Every load of a thread for the tile whose first zone (ring included) is (i0,
// j0), with no branch: threads outside the mesh read the nearest zone and use
// nothing of it.
template <typename T>
__device__ __forceinline__ void tile_load(const FusedArgs& a, const TileMesh& g, int i0, int j0, TileIn<T>& in) {
    const int i = i0 + ((int)threadIdx.x & (PN_TILE - 1)), j = j0 + (int)threadIdx.x / PN_TILE;
    const int ci = min(max(i, 0), g.nzx - 1), cj = min(max(j, g.pie), g.nzy - 1);
    const unsigned z = 8u * (unsigned)tile_zone(g, ci, cj), sb = (unsigned)tile_side(g, ci, cj);
    const unsigned p = (unsigned)tile_point(g, ci, cj), p0 = 8u * p, p3 = p0 + 8u * (unsigned)(g.nzx + 1);
    auto points = [&](const double* x, const double* y, d2 (&v)[4]) {
        v[0] = mk(at_byte<double>(x, p0), at_byte<double>(y, p0));
        v[1] = mk(at_byte<double, 8>(x, p0), at_byte<double, 8>(y, p0));
        v[2] = mk(at_byte<double, 8>(x, p3), at_byte<double, 8>(y, p3));
        v[3] = mk(at_byte<double>(x, p3), at_byte<double>(y, p3));
    };
    if constexpr (sizeof(T) == 8) {
        points(a.pxx, a.pxy, in.z.x);
        points(a.pux, a.puy, in.z.u);
        in.z.zm = at_byte<double>(a.zm, z);
        in.z.zr = at_byte<double>(a.zr, z);
        in.z.ze = at_byte<double>(a.ze, z);
        in.z.zvol = at_byte<double>(a.zvol, z);
        in.z.zwr = at_byte<double>(a.zwrate, z);
        const f64x2u m0 = at_byte<f64x2u>(a.smf, 8u * sb), m1 = at_byte<f64x2u, 16>(a.smf, 8u * sb);
        in.z.mf[0] = m0[0]; in.z.mf[1] = m0[1]; in.z.mf[2] = m1[0]; in.z.mf[3] = m1[1];
    } else {
        points(a.pxx, a.pxy, in.x);
        points(a.pux, a.puy, in.u);
        in.zm = at_byte<double>(a.zm, z);
        in.zvol = at_byte<double>(a.zvol, z);
        in.zwrate = at_byte<double>(a.zwrate, z);
        in.mf = at_byte<f32x4u>(a.fsmf, 4u * sb);
    }
    in.et = at_byte<double>(a.zetot, z);
    in.bits = at_byte<unsigned char>(a.pbc, p);
}

// The tile whose first zone (ring included) is (i0, j0), loaded in `in`; its
// dt limit, dvol ratio and bad sides go into slots as block `at`'s.  Returns
// whether a CL_FLAG tile has a zone for the network: such a tile is left to the
// list kernel and stores nothing.
template <typename T, int CL>
__device__ __forceinline__ bool tile_body(const FusedArgs& a, const TileOut& o, const TileMesh& g, int i0, int j0,
                                          const TileIn<T>& in, slot_t* slots, int at, double dt, bool zre,
                                          ClCount& total) {
    __shared__ T crn[12][PN_BLOCK];
    __shared__ double pts[sizeof(T) == 8 ? 5 : 4][PN_BLOCK];
    __shared__ struct {
        double dt[PN_BLOCK / 64], dv[PN_BLOCK / 64];
        int bad[PN_BLOCK / 64];
    } lds;
    const int tid = threadIdx.x;
    const int ti = tid & (PN_TILE - 1), tj = tid / PN_TILE;
    const int i = i0 + ti, j = j0 + tj;
    const bool zin = i >= 0 && i < g.nzx && j >= 0 && j < g.nzy;
    const bool tri = zin && j < g.pie;                       // a triangle of its own pass
    const bool quad = zin && !tri;
    const bool inner = ti >= 1 && ti <= PN_TIN && tj >= 1 && tj <= PN_TIN;
    const bool own = quad && inner;
    const bool pin = i >= 0 && i <= g.nzx && j >= g.pie && j <= g.nzy;   // point (i, j) exists
    PointIn q;
    double dtz = 1.e99, zm, zvol0;
    const double et = in.et;
    int bad = 0;
    ClCount cnt;
    TileKeep<T> keep;
    keep.c = &crn[0][tid];
    q.bits = in.bits;
    if constexpr (sizeof(T) == 8) {
        zm = in.z.zm;
        zvol0 = in.z.zvol;
        q.x0 = in.z.x[0];
        q.u0 = in.z.u[0];
        if (quad) dtz = zone_pred_core<4>(a, in.z, dt, bad, keep);
    } else {
        ZoneState st;
        st.zm = zm = in.zm;
        st.zvol = zvol0 = in.zvol;
        st.zwrate = in.zwrate;
        if (zre) {
            const int z = tile_zone(g, min(max(i, 0), g.nzx - 1), min(max(j, g.pie), g.nzy - 1));
            st.zr = a.zr[z];
            st.ze = a.ze[z];
        } else {
            // the mixed corrector stored neither; these are its quotients
            st.zr = zm / zvol0;
            st.ze = et / (zm + 1.e-99);
        }
        float mf[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) mf[k] = in.mf[k];
        q.x0 = in.x[0];
        q.u0 = in.u[0];
        // the network runs across the wave, so every lane takes part
        if (CL == CL_PACKED || CL == CL_LEAN || quad)
            dtz = zone_pred_mixed_core<4, CL>(a, in.x, in.u, st, mf, dt, bad, quad, cnt, keep);
    }
    if (tri) {
        // the corners of triangle i at points (i + 1, 1) and (i, 1), where a
        // quad has its corners 2 and 3
        const int s0 = g.so + 3 * i;
#pragma unroll
        for (int k = 2; k < 4; ++k) {
            const int sl = a.pcpos[s0 + k - 1];
            if constexpr (sizeof(T) == 8) {
                keep.force(k, mk(a.cfx[sl], a.cfy[sl]));
                keep.mass(k, a.cmass[sl]);
            } else {
                keep.force(k, a.fcrn[3 * sl], a.fcrn[3 * sl + 1]);
                keep.mass(k, a.fcrn[3 * sl + 2]);
            }
        }
    }
    if (!zin) {
        // outside the mesh: corners that add nothing
#pragma unroll
        for (int k = 0; k < 12; ++k) crn[k][tid] = (T)0;
    }
    if constexpr (CL == CL_FLAG) {
        if (__syncthreads_or(quad && cnt.flag)) return true;
    } else {
        __syncthreads();
    }
    if constexpr (CL == CL_PACKED || CL == CL_LEAN) {
        if (own) {
            total.learned += cnt.learned;
            total.fallback += cnt.fallback;
        }
    }
    if (pin && ti >= 1 && tj >= 1) {
        const int p = tile_point(g, i, j);
        if (!quad) q = load_point(a, p);     // the last column and row of points
        // the point's corners in ascending side order, every read first; one
        // that does not exist is zero, and adding zero to a sum that starts
        // from zero leaves its bits
        const int from[4] = {tid - PN_TILE - 1, tid - PN_TILE, tid - 1, tid};
        constexpr int at[4] = {2, 3, 1, 0};
        T cx[4], cy[4], cm[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            cx[k] = crn[3 * at[k]][from[k]];
            cy[k] = crn[3 * at[k] + 1][from[k]];
            cm[k] = crn[3 * at[k] + 2][from[k]];
        }
        double mass = 0.;
        d2 f = mk(0., 0.);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            mass += (double)cm[k];
            f = add(f, mk((double)cx[k], (double)cy[k]));
        }
        const PointOut w = point_new<T>(a, q, mass, f, dt);
        pts[0][tid] = w.x.x;
        pts[1][tid] = w.x.y;
        pts[2][tid] = w.vs.x;
        pts[3][tid] = w.vs.y;
        if constexpr (sizeof(T) == 8) pts[4][tid] = w.xpx;
        // a point belongs to the tile whose inner zones it is the first point
        // of; the mesh's last column and row go with the tiles they end
        if ((ti <= PN_TIN || i == g.nzx) && (tj <= PN_TIN || j == g.nzy)) {
            const unsigned o8 = 8u * (unsigned)p;
            put_byte(a.oxx, o8, w.x.x);
            put_byte(a.oxy, o8, w.x.y);
            put_byte(a.oux, o8, w.u.x);
            put_byte(a.ouy, o8, w.u.y);
            if (g.pie && j == 1) store_work_point<T>(a, p, w);   // for the triangles' corrector
        }
    }
    __syncthreads();
    double dvov = 1.e-99, dtm = 1.e99;
    int badc = 0;
    if (own) {
        const int at[4] = {tid, tid + 1, tid + PN_TILE + 1, tid + PN_TILE};
        d2 x[4], vs[4], sfw[4];
        double xp[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            x[k] = mk(pts[0][at[k]], pts[1][at[k]]);
            vs[k] = mk(pts[2][at[k]], pts[3][at[k]]);
            if constexpr (sizeof(T) == 8) xp[k] = pts[4][at[k]];
            sfw[k] = mk((double)keep.sfw[k].x, (double)keep.sfw[k].y);
        }
        const unsigned z = 8u * (unsigned)tile_zone(g, i, j);
        const CorrOut r = corr_core<4, T>(et, zvol0, zm, keep.p, sfw, x, vs, xp, dt, badc, dvov);
        put_byte(o.zwrate, z, r.zwrate);
        put_byte(o.zetot, z, r.zetot);
        if constexpr (sizeof(T) == 8) {
            put_byte(o.ze, z, r.ze);
            put_byte(o.zr, z, r.zr);
        }
        put_byte(o.zvol, z, r.zvol);
        put_byte(a.zp, z, keep.p);
        dtm = (dtz < dtm) ? dtz : dtm;       // a NaN never replaces the minimum
    }
    // the tile's partials; the counts share a register (at most 784 each), and
    // their fold is skipped by a wave that has none
    int bads = (own ? bad : 0) + (badc << 16);
    dtm = wave_min(dtm);
    dvov = wave_max(dvov);
    if (__any(bads)) bads = wave_sum(bads);
    if ((tid & 63) == 0) {
        lds.dt[tid >> 6] = dtm;
        lds.dv[tid >> 6] = dvov;
        lds.bad[tid >> 6] = bads;
    }
    __syncthreads();
    if (tid == 0) {
#pragma unroll
        for (int w = 1; w < PN_BLOCK / 64; ++w) {
            dtm = (lds.dt[w] < dtm) ? lds.dt[w] : dtm;
            dvov = (lds.dv[w] > dvov) ? lds.dv[w] : dvov;
            bads += lds.bad[w];
        }
        slots_dt(slots, at, dtm, bads & 0xffff);
        slots_dv(slots, at, dvov, bads >> 16);
    }
    return false;
}

// The second cycle of a pair when the first ended the run: the tile's own
// part of the state goes back to the problem's arrays.
template <typename T>
__device__ __forceinline__ void tile_copy(const FusedArgs& a, const TileOut& o, const TileMesh& g, int i0, int j0) {
    const int ti = threadIdx.x & (PN_TILE - 1), tj = threadIdx.x / PN_TILE;
    const int i = i0 + ti, j = j0 + tj;
    if (ti < 1 || tj < 1 || i > g.nzx || j > g.nzy) return;
    if ((ti <= PN_TIN || i == g.nzx) && (tj <= PN_TIN || j == g.nzy)) {
        const int p = tile_point(g, i, j);
        a.oxx[p] = a.pxx[p];
        a.oxy[p] = a.pxy[p];
        a.oux[p] = a.pux[p];
        a.ouy[p] = a.puy[p];
    }
    if (ti <= PN_TIN && tj <= PN_TIN && i < g.nzx && j < g.nzy) {
        const int z = tile_zone(g, i, j);
        o.zetot[z] = a.zetot[z];
        o.zwrate[z] = a.zwrate[z];
        o.zvol[z] = a.zvol[z];
        if constexpr (sizeof(T) == 8) {
            o.zr[z] = a.zr[z];
            o.ze[z] = a.ze[z];
        }
    }
}

struct TileArgs {
    TileOut o;
    TileMesh g;
    int ntx, ntiles;
    int back;                    // the second cycle of a pair
    CycleStep step;              // linked cycles: the place in their chain; others: `in` is current
    int* list;                   // learned form: tiles left to the list kernel, and their number
    int* nlist;
    int* nlist_clear;            // a chain's next cycle's number
};
__device__ __forceinline__ void tile_at(const TileArgs& t, int tile, int& i0, int& j0) {
    const int tj = tile / t.ntx, ti = tile - tj * t.ntx;
    i0 = ti * PN_TIN - 1;
    j0 = t.g.pie + tj * PN_TIN - 1;
}

// The block's tile of n: each XCD takes a contiguous share (blocks after the
// n-th have other work).
__device__ __forceinline__ int xcd_tile(int n) {
    const int b = blockIdx.x, q = n >> 3, r = n & 7, x = b & 7;
    return x * q + (x < r ? x : r) + (b >> 3);
}

// One block per tile, the tiles of each XCD a contiguous share in row order
// (neighbouring tiles share their rings through its L2); a pie's origin takes
// one block more.  The flagging form needs 147 VGPRs: at four waves per SIMD it
// spills 9 and takes 142 us on Sedov 1440^2, at three 121 us.
template <typename T, int CL, bool LINK>
__global__ void __launch_bounds__(PN_BLOCK)
__attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 ? 2 : (LINK || CL == CL_FLAG ? 3 : 4))))
k_tile(FusedArgs a, TileArgs t) {
    if ((int)blockIdx.x == t.ntiles) {
        const Ctl* c = t.step.in;
        if (LINK) {
            cycle_step(t.step);
            if (CL == CL_FLAG && threadIdx.x == 0) *t.nlist_clear = 0;
            return;
        }
        const int done = c->done;
        if (done && !(t.back && c->cur)) return;
        const double dt = c->dt;
        if (done) {
            if (threadIdx.x == 0) {
                const int p = t.g.po;
                a.oxx[p] = a.pxx[p]; a.oxy[p] = a.pxy[p]; a.oux[p] = a.pux[p]; a.ouy[p] = a.puy[p];
            }
        } else {
            point_heavy<T>(a, t.g.po, dt);
        }
        return;
    }
    const int tile = xcd_tile(t.ntiles);
    int i0, j0;
    tile_at(t, tile, i0, j0);
    // the loads do not wait for the control block, which another XCD has just
    // written: Sedov 1440^2 FP64 217 -> 209 us a cycle, mixed 116 -> 108,
    // learned 158 -> 153
    TileIn<T> in;
    tile_load<T>(a, t.g, i0, j0, in);
    auto body = [&](double dt, bool zre) {
        ClCount none;
        const bool left = tile_body<T, CL>(a, t.o, t.g, i0, j0, in, t.step.put, tile, dt, zre, none);
        if (CL == CL_FLAG && left && threadIdx.x == 0) t.list[atomicAdd(t.nlist, 1)] = tile;
    };
    if constexpr (LINK) {
        const CycleNow now = cycle_now(t.step);
        if (!now.done)
            body(now.dt, now.zre != 0);
        else if (t.back && now.ended)
            tile_copy<T>(a, t.o, t.g, i0, j0);
    } else {
        // (dt and zre_valid are read here and not before the branch: held
        // across it, the mixed kernel spills 8 registers)
        const Ctl* c = t.step.in;
        if (!c->done)
            body(c->dt, c->zre_valid != 0);
        else if (t.back && c->cur)
            tile_copy<T>(a, t.o, t.g, i0, j0);
    }
}

// The triangles of a pie's linked cycle, before and after its tiles: their
// predictor, which also ends the cycle before (one block more writes the
// control block), and their corrector.  A finalize of its own had taken 4.6 us
// and a launch (Noh pie 1024^2 FP64 118.6 -> 114.7 us a
// cycle, mixed 68 -> 64; 300^2 27.4 -> 24.4 and 20.9 -> 17.9).
template <typename T>
__global__ void __launch_bounds__(PN_BLOCK) k_tri_pred(FusedArgs a, CycleStep s, int nt, int back) {
    if (blockIdx.x == gridDim.x - 1) {
        cycle_step(s, back);
        return;
    }
    const CycleNow now = cycle_now(s);
    if (now.done) return;
    const int z = blockIdx.x * PN_BLOCK + threadIdx.x;
    double m = 1.e99;
    int bad = 0;
    if (z < nt) {
        int pp[3];
        load_pp<3>(a, 3 * z, pp);
        const SideW sw = side_w(z, 0, nt, 0, 3);
        ClCount cnt;
        double v;
        if constexpr (sizeof(T) == 8)
            v = zone_pred<3>(a, z, 3 * z, sw, pp, now.dt, bad);
        else
            v = zone_pred_mixed<3, CL_EXACT>(a, z, 3 * z, sw, pp, now.dt, bad, true, cnt, now.zre != 0);
        m = (v < m) ? v : m;
    }
    m = block_min(m);
    bad = block_sum(bad);
    if (threadIdx.x == 0) slots_dt(s.put, blockIdx.x, m, bad);
}
template <typename T>
__global__ void __launch_bounds__(PN_BLOCK) k_tri_corr(FusedArgs a, CycleStep s, int nt) {
    if (s.out->done) return;
    const int z = blockIdx.x * PN_BLOCK + threadIdx.x;
    double m = 1.e-99;
    int bad = 0;
    if (z < nt) corr_zone<3, T>(a, z, 3 * z, side_w(z, 0, nt, 0, 3), s.out->dt, bad, m);
    m = block_max(m);
    bad = block_sum(bad);
    if (threadIdx.x == 0) slots_dv(s.put, blockIdx.x, m, bad);
}

// The learned form's tiles that have a zone for the network (in the ring or
// inside): the whole tile again, the network evaluated for the wave's gated
// corners packed together.  Their order in the list is not fixed, their
// results are.  Where many tiles may be listed, two waves per SIMD and the lean
// evaluation (240 VGPRs; two groups of corners in one stream spilled 31 there).
// Learned Sedov 1440^2, a cycle after 900 cycles 137 -> 134 us, after 37600 208 ->
// 187, after 50000 232 -> 203; the separate passes take 192, 202 and 204.  On the
// small rects of linked cycles, whose listed tiles all run at once, one wave and
// both groups in one stream, without spills: learned 333 x 217 26.6 -> 24.8 us a
// cycle, 420^2 36.5 -> 32.9, tube 1024 x 128 32.6 -> 29.6 (lean 31.4 -> 32.7 on
// 420^2, 29.2 -> 31.0 on the tube).
template <bool LINK>
__global__ void __launch_bounds__(PN_BLOCK) __attribute__((amdgpu_waves_per_eu(LINK ? 1 : 2)))
k_tile_list(FusedArgs a, TileArgs t) {
    const Ctl* c = LINK ? t.step.out : t.step.in;
    const int done = c->done, n = *t.nlist;
    const double dt = c->dt;
    const bool zre = c->zre_valid != 0;
    if (done || (int)blockIdx.x >= n) return;
    constexpr int NQ = (int)(sizeof(ClosurePack) / 16);
    __shared__ ClosurePack wp;
    {
        const uint4* src = reinterpret_cast<const uint4*>(a.pack);
        uint4* dst = reinterpret_cast<uint4*>(&wp);
        for (int k = threadIdx.x; k < NQ; k += PN_BLOCK) dst[k] = src[k];
    }
    __syncthreads();
    FusedArgs b = a;
    b.pack = &wp;
    ClCount cnt;
    for (int k = blockIdx.x; k < n; k += gridDim.x) {
        const int tile = t.list[k];
        int i0, j0;
        tile_at(t, tile, i0, j0);
        TileIn<float> in;
        tile_load<float>(b, t.g, i0, j0, in);
        (void)tile_body<float, LINK ? CL_PACKED : CL_LEAN>(b, t.o, t.g, i0, j0, in, t.step.put, tile, dt, zre, cnt);
    }
    const int nl = block_sum(cnt.learned);
    const int nf = block_sum(cnt.fallback);
    if (threadIdx.x == 0 && (nl | nf)) {
        atomicAdd(a.cl_stats, (unsigned long long)nl);
        atomicAdd(a.cl_stats + 1, (unsigned long long)nf);
    }
}

// K4 of a tile cycle that is not linked, from the tiles' slots, which it
// empties, and npart partials of a pie's triangles (none: 64 threads do); says
// where the state is now (cur: 1 after the first cycle of a pair) and empties
// the learned form's lists.
__global__ void __launch_bounds__(PN_FIN_BLOCK) k_finalize_tile(FusedArgs a, int npart, slot_t* slots, DtParams q, int zre,
                                                                int cur, int* nlist) {
    Ctl* c = a.ctl;
    const CtlSnap v = snap_ctl(c);
    double mn = 1.e99, mx = 1.e-99;
    int bp = 0, bc = 0;
    SlotFold f = {1.e99, 1.e-99, 0, 0};
    if (threadIdx.x < 64) f = slots_fold(slots_load(slots));
    if (npart > 0) {
        fold_partials<PN_FIN_BLOCK>(a.part_dt, a.part_bp, npart, a.part_dv, a.part_bc, npart, mn, bp, mx, bc);
        blk_fold_fin<PN_FIN_BLOCK>(mn, mx, bp, bc);
    }
    slots_reset(slots);
    if (a.zcount)
        for (int k = threadIdx.x; k < a.nzruns * PN_LSLICES; k += blockDim.x) a.zcount[k * PN_LSTRIDE] = 0u;
    if (threadIdx.x != 0) return;
    if (nlist) *nlist = 0;
    if (v.done) {
        if (!cur) c->cur = 0;                // copied back
        return;
    }
    mn = (f.mn < mn) ? f.mn : mn;
    mx = (f.mx > mx) ? f.mx : mx;
    c->zre_valid = zre;
    end_cycle(c, v, mn, mx, bp + f.bp, bc + f.bc, q);
    c->cur = cur;
}

FusedArgs make_args(pennant_problem* pb) {
    FusedArgs a;
    const Params& q = pb->prm;
    a.mapsp1 = pb->dm.mapsp1; a.pcbeg = pb->dm.pcbeg; a.pcpos = pb->pcpos;
    a.smf = pb->f("smf"); a.nump = pb->dm.nump; a.npown = own_points(pb); a.la_npred = 0;
    a.pxx = pb->f("px", 0); a.pxy = pb->f("px", 1); a.pux = pb->f("pu", 0); a.puy = pb->f("pu", 1);
    a.oxx = a.pxx; a.oxy = a.pxy; a.oux = a.pux; a.ouy = a.puy;
    a.zr = pb->f("zr"); a.ze = pb->f("ze"); a.zetot = pb->f("zetot"); a.zwrate = pb->f("zwrate");
    a.zvol = pb->f("zvol"); a.zp = pb->f("zp"); a.zm = pb->f("zm");
    a.cfx = pb->cfx; a.cfy = pb->cfy; a.cmass = pb->cmass; a.sfwx = pb->sfwx; a.sfwy = pb->sfwy;
    a.fcrn = pb->fcrn; a.fsfw = pb->fsfw; a.fsmf = pb->fsmf; a.zpn = pb->zpn;
    a.vs2 = pb->vs2; a.pxpx = pb->pxpx; a.pbc = pb->pbc;
    a.heavy = pb->heavy; a.nheavy = pb->nheavy;
    a.part_dt = pb->part_d; a.part_dv = pb->part_d + pb->npart_pred;
    a.part_bp = pb->part_i; a.part_bc = pb->part_i + pb->npart_pred;
    a.ctl = pb->ctl;
    a.gamma = q.gamma; a.ssmin = q.ssmin; a.alfa = q.alfa; a.qgamma = q.qgamma;
    a.q1 = q.q1; a.q2 = q.q2; a.cfl = q.cfl;
    a.nbcs = pb->nbcs;
    a.bcv = pb->bcv_dev;
    a.xcd = pb->tune.xcd;
    a.pack = (const ClosurePack*)pb->closure;
    a.cap_buf = pb->cap_buf;
    a.cap = pb->cap;
    a.cap_count = pb->cl_counters;
    a.cl_stats = pb->cl_counters + 1;
    a.rect_nzx = (pb->tune.rect_maps && pb->rect_nzx > 0) ? pb->rect_nzx : 0;
    a.rect_m = pb->rect_m;
    a.rect_sh = pb->rect_sh;
    a.rect_so = 0;
    a.rect_po = 0;
    a.zlist = pb->zlist;
    a.zcount = pb->zcount;
    a.nzruns = (int)pb->zruns.size() / 3;
    return a;
}

__global__ void __launch_bounds__(PN_BLOCK) k_to_float(int n, const double* src, float* dst) {
    const int i = blockIdx.x * PN_BLOCK + threadIdx.x;
    if (i < n) dst[i] = (float)src[i];
}

// zr and ze as the FP64 corrector stores them (zr = zm / zvol, ze = zetot /
// (zm + 1e-99)), where mixed cycles left them to be derived; then the flag.
__global__ void __launch_bounds__(PN_BLOCK) k_zre(FusedArgs a, int nz) {
    if (a.ctl->zre_valid) return;
    const int z = blockIdx.x * PN_BLOCK + threadIdx.x;
    if (z < nz) {
        const double zm = a.zm[z];
        a.zr[z] = zm / a.zvol[z];
        a.ze[z] = a.zetot[z] / (zm + 1.e-99);
    }
}
__global__ void __launch_bounds__(64) k_zre_done(Ctl* c, int n) {
    for (int i = threadIdx.x; i < n; i += 64) c[i].zre_valid = 1;
}

// Small fills (kernels rather than memsets, so captured graphs hold kernel
// nodes only); one block of 64 threads.
__global__ void __launch_bounds__(64) k_zero_u32(unsigned* p, int n) {
    for (int i = threadIdx.x; i < n; i += 64) p[i] = 0u;
}
__global__ void __launch_bounds__(64) k_zero_u64(unsigned long long* p, int n) {
    if ((int)threadIdx.x < n) p[threadIdx.x] = 0ull;
}

int grid_for(int needed, int cap) { return needed < 1 ? 1 : (needed < cap ? needed : cap); }

// blocks of each K1 / K3 launch for a run of nz zones with NS sides
int pred_grid(const pennant_problem* pb, int nz, int ns, int form) {
    const int per = (form == FORM_FP64 && pb->tune.k1_layout == 1) ? (PN_BLOCK / 64) * (64 / ns) : PN_BLOCK;
    return grid_for((nz + per - 1) / per, pb->tune.max_blocks);
}
int corr_grid(const pennant_problem* pb, int nz) {
    return grid_for(nblocks(nz), pb->tune.max_blocks);
}

template <int NS>
void launch_pred(const pennant_problem* pb, const FusedArgs& a, int zb, int ze, int sb, int poff,
                 int form, int run, hipStream_t s) {
    const dim3 grid(pred_grid(pb, ze - zb, NS, form));
    if (form == FORM_LEARNED)
        hipLaunchKernelGGL((k_pred_mixed<NS, true>), grid, dim3(PN_BLOCK), 0, s, a, zb, ze, sb, poff, run);
    else if (form == FORM_MIXED && a.cap_buf)
        hipLaunchKernelGGL((k_pred_cl<NS, CL_CAPTURE>), grid, dim3(PN_BLOCK), 0, s, a, zb, ze, sb, poff);
    else if (form == FORM_MIXED)
        hipLaunchKernelGGL((k_pred_mixed<NS, false>), grid, dim3(PN_BLOCK), 0, s, a, zb, ze, sb, poff, run);
    else if (pb->tune.k1_layout == 1)
        hipLaunchKernelGGL(k_pred_corner<NS>, grid, dim3(PN_BLOCK), 0, s, a, zb, ze, sb, poff);
    else
        hipLaunchKernelGGL(k_pred_zone<NS>, grid, dim3(PN_BLOCK), 0, s, a, zb, ze, sb, poff);
}
template <int NS>
void launch_corr(const pennant_problem* pb, const FusedArgs& a, int zb, int ze, int sb, int poff,
                 int form, hipStream_t s) {
    const dim3 grid(corr_grid(pb, ze - zb));
    if (form != FORM_FP64)
        hipLaunchKernelGGL((k_corr<NS, float>), grid, dim3(PN_BLOCK), 0, s, a, zb, ze, sb, poff);
    else
        hipLaunchKernelGGL((k_corr<NS, double>), grid, dim3(PN_BLOCK), 0, s, a, zb, ze, sb, poff);
}

// ---------------------------------------------------------------------------
// Batched problems: one launch per phase over the units of every problem.
// Each zone unit lies in one side-count run of one problem, so a block works
// on one problem (its dt, parameters and stop flag) at a time and writes one
// partial per unit; K4 runs one block per problem over that problem's units.

struct BatchArgs {
    FusedArgs a;                   // arena arrays; per-problem scalars come from probs
    const BUnit* units;
    int nunits;
    const PUnit* punits;
    int npunits;
    const BHeavy* heavy;
    int nheavy;
    const BProb* probs;
    Ctl* ctls;
    int rect_maps;                 // rect problems: points and corner slots computed
};

__device__ __forceinline__ void apply_prob(FusedArgs& a, const BProb& q) {
    a.gamma = q.gamma; a.ssmin = q.ssmin; a.alfa = q.alfa; a.qgamma = q.qgamma;
    a.q1 = q.q1; a.q2 = q.q2; a.cfl = q.cfl;
    a.nbcs = q.nbcs;
    a.bcv = q.bcvx;            // q.bcvy follows q.bcvx in memory
}
// A rect problem's zone kernels compute its zones' points and corner slots
// (offset to the problem's place in the arena) when `on`.
__device__ __forceinline__ void apply_rect(FusedArgs& a, const BProb& q, int on) {
    a.rect_nzx = on ? q.rect_nzx : 0;
    a.rect_m = q.rect_m;
    a.rect_sh = q.rect_sh;
    a.rect_so = q.so;
    a.rect_po = q.po;
}

// A batch unit's side work force slots: the unit's zones are a PN_BLOCK
// chunk of one side-count run, as side_w takes them.
__device__ __forceinline__ SideW unit_w(const BUnit& U, int z) {
    SideW w;
    w.u0 = U.sb;
    w.i = z - U.zb;
    w.n = U.ze - U.zb;
    return w;
}

template <int NS, int FORM, int CL>
__device__ __forceinline__ void pred_unit(const FusedArgs& a, const BUnit& U, double dt,
                                          double& dtmin, int& bad, ClCount& cnt) {
    const int z = U.zb + (int)threadIdx.x;
    const bool valid = z < U.ze;
    if constexpr (FORM == FORM_FP64) {
        if (valid) {
            const double d = zone_pred<NS>(a, z, U.sb + (z - U.zb) * NS, unit_w(U, z), dt, bad);
            dtmin = (d < dtmin) ? d : dtmin;
        }
    } else if constexpr (CL == CL_EXACT) {
        if (valid) {
            const double d = zone_pred_mixed<NS, CL_EXACT>(a, z, U.sb + (z - U.zb) * NS, unit_w(U, z), dt,
                                                           bad, true, cnt, a.ctl->zre_valid != 0);
            dtmin = (d < dtmin) ? d : dtmin;
        }
    } else {
        const int zc = valid ? z : U.ze - 1;
        const double d = zone_pred_mixed<NS, CL>(a, zc, U.sb + (zc - U.zb) * NS, unit_w(U, zc), dt, bad,
                                                 valid, cnt, a.ctl->zre_valid != 0);
        if (valid) dtmin = (d < dtmin) ? d : dtmin;
    }
}

template <int FORM, int CL>
__global__ void __launch_bounds__(PN_BLOCK)
__attribute__((amdgpu_waves_per_eu((CL == CL_LEARNED) ? 2 : ((FORM == FORM_MIXED && CL == CL_EXACT) ? 4 : 1))))
k_pred_batch(BatchArgs B) {
    // the learned form reads the network's weights from an LDS copy of the
    // block's own
    constexpr int NQ = (CL == CL_LEARNED) ? (int)(sizeof(ClosurePack) / 16) : 1;
    __shared__ uint4 wq[NQ];
    if constexpr (CL == CL_LEARNED) {
        const uint4* src = reinterpret_cast<const uint4*>(B.a.pack);
        for (int i = threadIdx.x; i < NQ; i += PN_BLOCK) wq[i] = src[i];
        __syncthreads();
    }
    // a unit's header (its work unit and its problem's done flag and dt) is
    // loaded one unit ahead, so a unit's zone loads do not wait behind it
    Units w = block_units(B.nunits, B.a.xcd);
    BUnit Un;
    int dn = 1;
    double dtn = 0.;
    if (w.u < w.end) {
        Un = B.units[w.u];
        dn = B.ctls[Un.pid].done;
        dtn = B.ctls[Un.pid].dt;
    }
    for (; w.u < w.end; w.u += w.step) {
        const BUnit U = Un;
        const int done = dn;
        const double dt = dtn;
        if (w.u + w.step < w.end) {
            Un = B.units[w.u + w.step];
            dn = B.ctls[Un.pid].done;
            dtn = B.ctls[Un.pid].dt;
        }
        if (done) continue;
        Ctl* c = B.ctls + U.pid;
        FusedArgs a = B.a;
        if constexpr (CL == CL_LEARNED) a.pack = reinterpret_cast<const ClosurePack*>(wq);
        apply_prob(a, B.probs[U.pid]);
        apply_rect(a, B.probs[U.pid], B.rect_maps);
        a.ctl = c;                 // the problem's zr/ze flag for the predictor
        double dtmin = 1.e99;
        int bad = 0;
        ClCount cnt;
        if (U.ns == 4) pred_unit<4, FORM, CL>(a, U, dt, dtmin, bad, cnt);
        else pred_unit<3, FORM, CL>(a, U, dt, dtmin, bad, cnt);
        const double m = block_min(dtmin);
        const int nb = block_sum(bad);
        if constexpr (CL == CL_LEARNED) {
            const int nl = block_sum(cnt.learned);
            const int nf = block_sum(cnt.fallback);
            if (threadIdx.x == 0 && (nl | nf)) {
                atomicAdd(a.cl_stats, (unsigned long long)nl);
                atomicAdd(a.cl_stats + 1, (unsigned long long)nf);
            }
        }
        if (threadIdx.x == 0) {
            a.part_dt[U.slot] = m;
            a.part_bp[U.slot] = nb;
        }
    }
}

template <typename T>
__global__ void __launch_bounds__(PN_BLOCK) k_point_batch(BatchArgs B) {
    if ((int)blockIdx.x < B.nheavy) {
        const BHeavy h = B.heavy[blockIdx.x];
        const Ctl* c = B.ctls + h.pid;
        if (c->done) return;
        FusedArgs a = B.a;
        apply_prob(a, B.probs[h.pid]);
        point_heavy<T>(a, h.p, c->dt);
        return;
    }
    const PUnit U = B.punits[blockIdx.x - B.nheavy];
    const Ctl* c = B.ctls + U.pid;
    if (c->done) return;
    FusedArgs a = B.a;
    apply_prob(a, B.probs[U.pid]);
    const int p = U.pb + (int)threadIdx.x;
    if (p < U.pe) point_light<T>(a, p, c->dt);
}

template <typename T>
__global__ void __launch_bounds__(PN_BLOCK) k_corr_batch(BatchArgs B) {
    // a unit's header (its work unit and its problem's done flag and dt) is
    // loaded one unit ahead, so a unit's zone loads do not wait behind it
    Units w = block_units(B.nunits, B.a.xcd);
    BUnit Un;
    int dn = 1;
    double dtn = 0.;
    if (w.u < w.end) {
        Un = B.units[w.u];
        dn = B.ctls[Un.pid].done;
        dtn = B.ctls[Un.pid].dt;
    }
    for (; w.u < w.end; w.u += w.step) {
        const BUnit U = Un;
        const int done = dn;
        const double dt = dtn;
        if (w.u + w.step < w.end) {
            Un = B.units[w.u + w.step];
            dn = B.ctls[Un.pid].done;
            dtn = B.ctls[Un.pid].dt;
        }
        if (done) continue;
        double dvov = 1.e-99;
        int bad = 0;
        const int z = U.zb + (int)threadIdx.x;
        if (z < U.ze) {
            if (U.ns == 4) {
                FusedArgs a = B.a;
                apply_rect(a, B.probs[U.pid], B.rect_maps);
                corr_zone<4, T>(a, z, U.sb + (z - U.zb) * 4, unit_w(U, z), dt, bad, dvov);
            } else {
                corr_zone<3, T>(B.a, z, U.sb + (z - U.zb) * 3, unit_w(U, z), dt, bad, dvov);
            }
        }
        const double m = block_max(dvov);
        const int nb = block_sum(bad);
        if (threadIdx.x == 0) {
            B.a.part_dv[U.slot] = m;
            B.a.part_bc[U.slot] = nb;
        }
    }
}

__global__ void __launch_bounds__(PN_FIN_BLOCK) k_finalize_batch(BatchArgs B, int zre) {
    const BProb& q = B.probs[blockIdx.x];
    const int n = q.uend - q.ubeg;
    finalize_block(B.ctls + blockIdx.x, B.a.part_dt + q.ubeg, B.a.part_bp + q.ubeg, n,
                   B.a.part_dv + q.ubeg, B.a.part_bc + q.ubeg, n, q.cflv, q.cstop, q.dtmax,
                   q.dtfac, q.tstop, zre);
}

// Tile cycle of a batch of structured problems: one block per tile of any
// problem, then one per origin.  A tile's header holds its mesh, so that its
// loads wait for one read only.  The parameters of each problem cost registers
// that the single problem's kernel does not need: in mixed precision three
// waves per SIMD (no spills) measured 51.0 us a cycle and four 55.7, on 32
// problems of 32 to 512 zones a side (0.57 M zones); the separate passes 69.4
// (FP64 80 and 98).
struct TileBatch {
    TileOut o;
    const BTile* tiles;
    int ntiles;
    const BHeavy* origins;
    int back;                    // the second cycle of a pair
};

// A cycle's place in the problems' chains (CycleStep): control blocks by
// problem, three sets of slots a problem, and which of them.
struct BatchChain {
    const Ctl* in;
    Ctl* out;
    slot_t* sets;
    int prev, put, clear;        // prev -1: the chains' first cycle
    int zre;
};
__device__ __forceinline__ slot_t* batch_slots(const BatchChain& c, int pid, int set) {
    return c.sets + ((size_t)pid * 3 + set) * PN_SLOT_SET;
}
__device__ __forceinline__ DtParams batch_dt(const BProb& q) { return {q.cflv, q.dtmax, q.dtfac, q.tstop, q.cstop}; }
__device__ __forceinline__ CycleStep batch_step(const BatchArgs& B, const BatchChain& c, int pid) {
    CycleStep s;
    s.in = c.in + pid;
    s.out = c.out + pid;
    s.prev = c.prev < 0 ? nullptr : batch_slots(c, pid, c.prev);
    s.put = batch_slots(c, pid, c.put);
    s.clear = batch_slots(c, pid, c.clear);
    s.q = batch_dt(B.probs[pid]);
    s.zre = c.zre;
    return s;
}

// Before and after the tiles.  First the end of every problem's cycle before
// (a block each) and the predictor of the pies' triangles, whose blocks end their
// problem's by themselves; then the triangles' corrector.  With a K4 of partials
// between the cycles instead, 32 problems took 53.0 us a cycle instead of 51.0
// (mixed), 16 others 75.5 instead of 73.1 (FP64).
template <typename T>
__global__ void __launch_bounds__(PN_BLOCK) k_head_batch(BatchArgs B, BatchChain c, int nprob, int back) {
    if ((int)blockIdx.x < nprob) {
        cycle_step(batch_step(B, c, blockIdx.x), back);
        return;
    }
    const BUnit U = B.units[blockIdx.x - nprob];
    const CycleStep s = batch_step(B, c, U.pid);
    const CycleNow now = cycle_now(s);
    if (now.done) return;
    FusedArgs a = B.a;
    apply_prob(a, B.probs[U.pid]);
    const int z = U.zb + (int)threadIdx.x, sb = U.sb + 3 * (int)threadIdx.x;
    double m = 1.e99;
    int bad = 0;
    if (z < U.ze) {
        ClCount cnt;
        double v;
        if constexpr (sizeof(T) == 8) {
            v = zone_pred<3>(a, z, sb, unit_w(U, z), now.dt, bad);
        } else {
            int pp[3];
            load_pp<3>(a, sb, pp);
            v = zone_pred_mixed<3, CL_EXACT>(a, z, sb, unit_w(U, z), pp, now.dt, bad, true, cnt, now.zre != 0);
        }
        m = (v < m) ? v : m;
    }
    m = block_min(m);
    bad = block_sum(bad);
    if (threadIdx.x == 0) slots_dt(s.put, blockIdx.x, m, bad);
}
template <typename T>
__global__ void __launch_bounds__(PN_BLOCK) k_tail_batch(BatchArgs B, BatchChain c) {
    const BUnit U = B.units[blockIdx.x];
    const Ctl* q = c.out + U.pid;
    if (q->done) return;
    const int z = U.zb + (int)threadIdx.x;
    double m = 1.e-99;
    int bad = 0;
    if (z < U.ze) corr_zone<3, T>(B.a, z, U.sb + 3 * (int)threadIdx.x, unit_w(U, z), q->dt, bad, m);
    m = block_max(m);
    bad = block_sum(bad);
    if (threadIdx.x == 0) slots_dv(batch_slots(c, U.pid, c.put), blockIdx.x, m, bad);
}
// The ends of the problems' chains, a block each: c.in as the last cycle left
// it, c.put the set it filled.
__global__ void __launch_bounds__(64) k_chain_end_batch(BatchArgs B, BatchChain c) {
    const int pid = blockIdx.x;
    cycle_chain_end(B.ctls + pid, c.in + pid, batch_slots(c, pid, 0), c.put, batch_dt(B.probs[pid]), c.zre);
}
__global__ void __launch_bounds__(64) k_chain_begin_batch(slot_t* sets) {
    for (int k = 0; k < 3; ++k) slots_reset(sets + ((size_t)blockIdx.x * 3 + k) * PN_SLOT_SET);
}

template <typename T>
__global__ void __launch_bounds__(PN_BLOCK) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 ? 2 : 3)))
k_tile_batch(BatchArgs B, TileBatch t, BatchChain q) {
    if ((int)blockIdx.x >= t.ntiles) {
        const BHeavy h = t.origins[blockIdx.x - t.ntiles];
        const Ctl* c = q.out + h.pid;
        FusedArgs a = B.a;
        if (c->done) {
            if (t.back && c->cur && threadIdx.x == 0) {
                a.oxx[h.p] = a.pxx[h.p]; a.oxy[h.p] = a.pxy[h.p]; a.oux[h.p] = a.pux[h.p]; a.ouy[h.p] = a.puy[h.p];
            }
            return;
        }
        apply_prob(a, B.probs[h.pid]);
        point_heavy<T>(a, h.p, c->dt);
        return;
    }
    const int tile = xcd_tile(t.ntiles);
    const BTile U = t.tiles[tile];
    const TileMesh g = {U.nzx, U.nzy, U.pie, U.zo, U.so, U.po};
    TileIn<T> in;
    tile_load<T>(B.a, g, U.i0, U.j0, in);
    const Ctl* c = q.out + U.pid;
    FusedArgs a = B.a;
    if (c->done) {
        if (t.back && c->cur) tile_copy<T>(a, t.o, g, U.i0, U.j0);
        return;
    }
    apply_prob(a, B.probs[U.pid]);
    // scalar registers: as loaded they would take 16 vector registers, and this
    // kernel has none to spare
    a.gamma = uni(a.gamma); a.ssmin = uni(a.ssmin); a.alfa = uni(a.alfa); a.qgamma = uni(a.qgamma);
    a.q1 = uni(a.q1); a.q2 = uni(a.q2); a.cfl = uni(a.cfl);
    const double dt = uni(c->dt);
    ClCount none;
    (void)tile_body<T, CL_EXACT>(a, t.o, g, U.i0, U.j0, in, batch_slots(q, U.pid, q.put), tile, dt, c->zre_valid != 0,
                                 none);
}

// k_zre over the units of every problem whose flag is clear.
__global__ void __launch_bounds__(PN_BLOCK) k_zre_batch(BatchArgs B) {
    for (Units w = block_units(B.nunits, 0); w.u < w.end; w.u += w.step) {
        const BUnit U = B.units[w.u];
        if (B.ctls[U.pid].zre_valid) continue;
        const int z = U.zb + (int)threadIdx.x;
        if (z < U.ze) {
            const double zm = B.a.zm[z];
            B.a.zr[z] = zm / B.a.zvol[z];
            B.a.ze[z] = B.a.zetot[z] / (zm + 1.e-99);
        }
    }
}

BatchArgs make_batch_args(pennant_batch* b) {
    BatchArgs B;
    FusedArgs& a = B.a;
    std::memset(&a, 0, sizeof a);
    a.mapsp1 = b->mapsp1; a.pcbeg = b->pcbeg; a.pcpos = b->pcpos; a.smf = b->smf;
    a.nump = (int)b->nump;
    a.npown = a.nump;
    a.la_npred = 0;
    a.pxx = b->pxx; a.pxy = b->pxy; a.pux = b->pux; a.puy = b->puy;
    a.oxx = a.pxx; a.oxy = a.pxy; a.oux = a.pux; a.ouy = a.puy;
    a.zr = b->zr; a.ze = b->ze; a.zetot = b->zetot; a.zwrate = b->zwrate; a.zvol = b->zvol;
    a.zp = b->zp; a.zm = b->zm;
    a.cfx = b->cfx; a.cfy = b->cfy; a.cmass = b->cmass; a.sfwx = b->sfwx; a.sfwy = b->sfwy;
    a.fcrn = b->fcrn; a.fsfw = b->fsfw;
    a.fsmf = b->fsmf;
    a.vs2 = b->vs2; a.pxpx = b->pxpx; a.pbc = b->pbc;
    a.part_dt = b->part_d; a.part_dv = b->part_d + b->nunits;
    a.part_bp = b->part_i; a.part_bc = b->part_i + b->nunits;
    a.xcd = b->tune.xcd;
    a.pack = (const ClosurePack*)b->closure;
    a.cap_buf = b->cap_buf;
    a.cap = b->cap;
    a.cap_count = b->cl_counters;
    a.cl_stats = b->cl_counters + 1;
    a.rect_nzx = 0;
    a.rect_m = 0;
    a.rect_sh = 0;
    a.rect_so = 0;
    a.rect_po = 0;
    B.rect_maps = b->tune.rect_maps;
    B.units = b->units; B.nunits = b->nunits;
    B.punits = b->punits; B.npunits = b->npunits;
    B.heavy = b->heavy; B.nheavy = b->nheavy;
    B.probs = b->probs; B.ctls = b->ctls;
    return B;
}

}  // namespace

namespace pn {

// Builds the zone runs, the per-point BC bits, the heavy-point list and the
// fused-path buffers (partials sized for the largest grids the tuning
// allows).
int refresh_side_fracs(pennant_problem* pb) {
    const int64_t S = pb->hm.nums;
    if (S > 0)
        hipLaunchKernelGGL(k_to_float, dim3(nblocks(S)), dim3(PN_BLOCK), 0, pb->stream, (int)S,
                           (const double*)pb->f("smf"), const_cast<float*>(pb->fsmf));
    pb->smf_stale = false;
    return (int)hipGetLastError();
}

// Whether the mesh is a structured rect in the generator's numbering, so
// that the fused kernels may compute its zones' points and corner slots
// (rect_zone) instead of loading mapsp1 and pcpos: one run of quads, sides
// 4z .. 4z + 3, and every side's point and slot equal to the formula's
// (checked here, with the same integer arithmetic as the device's).
void rect_detect(pennant_problem* pb, const std::vector<int>& pcpos) {
    const HostMesh& h = pb->hm;
    pb->rect_nzx = 0;
    const long nzx = pb->prm.nzx;
    if (pb->prm.meshtype != "rect" || own_points(pb) != h.nump || pb->zruns.size() != 3 ||
        pb->zruns[2] != 4 || nzx < 1 || (long)h.numz % nzx != 0 || (int64_t)h.nums != 4 * (int64_t)h.numz)
        return;
    int sh = 0;
    while ((1L << sh) < nzx) ++sh;
    const unsigned long long m = ((1ull << (32 + sh)) / (unsigned long long)nzx) + 1ull;
    const long npx = nzx + 1;
    for (int z = 0; z < h.numz; ++z) {
        const long zy = (long)(((unsigned long long)(unsigned)z * m) >> (32 + sh));
        const long zx = z - zy * nzx;
        if (zy != z / nzx || h.zsbeg[z] != 4 * z) return;
        const long p0 = z + zy;
        const int left = zx >= 1, below = zy >= 1;
        const long pts[4] = {p0, p0 + 1, p0 + 1 + npx, p0 + npx};
        const int rank[4] = {(left & below) + below + left, below + (below & (zx + 1 < nzx)), 0, left};
        for (int k = 0; k < 4; ++k)
            if (h.mapsp1[4 * z + k] != pts[k] || pcpos[4 * z + k] != (long)rank[k] * h.nump + pts[k]) return;
    }
    pb->rect_nzx = (int)nzx;
    pb->rect_m = m;
    pb->rect_sh = 32 + sh;
}

int fused_setup(pennant_problem* pb) {
    const HostMesh& h = pb->hm;
    pb->zruns.clear();
    for (int z = 0; z < h.numz;) {
        int e = z + 1;
        while (e < h.numz && h.znump[e] == h.znump[z]) ++e;
        pb->zruns.push_back(z);
        pb->zruns.push_back(e);
        pb->zruns.push_back(h.znump[z]);
        z = e;
    }
    if (pb->bcs.size() > 8) return PENNANT_EINVAL;
    pb->nbcs = (int)pb->bcs.size();
    std::vector<unsigned char> bits((size_t)h.nump, 0);
    const double eps = 1.e-12;
    int bi = 0;
    auto mark = [&](double b, bool xplane) {
        for (int p = 0; p < h.nump; ++p) {
            const double c = xplane ? h.px[p] : h.py[p];
            if (std::fabs(c - b) < eps) bits[p] |= (unsigned char)(1u << bi);
        }
        pb->bcvx[bi] = xplane ? 1. : 0.;
        pb->bcvy[bi] = xplane ? 0. : 1.;
        ++bi;
    };
    for (double b : pb->prm.bcx) mark(b, true);
    for (double b : pb->prm.bcy) mark(b, false);
    std::vector<int> heavy;
    for (int p = 0; p < own_points(pb); ++p)
        if (h.pcbeg[p + 1] - h.pcbeg[p] > PN_HEAVY) heavy.push_back(p);
    auto al = [&](size_t n, size_t sz) -> void* { return problem_alloc(pb, n * sz); };
    const size_t S = h.nums, P = h.nump;
    // (a piece's master points list other pieces' corners too: more than its sides)
    const int64_t K = std::max((int64_t)S, (int64_t)h.pcside.size());
    if (!corner_slots_fit((int64_t)P, K)) return PENNANT_EINVAL;
    const size_t NC = (size_t)corner_slots((int64_t)P, K);
    pb->cfx = (double*)al(NC, 8); pb->cfy = (double*)al(NC, 8); pb->cmass = (double*)al(NC, 8);
    pb->sfwx = (double*)al(S, 8); pb->sfwy = (double*)al(S, 8);
    pb->vs2 = (double*)al(2 * P, 8); pb->pxpx = (double*)al(P, 8);
    pb->pbc = (unsigned char*)al(P, 1);
    pb->heavy = (int*)al(heavy.size(), 4);
    pb->nheavy = (int)heavy.size();
    // mixed-precision intermediates and the FP32 copy of smf
    pb->fcrn = (float*)al(3 * NC, 4);
    pb->fsfw = (float*)al(2 * S, 4);
    float* fsmf = (float*)al(S, 4);
    pb->fsmf = fsmf;
    if (!pb->fcrn || !pb->fsfw || !fsmf)
        return (int)hipErrorOutOfMemory;
    if (refresh_side_fracs(pb)) return (int)hipErrorUnknown;
    // K1 writes each corner's force and mass straight into its corner slot,
    // where K2 reads it.  (A piece's master point also lists the corners of
    // other pieces, pcside -1: their records arrive by the corner exchange.)
    std::vector<int> pcpos((size_t)h.nums);
    for (int p = 0; p < h.nump; ++p)
        for (int k = h.pcbeg[p]; k < h.pcbeg[p + 1]; ++k)
            if (h.pcside[k] >= 0) pcpos[h.pcside[k]] = (int)corner_slot((int64_t)P, p, k - h.pcbeg[p], k);
    pb->pcpos = (int*)al(S, 4);
    if (pb->pcpos &&
        hipMemcpy(pb->pcpos, pcpos.data(), S * 4, hipMemcpyHostToDevice) != hipSuccess)
        return (int)hipErrorUnknown;
    rect_detect(pb, pcpos);
    // partial slots: one per block of every K1 (resp. K3) launch of a cycle,
    // at the largest grid any tuning allows
    const int nruns = (int)pb->zruns.size() / 3;
    pb->npart_pred = nruns * PN_MAX_GRID;
    pb->npart_corr = nruns * PN_MAX_GRID;
    pb->cl_counters = (unsigned long long*)al(5, 8);
    pb->zpn = (double*)al((size_t)h.numz, 8);
    pb->zlist = (int*)al((size_t)h.numz, 4);
    pb->zcount = (unsigned*)al(pb->zruns.size() / 3 * PN_LSLICES * PN_LSTRIDE + 1, 4);
    if (!pb->cl_counters || !pb->zlist || !pb->zcount || !pb->zpn) return (int)hipErrorOutOfMemory;
    pb->part_d = (double*)al((size_t)pb->npart_pred + pb->npart_corr, 8);
    pb->part_i = (int*)al((size_t)pb->npart_pred + pb->npart_corr, 4);
    if (!pb->cfx || !pb->cfy || !pb->cmass || !pb->sfwx || !pb->sfwy || !pb->vs2 ||
        !pb->pxpx || !pb->pbc || !pb->heavy || !pb->pcpos || !pb->part_d || !pb->part_i)
        return (int)hipErrorOutOfMemory;
    if (!heavy.empty() &&
        hipMemcpy(pb->heavy, heavy.data(), heavy.size() * 4, hipMemcpyHostToDevice) != hipSuccess)
        return (int)hipErrorUnknown;
    double bcv[16];
    for (int i = 0; i < 8; ++i) { bcv[i] = pb->bcvx[i]; bcv[8 + i] = pb->bcvy[i]; }
    pb->bcv_dev = (double*)al(16, 8);
    if (!pb->bcv_dev || hipMemcpy(pb->bcv_dev, bcv, sizeof bcv, hipMemcpyHostToDevice) != hipSuccess)
        return (int)hipErrorOutOfMemory;
    if (const int rc = tile_setup(pb)) return rc;
    return (int)hipMemcpy(pb->pbc, bits.data(), bits.size(), hipMemcpyHostToDevice);
}

namespace {

// The learned pass over the zones a flagging predictor listed; with
// `pending` its counts go to the pending counters.
int launch_learned_pass(const pennant_problem* pb, const FusedArgs& a, bool pending, hipStream_t s) {
    FusedArgs b = a;
    if (pending) b.cl_stats = pb->cl_counters + 3;
    const HostMesh& h = pb->hm;
    for (size_t r = 0; r < pb->zruns.size(); r += 3) {
        const int zb = pb->zruns[r], ze = pb->zruns[r + 1], ns = pb->zruns[r + 2];
        const int sb = h.zsbeg[zb];
        // the learned pass holds 2 blocks per CU (registers): 512 blocks
        // fill the chip without dispatching blocks that find no work
        const int g = pred_grid(pb, ze - zb, ns, FORM_LEARNED);
        const dim3 grid(g < 512 ? g : 512), blk(PN_BLOCK);
        const int run = (int)(r / 3);
        switch (ns) {
            case 3: hipLaunchKernelGGL(k_pred_list<3>, grid, blk, 0, s, b, zb, ze, sb, run); break;
            case 4: hipLaunchKernelGGL(k_pred_list<4>, grid, blk, 0, s, b, zb, ze, sb, run); break;
            case 5: hipLaunchKernelGGL(k_pred_list<5>, grid, blk, 0, s, b, zb, ze, sb, run); break;
            case 6: hipLaunchKernelGGL(k_pred_list<6>, grid, blk, 0, s, b, zb, ze, sb, run); break;
            case 7: hipLaunchKernelGGL(k_pred_list<7>, grid, blk, 0, s, b, zb, ze, sb, run); break;
            case 8: hipLaunchKernelGGL(k_pred_list<8>, grid, blk, 0, s, b, zb, ze, sb, run); break;
            default: return PENNANT_EINVAL;
        }
    }
    return 0;
}

}  // namespace

int launch_cycle_points(pennant_problem* pb, Ctl* ctl) {
    FusedArgs a = make_args(pb);
    a.ctl = ctl;
    const TaskPoints t = {pb->vv("px0"), pb->vv("pu0"), pb->vv("pxp"), pb->vv("pf"), pb->vv("pap"), pb->f("pmaswt")};
    const int nb = pb->nheavy + nblocks(own_points(pb));
    if (nb > 0) hipLaunchKernelGGL(k_cycle_points, dim3(nb), dim3(PN_BLOCK), 0, pb->stream, a, t);
    return (int)hipGetLastError();
}

int fused_cycle(pennant_problem* pb, hipEvent_t* ev, int form) {
    if (form == FORM_LEARNED && !pb->closure) return PENNANT_EINVAL;
    const bool mixed = (form != FORM_FP64);
    const FusedArgs a = make_args(pb);
    const Params& q = pb->prm;
    hipStream_t s = pb->stream;
    const HostMesh& h = pb->hm;
    if (ev) (void)hipEventRecord(ev[0], s);
    int poff = 0;
    for (size_t r = 0; r < pb->zruns.size(); r += 3) {
        const int zb = pb->zruns[r], ze = pb->zruns[r + 1], ns = pb->zruns[r + 2];
        const int sb = h.zsbeg[zb];
        switch (ns) {
            case 3: launch_pred<3>(pb, a, zb, ze, sb, poff, form, (int)(r / 3), s); break;
            case 4: launch_pred<4>(pb, a, zb, ze, sb, poff, form, (int)(r / 3), s); break;
            case 5: launch_pred<5>(pb, a, zb, ze, sb, poff, form, (int)(r / 3), s); break;
            case 6: launch_pred<6>(pb, a, zb, ze, sb, poff, form, (int)(r / 3), s); break;
            case 7: launch_pred<7>(pb, a, zb, ze, sb, poff, form, (int)(r / 3), s); break;
            case 8: launch_pred<8>(pb, a, zb, ze, sb, poff, form, (int)(r / 3), s); break;
            default: return PENNANT_EINVAL;
        }
        poff += pred_grid(pb, ze - zb, ns, form);
    }
    const int npred = poff;
    if (ev) (void)hipEventRecord(ev[1], s);
    if (form == FORM_LEARNED) {
        const int rc = launch_learned_pass(pb, a, false, s);
        if (rc) return rc;
    }
    if (ev) (void)hipEventRecord(ev[2], s);
    const dim3 pgrid(pb->nheavy + nblocks(own_points(pb)));
    if (mixed)
        hipLaunchKernelGGL(k_point<float>, pgrid, dim3(PN_BLOCK), 0, s, a);
    else
        hipLaunchKernelGGL(k_point<double>, pgrid, dim3(PN_BLOCK), 0, s, a);
    if (ev) (void)hipEventRecord(ev[3], s);
    poff = 0;
    for (size_t r = 0; r < pb->zruns.size(); r += 3) {
        const int zb = pb->zruns[r], ze = pb->zruns[r + 1], ns = pb->zruns[r + 2];
        const int sb = h.zsbeg[zb];
        switch (ns) {
            case 3: launch_corr<3>(pb, a, zb, ze, sb, poff, form, s); break;
            case 4: launch_corr<4>(pb, a, zb, ze, sb, poff, form, s); break;
            case 5: launch_corr<5>(pb, a, zb, ze, sb, poff, form, s); break;
            case 6: launch_corr<6>(pb, a, zb, ze, sb, poff, form, s); break;
            case 7: launch_corr<7>(pb, a, zb, ze, sb, poff, form, s); break;
            case 8: launch_corr<8>(pb, a, zb, ze, sb, poff, form, s); break;
            default: return PENNANT_EINVAL;
        }
        poff += corr_grid(pb, ze - zb);
    }
    const int ncorr = poff;
    if (ev) (void)hipEventRecord(ev[4], s);
    hipLaunchKernelGGL(k_finalize, dim3(1), dim3(PN_FIN_BLOCK), 0, s, a, npred, ncorr, q.cflv,
                       q.cstop, q.dtmax, q.dtfac, q.tstop, mixed ? 0 : 1);
    if (ev) (void)hipEventRecord(ev[5], s);
    return (int)hipGetLastError();
}

namespace {

// Predictor launches of the pipelined cycle (the prologue's, or with REDO
// the redo), writing zp to zpn; returns the number of partials.
template <bool REDO>
int launch_lookahead_pred(const pennant_problem* pb, const FusedArgs& a, int form, hipStream_t s) {
    FusedArgs b = a;
    b.zp = pb->zpn;
    const HostMesh& h = pb->hm;
    int poff = 0;
    for (size_t r = 0; r < pb->zruns.size(); r += 3) {
        const int zb = pb->zruns[r], ze = pb->zruns[r + 1], ns = pb->zruns[r + 2];
        const int sb = h.zsbeg[zb];
        const dim3 grid(pred_grid(pb, ze - zb, ns, form)), blk(PN_BLOCK);
        const int run = (int)(r / 3);
        const bool fl = (form == FORM_LEARNED);
#define PN_LA(NS)                                                                                  \
    if (fl) hipLaunchKernelGGL((k_pred_mixed<NS, true, REDO>), grid, blk, 0, s, b, zb, ze, sb, poff, run); \
    else hipLaunchKernelGGL((k_pred_mixed<NS, false, REDO>), grid, blk, 0, s, b, zb, ze, sb, poff, run);
        switch (ns) {
            case 3: PN_LA(3) break;
            case 4: PN_LA(4) break;
            case 5: PN_LA(5) break;
            case 6: PN_LA(6) break;
            case 7: PN_LA(7) break;
            case 8: PN_LA(8) break;
            default: return -1;
        }
#undef PN_LA
        poff += grid.x;
    }
    return poff;
}


}  // namespace

int fused_prologue(pennant_problem* pb, int form) {
    if (form == FORM_FP64 || (form == FORM_LEARNED && !pb->closure)) return PENNANT_EINVAL;
    const FusedArgs a = make_args(pb);
    hipStream_t s = pb->stream;
    const int nz = (int)pb->zruns.size() / 3;
    hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(64), 0, s, pb->zcount, nz * PN_LSLICES * PN_LSTRIDE);
    hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(64), 0, s, pb->cl_counters + 3, 2);
    const int npred = launch_lookahead_pred<false>(pb, a, form, s);
    if (npred < 0) return PENNANT_EINVAL;
    hipLaunchKernelGGL(k_finalize_la<false>, dim3(1), dim3(PN_FIN_BLOCK), 0, s, a, npred);
    if (form == FORM_LEARNED) {
        const int rc = launch_learned_pass(pb, a, true, s);
        if (rc) return rc;
    }
    return (int)hipGetLastError();
}

int fused_cycle_pipe(pennant_problem* pb, hipEvent_t* ev, int form) {
    if (form == FORM_FP64 || (form == FORM_LEARNED && !pb->closure)) return PENNANT_EINVAL;
    const FusedArgs a = make_args(pb);
    const DtParams q = dt_params(pb);
    hipStream_t s = pb->stream;
    const HostMesh& h = pb->hm;
    const bool fl = (form == FORM_LEARNED);
    // partials of one predictor pass (the zone pass's, or its redo's)
    int nparts = 0;
    for (size_t r = 0; r < pb->zruns.size(); r += 3)
        nparts += pred_grid(pb, pb->zruns[r + 1] - pb->zruns[r], pb->zruns[r + 2], form);
    if (ev) (void)hipEventRecord(ev[0], s);
    {
        FusedArgs a2 = a;
        a2.la_npred = nparts;   // and one block more, for the look-ahead fold
        hipLaunchKernelGGL(k_point<float>, dim3(pb->nheavy + nblocks(own_points(pb)) + 1), dim3(PN_BLOCK), 0, s,
                           a2);
    }
    if (ev) (void)hipEventRecord(ev[1], s);
    int poff = 0;
    for (size_t r = 0; r < pb->zruns.size(); r += 3) {
        const int zb = pb->zruns[r], ze = pb->zruns[r + 1], ns = pb->zruns[r + 2];
        const int sb = h.zsbeg[zb];
        const dim3 grid(pred_grid(pb, ze - zb, ns, form)), blk(PN_BLOCK);
        const int run = (int)(r / 3);
#define PN_ZP(NS)                                                                                  \
    if (fl) hipLaunchKernelGGL((k_zone_pipe<NS, true>), grid, blk, 0, s, a, zb, ze, sb, poff, run, q); \
    else hipLaunchKernelGGL((k_zone_pipe<NS, false>), grid, blk, 0, s, a, zb, ze, sb, poff, run, q);
        switch (ns) {
            case 3: PN_ZP(3) break;
            case 4: PN_ZP(4) break;
            case 5: PN_ZP(5) break;
            case 6: PN_ZP(6) break;
            case 7: PN_ZP(7) break;
            case 8: PN_ZP(8) break;
            default: return PENNANT_EINVAL;
        }
#undef PN_ZP
        poff += grid.x;
    }
    if (ev) (void)hipEventRecord(ev[2], s);
    hipLaunchKernelGGL(k_finalize_pipe, dim3(1), dim3(PN_FIN_BLOCK), 0, s, a, poff, poff, q);
    // the redo, when the look-ahead dt was not the cycle's dt; its partials
    // are folded by the next cycle's K2 (every launch sequence that does not
    // continue with this form's cycles starts again from the prologue)
    const int npred = launch_lookahead_pred<true>(pb, a, form, s);
    if (npred != poff || npred != nparts) return PENNANT_EINVAL;
    if (ev) (void)hipEventRecord(ev[3], s);
    if (fl) {
        const int rc = launch_learned_pass(pb, a, true, s);
        if (rc) return rc;
    }
    if (ev) (void)hipEventRecord(ev[4], s);
    return (int)hipGetLastError();
}

namespace {

// The tile cycle's arguments, with the points and zones read from the state
// that cycle `second` of a pair starts from.
TileArgs tile_args(const pennant_problem* pb, int second, FusedArgs& a) {
    TileArgs t;
    const TileState& q = pb->tile;
    double* const own[9] = {a.pxx, a.pxy, a.pux, a.puy, a.zr, a.ze, a.zetot, a.zwrate, a.zvol};
    double* const* src = second ? q.alt : own;
    double* const* dst = second ? own : q.alt;
    a.pxx = src[0]; a.pxy = src[1]; a.pux = src[2]; a.puy = src[3];
    a.zr = src[4]; a.ze = src[5]; a.zetot = src[6]; a.zwrate = src[7]; a.zvol = src[8];
    a.oxx = dst[0]; a.oxy = dst[1]; a.oux = dst[2]; a.ouy = dst[3];
    t.o = {dst[4], dst[5], dst[6], dst[7], dst[8]};
    t.g = {q.nzx, q.nzy, q.pie, 0, 0, 0};
    t.ntx = (q.nzx + PN_TIN - 1) / PN_TIN;
    t.ntiles = t.ntx * ((q.nzy - q.pie + PN_TIN - 1) / PN_TIN);
    t.back = second;
    t.list = q.list;
    a.part_dt = q.part_d;
    a.part_dv = q.part_d + q.npart;
    a.part_bp = q.part_i;
    a.part_bc = q.part_i + q.npart;
    return t;
}

}  // namespace

template <bool LINK>
static void launch_tiles(const FusedArgs& a, const TileArgs& t, int blocks, int form, hipStream_t s) {
    const dim3 grid(blocks), blk(PN_BLOCK);
    if (form == FORM_FP64)
        hipLaunchKernelGGL((k_tile<double, CL_EXACT, LINK>), grid, blk, 0, s, a, t);
    else if (form == FORM_MIXED)
        hipLaunchKernelGGL((k_tile<float, CL_EXACT, LINK>), grid, blk, 0, s, a, t);
    else {
        hipLaunchKernelGGL((k_tile<float, CL_FLAG, LINK>), grid, blk, 0, s, a, t);
        hipLaunchKernelGGL(k_tile_list<LINK>, dim3(t.ntiles < 512 ? t.ntiles : 512), blk, 0, s, a, t);
    }
}

// Cycle k of n.  Linked cycles are a chain: each ends the cycle before it by
// itself (a rect's tile kernel, a pie's triangles' predictor), one block more
// writes the control block, and the last is ended when the run of n is.
static int tile_cycle(pennant_problem* pb, int form, int k, bool linked) {
    const int second = k & 1, zre = form == FORM_FP64 ? 1 : 0;
    FusedArgs a = make_args(pb);
    FusedArgs tri = a;                       // the triangles' own state stays in the problem's arrays
    TileArgs t = tile_args(pb, second, a);
    hipStream_t s = pb->stream;
    t.step = chain_step(pb, pb->tile.chain, linked ? k : 0, zre);
    t.nlist = pb->tile.nlist + (linked ? k & 1 : 0);
    t.nlist_clear = pb->tile.nlist + ((k + 1) & 1);
    const int nt = t.g.pie ? t.g.nzx : 0;    // triangles
    if (linked && !nt) {
        launch_tiles<true>(a, t, t.ntiles + 1, form, s);
        return (int)hipGetLastError();
    }
    tri.part_dt = a.part_dt; tri.part_dv = a.part_dv; tri.part_bp = a.part_bp; tri.part_bc = a.part_bc;
    tri.pxx = a.pxx; tri.pxy = a.pxy; tri.pux = a.pux; tri.puy = a.puy;
    if (linked) {
        const CycleStep step = t.step;
        const dim3 blk(PN_BLOCK), g(nblocks(nt)), g1(nblocks(nt) + 1);
        if (form == FORM_FP64)
            hipLaunchKernelGGL(k_tri_pred<double>, g1, blk, 0, s, tri, step, nt, second);
        else
            hipLaunchKernelGGL(k_tri_pred<float>, g1, blk, 0, s, tri, step, nt, second);
        t.step.in = step.out;                // as the triangles' kernel left it
        launch_tiles<false>(a, t, t.ntiles + 1, form, s);
        tri.pxx = a.oxx; tri.pxy = a.oxy; tri.pux = a.oux; tri.puy = a.ouy;
        if (form == FORM_FP64)
            hipLaunchKernelGGL(k_tri_corr<double>, g, blk, 0, s, tri, step, nt);
        else
            hipLaunchKernelGGL(k_tri_corr<float>, g, blk, 0, s, tri, step, nt);
        return (int)hipGetLastError();
    }
    int npart = 0;
    if (nt) {                                // (the learned form's)
        launch_pred<3>(pb, tri, 0, nt, 0, 0, form, 0, s);
        // one partial index per block of both halves
        npart = pred_grid(pb, nt, 3, form);
        if (npart != corr_grid(pb, nt)) return PENNANT_EINVAL;
        hipLaunchKernelGGL(k_pred_list<3>, dim3(npart < 512 ? npart : 512), dim3(PN_BLOCK), 0, s, tri, 0, nt, 0, 0);
    }
    launch_tiles<false>(a, t, t.ntiles + (nt ? 1 : 0), form, s);
    if (nt) {
        tri.pxx = a.oxx; tri.pxy = a.oxy; tri.pux = a.oux; tri.puy = a.ouy;
        launch_corr<3>(pb, tri, 0, nt, 0, 0, form, s);
    }
    hipLaunchKernelGGL(k_finalize_tile, dim3(1), dim3(npart ? PN_FIN_BLOCK : 64), 0, s, a, npart, t.step.put, t.step.q, zre,
                       second ? 0 : 1, form == FORM_LEARNED ? t.nlist : nullptr);
    return (int)hipGetLastError();
}

int tile_cycles(pennant_problem* pb, int form, int n) {
    const TileState& q = pb->tile;
    if (!q.nzx || (n & 1) || (form == FORM_LEARNED && !pb->closure)) return PENNANT_EINVAL;
    const int64_t tiles = (int64_t)((q.nzx + PN_TIN - 1) / PN_TIN) * ((q.nzy - q.pie + PN_TIN - 1) / PN_TIN);
    // a pie's few blocks of triangles always pay for the fold; the learned
    // form's triangles have a list pass of their own
    const bool linked = n > 0 && (q.pie ? form != FORM_LEARNED : tiles <= PN_LINK_TILES);
    // an error that another call has left is not to end a pair halfway
    if (const int rc = (int)hipGetLastError()) return rc;
    for (int k = 0; k < n; ++k)
        if (const int rc = tile_cycle(pb, form, k, linked)) return rc;
    return linked ? chain_end(pb, q.chain, n, form == FORM_FP64 ? 1 : 0) : 0;
}

// Whether the mesh is one the tile cycle takes: a rect (rect_detect has
// checked every side) or a pie of at least two rows in the generator's
// numbering, every side's point checked here against the formula the kernel
// uses.  Allocates the second set of state arrays, the partials and the
// learned form's list; where there is no memory for them (72 bytes a zone) the
// problem runs as separate passes.
int tile_setup(pennant_problem* pb) {
    const HostMesh& h = pb->hm;
    TileState& q = pb->tile;
    q.nzx = 0;
    const int64_t nzx = pb->prm.nzx;
    const bool pie = pb->prm.meshtype == "pie" && own_points(pb) == h.nump;
    if (!pie && pb->rect_nzx == 0) return 0;
    const int64_t nzy = nzx > 0 ? h.numz / nzx : 0;
    if (pie) {
        if (nzx < 1 || nzy < 2 || nzx * nzy != h.numz || h.nump != (nzx + 1) * nzy + 1 ||
            (int64_t)h.nums != 3 * nzx + 4 * nzx * (nzy - 1))
            return 0;
        for (int64_t j = 0; j < nzy; ++j)
            for (int64_t i = 0; i < nzx; ++i) {
                const int64_t z = j * nzx + i, sb = j ? 4 * z - nzx : 3 * i;
                const int64_t p = j * (nzx + 1) + i - nzx;        // the quad's first point
                const int64_t quad[4] = {p, p + 1, p + nzx + 2, p + nzx + 1}, tri[3] = {0, i + 2, i + 1};
                if (h.zsbeg[z] != sb || h.znump[z] != (j ? 4 : 3)) return 0;
                for (int k = 0; k < (j ? 4 : 3); ++k)
                    if (h.mapsp1[sb + k] != (j ? quad[k] : tri[k])) return 0;
            }
    }
    const int64_t tiles = ((nzx + PN_TIN - 1) / PN_TIN) * ((nzy - pie + PN_TIN - 1) / PN_TIN);
    const int64_t P = h.nump, Z = h.numz;
    q.npart = pie ? PN_MAX_GRID : 0;         // the triangles'
    const size_t bytes = PN_CHAIN_BYTES + (size_t)(4 * P + 5 * Z + 2 * (int64_t)q.npart) * 8 +
                         (size_t)(2 * (int64_t)q.npart + tiles + 2) * 4;
    char* m = (char*)problem_alloc(pb, bytes);
    if (!m) {
        (void)hipGetLastError();
        return 0;
    }
    q.chain = m;
    double* d = (double*)(m + PN_CHAIN_BYTES);
    for (int k = 0; k < 9; ++k) {
        q.alt[k] = d;
        d += k < 4 ? P : Z;
    }
    q.part_d = d;
    q.part_i = (int*)(d + 2 * (int64_t)q.npart);
    q.nlist = q.part_i + 2 * (int64_t)q.npart;
    q.list = q.nlist + 2;
    hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(64), 0, pb->stream, (unsigned*)q.nlist, 2);
    hipLaunchKernelGGL(k_chain_begin, dim3(1), dim3(64), 0, pb->stream, chain_sets(q.chain));
    q.nzx = (int)nzx;
    q.nzy = (int)nzy;
    q.pie = pie ? 1 : 0;
    return (int)hipGetLastError();
}

int reset_zone_lists(pennant_problem* pb) {
    const int nz = (int)pb->zruns.size() / 3;
    if (pb->zcount && nz > 0)
        hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(64), 0, pb->stream, pb->zcount, nz * PN_LSLICES * PN_LSTRIDE);
    return (int)hipGetLastError();
}

int materialize_zre(pennant_problem* pb) {
    if (!pb->zre_stale) return 0;
    const FusedArgs a = make_args(pb);
    const int nz = pb->hm.numz;
    hipLaunchKernelGGL(k_zre, dim3(nblocks(nz)), dim3(PN_BLOCK), 0, pb->stream, a, nz);
    hipLaunchKernelGGL(k_zre_done, dim3(1), dim3(64), 0, pb->stream, pb->ctl, 1);
    pb->zre_stale = false;
    return (int)hipGetLastError();
}

int batch_materialize_zre(pennant_batch* b) {
    if (!b->zre_stale) return 0;
    const BatchArgs B = make_batch_args(b);
    hipLaunchKernelGGL(k_zre_batch, dim3(grid_for(b->nunits, PN_MAX_GRID)), dim3(PN_BLOCK), 0,
                       b->stream, B);
    hipLaunchKernelGGL(k_zre_done, dim3(1), dim3(64), 0, b->stream, b->ctls, b->nprob);
    b->zre_stale = false;
    return (int)hipGetLastError();
}

int launch_to_float(const double* src, float* dst, int64_t n, hipStream_t s) {
    if (n > 0)
        hipLaunchKernelGGL(k_to_float, dim3(nblocks(n)), dim3(PN_BLOCK), 0, s, (int)n, src, dst);
    return (int)hipGetLastError();
}

int batch_cycle(pennant_batch* b, int form) {
    if (form == FORM_LEARNED && !b->closure) return PENNANT_EINVAL;
    const BatchArgs B = make_batch_args(b);
    hipStream_t s = b->stream;
    const dim3 zg(grid_for(b->nunits, b->tune.max_blocks)), blk(PN_BLOCK);
    if (form == FORM_FP64)
        hipLaunchKernelGGL((k_pred_batch<FORM_FP64, CL_EXACT>), zg, blk, 0, s, B);
    else if (form == FORM_LEARNED)
        hipLaunchKernelGGL((k_pred_batch<FORM_MIXED, CL_LEARNED>), zg, blk, 0, s, B);
    else if (b->cap_buf)
        hipLaunchKernelGGL((k_pred_batch<FORM_MIXED, CL_CAPTURE>), zg, blk, 0, s, B);
    else
        hipLaunchKernelGGL((k_pred_batch<FORM_MIXED, CL_EXACT>), zg, blk, 0, s, B);
    const dim3 pg(b->nheavy + b->npunits);
    if (form == FORM_FP64) {
        hipLaunchKernelGGL(k_point_batch<double>, pg, blk, 0, s, B);
        hipLaunchKernelGGL(k_corr_batch<double>, zg, blk, 0, s, B);
    } else {
        hipLaunchKernelGGL(k_point_batch<float>, pg, blk, 0, s, B);
        hipLaunchKernelGGL(k_corr_batch<float>, zg, blk, 0, s, B);
    }
    hipLaunchKernelGGL(k_finalize_batch, dim3(b->nprob), dim3(PN_FIN_BLOCK), 0, s, B,
                       form == FORM_FP64 ? 1 : 0);
    return (int)hipGetLastError();
}

int batch_tile_setup(pennant_batch* b, const std::vector<TileState>& meshes) {
    b->ntiles = 0;
    for (const TileState& m : meshes)
        if (m.nzx == 0) return 0;            // some problem needs the separate passes
    std::vector<BTile> tiles;
    std::vector<BUnit> tri;
    std::vector<BHeavy> origins;
    for (size_t k = 0; k < meshes.size(); ++k) {
        const TileState& m = meshes[k];
        const int zo = (int)b->zoff[k], so = (int)b->soff[k], po = (int)b->poff[k], pid = (int)k;
        if (m.pie) {
            for (int z = 0; z < m.nzx; z += PN_BLOCK) {
                BUnit U = {};
                U.zb = zo + z;
                U.ze = zo + (z + PN_BLOCK < m.nzx ? z + PN_BLOCK : m.nzx);
                U.sb = so + 3 * z;
                U.ns = 3;
                U.pid = pid;
                tri.push_back(U);
            }
            origins.push_back({po, pid});
        }
        for (int j = 0; j < m.nzy - m.pie; j += PN_TIN)
            for (int i = 0; i < m.nzx; i += PN_TIN)
                tiles.push_back({i - 1, m.pie + j - 1, m.nzx, m.nzy, m.pie, zo, so, po, pid});
    }
    const size_t P = (size_t)b->nump, Z = (size_t)b->numz;
    const size_t N = meshes.size();
    const size_t bytes = N * PN_CHAIN_BYTES + (4 * P + 5 * Z) * 8 + tiles.size() * sizeof(BTile) +
                         tri.size() * sizeof(BUnit) + origins.size() * sizeof(BHeavy);
    char* m = nullptr;
    if (hipMalloc((void**)&m, bytes) != hipSuccess) {
        (void)hipGetLastError();
        return 0;                            // no memory for a second state: separate passes
    }
    b->allocs.push_back(m);
    b->chain = m;                            // the problems' slots, then their second control blocks
    double* d = (double*)(m + N * PN_CHAIN_BYTES);
    for (int k = 0; k < 9; ++k) {
        b->alt[k] = d;
        d += k < 4 ? P : Z;
    }
    b->tiles = (BTile*)d;
    b->tunits = (BUnit*)(b->tiles + tiles.size());
    b->origins = (BHeavy*)(b->tunits + tri.size());
    b->ntunits = (int)tri.size();
    b->norigins = (int)origins.size();
    int rc = (int)hipMemcpy(b->tiles, tiles.data(), tiles.size() * sizeof(BTile), hipMemcpyHostToDevice);
    if (!rc && !tri.empty()) rc = (int)hipMemcpy(b->tunits, tri.data(), tri.size() * sizeof(BUnit), hipMemcpyHostToDevice);
    if (!rc && !origins.empty())
        rc = (int)hipMemcpy(b->origins, origins.data(), origins.size() * sizeof(BHeavy), hipMemcpyHostToDevice);
    hipLaunchKernelGGL(k_chain_begin_batch, dim3((unsigned)N), dim3(64), 0, b->stream, (slot_t*)b->chain);
    if (!rc) rc = (int)hipGetLastError();
    if (!rc) b->ntiles = (int)tiles.size();
    return rc;
}

// Step k of the problems' chains (as chain_step).
static BatchChain batch_chain(pennant_batch* b, int k, int zre) {
    slot_t* sets = (slot_t*)b->chain;
    Ctl* c[2] = {b->ctls, (Ctl*)(sets + (size_t)b->nprob * 3 * PN_SLOT_SET)};
    return {c[k & 1], c[(k + 1) & 1], sets, k ? (k - 1) % 3 : -1, k % 3, (k + 1) % 3, zre};
}

// Cycle k of a run, the second of a pair where k is odd.  The triangles' own
// state stays in the batch's arrays, as in tile_cycle; their point values come
// from the state the cycle starts from and go with the one it writes.
static int batch_tile_cycle(pennant_batch* b, int form, int k) {
    const int second = k & 1;
    BatchArgs B = make_batch_args(b);
    FusedArgs& a = B.a;
    BatchArgs T = B;                         // triangles
    double* const own[9] = {a.pxx, a.pxy, a.pux, a.puy, a.zr, a.ze, a.zetot, a.zwrate, a.zvol};
    double* const* src = second ? b->alt : own;
    double* const* dst = second ? own : b->alt;
    a.pxx = src[0]; a.pxy = src[1]; a.pux = src[2]; a.puy = src[3];
    a.zr = src[4]; a.ze = src[5]; a.zetot = src[6]; a.zwrate = src[7]; a.zvol = src[8];
    a.oxx = dst[0]; a.oxy = dst[1]; a.oux = dst[2]; a.ouy = dst[3];
    const TileBatch t = {{dst[4], dst[5], dst[6], dst[7], dst[8]}, b->tiles, b->ntiles, b->origins, second};
    T.units = b->tunits;
    T.nunits = b->ntunits;
    hipStream_t s = b->stream;
    const dim3 blk(PN_BLOCK), head(b->nprob + b->ntunits), tail(b->ntunits), grid(b->ntiles + b->norigins);
    const bool fp64 = form == FORM_FP64;
    const BatchChain c = batch_chain(b, k, fp64 ? 1 : 0);
    T.a.pxx = src[0]; T.a.pxy = src[1]; T.a.pux = src[2]; T.a.puy = src[3];
    if (fp64) hipLaunchKernelGGL(k_head_batch<double>, head, blk, 0, s, T, c, b->nprob, second);
    else hipLaunchKernelGGL(k_head_batch<float>, head, blk, 0, s, T, c, b->nprob, second);
    if (fp64) hipLaunchKernelGGL(k_tile_batch<double>, grid, blk, 0, s, B, t, c);
    else hipLaunchKernelGGL(k_tile_batch<float>, grid, blk, 0, s, B, t, c);
    if (b->ntunits) {
        T.a.pxx = dst[0]; T.a.pxy = dst[1]; T.a.pux = dst[2]; T.a.puy = dst[3];
        if (fp64) hipLaunchKernelGGL(k_tail_batch<double>, tail, blk, 0, s, T, c);
        else hipLaunchKernelGGL(k_tail_batch<float>, tail, blk, 0, s, T, c);
    }
    return (int)hipGetLastError();
}

int batch_tile_cycles(pennant_batch* b, int form, int n) {
    if (!b->ntiles || (n & 1) || form == FORM_LEARNED) return PENNANT_EINVAL;
    if (n < 1) return 0;
    if (const int rc = (int)hipGetLastError()) return rc;    // as tile_cycles
    for (int k = 0; k < n; ++k)
        if (const int rc = batch_tile_cycle(b, form, k)) return rc;
    BatchChain c = batch_chain(b, n, form == FORM_FP64 ? 1 : 0);
    c.put = c.prev;
    hipLaunchKernelGGL(k_chain_end_batch, dim3(b->nprob), dim3(64), 0, b->stream, make_batch_args(b), c);
    return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------
// Several pieces of one mesh on one device (src/Mesh.cc:432-617 partitions
// the points into private, master and ghost sets; src/Hydro.cc:450-455,
// 571-574, 766-769, 866-867, 902-906 read ghosts and reduce shared points).
// Each piece runs the fused K1 / K2 / K3 over its own arrays.  Between them:
//   corner exchange  each corner a piece's zones have at a ghost point is
//                    copied from the slot the piece's K1 wrote to the slot of
//                    the owner's corner list that holds it; the owner lists a
//                    master point's corners from every piece in ascending
//                    one-piece side order, so K2's ordered sum is the
//                    one-piece run's sum, bit for bit;
//   halo             after K2 the owners' new point state (px, pu and the
//                    calcWork point values) goes to the ghost copies, which
//                    K3 and the next cycle's K1 read.
// The pieces share one control block and one array of block partials, so a
// single finalize folds every piece's dt, dvol and bad-side partials.

namespace {

template <typename T>
__global__ void __launch_bounds__(PN_BLOCK) k_corner_xchg(const PieceTab* tab, const XEnt* x, int n,
                                                          const Ctl* ctl) {
    if (ctl->done) return;
    const int i = blockIdx.x * PN_BLOCK + threadIdx.x;
    if (i >= n) return;
    const XEnt e = x[i];
    const PieceTab& a = tab[e.sp];
    const PieceTab& b = tab[e.dp];
    if constexpr (sizeof(T) == 4) {
        const int64_t u = 3 * (int64_t)e.src, v = 3 * (int64_t)e.dst;
        b.fcrn[v] = a.fcrn[u];
        b.fcrn[v + 1] = a.fcrn[u + 1];
        b.fcrn[v + 2] = a.fcrn[u + 2];
    } else {
        b.cfx[e.dst] = a.cfx[e.src];
        b.cfy[e.dst] = a.cfy[e.src];
        b.cmass[e.dst] = a.cmass[e.src];
    }
}

template <typename T>
__global__ void __launch_bounds__(PN_BLOCK) k_halo(const PieceTab* tab, const XEnt* x, int n,
                                                   const Ctl* ctl) {
    if (ctl->done) return;
    const int i = blockIdx.x * PN_BLOCK + threadIdx.x;
    if (i >= n) return;
    const XEnt e = x[i];
    const PieceTab& a = tab[e.sp];
    const PieceTab& b = tab[e.dp];
    b.pxx[e.dst] = a.pxx[e.src];
    b.pxy[e.dst] = a.pxy[e.src];
    b.pux[e.dst] = a.pux[e.src];
    b.puy[e.dst] = a.puy[e.src];
    b.vs2[2 * (int64_t)e.dst] = a.vs2[2 * (int64_t)e.src];
    b.vs2[2 * (int64_t)e.dst + 1] = a.vs2[2 * (int64_t)e.src + 1];
    if constexpr (sizeof(T) == 8) b.pxpx[e.dst] = a.pxpx[e.src];
}

FusedArgs piece_args(pennant_pieces* pp, int q) {
    FusedArgs a = make_args(pp->pc[q]);
    a.ctl = pp->pc[0]->ctl;
    a.part_dt = pp->part_d;
    a.part_dv = pp->part_d + pp->nunits;
    a.part_bp = pp->part_i;
    a.part_bc = pp->part_i + pp->nunits;
    // no learned pass or tuple capture in a multi-piece run; the pieces'
    // maps are loaded
    a.rect_nzx = 0;
    a.zlist = nullptr;
    a.zcount = nullptr;
    a.nzruns = 0;
    a.cap_buf = nullptr;
    return a;
}

}  // namespace

// A phase of the piece cycle is one launch over the units of every piece (a
// unit is at most PN_BLOCK zones of one side-count run, or points, of one
// piece), which reads its piece's arrays from a table.  What bounds a cycle is
// the latency of its six dependent launches.  Noh pie 640 x 480 in 6 pieces,
// FP64, 100 cycles and the results' copies: 179 -> 81 us a cycle.  Before, with
// a launch per piece and run on the pieces' own streams, forked and joined
// around each phase, it was 34 launches and 30 event waits.  A run in one piece
// has nothing to gain from the tables and takes the launches of a problem (mixed,
// Sedov 1440^2: 188 us a cycle through the tables, 170 without).
namespace {

template <int FORM>
__global__ void __launch_bounds__(PN_BLOCK) __attribute__((amdgpu_waves_per_eu(FORM == FORM_MIXED ? 4 : 1)))
k_pred_pieces(const FusedArgs* A, const BUnit* units, double* part_dt, int* part_bp) {
    const BUnit U = units[blockIdx.x];
    const FusedArgs a = A[U.pid];
    if (a.ctl->done) return;
    const double dt = a.ctl->dt;
    double dtmin = 1.e99;
    int bad = 0;
    ClCount cnt;
    if (U.ns == 4) pred_unit<4, FORM, CL_EXACT>(a, U, dt, dtmin, bad, cnt);
    else pred_unit<3, FORM, CL_EXACT>(a, U, dt, dtmin, bad, cnt);
    const double m = block_min(dtmin);
    const int b = block_sum(bad);
    if (threadIdx.x == 0) {
        part_dt[blockIdx.x] = m;
        part_bp[blockIdx.x] = b;
    }
}

template <typename T>
__global__ void __launch_bounds__(PN_BLOCK) k_point_pieces(const FusedArgs* A, const PUnit* units, const BHeavy* heavy,
                                                           int nheavy) {
    if ((int)blockIdx.x < nheavy) {
        const BHeavy h = heavy[blockIdx.x];
        const FusedArgs a = A[h.pid];
        if (!a.ctl->done) point_heavy<T>(a, h.p, a.ctl->dt);
        return;
    }
    const PUnit U = units[blockIdx.x - nheavy];
    const FusedArgs a = A[U.pid];
    const int p = U.pb + (int)threadIdx.x;
    if (!a.ctl->done && p < U.pe) point_light<T>(a, p, a.ctl->dt);
}

template <typename T>
__global__ void __launch_bounds__(PN_BLOCK) k_corr_pieces(const FusedArgs* A, const BUnit* units, double* part_dv,
                                                          int* part_bc) {
    const BUnit U = units[blockIdx.x];
    const FusedArgs a = A[U.pid];
    if (a.ctl->done) return;
    const double dt = a.ctl->dt;
    double dvov = 1.e-99;
    int bad = 0;
    const int z = U.zb + (int)threadIdx.x;
    if (z < U.ze) {
        if (U.ns == 4) corr_zone<4, T>(a, z, U.sb + (z - U.zb) * 4, unit_w(U, z), dt, bad, dvov);
        else corr_zone<3, T>(a, z, U.sb + (z - U.zb) * 3, unit_w(U, z), dt, bad, dvov);
    }
    const double m = block_max(dvov);
    const int b = block_sum(bad);
    if (threadIdx.x == 0) {
        part_dv[blockIdx.x] = m;
        part_bc[blockIdx.x] = b;
    }
}

}  // namespace

// The pieces' argument table, their units and one partial per zone unit.
int pieces_setup(pennant_pieces* pp) {
    std::vector<BUnit> units;
    std::vector<PUnit> punits;
    std::vector<BHeavy> heavy;
    for (size_t q = 0; q < pp->pc.size(); ++q) {
        const pennant_problem* pb = pp->pc[q];
        const HostMesh& h = pb->hm;
        for (size_t r = 0; r < pb->zruns.size(); r += 3) {
            const int zb = pb->zruns[r], ze = pb->zruns[r + 1], ns = pb->zruns[r + 2];
            if (ns != 3 && ns != 4) return PENNANT_EINVAL;
            for (int u = zb; u < ze; u += PN_BLOCK) {
                BUnit U = {};
                U.zb = u;
                U.ze = u + PN_BLOCK < ze ? u + PN_BLOCK : ze;
                U.sb = h.zsbeg[(size_t)u];
                U.ns = ns;
                U.pid = (int)q;
                units.push_back(U);
            }
        }
        const int own = own_points(pb);
        for (int p = 0; p < own; p += PN_BLOCK)
            punits.push_back({p, p + PN_BLOCK < own ? p + PN_BLOCK : own, (int)q, 0});
        for (int p = 0; p < own; ++p)
            if (h.pcbeg[(size_t)p + 1] - h.pcbeg[(size_t)p] > PN_HEAVY) heavy.push_back({p, (int)q});
    }
    pp->nunits = (int)units.size();
    pp->npunits = (int)punits.size();
    pp->nheavy = (int)heavy.size();
    const size_t n = units.size(), bytes[] = {n * 2 * 8, n * 2 * 4, n * sizeof(BUnit), punits.size() * sizeof(PUnit),
                                              heavy.size() * sizeof(BHeavy), pp->pc.size() * sizeof(FusedArgs)};
    void** to[] = {(void**)&pp->part_d, (void**)&pp->part_i, (void**)&pp->units, (void**)&pp->punits,
                   (void**)&pp->heavy, &pp->args};
    for (int k = 0; k < 6; ++k) {
        if (hipMalloc(to[k], bytes[k] > 0 ? bytes[k] : 8) != hipSuccess) return (int)hipErrorOutOfMemory;
        pp->allocs.push_back(*to[k]);
    }
    std::vector<FusedArgs> A;
    for (size_t q = 0; q < pp->pc.size(); ++q) A.push_back(piece_args(pp, (int)q));
    int rc = (int)hipMemcpy(pp->units, units.data(), bytes[2], hipMemcpyHostToDevice);
    if (!rc) rc = (int)hipMemcpy(pp->punits, punits.data(), bytes[3], hipMemcpyHostToDevice);
    if (!rc && !heavy.empty()) rc = (int)hipMemcpy(pp->heavy, heavy.data(), bytes[4], hipMemcpyHostToDevice);
    if (!rc) rc = (int)hipMemcpy(pp->args, A.data(), bytes[5], hipMemcpyHostToDevice);
    return rc;
}

int pieces_cycle(pennant_pieces* pp, int form) {
    if (form == FORM_LEARNED || pp->pc.empty()) return PENNANT_EINVAL;
    const bool mixed = (form != FORM_FP64);
    if (pp->pc.size() == 1) {                // the whole mesh: a problem's own passes
        if (mixed) pp->zre_stale = true;
        return fused_cycle(pp->pc[0], nullptr, form);
    }
    hipStream_t s = pp->pc[0]->stream;
    const FusedArgs* A = (const FusedArgs*)pp->args;
    const Ctl* ctl = pp->pc[0]->ctl;
    const dim3 zg(pp->nunits), pg(pp->nheavy + pp->npunits), xg(nblocks(pp->ncx)), hg(nblocks(pp->nhalo)), blk(PN_BLOCK);
    double* dv = pp->part_d + pp->nunits;
    int* bc = pp->part_i + pp->nunits;
    if (mixed) {
        hipLaunchKernelGGL(k_pred_pieces<FORM_MIXED>, zg, blk, 0, s, A, pp->units, pp->part_d, pp->part_i);
        if (pp->ncx > 0) hipLaunchKernelGGL(k_corner_xchg<float>, xg, blk, 0, s, pp->tab, pp->cx, pp->ncx, ctl);
        hipLaunchKernelGGL(k_point_pieces<float>, pg, blk, 0, s, A, pp->punits, pp->heavy, pp->nheavy);
        if (pp->nhalo > 0) hipLaunchKernelGGL(k_halo<float>, hg, blk, 0, s, pp->tab, pp->halo, pp->nhalo, ctl);
        hipLaunchKernelGGL(k_corr_pieces<float>, zg, blk, 0, s, A, pp->units, dv, bc);
    } else {
        hipLaunchKernelGGL(k_pred_pieces<FORM_FP64>, zg, blk, 0, s, A, pp->units, pp->part_d, pp->part_i);
        if (pp->ncx > 0) hipLaunchKernelGGL(k_corner_xchg<double>, xg, blk, 0, s, pp->tab, pp->cx, pp->ncx, ctl);
        hipLaunchKernelGGL(k_point_pieces<double>, pg, blk, 0, s, A, pp->punits, pp->heavy, pp->nheavy);
        if (pp->nhalo > 0) hipLaunchKernelGGL(k_halo<double>, hg, blk, 0, s, pp->tab, pp->halo, pp->nhalo, ctl);
        hipLaunchKernelGGL(k_corr_pieces<double>, zg, blk, 0, s, A, pp->units, dv, bc);
    }
    const Params& q = pp->prm;
    hipLaunchKernelGGL(k_finalize, dim3(1), dim3(PN_FIN_BLOCK), 0, s, piece_args(pp, 0), pp->nunits, pp->nunits, q.cflv,
                       q.cstop, q.dtmax, q.dtfac, q.tstop, mixed ? 0 : 1);
    if (mixed) pp->zre_stale = true;
    return (int)hipGetLastError();
}

int pieces_materialize_zre(pennant_pieces* pp) {
    if (!pp->zre_stale || pp->pc.empty()) return 0;
    hipStream_t s = pp->pc[0]->stream;
    for (size_t q = 0; q < pp->pc.size(); ++q) {
        const int nz = pp->pc[q]->hm.numz;
        if (nz > 0)
            hipLaunchKernelGGL(k_zre, dim3(nblocks(nz)), dim3(PN_BLOCK), 0, s, piece_args(pp, (int)q), nz);
    }
    hipLaunchKernelGGL(k_zre_done, dim3(1), dim3(64), 0, s, pp->pc[0]->ctl, 1);
    pp->zre_stale = false;
    return (int)hipGetLastError();
}

}  // namespace pn
