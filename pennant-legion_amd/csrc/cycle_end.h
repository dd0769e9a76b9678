// The end of a cycle: calcDt (src/Hydro.cc:1647-1667), checkBadSides
// (src/Mesh.cc:1531-1550), the time and cycle update (src/Driver.cc:266-295),
// the stop test and calcGlobalDt (src/Driver.cc:213-245) for the next cycle,
// from the cycle's smallest dt limit, largest dvol ratio and bad-side counts;
// and the slots through which the blocks of a kernel hand these on.
// Included by every source file that ends cycles.
#pragma once

#include "common.h"
#include "problem.h"

namespace {

using pn::Ctl;

// The control block's fields that end a cycle
struct CtlSnap {
    double time, dt, la_dtnew;
    int cycle, la_bp, done;
};
// Relaxed atomic loads: vector loads (never scalar-cache loads), issued
// back to back with no wait between them.
__device__ __forceinline__ double ld_vec(const double* p) {
    return __builtin_bit_cast(double, __hip_atomic_load(reinterpret_cast<const unsigned long long*>(p),
                                                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}
__device__ __forceinline__ int ld_vec(const int* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Read through vector loads: the caller stores to the block later.
__device__ __forceinline__ CtlSnap snap_ctl(const Ctl* c) {
    CtlSnap v;
    v.time = ld_vec(&c->time);
    v.dt = ld_vec(&c->dt);
    v.la_dtnew = ld_vec(&c->la_dtnew);
    v.cycle = ld_vec(&c->cycle);
    v.la_bp = ld_vec(&c->la_bp);
    v.done = ld_vec(&c->done);
    return v;
}

struct DtParams {
    double cflv, dtmax, dtfac, tstop;
    int cstop;
};
inline DtParams dt_params(const pennant_problem* pb) {
    const pn::Params& q = pb->prm;
    DtParams d;
    d.cflv = q.cflv; d.dtmax = q.dtmax; d.dtfac = q.dtfac; d.tstop = q.tstop; d.cstop = q.cstop;
    return d;
}

// What follows a cycle that ran with dt from `time` as the `cycle`-th: dtrec,
// and when its sides were good the new time, cycle, next dt and done flag
// (with bad sides the run is done).
struct CycleEnd {
    double dtrec, time, dt;
    int cycle, done;
};
__device__ __forceinline__ CycleEnd cycle_end(double dt, double time, int cycle, double mn, double mx, int bad,
                                              const DtParams& q) {
    CycleEnd e;
    double r = 1.e99;
    if (mn < r) r = mn;
    const double d2v = dt * q.cflv / mx;
    if (d2v < r) r = d2v;
    e.dtrec = r;
    e.time = time + dt;
    e.cycle = cycle + 1;
    double nd = q.dtmax;
    const double dtrecover = q.dtfac * dt;
    if (dtrecover < nd) nd = dtrecover;
    if ((q.tstop - e.time) < nd) nd = q.tstop - e.time;
    if (r < nd) nd = r;
    e.dt = nd;
    e.done = (bad > 0 || e.cycle >= q.cstop || e.time >= q.tstop) ? 1 : 0;
    return e;
}

// Ends the cycle in the control block c, whose fields v were read before any
// store to it (a scalar-cache load is not ordered with a later vector store to
// the same address).  bp, bc: the predictor's and the corrector's bad sides.
// Returns the new done flag; *next_dt (when given) receives the next dt.
__device__ __forceinline__ int end_cycle(Ctl* c, const CtlSnap& v, double mn, double mx, int bp, int bc,
                                         const DtParams& q, double* next_dt = nullptr) {
    const CycleEnd e = cycle_end(v.dt, v.time, v.cycle, mn, mx, bp + bc, q);
    c->dtnew = mn;
    c->dvovmax = mx;
    c->numsbad_pred = bp;
    c->numsbad_corr = bc;
    c->dtrec = e.dtrec;
    c->done = e.done;
    if (bp > 0 || bc > 0) {
        c->err_cycle = v.cycle;
        c->err_pred = bp > 0 ? 1 : 0;
        return 1;
    }
    c->time = e.time;
    c->cycle = e.cycle;
    c->dtlast = v.dt;
    c->dt = e.dt;
    if (next_dt) *next_dt = e.dt;
    return e.done;
}

// ---------------------------------------------------------------------------
// Slots
//
// The blocks of a kernel fold their dt limits and dvol ratios into a set of
// slots by atomic minima (no value is returned, so nothing waits), and whoever
// needs the result folds the slots: a wave, with one load a lane.  With an
// array of partials a one-block kernel did that between every two cycles, 9.5
// us for 10600 tiles and 18 us for 32400 task tiles; one wave with the slots
// takes 3.5, or every block of the next kernel does it by itself while its own
// loads are under way (worth it with few blocks: PN_LINK_TILES, PN_LINK_TASKS).
//
// Doubles are held as integers of the same order; ratios as the complement, so
// that every slot takes a minimum (exact in any order).  A line per slot: 16
// for each, and one for the counts of bad sides.
#define PN_SLOTS 16
#define PN_SLOT_LINE 16                  // 64-bit words of a line
#define PN_SLOT_SET ((2 * PN_SLOTS + 1) * PN_SLOT_LINE)
typedef unsigned long long slot_t;

__device__ __forceinline__ slot_t slot_key(double v) {
    const slot_t b = __builtin_bit_cast(slot_t, v);
    return b ^ ((b >> 63) ? ~0ull : 1ull << 63);
}
__device__ __forceinline__ double slot_value(slot_t k) {
    return __builtin_bit_cast(double, k ^ ((k >> 63) ? 1ull << 63 : ~0ull));
}
// Block `b`'s contribution, by one thread.
__device__ __forceinline__ void slots_dt(slot_t* set, int b, double dt, int bp) {
    atomicMin(set + (b & (PN_SLOTS - 1)) * PN_SLOT_LINE, slot_key(dt));
    if (bp) atomicAdd(set + 2 * PN_SLOTS * PN_SLOT_LINE, (slot_t)(unsigned)bp);
}
__device__ __forceinline__ void slots_dv(slot_t* set, int b, double dv, int bc) {
    atomicMin(set + (PN_SLOTS + (b & (PN_SLOTS - 1))) * PN_SLOT_LINE, ~slot_key(dv));
    if (bc) atomicAdd(set + 2 * PN_SLOTS * PN_SLOT_LINE, (slot_t)(unsigned)bc << 32);
}
// Empties the set, by the first threads of a block of at least 64.
__device__ __forceinline__ void slots_reset(slot_t* set) {
    const int t = threadIdx.x;
    if (t <= 2 * PN_SLOTS)
        set[t * PN_SLOT_LINE] = t < PN_SLOTS ? slot_key(1.e99) : (t < 2 * PN_SLOTS ? ~slot_key(1.e-99) : 0ull);
}
// This lane's slot of the set, and the fold of a wave's: the same in all lanes.
__device__ __forceinline__ slot_t slots_load(const slot_t* set) {
    const int l = (int)(threadIdx.x & 63);
    return __hip_atomic_load(set + (l < 2 * PN_SLOTS ? l : 2 * PN_SLOTS) * PN_SLOT_LINE, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
}
struct SlotFold {
    double mn, mx;
    int bp, bc;
};
template <int ROR>
__device__ __forceinline__ slot_t row_min(slot_t v) {     // with the lane ROR further round its row of 16
    const unsigned lo = __builtin_amdgcn_mov_dpp((int)(unsigned)v, 0x120 + ROR, 0xf, 0xf, false);
    const unsigned hi = __builtin_amdgcn_mov_dpp((int)(unsigned)(v >> 32), 0x120 + ROR, 0xf, 0xf, false);
    const slot_t o = (slot_t)hi << 32 | lo;
    return o < v ? o : v;
}
__device__ __forceinline__ slot_t slot_lane(slot_t v, int l) {
    return (slot_t)(unsigned)__builtin_amdgcn_readlane((int)(unsigned)(v >> 32), l) << 32 |
           (unsigned)__builtin_amdgcn_readlane((int)(unsigned)v, l);
}
__device__ __forceinline__ SlotFold slots_fold(slot_t v) {
    const slot_t bad = slot_lane(v, 2 * PN_SLOTS);
    v = row_min<8>(v);
    v = row_min<4>(v);
    v = row_min<2>(v);
    v = row_min<1>(v);
    SlotFold f;
    f.mn = slot_value(slot_lane(v, 0));
    f.mx = slot_value(~slot_lane(v, PN_SLOTS));
    f.bp = (int)(unsigned)bad;
    f.bc = (int)(bad >> 32);
    return f;
}

// A kernel's place in a chain of cycles with no finalize between them.  Each
// reads the control block `in` and, unless it is the chain's first, the slots
// `prev` that the cycle before it filled; it fills `put`, empties `clear` (the
// set of the cycle before that) and leaves the control block as it is now in
// `out`.  Blocks of one kernel all read what none of them writes.
struct CycleStep {
    const Ctl* in;
    Ctl* out;
    const slot_t* prev;          // NULL: `in` is current
    slot_t *put, *clear;
    DtParams q;
    int zre;                     // Ctl::zre_valid after a cycle of the chain
};
struct CycleNow {
    double dt;
    int done, ended, zre;        // ended: the cycle before ended the run
};
__device__ __forceinline__ CycleNow cycle_now(const CycleStep& s) {
    CycleNow n = {s.in->dt, s.in->done, 0, s.in->zre_valid};
    if (s.prev) {
        const slot_t v = slots_load(s.prev);
        const double time = s.in->time;
        const int cycle = s.in->cycle;
        if (!n.done) {
            const SlotFold f = slots_fold(v);
            const CycleEnd e = cycle_end(n.dt, time, cycle, f.mn, f.mx, f.bp + f.bc, s.q);
            // (uniform: in scalar registers)
            n.dt = pn::uni(e.dt);
            n.done = n.ended = __builtin_amdgcn_readfirstlane(e.done);
            n.zre = s.zre;
        }
    }
    return n;
}
// The step's writes, by one block.  back: the state, where the cycle before
// ended the run, is in the second set of arrays and this one copies it back
// (Ctl::cur).
__device__ __forceinline__ void cycle_step(const CycleStep& s, int back = 0) {
    if (threadIdx.x < 64) {
        const CtlSnap v = snap_ctl(s.in);
        SlotFold f = {};
        if (s.prev) f = slots_fold(slots_load(s.prev));
        if (threadIdx.x == 0) {
            *s.out = *s.in;
            s.out->cur = 0;
            if (s.prev && !v.done) {
                s.out->zre_valid = s.zre;
                s.out->cur = end_cycle(s.out, v, f.mn, f.mx, f.bp, f.bc, s.q) && back;
            }
        }
    }
    slots_reset(s.clear);
}
// The end of a chain whose last cycle filled the first of the three sets
// `sets` + `last` and left its control block in `in`: c is current again and
// the sets are empty.  One block.
__device__ __forceinline__ void cycle_chain_end(Ctl* c, const Ctl* in, slot_t* sets, int last, const DtParams& q,
                                                int zre) {
    if (threadIdx.x < 64) {
        const CtlSnap v = snap_ctl(in);
        const SlotFold f = slots_fold(slots_load(sets + last * PN_SLOT_SET));
        if (threadIdx.x == 0) {
            if (c != in) *c = *in;
            c->cur = 0;
            if (!v.done) {
                c->zre_valid = zre;
                end_cycle(c, v, f.mn, f.mx, f.bp, f.bc, q);
            }
        }
    }
    __syncthreads();
    for (int k = 0; k < 3; ++k) slots_reset(sets + k * PN_SLOT_SET);
}
__global__ void __launch_bounds__(64) k_chain_end(Ctl* c, const Ctl* in, slot_t* sets, int last, DtParams q, int zre) {
    cycle_chain_end(c, in, sets, last, q, zre);
}
__global__ void __launch_bounds__(64) k_chain_begin(slot_t* sets) {
    for (int k = 0; k < 3; ++k) slots_reset(sets + k * PN_SLOT_SET);
}

// Memory of a chain: three sets of slots and a second control block.  (A
// batch's chains lie as all their slots and then an array of control blocks,
// with other arrays after it.)
#define PN_CHAIN_CTL 256
#define PN_CHAIN_BYTES (3 * PN_SLOT_SET * 8 + PN_CHAIN_CTL)
static_assert(sizeof(Ctl) <= PN_CHAIN_CTL, "a chain's second control block");
inline slot_t* chain_sets(void* m) { return static_cast<slot_t*>(m); }
inline Ctl* chain_ctl(void* m) { return reinterpret_cast<Ctl*>(static_cast<slot_t*>(m) + 3 * PN_SLOT_SET); }
// Step k of a chain on the problem's control block.
inline CycleStep chain_step(pennant_problem* pb, void* m, int k, int zre) {
    slot_t* s = chain_sets(m);
    Ctl* c[2] = {pb->ctl, chain_ctl(m)};
    CycleStep t;
    t.in = c[k & 1];
    t.out = c[(k + 1) & 1];
    t.prev = k ? s + (k - 1) % 3 * PN_SLOT_SET : nullptr;
    t.put = s + k % 3 * PN_SLOT_SET;
    t.clear = s + (k + 1) % 3 * PN_SLOT_SET;
    t.q = dt_params(pb);
    t.zre = zre;
    return t;
}
// Ends a chain of n steps, or (n = 0) one cycle that was not linked: step 0's
// slots and the problem's control block.
inline int chain_end(pennant_problem* pb, void* m, int n, int zre) {
    Ctl* c[2] = {pb->ctl, chain_ctl(m)};
    hipLaunchKernelGGL(k_chain_end, dim3(1), dim3(64), 0, pb->stream, pb->ctl, c[n & 1], chain_sets(m),
                       n ? (n - 1) % 3 : 0, dt_params(pb), zre);
    return (int)hipGetLastError();
}

}  // namespace
