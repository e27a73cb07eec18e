// sevc_dev.h -- device helpers shared by the time step and the adjoint
// window kernels (entity access, set operations on the trivalent mesh,
// areas and the analytic force).  Include after sevc_state.h/sevc_geom.h.
#pragma once
#include <hip/hip_runtime.h>
#include "sevc_state.h"
#include "sevc_geom.h"
#include "../../include/sevc.h"
#include "../../include/sevc_math.h"

namespace sevc {

enum { T_COMMON = 0, T_NUCLEATED = 1 };                                  // geometry.h:19
constexpr unsigned kStreamMcSite = 1u, kStreamMcPick = 2u, kStreamRate = 3u;
constexpr int kMaxStride = 128;   // largest grain-list stride supported

// ---------------------------------------------------------------------
// helpers
// ---------------------------------------------------------------------

// Map the hardware workgroup id so that each of the 8 XCDs (workgroups are
// dealt round-robin over XCDs) processes one contiguous slice of the table:
// neighbouring slots then share an L2.
__device__ __forceinline__ int xcd_remap(int b, int nb) {
    int q = nb >> 3, r = nb & 7, x = b & 7;
    return x * q + (x < r ? x : r) + (b >> 3);
}

// An event of member m met an inconsistent state or a full grain list: the
// member records the first such code and stops (its later event entries of
// the step are skipped, as after a failed check); the other members of a
// batch go on.
__device__ __forceinline__ void set_error(const Dev& d, int m, int code) {
    MState& M = d.ms[m];
    if (atomicCAS(&M.status, 0, code) == 0) {
        M.active = 0;
        M.done = 1;
    }
}

__device__ __forceinline__ int other_end(const Dev& d, int b, int v) {
    return d.bvx[2 * b] == v ? d.bvx[2 * b + 1] : d.bvx[2 * b];
}

// The set operations on vertex-grain triples run on values already loaded and
// keep their results in scalars: a result array filled at a run-time position
// would live in scratch memory (or in LDS, where the compiler finds room).

// geometry.h:837-848: the first two matches of (ga[i], gb[j]) in order of i,
// then j (-1 where there are fewer); the number found, at most 2.
__device__ __forceinline__ int triples_intersect(const int (&ga)[3], const int (&gb)[3], int& o0, int& o1) {
    int k = 0;
    o0 = o1 = -1;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) {
            const bool hit = ga[i] == gb[j];
            o1 = hit && k == 1 ? ga[i] : o1;
            o0 = hit && k == 0 ? ga[i] : o0;
            k += hit && k < 2 ? 1 : 0;
        }
    return k;
}

// geometry.h:886-898 (with grains_union, :863-875): the first two of the
// union (ga, then the first of gb not among them, -1 if none) that are not
// among the intersection (i0, i1).
__device__ __forceinline__ void triples_symdiff(const int (&ga)[3], const int (&gb)[3], int i0, int i1, int& o0, int& o1) {
    int fourth = -1;
    bool have = false;
#pragma unroll
    for (int j = 0; j < 3; j++) {
        const int g = gb[j];
        const bool other = !have && g != ga[0] && g != ga[1] && g != ga[2];
        fourth = other ? g : fourth;
        have = have || other;
    }
    const int gun[4] = {ga[0], ga[1], ga[2], fourth};
    int k = 0;
    o0 = o1 = -1;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const bool out = gun[i] != i0 && gun[i] != i1;
        o1 = out && k == 1 ? gun[i] : o1;
        o0 = out && k == 0 ? gun[i] : o0;
        k += out ? 1 : 0;
    }
}

__device__ __forceinline__ void load_triple(const int* a, int v, int (&t)[3]) {
#pragma unroll
    for (int q = 0; q < 3; q++) t[q] = a[3 * v + q];
}

__device__ __forceinline__ int grains_intersect(const Dev& d, int a, int b, int& o0, int& o1) {
    int ga[3], gb[3];
    load_triple(d.vg, a, ga);
    load_triple(d.vg, b, gb);
    return triples_intersect(ga, gb, o0, o1);
}

__device__ __forceinline__ int* glist(const Dev& d, int g) { return d.gvx + (size_t)g * d.S; }

// Member owning a vertex / grain / edge slot (members own consecutive slot
// ranges; a batch keeps the owner of every slot, one load).
__device__ __forceinline__ int member_of_vertex(const Dev& d, int v) { return d.B == 1 ? 0 : d.vmem[v]; }
__device__ __forceinline__ int member_of_grain(const Dev& d, int g) { return d.B == 1 ? 0 : d.gmem[g]; }
__device__ __forceinline__ int member_of_edge(const Dev& d, int e) { return d.B == 1 ? 0 : d.emem[e]; }

// geometry.h:703-710
// The list is read eight entries at a time (independent loads), then
// searched in order: the first index holding v, or -1.
__device__ __forceinline__ int grain_contains_vertex(const Dev& d, int g, int v) {
    const int* L = glist(d, g);
    const int n = d.glen[g];
    for (int i0 = 0; i0 < n; i0 += 8) {
        int x[8];
#pragma unroll
        for (int q = 0; q < 8; q++) x[q] = i0 + q < n ? L[i0 + q] : -2;
#pragma unroll
        for (int q = 0; q < 8; q++)
            if (x[q] == v) return i0 + q;
    }
    return -1;
}

// What a flip asks of a grain's list about its edge's ends a and b, from one
// reading of the list (eight entries and the next one at a time, the searches
// of all four grains around a flip in step): `ab` and `ba`, whether (a, b) /
// (b, a) come one after the other round the list (grain_contains_consecutive,
// geometry.h:724-734: 1 for the pair as asked, 2 for the other way round,
// whichever comes first, -1 for neither), and the first place of a and of b
// (-1: not in the list).
struct GrainFind {
    int ab, ba, a, b;
};

__device__ __forceinline__ GrainFind grain_find(const Dev& d, int g, int a, int b) {
    const int* L = glist(d, g);
    const int n = d.glen[g];
    // the first eight entries come with the length where the row has them
    const bool wide = d.S % 4 == 0 && d.S >= 8;
    int4 h0 = make_int4(-1, -1, -1, -1), h1 = h0;
    if (wide) {
        h0 = reinterpret_cast<const int4*>(L)[0];
        h1 = reinterpret_cast<const int4*>(L)[1];
    }
    const int l0 = wide ? h0.x : (n > 0 ? L[0] : -2);
    GrainFind f = {-1, -1, -1, -1};
#pragma unroll 1
    for (int i0 = 0; i0 < n; i0 += 8) {
        int x[9];
        if (wide && i0 == 0) {
            x[0] = h0.x; x[1] = h0.y; x[2] = h0.z; x[3] = h0.w;
            x[4] = h1.x; x[5] = h1.y; x[6] = h1.z; x[7] = h1.w;
            x[8] = n > 8 ? L[8] : -2;
        } else {
#pragma unroll
            for (int q = 0; q < 9; q++) x[q] = i0 + q < n ? L[i0 + q] : -2;
        }
#pragma unroll
        for (int q = 0; q < 9; q++) x[q] = i0 + q == n ? l0 : (i0 + q > n ? -2 : x[q]);
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const bool in = i0 + q < n;
            f.a = in && f.a < 0 && x[q] == a ? i0 + q : f.a;
            f.b = in && f.b < 0 && x[q] == b ? i0 + q : f.b;
            const int p = !in ? -1 : (x[q] == a && x[q + 1] == b) ? 1 : (x[q] == b && x[q + 1] == a) ? 2 : -1;
            f.ab = f.ab < 0 ? p : f.ab;
        }
    }
    // asked the other way round, the same first pair answers
    f.ba = f.ab < 0 ? -1 : 3 - f.ab;
    return f;
}

// geometry.h:548-550, pow(c,3) as c*c*c
__device__ __forceinline__ double gb_energy_func(double d_alpha, double eps) {
    double c = sevc_cos(4 * d_alpha);
    return (1 + 0.5 * eps * (1 - c * c * c));
}

// geometry.h:559-564
__device__ __forceinline__ double boundary_compute_energy(const Dev& d, int b, double eps) {
    int g0, g1;
    if (grains_intersect(d, d.bvx[2 * b], d.bvx[2 * b + 1], g0, g1) < 2) return 1.0;
    return gb_energy_func(d.gori[g0] - d.gori[g1], eps);
}

// geometry.h:513-517 plus the flip-threshold extension
__device__ __forceinline__ bool is_candidate(double te, double len, double dt, double thr) {
    if (te >= 0 && te <= dt) return true;
    // a zero-length edge (just flipped, t_ext = no-motion value) is not shrinking
    if (thr > 0 && te >= 0 && len > 0 && len < thr) return true;
    return false;
}

// The step's dt for a minimum extinction time of the given bits (nondecreasing
// in them).
__device__ __forceinline__ double dt_from_tau(const Params& P, unsigned long long bits) {
    if (!P.adaptive) return P.dt_max;
    if (bits == 0x7FF0000000000000ull) return P.dt_max;
    double tau = __longlong_as_double((long long)bits);
    double dt = P.dt_safety * tau;
    if (dt < P.dt_min) dt = P.dt_min;
    if (dt > P.dt_max) dt = P.dt_max;
    return dt;
}

__device__ __forceinline__ double member_dt(const Params& P, const MState& M) { return dt_from_tau(P, M.tau_bits); }

// compute_area of grain g (geometry.h:757-765 after :908-931) with the
// vertex positions X (2 doubles per vertex slot).
__device__ __forceinline__ double grain_area_at(const Dev& d, const double* X, int g, double D) {
    int n = d.glen[g];
    if (n <= 0) return 0.0;
    const int* L = glist(d, g);
    AreaAcc acc;
    int w = L[0];
    acc.start(X[2 * w], X[2 * w + 1]);
    for (int k = 1; k < n; k++) {
        w = L[k];
        acc.push(X[2 * w], X[2 * w + 1], D);
    }
    return acc.finish();
}

__device__ __forceinline__ double grain_area(const Dev& d, int g, double D) { return grain_area_at(d, d.pos, g, D); }

// geometry.h:369-376, as three 16-byte stores (grn, vrt, prev) and one
// 4-byte store (the four fix bytes) into the vertex's 64-byte record
__device__ __forceinline__ void reset_mods(const Dev& d, int v) {
    static_assert(offsetof(ModRec, grn) == 0 && offsetof(ModRec, vrt) == 16 && offsetof(ModRec, prev) == 32 &&
                      offsetof(ModRec, fix) == 48,
                  "record layout");
    int4* r = reinterpret_cast<int4*>(&d.mods[v]);
    r[0] = make_int4(-1, -1, -1, -1);
    r[1] = make_int4(-1, -1, -1, -1);
    r[2] = make_int4(-1, -1, -1, -1);
    *reinterpret_cast<unsigned*>(d.mods[v].fix) = 0x01010101u * (unsigned)FIX_NONE;
}

__device__ __forceinline__ void set_mod(const Dev& d, int v, int slot, int fix, int grn, int vrt) {
    d.mods[v].fix[slot] = (uint8_t)fix;
    d.mods[v].grn[slot] = grn;
    d.mods[v].vrt[slot] = vrt;
}

// A slot of a list whose length is *counter, for each active lane with
// `want` (-1 for the others), with one atomic per wave: lanes that append
// at the same point share it (the slots are consecutive in lane order).  The
// lists' order is unspecified, as with an atomic per lane; one atomic per
// wave keeps a step with thousands of events from queueing them on one
// address.
__device__ __forceinline__ int wave_slot(int* counter, bool want) {
    const unsigned long long m = __ballot(want);
    if (m == 0) return -1;
    const int lane = (int)(threadIdx.x & 63);
    const int leader = __ffsll((long long)m) - 1;
    int base = 0;
    if (lane == leader) base = atomicAdd(counter, (int)__popcll(m));
    base = __builtin_amdgcn_readlane(base, leader);
    return want ? base + (int)__popcll(m & ((1ull << lane) - 1ull)) : -1;
}

// Adds, for each active lane with `want`, one to the member counter
// `field` of member `mem`: one atomic per distinct member among the wave's
// lanes.
__device__ __forceinline__ void wave_count(const Dev& d, bool want, int mem, long long MState::*field) {
    unsigned long long m = __ballot(want);
    const int lane = (int)(threadIdx.x & 63);
    while (m) {
        const int leader = __ffsll((long long)m) - 1;
        const int k = __builtin_amdgcn_readlane(mem, leader);
        const unsigned long long same = __ballot(want && mem == k);
        if (lane == leader) atomicAdd(reinterpret_cast<unsigned long long*>(&(d.ms[k].*field)), (unsigned long long)__popcll(same));
        m &= ~same;
    }
}

// The per-table-block (enabled, free) slot counts follow every event that
// enables or disables a slot (k_count_all recounts them only after a host
// upload): one 64-bit atomic adds (+1, -1) or (-1, +1) to the pair.
__device__ __forceinline__ void slot_count_add(int2* bc, int blk, bool enable) {
    atomicAdd(reinterpret_cast<unsigned long long*>(&bc[blk]),
              enable ? 0xFFFFFFFF00000001ull : 0x00000000FFFFFFFFull);
}

// Where a member's slots and table blocks start (members own consecutive runs
// of kBlock slots from their offsets): loaded once per event, with its other
// data, for all the flags it changes.
struct SlotBase {
    int voff, eoff, goff, vf, ef, gf;
};
__device__ __forceinline__ SlotBase slot_base(const Dev& d, int m) {
    if (d.B == 1) return SlotBase{0, 0, 0, 0, 0, 0};
    const Params& P = d.prm[m];
    return SlotBase{P.voff, P.eoff, P.goff, d.vblk_first[m], d.eblk_first[m], d.gblk_first[m]};
}

// Set an enable flag whose value is known to be `was` (loaded by the caller
// with its other data), counting a change of state.  No other thread writes
// the same flag in the same launch (events that touch a slot are serial or
// disjoint).
__device__ __forceinline__ void set_vertex_enabled(const Dev& d, const SlotBase& S, int v, bool was, bool on) {
    if (was != on) {
        d.ven[v] = on ? 1 : 0;
        slot_count_add(d.bc_v, S.vf + (v - S.voff) / kBlock, on);
    }
}
__device__ __forceinline__ void set_edge_enabled(const Dev& d, const SlotBase& S, int e, bool was, bool on) {
    if (was != on) {
        d.benab[e] = on ? 1 : 0;
        slot_count_add(d.bc_e, S.ef + (e - S.eoff) / kBlock, on);
    }
}
__device__ __forceinline__ void set_grain_enabled(const Dev& d, const SlotBase& S, int g, bool was, bool on) {
    if (was != on) {
        d.genab[g] = on ? 1 : 0;
        slot_count_add(d.bc_g, S.gf + (g - S.goff) / kBlock, on);
    }
}

// Flags the grains g[q] (where want[q]) for the fix stage `stage`
// (grain.fix = true) and lists each once.  The exchanges of all N are issued
// together, and one atomic per wave takes the list room of all its lanes, so
// the chain is two atomics long whatever N (one grain at a time took two for
// each: a flip's four took 8 us).
template <int N>
__device__ __forceinline__ void flag_grains(const Dev& d, const int (&g)[N], const bool (&want)[N], int stage) {
    int old[N];
#pragma unroll
    for (int q = 0; q < N; q++) old[q] = want[q] ? atomicExch(&d.gfix[g[q]], 1) : 1;
    unsigned long long m[N];
    int total = 0;
#pragma unroll
    for (int q = 0; q < N; q++) {
        m[q] = __ballot(old[q] == 0);
        total += (int)__popcll(m[q]);
    }
    if (total == 0) return;
    const int lane = (int)(threadIdx.x & 63);
    const int leader = __ffsll((long long)__ballot(1)) - 1;
    int base = 0;
    if (lane == leader) base = atomicAdd(&d.cnt[C_FIX0 + stage], total);
    base = __builtin_amdgcn_readlane(base, leader);
#pragma unroll
    for (int q = 0; q < N; q++) {
        if (old[q] == 0) d.l_fix[stage][base + (int)__popcll(m[q] & ((1ull << lane) - 1ull))] = g[q];
        base += (int)__popcll(m[q]);
    }
}

// A list counter read in the launch that fills it (an atomic load: the
// counters are only ever changed by atomics, which pass the vector cache).
__device__ __forceinline__ int cnt_now(const Dev& d, int c) {
    return __hip_atomic_load(&d.cnt[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Orders a wave's LDS accesses (its lanes run in step, so only the compiler
// has to keep them in order).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// An edit left grain g with three vertices: the next search for adjacent
// 3-sided pairs looks at it (tri_items).  Each of a step's three edit stages
// and its nucleations list a grain at most once, so 6 G entries hold them.
__device__ __forceinline__ void list_tri(const Dev& d, int g, bool want) {
    const int s = wave_slot(&d.cnt[C_TRI], want);
    if (want && (unsigned)s < 6u * (unsigned)d.G) d.l_tri[s] = g;
}

// Inclusive prefix sum of v over the 64 lanes of a wave (every lane active),
// by DPP lane moves: Hillis-Steele steps within each row of 16 lanes (row
// shifts by 1, 2, 4, 8; lanes shifted in from outside the row add 0), then
// the total of row 0 / row 2 (its lane 15, broadcast) into rows 1 / 3, and
// the total of rows 0-1 (lane 31, broadcast) into rows 2 and 3.  Rows that
// a broadcast does not write add 0.
__device__ __forceinline__ int wave_inclusive_scan(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);    // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);    // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);    // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);    // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);   // row_bcast:15 into rows 1, 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);   // row_bcast:31 into rows 2, 3
    return v;
}

// Sum of v over the 64 lanes of a wave (every lane active), in every lane.
__device__ __forceinline__ int wave_sum(int v) {
    return __builtin_amdgcn_readlane(wave_inclusive_scan(v), 63);
}

// Minimum of v over the 64 lanes of a wave (every lane active), in every
// lane: the row-shift and broadcast pattern of wave_inclusive_scan with min
// for sum, on both 32-bit halves; lanes with no source keep the identity
// (all ones).
__device__ __forceinline__ unsigned long long wave_min_u64(unsigned long long v) {
#define SEVC_MIN_STEP(ctrl, rows)                                                                        \
    {                                                                                                    \
        const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(-1, (int)(unsigned)v, ctrl, rows, 0xf, false);  \
        const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(-1, (int)(unsigned)(v >> 32), ctrl, rows, 0xf, false); \
        const unsigned long long s = ((unsigned long long)hi << 32) | lo;                                \
        v = s < v ? s : v;                                                                               \
    }
    SEVC_MIN_STEP(0x111, 0xf)   // row_shr:1
    SEVC_MIN_STEP(0x112, 0xf)   // row_shr:2
    SEVC_MIN_STEP(0x114, 0xf)   // row_shr:4
    SEVC_MIN_STEP(0x118, 0xf)   // row_shr:8
    SEVC_MIN_STEP(0x142, 0xa)   // row_bcast:15 into rows 1, 3
    SEVC_MIN_STEP(0x143, 0xc)   // row_bcast:31 into rows 2, 3
#undef SEVC_MIN_STEP
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)v, 63);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(v >> 32), 63);
    return ((unsigned long long)hi << 32) | lo;
}

// Block lb of one of the three entity tables.  A single member's table is
// runs of kBlock consecutive slots from 0, so its bounds are computed: the
// block's own loads then need not wait for a table load.
__device__ __forceinline__ Blk table_blk(const Dev& d, const Blk* tbl, int lb) {
    if (d.B == 1 && (tbl == d.vblk || tbl == d.eblk || tbl == d.gblk)) {
        const int total = tbl == d.vblk ? d.V : (tbl == d.eblk ? d.E : d.G);
        const int b = lb * kBlock;
        return Blk{0, b, min(b + kBlock, total)};
    }
    return tbl[lb];
}

#define TABLE_BLOCK(tbl, nblk)                                   \
    int lb_ = xcd_remap((int)blockIdx.x, (int)gridDim.x);        \
    if (lb_ >= (nblk)) return;                                   \
    const Blk bd_ = table_blk(d, (tbl), lb_);                    \
    const Params& P = d.prm[bd_.m];                              \
    MState& M = d.ms[bd_.m];                                     \
    (void)P; (void)M;                                            \
    const int i = bd_.b + (int)threadIdx.x;

// Analytic -grad E at vertex v (extension; the adjoint differentiates
// exactly this): edges contribute -gamma_b wrap(p_v - p_nb)/L_b, grains
// -SE_g sign(A_g) dA_g/dp_v with dA/dx_k = (dy_prev + dy_next)/2 and
// dA/dy_k = -(dx_prev + dx_next)/2, d_prev = wrap(p_k - p_{k-1}),
// d_next = wrap(p_{k+1} - p_k).  Positions X, grain areas A.
__device__ __forceinline__ void analytic_force_at(const Dev& d, const double* X, const double* A, const Params& P,
                                                  int v, double* fx, double* fy) {
    const double D = P.D;
    double x = X[2 * v], y = X[2 * v + 1];
    double ex = 0.0, ey = 0.0, gx = 0.0, gy = 0.0;
    for (int j = 0; j < 3; j++) {
        int b = d.vb[3 * v + j];
        int nb = other_end(d, b, v);
        double dx = wrapd(x, X[2 * nb], D), dy = wrapd(y, X[2 * nb + 1], D);
        double L = mag(dx, dy);
        if (L > 0) {
            ex += d.ben[b] * (dx / L);
            ey += d.ben[b] * (dy / L);
        }
    }
    for (int j = 0; j < 3; j++) {
        int g = d.vg[3 * v + j];
        int n = d.glen[g];
        int k = grain_contains_vertex(d, g, v);
        if (k < 0 || n < 3) continue;
        const int* L = glist(d, g);
        int wp = L[(k + n - 1) % n], wn = L[(k + 1) % n];
        double dpx = wrapd(x, X[2 * wp], D), dpy = wrapd(y, X[2 * wp + 1], D);
        double dnx = wrapd(X[2 * wn], x, D), dny = wrapd(X[2 * wn + 1], y, D);
        double sg = A[g] < 0 ? -1.0 : 1.0;
        double c = d.gse[g] * sg * 0.5;
        gx += c * (dpy + dny);
        gy += c * (-(dpx + dnx));
    }
    *fx = -(ex + gx);
    *fy = -(ey + gy);
}

}  // namespace sevc
