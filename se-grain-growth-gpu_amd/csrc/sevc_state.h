// sevc_state.h -- device state of a (batched) vertex-model simulation.
//
// All members of a batch live in one set of structure-of-arrays buffers;
// topology indices are global slot ids (member offset added at upload), so
// every per-entity kernel covers all members in one launch.  Per-member
// parameters and loop state are small device arrays read once per
// workgroup through the block tables.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sevc {

constexpr int kBlock = 256;          // elements per table block (one workgroup)
constexpr int kFixStages = 3;        // 0: two-grain, 1: T2 removal, 2: flips
constexpr int kTile = 64;            // grains per velocity tile (pass 1)
constexpr int kMaxHistBins = 64;     // bins of the device area histogram
constexpr int kNuclThreads = 1024;   // workgroup of the nucleation manager (one per member)
constexpr int kPollFast = 2048;      // candidate lists up to this length poll with registers and LDS (two per lane)
constexpr int kPollBig = 16384;      // lists up to this length poll with flags and t_ext in LDS
// A step that lists more edges than kBusyOver makes the state busy, one that
// lists fewer than kBusyUnder makes it calm (end_lists): a calm state's events
// run in one workgroup (k_events), a busy one's in a launch per stage.  The
// edges of all members count together, as one workgroup runs them all.  The line
// lies where both cost the same, which is near kEvMax at every size, in batches
// and for flips, removals and nucleations alike: past it the one workgroup runs
// the launches' stages.  A step, one workgroup / a launch per stage, in us:
//     listed edges                      80-95     125-145   153-176   190-205   215-245
//     2,000 grains, flips              94 / 104  109 / 112 111 / 111 135 / 116 162 / 118
//     20,000, flips                   101 / 114  121 / 124           170 / 126
//     250,000, flips                  157 / 173            183 / 176           258 / 183
//     1,000,000, flips                336 / 354  350 / 362 353 / 357
//     400,000 to 500,000, nucleations            243 / 266 271 / 264 282 / 268 328 / 285
//     8 of 2,000, flips                          113 / 116 117 / 115 165 / 119 180 / 125
//     32 of 2,000, nucleations        157 / 183  177 / 192
constexpr int kEvMax = 192;          // longest candidate list that k_events runs in LDS
constexpr int kEvThreads = 512;     // workgroup of k_events
constexpr int kHeadGrains = 8192;    // largest member whose candidates k_head draws itself
constexpr int kHeadEvents = 8;       // most nucleations a member may expect for k_head to apply them itself
constexpr int kBusyOver = 180, kBusyUnder = 150;
constexpr int kCountWaves = 4;       // table blocks per workgroup of k_count_all (one wave each)

// What k_head does besides the nucleation's selection.
enum { HEAD_BEGIN = 1, HEAD_SELECT = 2, HEAD_DRAW = 4, HEAD_INSERT = 8, HEAD_RESCALE = 16 };

// Per-member run parameters (from sevc_options).
struct Params {
    double D, dt_max, dt_min, dt_safety, flip_thr, mobility;
    double gb_eps, gb_scaling, mc_k, nucl_rate, nucl_scaling, tmax;
    unsigned long long seed;
    int nmax, adaptive, nucl_mode, do_nucl, gap, events, vel_model, min_grains, n_grains0;
    int gate_grains;                 // MC nucleation opens once enabled grains <= this (5 n_grains0 / 6)
    int debug;                       // debug_lvl: >= 1 runs the checks of check_data inside the step
    int cap;                         // max_vrt_per_grn of this member (lists are stored at the batch's stride S >= cap)
    int voff, nv, eoff, ne, goff, ng;
};

// Per-member loop state (main.cu:30-113), updated on the device.
struct MState {
    int n, active, done, curr_grains, allow_nucl, nucl_now, status, n_venabled;
    int chk_phase;                   // phase of a failed check (debug_lvl >= 1), else 0
    int open;                        // a step has begun and is not yet summed up (end_member)
    double t, dt;
    unsigned long long tau_bits;     // min positive t_ext (as ordered bits)
    long long flips, removals, two, nucl, vsteps, steps;
    double nucl_area_pct;
    double lab_dt;                   // dt of the last step that labelled this member's edges
};

// A workgroup's range of one member's entities: [b, e).
struct Blk { int m, b, e; };

enum Counter {
    C_CAND = 0, C_TWO, C_T2, C_T2C, C_FLIPC,
    C_FIX0, C_FIX1, C_FIX2, C_DIRTY, C_CONF, C_VFALL, C_BIGR, C_RAN,
    C_COUNT,                          // the counters above are cleared when the next step begins
    C_NUCL = C_COUNT,                 // these once they have been read:
    C_NEV, C_TRI,
    C_TOTAL
};

enum { FIX_ADD = 0, FIX_REMOVE = 1, FIX_REPLACE = 2, FIX_NONE = 3 };   // geometry.h:17

// A vertex's four deferred grain-list edits (mod_t, geometry.h:26-31), in
// one 64-byte record so that reading or clearing them touches one line.
struct alignas(64) ModRec {
    int grn[4], vrt[4], prev[4];
    uint8_t fix[4];
};
static_assert(sizeof(ModRec) == 64, "one line per vertex");

struct Dev {
    // vertices
    double* pos; double* vel; int* vb; int* vg; uint8_t* ven;
    double* venergy; double* vparts;
    ModRec* mods;                        // deferred grain-list edits, one 64-B record per vertex
    double* nucl_r; double* nucl_ori; double* dE; double* nfac; uint8_t* vnuc;
    // boundaries
    int* bvx; double* ben; double* blen; double* bt; uint8_t* benab; uint8_t* bcand; int* conf;
    int* pgat; double* pgt;          // polling gathers: 25 columns of kPollBig, t_ext
    uint8_t* blab;                  // per edge: bit 0 candidate (enabled), bit 1 enabled when labelled, bit 2 label after polling
    int* l_flipped; int* n_flipped;  // edges flipped since the last step start (energies to rescale)
    int* vmem; int* emem; int* gmem;  // owning member of each vertex / edge / grain slot (batches)
    // grains
    int* gvx; int* glen; double* garea; double* gdadt; double* gori; double* gse;
    uint8_t* genab; uint8_t* gtype; uint8_t* gcand; int* gfix;
    int S;
    int V, E, G;                          // total slots over members
    // members
    const Params* prm; MState* ms; int B;
    const Blk* vblk; const Blk* eblk; const Blk* gblk;
    int nvb, neb, ngb;
    const Blk* gtile; int ntile;         // tiles of tile_T consecutive grains of one member (velocity pass 1)
    int tile_T;
    const Blk* vtile; int nvtile;        // vertex tiles of the one-pass velocity
    double* vterm;                       // 6 per vertex: stored-energy terms (x,y) per grain slot
    int4* slist;                         // free-slot search: (kind, block, rank) lists, ngb+neb+nvb entries
    int* vblk_first; int* eblk_first; int* gblk_first;   // first table block of each member (B+1)
    // work lists and scratch
    int* cnt;
    int* l_cand; int* l_two; int* l_t2; int* l_t2c; int* l_flipc;
    int* l_fix[kFixStages]; int* l_dirty; int* l_nucl; int* l_conf; int* l_vfall;
    int4* c_id; double2* c_te;            // the first kEvMax listed edges: (edge, its ends, member), (t_ext, length)
    int* l_tri;                           // grains that an edit left with three vertices (next two-triangle search)
    int* l_bigr;                          // grains longer than the lane-per-grain velocity pass holds
    int* nrec; double* nal;               // rate-mode candidate sites: (site or -1, its 3 grains), shortest edge
    int* l_nev;                           // nucleation events of the step: (member, A, B, C, AB, BC, CA, g)
    int2* bc_v; int2* bc_e; int2* bc_g;   // per table block: (enabled, free) slot counts
    double* partial;                      // per grain block partial sums (2 levels)
    int* nscr;                            // nucleation scratch, 12 ints per grain slot
    int diag;                             // compute export diagnostics this step
    int debug;                            // a member runs the checks of check_data (debug_lvl >= 1)
    int* chk_bad;                         // violations per member found by the last check
    int poll_fast;                        // longest candidate list polled from registers (<= kPollFast)
    int poll_lds;                         // longest candidate list polled from LDS (<= kPollBig)
    int* busy;                            // 1: many edges listed per step (device copy of *busy_host)
    int* busy_host;                       // the same in pinned host memory, written when it changes
    int quiet;                            // the step's list does not change the word
    int free_rows;                        // blocks per kind of one free-slot search round (0: the default)
};

// The grains of each vertex table block and their lists, for the steps of a
// topology-fixed window (sevc_adjoint.hip); null without.
constexpr int kWinBlockGrains = 3 * kBlock;
struct WinBlocks {
    int* loc;
    int* count;
    int2* grain;
    int4* list;
};

// One array of a mesh download (k_pack): n items of `src` go to byte `dst` of
// the staging buffer.  PACK_RAW copies n 4-byte words, PACK_BYTE n bytes,
// PACK_ID n ids (off taken from those >= 0); PACK_ROW takes the first `row`
// ids of each `stride` of src, n ids in all.
enum { PACK_RAW = 0, PACK_BYTE, PACK_ID, PACK_ROW };
struct PackSeg {
    const void* src;
    unsigned long long dst, n;
    int kind, off, row, stride;
};
constexpr int kPackSegs = 24;
struct PackList {
    PackSeg seg[kPackSegs];
    int n;
};

// The arrays of a checkpoint or a restore (k_copy_arrays): n bytes from src to
// dst, both 16-byte aligned, by the workgroups from `first` on.
struct CopySeg {
    const char* src;
    char* dst;
    unsigned long long n;
    int first;
};
constexpr int kCopySegs = 48, kCopyChunk = 16384;     // bytes per workgroup
struct CopyList {
    CopySeg seg[kCopySegs];
    int n;
    int* word;                           // set to `value` besides (null: none)
    int value;
};

}  // namespace sevc
