// kernels.h -- host-callable launchers for the HIP kernels in kernels.hip.
#pragma once
#include <hip/hip_runtime.h>

#include "convert.h"
#include "movegen.h"

namespace pf {

// Device view of the slider tables (pointers into one device blob).
struct DevTables {
    const SliderTables* t;
};

// One breadth-first level: parents `in[0..n_in)` with their root ids.
struct LevelArgs {
    const Board* in;
    const u32* in_root;
    u32 n_in;
    Board* out;          // children (expand-and-write mode only)
    u32* out_root;
    u64 out_cap;         // capacity of out / out_root in nodes
    u32* out_count;      // device bump counter for out
    unsigned long long* root_sums;  // per-root accumulators (nullptr: skip)
    unsigned long long* total;      // sum over all children (nullptr: skip)
    u32* tile_ctr;       // persistent tile queue counter (zero before launch)
    u32* err;            // set non-zero on capacity overflow
    u32 tile_parents;    // parents per tile, at most the shape's (0: the shape's); a small level
                         // uses fewer, so that it spreads over more workgroups
    bool uncounted = false;  // the children's moves are not counted (no total, no root_sums)
};

// Parents per tile for a level of n parents on `grid` workgroups of a shape
// with at most tp_max parents per tile: enough tiles for every workgroup, but
// at least four parents (about 120 children, two waves of them) each.  With
// fewer, a tile takes as long and a small level has more of them to add to the
// level's counters, some 9 ns each: one root at perft 4 49 -> 41 us, 32 roots
// 78 -> 65 (eight parents: 43 and 70).
PF_HD u32 level_tile_parents(u64 n, u64 grid, u32 tp_max) {
    const u64 g = grid ? grid : 1, t = (n + g - 1) / g;
    return (u32)(t < 4 ? 4 : t > tp_max ? tp_max : t);
}

// A leaf level runs by sets (leaf.h) from this many parents per workgroup.
constexpr u32 kLeafSetsMinParents = 32;
constexpr u32 kLeafSetsTile = 256;  // its parents per tile

enum ExpandMode : int { kLeaf = 0, kWrite = 1 };

// Occupancy-derived grid size for the expand kernel (workgroups); small = 1
// for the shape the level loop uses on small levels.
int expand_grid(int backend, int mode, int small, int n_cu);

hipError_t launch_init_roots(int backend, const DevTables& dt, Board* roots, u32 n,
                             unsigned long long* root_sums, hipStream_t s);
hipError_t launch_expand(int backend, int mode, int small, const DevTables& dt, const LevelArgs& a,
                         int grid, hipStream_t s);
hipError_t launch_range_count(const Board* b, u32 n, unsigned long long* out, hipStream_t s);
// Roots already in device memory (reference layout) -> boards + root ids.
hipError_t launch_pos_to_board(const pf_pos48* in, u32 n, Board* out, u32* rid, hipStream_t s);

// Whole-batch breadth-first perft in one cooperative launch (grid barrier
// between levels).  Levels 1..depth-2 are bump-allocated in `arena`.
struct PersistCtl {
    u32 tile_ctr[20];
    u32 out_count[20];
    u32 err;
    u32 pad[3];
    unsigned long long totals[20];  // totals[L] = number of nodes of level L
    unsigned long long lvl_off[20];  // stream-ordered form: arena offset of level L
    unsigned long long t0;           // stream-ordered form, small batches: device clock at its begin kernel
};
struct PersistArgs {
    Board* roots;
    u32* root_ids;
    u32 n_roots;
    int depth;
    char* arena;
    u64 arena_bytes;
    PersistCtl* ctl;
    unsigned long long* sums;
    u32 leaf_grid = 0;  // stream-ordered form: workgroups of a leaf level that runs by sets
};
// Tile-shape variants of the persistent kernel (kernels.hip, PCfg) and the
// most workgroups per CU that can be resident for one of them.
constexpr int kPersistVariants = 3;
int persistent_max_bpc(int backend, int variant);
hipError_t launch_persistent(int backend, int variant, const DevTables& dt, const PersistArgs& a, int grid,
                             hipStream_t s);
// The same batch as one launch per level on stream s (levels sized and placed
// on the device; no host round trip): the root count, then depth - 1 level
// launches of grid[kWrite] / grid[kLeaf] workgroups of the level kernel's
// form variant[kWrite] / variant[kLeaf].  Write levels have two forms, the leaf
// level one, by sets; both have one more for the byte backend.  (The numbers
// are those of tune files.)
constexpr int kStreamWrite8192 = 0;      // 256 parents x 8192 moves a tile
constexpr int kStreamWrite4096 = 3;      // 256 x 4096
constexpr int kStreamByteLds = 6;        // byte backend only: its tables staged in LDS (both modes)
constexpr int kStreamLeafSets = 7;       // leaf level by sets (leaf.h); below kLeafSetsMinParents move by move
constexpr int kStreamWriteDefault = kStreamWrite4096;
int stream_grid(int backend, int mode, int variant, int n_cu);
hipError_t launch_stream(int backend, const DevTables& dt, const PersistArgs& a, const int grid[2],
                         const int variant[2], hipStream_t s);

// A batch of at most kStreamSmall roots: `pos` (reference layout; coherent
// host or device memory) is converted, counted and its control block cleared
// by one launch of one workgroup in front of the levels (depth >= 1), and its
// outcome posted to the host's StreamIO by one behind them, in place of three
// clears, two or three copies and their waits.  One position (whose levels
// the host sized one by one before) at depth 3 133 -> 35 us and at depth 5 230
// -> 81, a divide at depth 5 159 -> 87, 37 positions at perft 4 179 -> 104, 100
// in device memory 141 -> 128.  1024 is one workgroup's threads: the begin of
// more roots would wait on passes of a single CU.
constexpr u32 kStreamSmall = 1024;
struct StreamIO {  // coherent host memory
    u32 done;      // the call's number, written after the rest
    u32 err;       // PersistCtl::err
    unsigned long long t0, t1;  // device clock at the begin and the post kernel
    unsigned long long used;    // arena bytes of the levels written
    unsigned long long sums[kStreamSmall];
    pf_pos48 pos[kStreamSmall];
};
// The levels as above, behind the begin kernel.
hipError_t launch_stream_small(int backend, const DevTables& dt, const PersistArgs& a, const pf_pos48* pos,
                               const int grid[2], const int variant[2], hipStream_t s);
// The sums to dev_out (null: io->sums; a.sums: they are there), then the rest
// of *io, then io->done = seq.
hipError_t launch_stream_post(const PersistArgs& a, unsigned long long* dev_out, StreamIO* io, u32 seq, hipStream_t s);

}  // namespace pf
