// gen_dev.h -- the moves of a few parents by a whole workgroup.
#pragma once
#include <hip/hip_runtime.h>

#include "movegen.h"
#include "wave.h"

namespace pf {

// A tile of at most this many parents generates its moves with the whole
// workgroup.  A small level waits on one tile's chain of dependent steps, and
// one lane walking through its parent's pieces was half of it (4.3 of a write
// level's 8.7 us).  One position at depth 3 35.6 -> 33.8 us, 37 positions at
// perft 4 97 -> 91, 100 positions 126 -> 119.  The table's tiles, whose kernels
// have no registers left for it, keep a lane per parent: one served request at
// depth 4 went from 95 to 100 us with it.
constexpr u32 kCoopParents = 8;

// The moves of the np <= kCoopParents parents `b`, tagged with the parent << 16,
// into list[off[parent] ..): 32 lanes a parent with two squares each, or 64
// with one, each generating the moves of the pieces there.  Every thread of
// the workgroup calls it, with the arrays stored and a barrier behind them.
template <int WG, int CAP, class SL>
__device__ __forceinline__ void coop_generate(const SL& sl, const Board* boards, const u32* off, const u32 np,
                                              u32* list) {
    static_assert(CAP >= (int)kCoopParents * 218, "their moves fit the list");
    static_assert(WG == 256, "32 threads for each of kCoopParents parents");
    const u32 tid = threadIdx.x, lane = tid & 63;
    const bool wide = np <= kCoopParents / 2;
    const u32 par = wide ? tid >> 6 : tid >> 5;
    const u64 who = wide ? bit((int)lane) : 0x100000001ULL << (tid & 31);
    const bool work = par < np;
    Board b = {};
    PosInfo pi = {};
    EmitCount n{0};
    if (work) {
        b = boards[par];
        analyse(b, sl, pi);
        generate(b, sl, pi, n, who);
    }
    const u32 incl = wave_incl_scan(n.n);
    const u32 low = (u32)__builtin_amdgcn_readlane((int)incl, 31);  // of the lower half's parent
    if (n.n) {
        struct Store {
            u32* list;
            u32 at, tag;
            __device__ __forceinline__ void operator()(u32 m) {
                if (at < (u32)CAP) list[at] = m | tag;
                at++;
            }
        } e{list, off[par] + incl - n.n - (!wide && lane >= 32 ? low : 0u), par << 16};
        generate(b, sl, pi, e, who);
    }
}

}  // namespace pf
