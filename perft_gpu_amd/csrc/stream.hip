// stream.hip -- the batch as a sequence of launches on one stream, one per
// level (PF_MODE_STREAM, and PF_MODE_AUTO's table-free single pass).
//
// The levels are sized and placed on the device exactly as in k_persistent
// (the totals and level offsets live in PersistCtl), so nothing returns to
// the host between levels, and the launch boundary replaces the grid barrier
// (the reference syncs the device after every level, perft_bb.h:1071-1135).
// Every workgroup of a level launch derives the same placement from words
// the previous launch finished writing.
//
// The write kernel is built in two forms, a move window of 8192 and one of
// 4096, of which the autotuner picks one per backend (the reference fixes its
// launch shape at compile time, perft_bb.h:327-329, switches.h:14-21).  Their
// LDS and registers (124 VGPRs) hold them at three and four workgroups per CU;
// asked for four or five waves per SIMD the first compiles to the same
// instructions, the second for four too, and for five (96 VGPRs) it spills.
// The leaf level runs by sets (leaf.h).
//
// The leaf level's kernels are built for three waves per SIMD, the most that
// needs no spills (tests/test_no_spills.py).  Built for four (128 VGPRs, 36 B
// of spills per lane, record pools and move list cut so that four workgroups
// fit a CU) 256 positions at perft 5 take 2.61 ms instead of 2.53, with equal
// sums: 40 batches of all backends, eight runs each.
#include <hip/hip_runtime.h>

#include "convert.h"
#include "level_dev.h"

namespace pf {

template <int B>
__global__ __launch_bounds__(kWG) void k_stream_roots(const SliderTables* tabs, PersistArgs p) {
    const auto sl = SlOf<B>::make(tabs);
    const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
    unsigned long long c = 0;
    if (i < p.n_roots) {
        const Board b = p.roots[i];
        c = count_moves(b, sl);
        p.roots[i] = with_count(b, (u32)c);
        if (p.depth == 1) p.sums[p.root_ids[i]] = c;
    }
    c = wave_sum64(c);
    if ((threadIdx.x & 63) == 0 && c) atomicAdd(&p.ctl->totals[1], c);
}

// Begin of a small batch: one workgroup of a thread per root.
template <int B>
__global__ __launch_bounds__(kStreamSmall) void k_stream_begin(const SliderTables* tabs, PersistArgs p,
                                                               const pf_pos48* __restrict__ pos) {
    __shared__ unsigned long long red[kStreamSmall / 64];
    constexpr u32 kWords = sizeof(PersistCtl) / 4;
    const u32 i = threadIdx.x;
    const unsigned long long t0 = wall_clock64();
    unsigned long long c = 0;
    if (i < p.n_roots) {
        const Board b = to_board(pos[i]);
        c = count_moves(b, SlOf<B>::make(tabs));
        p.roots[i] = with_count(b, (u32)c);
        p.root_ids[i] = i;
        p.sums[i] = p.depth == 1 ? c : 0;
    }
    for (u32 w = i; w < kWords; w += blockDim.x) reinterpret_cast<u32*>(p.ctl)[w] = 0;
    c = wave_sum64(c);
    if ((i & 63) == 0) red[i >> 6] = c;
    __syncthreads();  // (the words are cleared before two of them are set)
    if (i == 0) {
        unsigned long long t = 0;
        for (u32 w = 0; w < blockDim.x / 64; w++) t += red[w];
        p.ctl->totals[1] = t;
        p.ctl->t0 = t0;
    }
}

// Arena bytes of a level of n nodes: its boards, then its root ids.
__device__ __forceinline__ u64 level_bytes(u64 n) {
    return ((n * sizeof(Board) + 255) & ~255ULL) + ((n * sizeof(u32) + 255) & ~255ULL);
}

__global__ __launch_bounds__(kWG) void k_stream_post(const PersistCtl* ctl, int depth, const unsigned long long* sums,
                                                     u32 n, unsigned long long* out, StreamIO* io, u32 seq) {
    if (threadIdx.x == 0) {
        const int L = depth > 2 ? depth - 2 : 0;  // the last level written, behind the roots
        // (all read before the first is written)
        const u32 err = ctl->err;
        const unsigned long long t0 = ctl->t0, off = ctl->lvl_off[L], nodes = ctl->totals[L];
        io->err = err;
        io->t0 = t0;
        io->used = L ? off + level_bytes(nodes) : 0;
        io->t1 = wall_clock64();
    }
    for (u32 i = threadIdx.x; i < n; i += blockDim.x) out[i] = sums[i];
    __threadfence_system();  // this thread's writes reach the host before the barrier ...
    __syncthreads();
    if (threadIdx.x == 0)    // ... and so before done
        __hip_atomic_store(&io->done, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// One level for one workgroup of the launch.  `make_sl` builds the slider
// backend once the workgroup knows it has work (the byte backend's LDS form
// copies its tables into LDS there).
template <int MODE, bool SETS, int TP, int CAP, int WG, class MakeSl>
__device__ __forceinline__ void stream_level(const MakeSl& make_sl, const PersistArgs& p, int L,
                                             TileLds<TP, CAP, WG>& s, LeafLevelLds* sets) {
    PersistCtl* ctl = p.ctl;
    // What the previous launches left, read in one go: a small level waits on
    // each of these reads.
    const u64 nl = ctl->totals[L], lo = ctl->lvl_off[L], nn = ctl->totals[L + 1];
    // an earlier level did not fit: nothing below it is counted (one read per
    // workgroup, so that the whole workgroup leaves together)
    if (threadIdx.x == 0) s.ok = ctl->err;
    __syncthreads();
    if (s.ok) return;
    const Board* cur = p.roots;
    const u32* cur_r = p.root_ids;
    u64 n = p.n_roots, off = 0;
    if (L > 0) {
        n = nl;
        off = lo;
        cur = reinterpret_cast<const Board*>(p.arena + off);
        cur_r = reinterpret_cast<const u32*>(p.arena + off + ((n * sizeof(Board) + 255) & ~255ULL));
        off += level_bytes(n);
    }
    LevelArgs a;
    a.in = cur;
    a.in_root = cur_r;
    a.n_in = (u32)n;
    a.tile_ctr = &ctl->tile_ctr[L];
    a.err = &ctl->err;
    a.out_count = &ctl->out_count[L];
    a.tile_parents = level_tile_parents(n, gridDim.x, TP);
    // workgroups past the level's tile count leave at once (block 0 stays:
    // it places the next level); the others drain the tile queue
    const u64 ntiles = (n + a.tile_parents - 1) / a.tile_parents;
    if (MODE == kLeaf) {
        if (blockIdx.x >= ntiles) return;
        const auto sl = make_sl();
        a.out = nullptr;
        a.out_root = nullptr;
        a.out_cap = 0;
        a.root_sums = p.sums;
        a.total = nullptr;
        if constexpr (SETS) {
            if (a.tile_parents >= kLeafSetsMinParents) {
                leaf_level(sl, a, *sets);
                return;
            }
        }
        expand_level(sl, a, kLeaf, s);
        return;
    }
    const u64 bbytes = (nn * sizeof(Board) + 255) & ~255ULL, rbytes = (nn * sizeof(u32) + 255) & ~255ULL;
    if (nn > 0xFFFFFFFFull || off + bbytes + rbytes > p.arena_bytes) {
        if (blockIdx.x == 0 && threadIdx.x == 0) atomicOr(&ctl->err, 2u);
        return;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) ctl->lvl_off[L + 1] = off;
    if (blockIdx.x > 0 && blockIdx.x >= ntiles) return;
    const auto sl = make_sl();
    a.out = reinterpret_cast<Board*>(p.arena + off);
    a.out_root = reinterpret_cast<u32*>(p.arena + off + bbytes);
    a.out_cap = nn;
    a.root_sums = nullptr;
    a.total = &ctl->totals[L + 2];
    // A leaf level by sets needs no move counts of its parents, so the last write
    // level leaves them out.  Its 8.2 million children of 256 positions at perft 5
    // take 136 us instead of 264 (52 B each written: 3.1 TB/s), 24.6 million of
    // 701 positions with the fancy backend 331 instead of 869.
    if (L == p.depth - 3 && p.leaf_grid &&
        level_tile_parents(nn, p.leaf_grid, kLeafSetsTile) >= kLeafSetsMinParents) {
        a.uncounted = true;
        a.total = nullptr;
    }
    expand_level(sl, a, kWrite, s);
}

template <int B, int V>
__global__ __launch_bounds__(kWG) void k_stream_write(const SliderTables* tabs, PersistArgs p, int L) {
    using Shape = PCfg<B, V>;
    __shared__ TileLds<Shape::TP, Shape::CAP, kWG> s;
    stream_level<kWrite, false>([&] { return SlOf<B>::make(tabs); }, p, L, s, nullptr);
}

// The byte backend's LDS form (level_dev.h): one 768-thread workgroup per CU,
// tables staged in its LDS.
template <int MODE>
__global__ __launch_bounds__(kByteLdsWG) void k_stream_level_byte_lds(const SliderTables* tabs, PersistArgs p, int L) {
    extern __shared__ __align__(16) unsigned char dyn_lds[];
    __shared__ TileLds<kByteLdsTP, kByteLdsCap, kByteLdsWG> s;
    stream_level<MODE, false>([&] { return stage_byte_tables(tabs, dyn_lds); }, p, L, s, nullptr);
}

// The leaf level by sets; a level too small for it runs move by move.
template <int B>
__global__ __launch_bounds__(kWG) __attribute__((amdgpu_waves_per_eu(kLeafSetsWaves)))
void k_stream_leaf(const SliderTables* tabs, PersistArgs p, int L) {
    __shared__ union {
        TileLds<256, 4096, kWG> tile;
        LeafLevelLds sets;
    } s;
    static_assert(kLeafSetsTile == 256, "as many as the other form's");
    stream_level<kLeaf, true>([&] { return SlOf<B>::make(tabs); }, p, L, s.tile, &s.sets);
}

// ---- launch plumbing --------------------------------------------------------
template <int B>
static void* level_fn(int mode, int v) {
    if (mode == kLeaf) return reinterpret_cast<void*>(&k_stream_leaf<B>);
    return v == kStreamWrite8192 ? reinterpret_cast<void*>(&k_stream_write<B, 0>)
                                 : reinterpret_cast<void*>(&k_stream_write<B, 2>);
}
static void* pick_stream_level(int backend, int mode, int v) {
    if (backend == kByte && v == kStreamByteLds)
        return mode == kWrite ? reinterpret_cast<void*>(&k_stream_level_byte_lds<kWrite>)
                              : reinterpret_cast<void*>(&k_stream_level_byte_lds<kLeaf>);
    switch (backend) {
    case kKS: return level_fn<kKS>(mode, v);
    case kPlain: return level_fn<kPlain>(mode, v);
    case kFancy: return level_fn<kFancy>(mode, v);
    default: return level_fn<kByte>(mode, v);
    }
}
static void* pick_stream_roots(int backend) {
    switch (backend) {
    case kKS: return reinterpret_cast<void*>(&k_stream_roots<kKS>);
    case kPlain: return reinterpret_cast<void*>(&k_stream_roots<kPlain>);
    case kFancy: return reinterpret_cast<void*>(&k_stream_roots<kFancy>);
    default: return reinterpret_cast<void*>(&k_stream_roots<kByte>);
    }
}

// Workgroup size and dynamic LDS of a level kernel form.
static int stream_wg(int backend, int variant) {
    return backend == kByte && variant == kStreamByteLds ? kByteLdsWG : kWG;
}
static size_t stream_dyn(int backend, int variant) {
    return backend == kByte && variant == kStreamByteLds ? kByteLds : 0;
}

int stream_grid(int backend, int mode, int variant, int n_cu) {
    return blocks_per_cu(pick_stream_level(backend, mode, variant), stream_wg(backend, variant),
                         stream_dyn(backend, variant)) * n_cu;
}

// Levels 0..depth-2.
static hipError_t launch_levels(int backend, const SliderTables* t, const PersistArgs& a, const int grid[2],
                                const int variant[2], hipStream_t s) {
    PersistArgs args = a;
    args.leaf_grid = variant[kLeaf] == kStreamByteLds && backend == kByte ? 0u : (u32)grid[kLeaf];
    for (int L = 0; L <= a.depth - 2; L++) {
        const int mode = (L == a.depth - 2) ? kLeaf : kWrite;
        void* kargs[] = {(void*)&t, (void*)&args, (void*)&L};
        // (a form with dynamic LDS had the attribute set when its grid was sized)
        void* f = pick_stream_level(backend, mode, variant[mode]);
        const size_t dyn = stream_dyn(backend, variant[mode]);
        const hipError_t e = hipLaunchKernel(f, dim3(grid[mode]), dim3(stream_wg(backend, variant[mode])), kargs,
                                             dyn, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_stream(int backend, const DevTables& dt, const PersistArgs& a, const int grid[2],
                         const int variant[2], hipStream_t s) {
    PersistArgs args = a;
    const SliderTables* t = dt.t;
    void* kargs[] = {(void*)&t, (void*)&args};
    const hipError_t e = hipLaunchKernel(pick_stream_roots(backend), dim3((a.n_roots + kWG - 1) / kWG), dim3(kWG),
                                         kargs, 0, s);
    return e != hipSuccess ? e : launch_levels(backend, t, a, grid, variant, s);
}

hipError_t launch_stream_small(int backend, const DevTables& dt, const PersistArgs& a, const pf_pos48* pos,
                               const int grid[2], const int variant[2], hipStream_t s) {
    if (a.n_roots > kStreamSmall) return hipErrorInvalidValue;
    const dim3 wg((a.n_roots + 63) / 64 * 64);
    switch (backend) {
    case kKS: hipLaunchKernelGGL(k_stream_begin<kKS>, dim3(1), wg, 0, s, dt.t, a, pos); break;
    case kPlain: hipLaunchKernelGGL(k_stream_begin<kPlain>, dim3(1), wg, 0, s, dt.t, a, pos); break;
    case kFancy: hipLaunchKernelGGL(k_stream_begin<kFancy>, dim3(1), wg, 0, s, dt.t, a, pos); break;
    default: hipLaunchKernelGGL(k_stream_begin<kByte>, dim3(1), wg, 0, s, dt.t, a, pos); break;
    }
    const hipError_t e = hipGetLastError();
    return e != hipSuccess ? e : launch_levels(backend, dt.t, a, grid, variant, s);
}

hipError_t launch_stream_post(const PersistArgs& a, unsigned long long* dev_out, StreamIO* io, u32 seq, hipStream_t s) {
    const u32 n = dev_out == a.sums ? 0u : a.n_roots;  // counts to move
    if (!dev_out && n > kStreamSmall) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_stream_post, dim3(1), dim3(n > 64 ? kWG : 64), 0, s, a.ctl, a.depth, a.sums, n,
                       dev_out ? dev_out : io->sums, io, seq);
    return hipGetLastError();
}

}  // namespace pf
