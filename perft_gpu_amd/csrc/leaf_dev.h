// leaf_dev.h -- the leaf level for one workgroup: perft 2 of a tile of
// parents held in LDS (leaf.h), shared by the table-free and table kernels.
#pragma once
#include <hip/hip_runtime.h>

#include "kernels.h"
#include "leaf.h"
#include "wave.h"

namespace pf {

// A value that is the same in all lanes, in a scalar register.
__device__ __forceinline__ u32 uniform(u32 x) { return __builtin_amdgcn_readfirstlane(x); }

// Records that a wave's 64 parents hand out: those of which the replies of
// the opponent's king are missing from the start, the others from the end.
template <int N>
struct LeafPool {
    u64 to[N];
    u16 meta[N];  // the record's meta | lane << kLeafMetaBits
};

template <int TP, int N, int CAP, int WG>
struct LeafLds {
    Board b[TP];
    u32 sum[TP];
    LeafPool<N> pool[WG / 64];
    u32 mv[CAP];  // move | parent << 16
    u32 wtot[WG / 64];
    u32 more[WG / 64];  // waves with calls left undone
};

// Collects a wave's records.  Every lane of the wave takes part in each call
// (with empty sets where it has none), so the fill counts are the same in all
// lanes and need no atomics.  A call that does not fit is left undone with
// all later ones; the next round skips the `done` ones.
template <int N>
struct LeafEmit {
    LeafPool<N>* pool;
    u32 tag;  // lane << kLeafMetaBits
    u32 nk, nf, call, done;
    bool more;  // calls were left undone
    __device__ __forceinline__ static u32 below(u64 m) {
        return __builtin_amdgcn_mbcnt_hi((u32)(m >> 32), __builtin_amdgcn_mbcnt_lo((u32)m, 0));
    }
    __device__ __forceinline__ void operator()(u64 k, u64 f, u32 meta) {
        const u64 mk = __ballot(k != 0), mf = __ballot(f != 0);
        if (!(mk | mf)) return;
        const u32 ck = uniform(nk), cf = uniform(nf);
        const u32 ek = ck + (u32)__popcll(mk), ef = cf + (u32)__popcll(mf);
        call++;
        if (call <= done) return;
        more = more || ek + ef > (u32)N;
        if (more) return;
        if (k) {
            u32 at = ck + below(mk);
            pool->to[at] = k;
            pin(at);  // (else meta's address is made from to's by a 64-bit multiply)
            pool->meta[at] = (u16)(meta | tag);
        }
        if (f) {
            u32 at = N - 1 - cf - below(mf);
            pool->to[at] = f;
            pin(at);
            pool->meta[at] = (u16)(meta | tag);
        }
        nk = ek;
        nf = ef;
        done = call;
    }
};

// Makes and counts the moves of the waves' records [r0, r1) (KING: only the
// replies of the opponent's king are counted), adding to the parents' sums.
// Ends with a barrier behind the last use of every LDS array; returns the
// number of moves.
template <bool KING, class SL, int TP, int N, int CAP, int WG>
__device__ __forceinline__ u32 leaf_records(const SL& sl, const u32 r0, const u32 r1, LeafLds<TP, N, CAP, WG>& s) {
    u32 tid = threadIdx.x;
    pin(tid);  // addresses made from it are made again here, not kept in registers through the tile
    const u32 lane = tid & 63, wid = uniform(tid >> 6);
    const LeafPool<N>& pool = s.pool[wid];
    u32 cnt = 0;
    for (u32 r = r0 + lane; r < r1; r += 64) {
        u32 q = r;
        pin(q);  // (as in LeafEmit)
        cnt += leaf_rec_moves(pool.to[r], pool.meta[q]);
    }
    const u32 incl = wave_incl_scan(cnt);
    if (lane == 63) s.wtot[wid] = incl;
    __syncthreads();
    u32 woff = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < WG / 64; w++) {
        const u32 t = uniform(s.wtot[w]);
        woff += (w < (int)wid) ? t : 0;
        tot += t;
    }
    for (u32 w0 = 0; w0 < tot; w0 += CAP) {
        u32 pos = woff + incl - cnt - w0;  // of the lane's next move, wrapping below the window
        for (u32 r = r0 + lane; r < r1; r += 64) {
            u32 q = r;
            pin(q);
            const u32 meta = pool.meta[q], tag = ((meta >> kLeafMetaBits) | (wid << 6)) << 16;
            LeafRecIter it{pool.to[r], meta, 0};
            while (!it.done()) {
                const u32 m = it.next();
                if (pos < (u32)CAP) s.mv[pos] = m | tag;
                pos++;
            }
        }
        __syncthreads();
        const u32 m = min((u32)CAP, tot - w0);
        for (u32 j = tid; j < m; j += WG) {
            const u32 x = s.mv[j], par = x >> 16;
            const Board& b = *reinterpret_cast<const Board*>(reinterpret_cast<const char*>(s.b) +
                                                             mul24(par, sizeof(Board)));
            const u32 c = KING ? leaf_king_replies(b, x & 0xFFFFu) : count_moves(make_move(b, x & 0xFFFFu), sl);
            atomicAdd(&s.sum[par], c);
        }
        __syncthreads();
    }
    __syncthreads();
    return tot;
}

// s.sum[i] = perft 2 of s.b[i] for i < np (np <= TP <= WG).  Every thread of
// the workgroup calls it, with the boards stored (empty ones from np on to
// the end of the last wave with parents) and a barrier behind them; it ends
// with a barrier.  `made` (when not null) grows by the parents' moves, summed
// over the threads.
template <class SL, int TP, int N, int CAP, int WG>
__device__ __forceinline__ void leaf_tile(const SL& sl, const u32 np, LeafLds<TP, N, CAP, WG>& s,
                                          u32* made = nullptr) {
    static_assert(TP == WG, "one parent per thread");
    static_assert(N >= 128, "one call of a whole wave fits");
    u32 tid = threadIdx.x;
    pin(tid);
    const u32 wid = uniform(tid >> 6);
    LeafEmit<N> e{&s.pool[wid], (tid & 63) << kLeafMetaBits, 0, 0, 0, 0, false};
    const bool work = (wid << 6) < np;  // of the wave
    bool again = false;
    do {
        e.nk = e.nf = e.call = 0;
        e.more = false;
        if (work) {
            u32 summed = 0;
            const u32 sum = leaf_sum(s.b[tid], sl, e, made ? &summed : nullptr);
            if (!again) {
                s.sum[tid] = sum;
                if (made) *made += summed;
            }
        }
        if ((tid & 63) == 0) s.more[wid] = e.more;
        const u32 full = leaf_records<false>(sl, N - e.nf, N, s);
        if (made && tid == 0) *made += full;
        // (read between barriers, so that no wave writes the next round's yet)
        u32 m = 0;
#pragma unroll
        for (int w = 0; w < WG / 64; w++) m |= s.more[w];
        again = uniform(m) != 0;
        leaf_records<true>(sl, 0, e.nk, s);
    } while (again);
}

}  // namespace pf
