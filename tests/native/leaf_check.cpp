// leaf_check.cpp -- TEST HARNESS ONLY (built by tests/test_leaf.py): the leaf
// sums of perft_gpu_amd/csrc/leaf.h on the CPU, against the same header set's
// move-by-move counts.  Not part of the product library.
#include <stdint.h>

#include "../../perft_gpu_amd/csrc/convert.h"
#include "../../perft_gpu_amd/csrc/leaf.h"

using namespace pf;

namespace {

const KSBackend sl{};

struct Sum {  // counts the records' moves
    const Board* b;
    uint64_t n = 0;
    int recs = 0, king = 0, full = 0, bad = 0;
    void one(u64 to, u32 meta, bool is_king) {
        if (!to) return;
        recs++;
        u32 k = 0;
        for (LeafRecIter it{to, meta, 0}; !it.done(); k++) {
            const u32 m = it.next();
            n += is_king ? leaf_king_replies(*b, m) : count_moves(make_move(*b, m), sl);
        }
        if (k != leaf_rec_moves(to, meta)) bad++;
        (is_king ? king : full) += (int)k;
    }
    void operator()(u64 k, u64 f, u32 meta) {
        one(k, meta, true);
        one(f, meta, false);
    }
};

uint64_t g_rng = 88172645463325252ULL;
u64 rnd() {
    g_rng ^= g_rng << 13;
    g_rng ^= g_rng >> 7;
    g_rng ^= g_rng << 17;
    return g_rng;
}

}  // namespace

extern "C" {

// perft 2 by sets; stats: records, moves whose king replies were counted,
// moves made and counted, records whose move number was wrong (and 1 if the
// moves summed and handed out are not all)
uint64_t lc_perft2(const pf_pos48* p, int* stats) {
    const Board b = to_board(*p);
    Sum e{&b};
    u32 summed = 0;
    const uint64_t s = leaf_sum(b, sl, e, &summed);
    if (summed + (u32)e.full != count_moves(b, sl)) e.bad++;
    if (stats) stats[0] = e.recs, stats[1] = e.king, stats[2] = e.full, stats[3] = e.bad;
    return s + e.n;
}

// perft 2 move by move
uint64_t lc_perft2_moves(const pf_pos48* p) {
    const Board b = to_board(*p);
    PosInfo pi;
    analyse(b, sl, pi);
    uint64_t s = 0;
    auto emit = [&](u32 m) { s += count_moves(make_move(b, m), sl); };
    generate(b, sl, pi, emit);
    return s;
}

// whether the side to move could capture the other side's king, or a castling
// right stands without its king and rook at home: the replies are then no
// chess moves, and host and GPU counts of them need not agree
int lc_unsound(const pf_pos48* p) {
    const Board b = to_board(*p);
    const int r = st_rights(b);
    auto home = [&](int king, int rook, u64 side) { return (b.kings & side & bit(king)) && (b.rooks & ~b.bishops & side & bit(rook)); };
    const u64 them0 = occupancy(b) & ~b.us;
    if (((r & 1) && !home(4, 7, b.us)) || ((r & 2) && !home(4, 0, b.us)) || ((r & 4) && !home(60, 63, them0)) ||
        ((r & 8) && !home(60, 56, them0)))
        return 1;
    PosInfo pi;
    analyse(b, sl, pi);
    const u64 them = pi.them, att = rook_fill(b.rooks & pi.us, ~pi.occ) | bishop_fill(b.bishops & pi.us, ~pi.occ) |
                                    knight_fill(b.knights & pi.us) | king_fill(pi.K) | pawn_hits(pi.pawns & pi.us);
    return (att & b.kings & them) != 0;
}

// n positions of randomly placed pieces (one king a side), most of them
// unreachable: adjacent kings, either side in check, many queens
void lc_random(uint64_t seed, int n, pf_pos48* out) {
    g_rng = seed * 0x9E3779B97F4A7C15ULL + 1;
    for (int i = 0; i < n; i++) {
        Board b{};
        u64 used = 0;
        auto put = [&](u64 mask) {
            for (;;) {
                const u64 x = bit((int)(rnd() & 63)) & mask;
                if (x && !(x & used)) { used |= x; return x; }
            }
        };
        auto own = [&](u64 x) { if (rnd() & 1) b.us |= x; };
        const u64 k = put(~0ULL);
        b.us = k;
        b.kings = k | put(~0ULL);
        const int np = (int)(rnd() % 12), nn = (int)(rnd() % 5), nb = (int)(rnd() % 5), nr = (int)(rnd() % 5);
        const int nq = (int)(rnd() % ((rnd() % 8) ? 3 : 12));
        for (int j = 0; j < np; j++) { const u64 x = put(kRanks2to7); b.pawns |= x; own(x); }
        for (int j = 0; j < nn; j++) { const u64 x = put(~0ULL); b.knights |= x; own(x); }
        for (int j = 0; j < nb; j++) { const u64 x = put(~0ULL); b.bishops |= x; own(x); }
        for (int j = 0; j < nr; j++) { const u64 x = put(~0ULL); b.rooks |= x; own(x); }
        for (int j = 0; j < nq; j++) { const u64 x = put(~0ULL); b.bishops |= x; b.rooks |= x; own(x); }
        if (rnd() % 4 == 0) b.pawns |= rnd() & 15;
        if (rnd() % 8 == 0) b.pawns |= (u64)(rnd() % 9) << 4;
        out[i] = to_pos48(b, (int)(rnd() & 1));
    }
}

}
