// kings_check.cpp -- TEST HARNESS ONLY (built by tests/test_kings.py): boards
// on which a side has no king or several, through every form in which the
// kernels generate and count moves.  Not part of the product library.
#include <stdint.h>

#include <algorithm>
#include <vector>

#include "../../perft_gpu_amd/csrc/convert.h"
#include "../../perft_gpu_amd/csrc/leaf.h"

using namespace pf;

namespace {

const KSBackend sl{};

std::vector<u32> moves(const Board& b, u64 who) {
    PosInfo pi;
    analyse(b, sl, pi);
    std::vector<u32> v;
    auto emit = [&](u32 m) { v.push_back(m); };
    generate(b, sl, pi, emit, who);
    return v;
}

struct Sum {
    const Board* b;
    u64 n = 0;
    void one(u64 to, u32 meta, bool king) {
        for (LeafRecIter it{to, meta, 0}; !it.done();) {
            const u32 m = it.next();
            n += king ? leaf_king_replies(*b, m) : count_moves(make_move(*b, m), sl);
        }
    }
    void operator()(u64 k, u64 f, u32 meta) {
        one(k, meta, true);
        one(f, meta, false);
    }
};

}  // namespace

extern "C" {

// Bits of what disagrees, on a board or one of its children (`depth` plies),
// with generate() over the whole board: 1 the moves of its squares taken one
// by one, 2 in pairs (as coop_generate's lanes do), 4 count_moves, 8 perft 2
// by sets.
static int disagree(const Board& b, int depth) {
    std::vector<u32> all = moves(b, ~0ULL);
    std::sort(all.begin(), all.end());
    int bad = 0;
    for (int pairs = 0; pairs < 2; pairs++) {
        std::vector<u32> v;
        for (int i = 0; i < (pairs ? 32 : 64); i++)
            for (u32 m : moves(b, pairs ? 0x100000001ULL << i : bit(i))) v.push_back(m);
        std::sort(v.begin(), v.end());
        if (v != all) bad |= 1 << pairs;
    }
    if (count_moves(b, sl) != all.size()) bad |= 4;
    u64 want = 0;
    for (u32 m : all) want += count_moves(make_move(b, m), sl);
    Sum e{&b};
    const u64 s = leaf_sum(b, sl, e);
    if (s + e.n != want) bad |= 8;
    for (size_t i = 0; depth && i < all.size(); i++) bad |= disagree(make_move(b, all[i]), depth - 1);
    return bad;
}
int kc_disagree(const pf_pos48* p, int depth) { return disagree(to_board(*p), depth); }
}
