// refill_check.cpp -- TEST HARNESS ONLY (built by tests/test_leaf_refill.py):
// how many records the leaf sums of a position hand out.  Not part of the
// product library.
#include <stdint.h>

#include "../../perft_gpu_amd/csrc/convert.h"
#include "../../perft_gpu_amd/csrc/leaf.h"

using namespace pf;

namespace {
const KSBackend sl{};
struct Count {
    int n = 0;
    void operator()(u64 k, u64 f, u32) { n += (k != 0) + (f != 0); }
};
int records(const Board& b) {
    Count c;
    leaf_sum(b, sl, c);
    return c.n;
}
template <class F>
void each_child(const Board& b, F f) {
    PosInfo pi;
    analyse(b, sl, pi);
    auto emit = [&](u32 m) { f(make_move(b, m)); };
    generate(b, sl, pi, emit);
}
}  // namespace

extern "C" {
int rc_records(const pf_pos48* p) { return records(to_board(*p)); }
// over the positions two plies below: their records, and how many they are
int rc_below(const pf_pos48* p, int* n) {
    int sum = 0;
    *n = 0;
    each_child(to_board(*p), [&](const Board& c) {
        each_child(c, [&](const Board& g) {
            sum += records(g);
            (*n)++;
        });
    });
    return sum;
}
}
