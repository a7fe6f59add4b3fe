// noalloc_check.cpp -- TEST HARNESS ONLY (built by tests/test_noalloc_errors.py):
// the host side of pf_perft_batch_noalloc (noalloc.hip) with the HIP calls and
// the launchers replaced by ones that record what was queued and fail on
// demand.  Nothing runs on a GPU.  Not part of the product library.
#include "../../perft_gpu_amd/csrc/engine.h"

namespace {
int g_step, g_fail, g_queued, g_unfinished;  // launches are numbered from 1; the g_fail-th does not start
hipError_t queue() {
    if (++g_step == g_fail) return hipErrorLaunchFailure;
    g_queued++;
    g_unfinished = 1;
    return hipSuccess;
}
hipError_t g_last;
hipError_t fake_set_device(int) { return hipSuccess; }
hipError_t fake_symbol(void** p) {
    *p = nullptr;  // (only passed on)
    return hipSuccess;
}
hipError_t fake_sync(hipStream_t) {
    g_unfinished = 0;
    return hipSuccess;
}
hipError_t fake_record() { return queue(); }
hipError_t fake_last() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
}  // namespace
#define hipSetDevice fake_set_device
#undef HIP_SYMBOL
#define HIP_SYMBOL(x) x
#define hipGetSymbolAddress(p, s) fake_symbol(p)
#define hipStreamSynchronize fake_sync
#define hipEventRecord(e, s) fake_record()
#define hipEventElapsedTime(p, a, b) (*(p) = 0.f, hipSuccess)
#define hipGetLastError fake_last
#undef hipLaunchKernelGGL
#define hipLaunchKernelGGL(...) (void)(g_last = queue())
#include "../../perft_gpu_amd/csrc/noalloc.hip"

namespace pf {
hipError_t launch_pos_to_board(const pf_pos48*, u32, Board*, u32*, hipStream_t) { return queue(); }
hipError_t launch_stream(int, const DevTables&, const PersistArgs& a, const int*, const int*, hipStream_t) {
    for (int i = 0; i < a.depth; i++)
        if (queue() != hipSuccess) return hipErrorLaunchFailure;
    return hipSuccess;
}
hipError_t launch_stream_small(int b, const DevTables& t, const PersistArgs& a, const pf_pos48*, const int* g,
                               const int* v, hipStream_t s) {
    return launch_stream(b, t, a, g, v, s);
}
hipError_t launch_stream_post(const PersistArgs&, unsigned long long*, StreamIO*, u32, hipStream_t) { return queue(); }
pf_status Engine::wait_small() {
    g_unfinished = 0;
    return PF_OK;
}
void Engine::add_small_time() {}
}  // namespace pf

extern "C" {
// Returns the call's status when its `fail`-th launch (from 1; 0: none) does
// not start; *queued the launches that did, *unfinished whether the call
// returned without waiting for them.
int nc_call(int n, int depth, int fail, int* queued, int* unfinished) {
    static pf::Engine e;
    g_step = g_queued = g_unfinished = 0;
    g_fail = fail;
    g_last = hipSuccess;
    const pf_status s = e.perft_noalloc(nullptr, n, depth, nullptr);
    *queued = g_queued;
    *unfinished = g_unfinished;
    return (int)s;
}
}
