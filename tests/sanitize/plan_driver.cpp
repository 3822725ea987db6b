// Host-only driver of the plan management (apr-cnn_amd/csrc/plan.hip, which holds no kernels): compiled with it and the APR
// builder into one executable under AddressSanitizer and UndefinedBehaviorSanitizer (tests/test_sanitizers.py).  The HIP
// runtime is replaced by the stand-in below, which keeps "device" memory on the heap (so that every copy is checked
// against the size of both buffers), has a settable amount of it, and records what happens to streams and events.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <vector>

#include "../../apr-cnn_amd/csrc/common.hpp"

#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); std::exit(1); } } while (0)

// ------------------------------------------------------------------------------------------------ stand-in runtime
static std::map<void*, size_t> g_mem;
static size_t g_free = (size_t)1 << 30;            // what hipMemGetInfo reports
static size_t g_fail_from = SIZE_MAX;              // hipMalloc fails from this size on, whatever is reported
static int g_mallocs = 0, g_frees = 0, g_syncs = 0, g_streams_made = 0, g_streams_destroyed = 0;
struct FakeEvent { hipStream_t on = nullptr; };
static std::set<hipStream_t> g_streams;
static std::map<hipEvent_t, FakeEvent> g_events;

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    ++g_mallocs;
    if (n > g_free || n >= g_fail_from) { *p = nullptr; return hipErrorOutOfMemory; }
    *p = std::calloc(1, n); g_mem[*p] = n; g_free -= n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    CHECK(g_mem.count(p) == 1);
    ++g_frees; g_free += g_mem[p]; g_mem.erase(p); std::free(p);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) { *f = g_free; *t = (size_t)1 << 31; return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stand-in"; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    ++g_streams_made; *s = (hipStream_t)std::malloc(1); g_streams.insert(*s);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    CHECK(g_streams.erase(s) == 1);
    for (auto& e : g_events) CHECK(e.second.on != s);          // no event may be left that was recorded on it
    ++g_streams_destroyed; std::free((void*)s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) { CHECK(!s || g_streams.count(s)); ++g_syncs; return hipSuccess; }
static bool g_capturing = false;
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* c) {
    *c = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) { CHECK(!s || g_streams.count(s)); CHECK(g_events.count(e)); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)std::malloc(1); g_events[*e]; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { CHECK(!s || g_streams.count(s)); g_events.at(e).on = s; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { CHECK(g_events.count(e)); ++g_syncs; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { CHECK(g_events.erase(e) == 1); std::free((void*)e); return hipSuccess; }

void* aprcore_create(int, int, int);
void aprcore_destroy(void*);
int aprcore_level_max(void*);
void aprcore_level_dims(void*, int, int32_t*);
int aprcore_build_from_levels(void*, const uint8_t*);
void aprcore_access_info(void*, int, int64_t*);
void aprcore_access_copy(void*, int, int32_t*, int32_t*, int32_t*, uint64_t*, uint64_t*, uint16_t*);
}
namespace aprnet {       // lists are built by kernels: none here
void free_lists(WinLists&) {}
void free_face_lists(FaceLists&) {}
void free_need_lists(NeedLists&) {}
}

// ------------------------------------------------------------------------------------------------ an APR on the host
struct Access {
    std::vector<int32_t> z, x, y;
    std::vector<uint64_t> lxz, xz_end;
    std::vector<uint16_t> yv;
    aprnet_access_desc d{};
    Access(void* h, int which) {
        const int lmax = aprcore_level_max(h);
        int64_t info[4];
        aprcore_access_info(h, which, info);
        z.resize(lmax + 1); x.resize(lmax + 1); y.resize(lmax + 1); lxz.resize(info[1] + 2); xz_end.resize(info[2]); yv.resize(info[3]);
        aprcore_access_copy(h, which, z.data(), x.data(), y.data(), lxz.data(), xz_end.data(), yv.data());
        d = {(int32_t)info[0], (int32_t)info[1], z.data(), x.data(), y.data(), lxz.data(), xz_end.data(), yv.data(), (uint64_t)info[2], (uint64_t)info[3]};
    }
};
static void* build(int zn, int xn, int yn, unsigned seed) {
    void* h = aprcore_create(zn, xn, yn);
    const int lmax = aprcore_level_max(h);
    int32_t dims[3];
    aprcore_level_dims(h, lmax - 1, dims);
    std::vector<uint8_t> want((size_t)dims[0] * dims[1] * dims[2], 0);
    for (auto& v : want) { seed = seed * 1664525u + 1013904223u; if ((seed >> 24) < 8) v = (uint8_t)(lmax - ((seed >> 16) & 1)); }
    aprcore_build_from_levels(h, want.data());
    return h;
}

using namespace aprnet;

// what a backward call does to its plan: scratch, side stream, fork and join
static void backward(aprnet_plan* p, hipStream_t st) {
    TileList tl;
    CHECK(get_tiles(p, 0, 2, 4, &tl, st) == 0 && tl.n > 0);
    ScratchLease lease;
    CHECK(lease.acquire(p, 4096, st) == 0);
    std::memset(p->d_scratch, 1, 4096);
    if (!p->side) {
        CHECK(side_stream_acquire(p->device, &p->side) == 0);
        CHECK(hipEventCreateWithFlags(&p->ev_fork, 0) == hipSuccess && hipEventCreateWithFlags(&p->ev_join, 0) == hipSuccess);
    }
    CHECK(hipEventRecord(p->ev_fork, st) == hipSuccess && hipStreamWaitEvent(p->side, p->ev_fork, 0) == hipSuccess);
    CHECK(hipEventRecord(p->ev_join, p->side) == hipSuccess && hipStreamWaitEvent(st, p->ev_join, 0) == hipSuccess);
}

// plans that come and go: the arrays of the APRs stay as they were built, side streams are shared by the plans that
// follow each other, nothing is left behind
static void plans_come_and_go() {
    hipStream_t st = nullptr;
    CHECK(hipStreamCreateWithFlags(&st, 0) == hipSuccess);
    g_streams_made = 0;
    for (int round = 0; round < 20; ++round) {
        void* h = build(9 + round, 21, 17 + 3 * round, 7u + (unsigned)round);
        Access apr(h, 0), tree(h, 1);
        aprcore_destroy(h);
        const std::vector<uint16_t> y0 = apr.yv, t0 = tree.yv;
        aprnet_plan* p[3] = {};
        for (auto& q : p) {
            CHECK(aprnet_plan_create(&apr.d, &tree.d, 0, &q) == 0);
            backward(q, st);
            std::vector<int32_t> children((size_t)8 * q->n_tree);
            CHECK(aprnet_plan_children(q, children.data()) == 0);
        }
        for (auto& q : p) aprnet_plan_destroy(q);
        CHECK(apr.yv == y0 && tree.yv == t0);
        CHECK(g_events.empty() && g_mem.empty());
    }
    CHECK(g_streams_made == 3 && g_streams_destroyed == 0);
    // more plans at once than idle streams are kept: the rest are destroyed, after their events
    void* h = build(9, 21, 17, 3u);
    Access apr(h, 0), tree(h, 1);
    aprcore_destroy(h);
    std::vector<aprnet_plan*> many(20, nullptr);
    for (auto& q : many) { CHECK(aprnet_plan_create(&apr.d, &tree.d, 0, &q) == 0); backward(q, st); }
    for (auto& q : many) aprnet_plan_destroy(q);
    CHECK(g_streams_made == 20 && g_streams_destroyed == 4);
    CHECK(g_events.empty() && g_mem.empty());
    CHECK(hipStreamDestroy(st) == hipSuccess);
}

// a request that the caller can do without costs nothing when it cannot be met
static void optional_scratch() {
    void* h = build(9, 21, 17, 5u);
    Access apr(h, 0), tree(h, 1);
    aprcore_destroy(h);
    aprnet_plan* p = nullptr;
    CHECK(aprnet_plan_create(&apr.d, &tree.d, 0, &p) == 0);
    const size_t big = (size_t)64 << 20, small = (size_t)1 << 20;
    CHECK(plan_scratch(p, small, nullptr) == 0);
    void* kept = p->d_scratch;
    const size_t room = g_free;
    auto untouched = [&](int rc) {
        CHECK(rc != 0 && p->d_scratch == kept && p->scratch_bytes == small);
        CHECK(g_mallocs == 0 && g_frees == 0 && g_syncs == 0);
    };
    // no room (what is reported as free and the buffer itself do not suffice), call after call
    g_free = big - small - 1;
    for (int i = 0; i < 3; ++i) { g_mallocs = g_frees = g_syncs = 0; untouched(plan_scratch(p, big, nullptr, true)); CHECK(plan_scratch(p, small, nullptr) == 0); }
    // memory has come back: granted
    g_free = room;
    CHECK(plan_scratch(p, big, nullptr, true) == 0 && p->scratch_bytes == big);
    // a refusal that is only seen when allocating is remembered: equal and larger ones are not tried again, a smaller one is
    g_fail_from = 2 * big;
    CHECK(plan_scratch(p, 2 * big, nullptr, true) != 0);
    CHECK(plan_scratch(p, small, nullptr) == 0);
    kept = p->d_scratch;
    g_mallocs = g_frees = g_syncs = 0;
    untouched(plan_scratch(p, 2 * big, nullptr, true));
    untouched(plan_scratch(p, 3 * big, nullptr, true));
    CHECK(plan_scratch(p, big, nullptr, true) == 0);
    // a call that cannot do without asks again, and its success clears the refusal
    g_fail_from = SIZE_MAX;
    CHECK(plan_scratch(p, 2 * big, nullptr) == 0 && p->scratch_refused == 0);
    CHECK(plan_scratch(p, 3 * big, nullptr, true) == 0);
    // a buffer that a graph may address stays, and does not count as room
    g_capturing = true;
    CHECK(plan_scratch(p, big, nullptr) == 0 && p->scratch_in_graph);
    CHECK(plan_scratch(p, 4 * big, nullptr) == APRNET_ERR_UNSUPPORTED);
    g_capturing = false;
    kept = p->d_scratch;
    g_free = 4 * big - 1;
    CHECK(plan_scratch(p, 4 * big, nullptr, true) != 0 && p->d_scratch == kept && p->retired.empty());
    g_free = 4 * big;
    CHECK(plan_scratch(p, 4 * big, nullptr, true) == 0 && p->d_scratch != kept && p->retired.size() == 1);
    aprnet_plan_destroy(p);
    CHECK(g_mem.empty() && g_events.empty());
}

int main() {
    optional_scratch();
    plans_come_and_go();
    std::printf("OK\n");
    return 0;
}
