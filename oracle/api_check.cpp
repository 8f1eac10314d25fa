// api_check.cpp -- test infrastructure: the library's host orchestration (fasted_amd/csrc/fasted_api.cpp, compiled as plain C++)
// over a stand-in for the HIP runtime and for the kernel launchers, so that what no GPU run can bring about or see -- memory
// that is refused, a wait that fails, which launch was asked for and what was waited for -- is checked on the CPU.  Device
// memory is host memory, every launch is over as soon as it is made but counts as under way until its stream is waited for,
// and a clock advances by a fixed time per launch.  Built with the address and undefined-behaviour sanitizers by
// `make -C oracle asan`; run with the name of a check.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <utility>
#include <vector>

#include "../fasted_amd/csrc/join_kernels.h"
#include "../include/fasted.h"

static int failures = 0;
#define CHECK(cond)                                                                       \
    do {                                                                                  \
        if (!(cond)) {                                                                    \
            std::fprintf(stderr, "%s:%d: check failed: %s\n", __FILE__, __LINE__, #cond); \
            ++failures;                                                                   \
        }                                                                                 \
    } while (0)

// ---- the stand-in ------------------------------------------------------------------------
namespace {

constexpr double kNormsMs = 1.0, kJoinMs = 10.0, kListMs = 5.0, kSortMs = 3.0;  // what a kernel takes
constexpr double kDispatchMs = 0.25;                                            // and what its launch does, before it
constexpr int kClockKHz = 100000;

struct World {
    double now = 1.0;                          // ms
    std::map<hipStream_t, int> underWay;       // launches and copies nobody has waited for
    std::vector<fasted::JoinLaunch> joins;
    int lists = 0, sorts = 0;
    unsigned long long found = 0;              // pairs of the next joins: the first of a row-major list of 0/1 columns
    unsigned foundPerQuery = 0;                // where set, `found` follows the number of query points
    size_t refuseFrom = ~(size_t)0;            // device allocations of so many bytes are refused
    int eventWaitsToFail = 0;                  // after how many waits for an event one fails (0: none)
    int pinnedAllocations = 0;
    size_t refusePinnedFrom = ~(size_t)0;      // pinned allocations of so many bytes are refused
    std::map<void*, size_t> pinned;
} world;

struct Event {
    double at = 0.0;
};

unsigned long long ticks() { return (unsigned long long)std::llround(world.now * kClockKHz); }

unsigned long long* host_words(unsigned long long* counters) {
    return reinterpret_cast<unsigned long long*>(counters[fasted::host_words_slot()]);
}

void write_pairs(void* to, unsigned long long cap) {
    auto* const p = static_cast<FastedPair*>(to);
    for (unsigned long long i = 0; i < world.found && i < cap; ++i) {
        p[i].QueryPoint = (int)(i / 2);
        p[i].CandidatePoint = (int)(i % 2);
    }
}

}  // namespace

extern "C" {
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = kClockKHz; return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { world.underWay.clear(); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { world.underWay.erase(s); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = reinterpret_cast<hipStream_t>(new char); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { world.underWay.erase(s); delete reinterpret_cast<char*>(s); return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = reinterpret_cast<hipEvent_t>(new Event); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { delete reinterpret_cast<Event*>(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { reinterpret_cast<Event*>(e)->at = world.now; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) {
    if (world.eventWaitsToFail > 0 && --world.eventWaitsToFail == 0) return hipErrorUnknown;
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) {
    *ms = (float)(reinterpret_cast<Event*>(b)->at - reinterpret_cast<Event*>(a)->at);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* freeB, size_t* total) { *freeB = *total = (size_t)4 << 30; return hipSuccess; }
hipError_t hipMalloc(void** p, size_t bytes) {
    if (bytes >= world.refuseFrom) return hipErrorOutOfMemory;
    *p = std::malloc(bytes);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) { world.underWay.clear(); std::free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
    if (bytes >= world.refusePinnedFrom) return hipErrorOutOfMemory;
    *p = std::calloc(1, bytes);
    world.pinned[*p] = bytes;
    ++world.pinnedAllocations;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) { world.pinned.erase(p); std::free(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { *d = h; return hipSuccess; }
hipError_t hipMemset(void* p, int v, size_t n) { std::memset(p, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t s) { ++world.underWay[s]; return hipMemset(p, v, n); }
hipError_t hipMemcpy(void* to, const void* from, size_t n, hipMemcpyKind) { std::memcpy(to, from, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* to, const void* from, size_t n, hipMemcpyKind k, hipStream_t s) { ++world.underWay[s]; return hipMemcpy(to, from, n, k); }
hipError_t hipMemcpy2D(void* to, size_t toPitch, const void* from, size_t fromPitch, size_t width, size_t rows, hipMemcpyKind k) {
    for (size_t r = 0; r < rows; ++r) (void)hipMemcpy(static_cast<char*>(to) + r * toPitch, static_cast<const char*>(from) + r * fromPitch, width, k);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* symbol) { *p = const_cast<void*>(symbol); return hipSuccess; }
}

namespace fasted {
int counter_words() { return 160; }
int band_words() { return 5120; }
int host_words_slot() { return 144; }
const char* build_tag() { return ""; }
size_t bits_bytes(int nQ, int nC) { return (size_t)tile_count(nQ, nC) * 8192; }
unsigned long long tile_count(long long nQ, long long nC) { return (unsigned long long)((nQ + 255) / 256) * ((nC + 255) / 256); }
unsigned long long raster_count(long long, long long, bool) { return 0; }
int raster_coord(unsigned long long, long long, long long, bool, int*, int*) { return 0; }
int lds_chunk_slot(int, int) { return 0; }
size_t sort_scratch_bytes(unsigned long long count) { return count * 8; }
void SortBuffers::release() {}

hipError_t launch_sum_squared(const NormPoints&, const NormPoints*, int, float, unsigned long long* counters, hipStream_t s,
                              unsigned long long, Reset reset) {
    world.now += kDispatchMs;
    if (counters && reset != Reset::kNothing) counters[2] = ticks();
    world.now += kNormsMs;
    ++world.underWay[s];
    return hipSuccess;
}
hipError_t launch_halves(const float*, int, float, float*, unsigned long long* counters, hipStream_t s, unsigned long long, Reset reset) {
    return launch_sum_squared(NormPoints{}, nullptr, 64, 0.f, counters, s, 1, reset);
}
hipError_t launch_pad_rows(const void*, int, void*, int, long long, hipStream_t s) { ++world.underWay[s]; return hipSuccess; }
hipError_t launch_padding_check(const void*, long long, int, int, int, unsigned long long*, hipStream_t) { return hipSuccess; }
hipError_t launch_reset_counters(unsigned long long*, bool, hipStream_t s) { ++world.underWay[s]; return hipSuccess; }
hipError_t launch_offset_appended_pairs(void*, unsigned long long*, const unsigned long long*, unsigned long long, int, int, hipStream_t s) {
    ++world.underWay[s];
    return hipSuccess;
}
hipError_t launch_pair_distances(const void*, long long, int, const void*, long long, int, int, const void*, unsigned long long count,
                                 float* out, hipStream_t s) {
    std::fill(out, out + count, 0.f);
    ++world.underWay[s];
    return hipSuccess;
}
hipError_t launch_join(const JoinLaunch& l, hipStream_t s, BitsLayout*) {
    world.joins.push_back(l);
    if (world.foundPerQuery) world.found = (unsigned long long)world.foundPerQuery * l.nQ;
    world.now += kDispatchMs;
    unsigned long long* const w = host_words(l.counters);
    if (w) {
        w[1] = l.counters[2];
        w[2] = ticks();
    }
    world.now += kJoinMs;
    ++world.underWay[s];
    if (l.bits) return hipSuccess;  // (the list kernel reports)
    write_pairs(l.pairs, l.cap);
    l.counters[0] = world.found;
    if (w) {
        w[0] = world.found;
        w[3] = ticks();
    }
    return hipSuccess;
}
hipError_t launch_expand_bits(const unsigned*, const BitsLayout&, int, int, unsigned long long* counters, void* pairs, unsigned long long cap,
                              hipStream_t s) {
    ++world.lists;
    world.now += kDispatchMs;
    unsigned long long* const w = host_words(counters);
    write_pairs(pairs, cap);
    w[0] = counters[0] = world.found;
    w[3] = ticks();
    world.now += kListMs;
    w[4] = ticks();
    ++world.underWay[s];
    return hipSuccess;
}
hipError_t sort_pairs_row_major(void*, unsigned long long, hipStream_t s, SortBuffers*, long long, long long, long long) {
    ++world.sorts;
    world.now += kSortMs;
    world.underWay.erase(s);  // (it waits for its stream)
    return hipSuccess;
}
}  // namespace fasted

// ---- the checks --------------------------------------------------------------------------
namespace {

// Two sets of points, neither with more workgroups than a launch may hold, that together have more: two launches.
void check_norms_of_two_large_sets() {
    using namespace fasted;
    for (int dPad : {64, 128, 256, 512, 4096}) {
        const int rows = kNormThreads / norm_lanes(dPad);  // of a workgroup
        const long long most = ((1ll << 32) / kNormThreads - 1) * rows;
        if (most + 1 > INT32_MAX) continue;
        CHECK(norm_groups((int)most, dPad) * (unsigned long long)kNormThreads < 1ull << 32);
        CHECK(norms_fit_one_launch((int)most - rows, rows, dPad) && norms_fit_one_launch(rows, (int)most - rows, dPad));
        CHECK(!norms_fit_one_launch((int)most, 1, dPad) && !norms_fit_one_launch(1, (int)most, dPad));
        CHECK(!norms_fit_one_launch((int)most, (int)most, dPad));
    }
    CHECK(norm_lanes(64) == 8 && norm_lanes(192) == 16 && norm_lanes(512) == 64 && norm_lanes(4096) == 64);
    CHECK(norm_groups(1, 64) == 1 && norm_groups(32, 64) == 1 && norm_groups(33, 64) == 2 && norm_groups(5, 512) == 2);
    CHECK(!norms_fit_one_launch(34000000, 34000000, 512) && norms_fit_one_launch(34000000, 33000000, 512));
}

// A sorted call returns with its stream drained, however few pairs there are to sort and whoever reported them.
void check_sorted_joins_drain_the_stream() {
    const hipStream_t stream = reinterpret_cast<hipStream_t>(&world);
    // up to 512 tiles, more, more than report themselves; hit bits
    for (auto [nQ, nC] : {std::pair<long long, long long>{256, 30000}, {30000, 256}, {30000, 2560}, {30000, 400000}, {300, 300}})
        for (unsigned long long found : {0ull, 1ull, 2ull, 4ull})
            for (unsigned more : {0u, (unsigned)FASTED_EVENT_TIMING})
                for (bool wantStats : {true, false}) {
                    world.found = found;
                    alignas(16) static char points[64];
                    FastedPair pairs[4];
                    FastedJoinStats st{};
                    CHECK(fasted_join_device(points, nQ, 64, points, nC, 64, 64, 1.0, nullptr, nullptr, pairs, 4, FASTED_SORT_PAIRS | more, stream,
                                             wantStats ? &st : nullptr) == 0);
                    CHECK(world.underWay.count(stream) == 0);
                    CHECK(!wantStats || st.pairsStored == found);
                }
}

// The join's time spans the writing of its pairs, whoever writes them and whatever it is timed with; a sort is not part of it.
void check_join_time_spans_the_writing_of_the_pairs() {
    alignas(16) static char points[64];
    FastedPair pairs[4];
    auto near = [](double a, double b) { return std::fabs(a - b) < 1e-3; };
    for (unsigned long long found : {0ull, 3ull})
        for (unsigned more : {0u, (unsigned)FASTED_EVENT_TIMING, (unsigned)FASTED_FULL_MATRIX})
            for (long long n : {100, 5000, 20224, 20225, 90000, 200000}) {
                world.found = found;
                world.sorts = 0;
                const int listsBefore = world.lists;
                FastedJoinStats st{};
                CHECK(fasted_self_join_device(points, n, 64, 64, 1.0, nullptr, pairs, 4, FASTED_SORT_PAIRS | more, nullptr, &st) == 0);
                const bool list = n <= 20224, events = more & FASTED_EVENT_TIMING || n > 92672;
                const double before = events ? kDispatchMs : 0.0, between = events ? 0.0 : kDispatchMs;
                CHECK(world.lists - listsBefore == (list ? 1 : 0) && world.sorts == (!list && found > 1 ? 1 : 0));
                CHECK(near(st.sumSquaredMs, before + kNormsMs + between) &&
                      near(st.joinMs, before + kJoinMs + (list ? kDispatchMs + kListMs : 0.0)));
                CHECK(!list || st.sortMs == 0.0f);
                CHECK(fasted_self_join_device(points, n, 64, 64, 1.0, nullptr, pairs, 4, more, nullptr, &st) == 0);
                CHECK(near(st.sumSquaredMs, before + kNormsMs + between) && near(st.joinMs, before + kJoinMs) && st.sortMs == 0.0f);
            }
}

// Results.TFLOPS: 2 N^2 D over the time between events, as the reference has it, for all but the smallest joins, whose calls
// three event records would lengthen by a third.
void check_results_are_timed_with_events() {
    world.found = 3;
    for (int n : {300, 5632, 5633, 20225}) {
        const Results r = runFromExponentialDataset(n, 2, 40.0, 1.0, 0.1, false);
        const double list = n <= 20224 ? kDispatchMs + kListMs : 0.0;
        const double ms = kDispatchMs + kNormsMs + kJoinMs + list + (n <= 5632 ? 0.0 : kDispatchMs);
        CHECK(std::fabs(r.TFLOPS * ms / (2.0 * n * n * 2 / 1e9) - 1.0) < 1e-4);
        CHECK(r.pairsFound == 3 && r.pairsStored == 3);
    }
}

// Every entry tells the join how many dimensions there are, so that none multiplies padding where a kernel can leave it out.
void check_every_join_is_told_the_dimensionality() {
    constexpr int n = 700, d = 65, dPad = 128;
    std::vector<uint16_t> points((size_t)n * dPad, 0);
    FastedPair pairs[4];
    unsigned long long found = 0, stored = 0;
    double epsilon = 0.0, selectivity = 0.0;
    int probes = 0, rows = 0;
    const std::function<void()> entries[] = {
        [&] { (void)runFromExponentialDataset(n, d, 40.0, 1.0, 0.1, false); },
        [&] { (void)reRun(0.2, false); },
        [&] { CHECK(fasted_count_pairs(0.1, &found, nullptr) == 0); },
        [&] { CHECK(fasted_count_pairs_sampled(0.1, 100, &found, &rows, nullptr) == 0); },
        [&] { CHECK(fasted_find_epsilon(1.0, 0.1, &epsilon, &selectivity, &probes) == 0); },
        [&] { CHECK(fasted_find_epsilon_sampled(1.0, 0.1, 100, &epsilon, &selectivity, &probes) == 0); },
        [&] { CHECK(fasted_find_epsilon_volumetric(1.0, 0.1, &epsilon, &selectivity, &probes) == 0); },
        [&] { CHECK(fasted_self_join(points.data(), n, d, 0.1, pairs, 4, &found, &stored) == 0); },
        [&] { CHECK(fasted_self_join_blocked(points.data(), n, d, 0.1, 256, pairs, 4, &found, &stored) == 0); },
        [&] { CHECK(fasted_self_join_device(points.data(), n, d, dPad, 0.1, nullptr, pairs, 4, 0, nullptr, nullptr) == 0); },
        [&] { CHECK(fasted_self_join_device_noalloc(points.data(), n, d, dPad, 0.1, pairs, 4, 0, nullptr, nullptr) == 0); },
        [&] { CHECK(fasted_join_device(points.data(), n, dPad, points.data(), n, dPad, d, 0.1, nullptr, nullptr, pairs, 4, 0, nullptr, nullptr) == 0); },
    };
    int entry = 0;
    for (const auto& call : entries) {
        world.joins.clear();
        world.foundPerQuery = 2;  // (the selectivity the searches look for)
        call();
        CHECK(!world.joins.empty());
        for (const fasted::JoinLaunch& l : world.joins)
            if (l.d != d || l.dPad != dPad) {
                std::fprintf(stderr, "entry %d: %d dimensions of %d\n", entry, l.d, l.dPad);
                ++failures;
                break;
            }
        ++entry;
    }
}

// Pinned pieces with a transfer that nobody has waited for are not used again: not by the next call, and not by one that
// follows on another stream.
void check_a_failed_download_gives_up_its_pieces() {
    constexpr int n = 4000;
    constexpr unsigned long long cap = 1000000;  // 8 MB, four pieces
    std::vector<uint16_t> points((size_t)n * 64, 0);
    std::vector<FastedPair> pairs(cap);
    unsigned long long found = 0, stored = 0;
    world.found = cap;
    auto join = [&](bool blocked) {
        std::fill(pairs.begin(), pairs.end(), FastedPair{-1, -1});
        return blocked ? fasted_self_join_blocked(points.data(), n, 64, 1.0, 8192, pairs.data(), cap, &found, &stored)
                       : fasted_self_join(points.data(), n, 64, 1.0, pairs.data(), cap, &found, &stored);
    };
    auto whole = [&] {
        for (unsigned long long i = 0; i < cap; ++i)
            if (pairs[i].QueryPoint != (int)(i / 2) || pairs[i].CandidatePoint != (int)(i % 2)) return false;
        return true;
    };
    for (bool blocked : {false, true}) {
        CHECK(join(blocked) == 0 && stored == cap && whole());
        const int allocations = world.pinnedAllocations;
        const size_t held = world.pinned.size();
        CHECK(join(blocked) == 0 && whole() && world.pinnedAllocations == allocations);  // kept
        for (int wait : {1, 2, 4}) {
            const int before = world.pinnedAllocations;
            world.eventWaitsToFail = wait;
            CHECK(join(blocked) != 0 && world.pinned.size() == held - 1);
            CHECK(join(blocked) == 0 && whole() && world.pinnedAllocations == before + 1 && world.pinned.size() == held);
        }
    }
}

// Long lists come down without pinned memory where there is none to be had.
void check_lists_come_down_without_pinned_memory() {
    constexpr int n = 1000;
    constexpr unsigned long long cap = 700000;  // 5.6 MB
    std::vector<uint16_t> points((size_t)n * 64, 0);
    std::vector<FastedPair> pairs(cap, FastedPair{-1, -1});
    unsigned long long found = 0, stored = 0;
    world.found = cap;
    world.refusePinnedFrom = (size_t)1 << 20;
    CHECK(fasted_self_join(points.data(), n, 64, 1.0, pairs.data(), cap, &found, &stored) == 0 && stored == cap);
    for (unsigned long long i = 0; i < cap && failures == 0; ++i) CHECK(pairs[i].QueryPoint == (int)(i / 2) && pairs[i].CandidatePoint == (int)(i % 2));
}

// Without memory for the hit bits a sorted join of few points stages its pairs and sorts them; with it again, it leaves bits.
void check_without_memory_for_hit_bits_the_pairs_are_sorted() {
    alignas(16) static char points[64];
    FastedPair pairs[4];
    world.found = 4;
    auto join = [&](long long n, bool inBits) {
        const int lists = world.lists, sorts = world.sorts;
        FastedJoinStats st{};
        std::fill(pairs, pairs + 4, FastedPair{-1, -1});
        CHECK(fasted_self_join_device(points, n, 64, 64, 1.0, nullptr, pairs, 4, FASTED_SORT_PAIRS, nullptr, &st) == 0);
        CHECK(st.pairsFound == 4 && st.pairsStored == 4 && pairs[3].QueryPoint == 1 && pairs[3].CandidatePoint == 1);
        CHECK(world.lists - lists == (inBits ? 1 : 0) && world.sorts - sorts == (inBits ? 0 : 1));
        CHECK((world.joins.back().bits != nullptr) == inBits);
        CHECK(std::fabs(st.joinMs - (inBits ? kJoinMs + kDispatchMs + kListMs : kJoinMs)) < 1e-3);
    };
    join(1000, true);
    world.refuseFrom = (size_t)1 << 20;
    join(1000, true);  // (the megabyte that is there does)
    join(8000, false);
    join(1000, false);  // (it has been given back)
    world.refuseFrom = ~(size_t)0;
    join(8000, true);
    join(20224, true);
}

const std::map<std::string, std::function<void()>> kChecks = {
    {"without_memory_for_hit_bits_the_pairs_are_sorted", check_without_memory_for_hit_bits_the_pairs_are_sorted},
    {"lists_come_down_without_pinned_memory", check_lists_come_down_without_pinned_memory},
    {"a_failed_download_gives_up_its_pieces", check_a_failed_download_gives_up_its_pieces},
    {"every_join_is_told_the_dimensionality", check_every_join_is_told_the_dimensionality},
    {"results_are_timed_with_events", check_results_are_timed_with_events},
    {"join_time_spans_the_writing_of_the_pairs", check_join_time_spans_the_writing_of_the_pairs},
    {"sorted_joins_drain_the_stream", check_sorted_joins_drain_the_stream},
    {"norms_of_two_large_sets", check_norms_of_two_large_sets},
};

}  // namespace

int main(int argc, char** argv) {
    setenv("FASTED_QUIET", "1", 1);
    const auto it = argc == 2 ? kChecks.find(argv[1]) : kChecks.end();
    if (it == kChecks.end()) {
        for (const auto& c : kChecks) std::printf("%s\n", c.first.c_str());
        return argc == 1 ? 0 : 2;
    }
    it->second();
    releaseResources();
    if (failures == 0) std::printf("all checks held\n");
    return failures != 0;
}
