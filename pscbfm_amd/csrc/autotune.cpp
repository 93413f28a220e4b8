// Launch-shape autotuner (see autotune.h).
#include "autotune.h"

#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <stdexcept>
#include <tuple>

#include "batch.h"
#include "device_system.h"

namespace pscbfm {

namespace {

// Signature of a workload for the cache: lattice kind, box exponents, and
// the rounded log2 of the monomer count, species size, degree and count of
// systems (batches).
using Key = std::tuple<int, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t>;

uint32_t log2_ceil(uint64_t v) {
    uint32_t r = 0;
    while ((uint64_t(1) << r) < v) ++r;
    return r;
}

Key system_key(int mode, const SystemLayout& L, uint32_t kind, uint32_t count) {
    uint32_t deg = 0;
    for (const ColorInfo& c : L.colors) deg = std::max(deg, c.maxDegree);
    return Key{mode, kind, L.codec.log2L[0], L.codec.log2L[1], L.codec.log2L[2], log2_ceil(L.nMonomers),
               log2_ceil(L.maxColorCount), deg, count};
}

std::mutex g_cacheMutex;
std::map<Key, TuneResult>& cache() {
    static std::map<Key, TuneResult> c;
    return c;
}

struct Events {
    hipEvent_t a = nullptr, b = nullptr;
    Events() {
        hip_check(hipEventCreate(&a), "hipEventCreate");
        hip_check(hipEventCreate(&b), "hipEventCreate");
    }
    ~Events() {
        (void)hipEventDestroy(a);
        (void)hipEventDestroy(b);
    }
    double ms() const {
        float v = 0;
        hip_check(hipEventElapsedTime(&v, a, b), "hipEventElapsedTime");
        return v;
    }
};

// Times `mcs` sweeps of a scratch copy of L at shape s (graph replay).
double time_system(const SystemLayout& L, uint32_t kind, uint64_t seed, LaunchShape s, uint32_t mcs,
                   hipStream_t st) {
    DeviceSystem dev;
    dev.allocate(L, kind, seed, /*withLists=*/true, uint32_t(max_grid(L.maxColorCount)), st);
    s.grid = grid_for(L.maxColorCount, s.block * s.slots);
    s.performBlock = automatic_perform_block(L, s.block, s.slots);
    s.clearPass = automatic_clear_pass(L, kind);
    const uint32_t nc = std::max<uint32_t>(1u, uint32_t(L.colors.size()));
    const uint32_t g = nc;  // one sweep per replay
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    hip_check(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal), "hipStreamBeginCapture");
    hipError_t err = hipSuccess;
    for (uint32_t k = 0; k < g && err == hipSuccess; ++k) {
        err = launch_check(dev.desc, k, s, st);
        if (err == hipSuccess) err = launch_perform(dev.desc, k, s, st);
    }
    if (err == hipSuccess) err = launch_advance(dev.desc.state, g, st);
    const hipError_t endErr = hipStreamEndCapture(st, &graph);
    if (err != hipSuccess) hip_fail(err, "kernel launch during capture");
    hip_check(endErr, "hipStreamEndCapture");
    const hipError_t ie = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    hip_check(ie, "hipGraphInstantiate");
    Events ev;
    hipError_t runErr = hipGraphLaunch(exec, st);  // warm-up sweep
    if (runErr == hipSuccess) runErr = hipEventRecord(ev.a, st);
    for (uint32_t r = 0; r < mcs && runErr == hipSuccess; ++r) runErr = hipGraphLaunch(exec, st);
    if (runErr == hipSuccess) runErr = hipEventRecord(ev.b, st);
    if (runErr == hipSuccess) runErr = hipStreamSynchronize(st);
    (void)hipGraphExecDestroy(exec);
    hip_check(runErr, "autotune sweep");
    return ev.ms() / std::max<uint32_t>(mcs, 1u);
}

TuneResult pick(std::vector<TuneTrial> trials) {
    TuneResult r;
    r.trials = std::move(trials);
    auto it = std::min_element(r.trials.begin(), r.trials.end(),
                               [](const TuneTrial& a, const TuneTrial& b) { return a.msPerMcs < b.msPerMcs; });
    r.best = it->shape;
    r.bestMsPerMcs = it->msPerMcs;
    return r;
}

}  // namespace

namespace {
double occupied_fraction(const SystemLayout& L) {
    const uint32_t log2Cells = L.codec.log2L[0] + L.codec.log2L[1] + L.codec.log2L[2];
    return 8.0 * double(L.nMonomers) / std::ldexp(1.0, int(log2Cells));
}
}  // namespace

void automatic_shape(const SystemLayout& L, uint32_t latticeKind, uint32_t* block, uint32_t* slots) {
    // Two monomers per thread keep more loads in flight per wave, one gives
    // twice the waves.  Measured, 256 x 2 against the choice, us per substep
    // by members of a species:
    //   up to 20,000, 64 x 1: 8192 6.7 and 5.6 (uint8 7.5 and 5.8); 128 x 1
    //     takes 5.7 (6.0), at 11,800 5.84 against 5.80 (6.35 and 6.15), at
    //     19,700 6.13 against 5.93 (6.53 and 6.32);
    //   up to 2^15, 128 x 1: 32768 6.7 and 5.7 (7.5 and 6.0); 64 x 1 takes
    //     5.8 there, 256 x 1 5.7 and 6.1;
    //   else 256 x 1: 65536 6.8 and 6.3, 2^18 8.3 and 8.2, uint8 2^19 12.8 and
    //     12.3, dense network of 374,400 11.2 and 10.9, at occupied fraction
    //     0.2 839,000 19.6 and 18.3, 1.7 million 30.1 and 28.6, uint8 2^22 55.9
    //     and 55.1;
    //   but 256 x 2 for more than 400,000 on the bit lattice at 0.4 or denser,
    //     where the waves of 256 x 1 share the caches worse: 2^19 10.6 to 11.1
    //     with 256 x 1 and 10.7, 2^20 15.4 and 15.2, 2^21 23.9 and 23.4.
    const bool pairs = latticeKind == kLatticeBit && L.maxColorCount > 400000u && occupied_fraction(L) >= 0.4;
    *block = L.maxColorCount <= 20000u ? 64u : (L.maxColorCount <= (1u << 15) ? 128u : 256u);
    *slots = pairs ? 2u : 1u;
}

namespace {
uint32_t max_degree(const SystemLayout& L) {
    uint32_t v = 0;
    for (const ColorInfo& ci : L.colors) v = std::max(v, ci.maxDegree);
    return v;
}
}  // namespace

uint32_t automatic_perform_block(const SystemLayout& L, uint32_t block, uint32_t slots) {
    // Pass 2 walks one compacted pass-1 list per workgroup.  With one monomer
    // per pass-1 thread, or in a dense system (at least a quarter of the cells
    // occupied), a list of a 256-thread workgroup has about 128 entries or
    // fewer: 128 threads against 256, us per substep, 18.3 and 18.7 (839,000
    // members, fraction 0.2, 256 x 1), 38.8 and 39.2 (512^3 melt).  Dilute systems
    // with two monomers per thread have fuller lists and keep the pass-1 block.
    // In a dense network fewer moves still pass the bond test: 64 threads against
    // 128, fraction 0.7, 10.2 and 10.4 (uint8 11.5 and 11.6); the 256^3 melt, 0.5,
    // 11.0 and 10.1.
    if (block <= 128u) return 0u;
    if (slots == 1u && max_degree(L) > 2u && occupied_fraction(L) >= 0.4) return 64u;
    return slots == 1u || occupied_fraction(L) >= 0.25 ? 128u : 0u;
}

uint32_t automatic_clear_pass(const SystemLayout& L, uint32_t latticeKind) {
    // The clear (16 bytes per thread and step) goes into pass 1, which has issue
    // slots to spare, on the bit lattice; the uint8 lattice's pass 1 moves eight
    // times the plane bytes, so it clears in pass 2.  us per substep, pass 1
    // against pass 2: 512^3 melt 39.1 and 39.8, 839,000 members at fraction 0.2
    // 16.5 and 17.4, dense star network 10.4 and 10.6, 128^3 melt 5.9 either way;
    // uint8, 256^3 melt 12.3 and 11.9.  Dense melts of some hundred thousand
    // members on the bit lattice are the exception: 104,800 at 0.4 6.9 and 6.6, 2^18
    // at 0.5 8.4 and 8.1, 2^19 10.2 and 10.1; 2^20 14.6 either way.
    if (latticeKind != kLatticeBit) return 2u;
    const bool middle = L.maxColorCount > (1u << 16) && L.maxColorCount <= (1u << 19);
    return middle && max_degree(L) <= 2u && occupied_fraction(L) >= 0.4 ? 2u : 1u;
}

const std::vector<LaunchShape>& tune_candidates() {
    static const std::vector<LaunchShape> c = [] {
        std::vector<LaunchShape> v;
        for (uint32_t block : {64u, 128u, 192u, 256u})
            for (uint32_t slots : {1u, 2u, 4u}) {
                LaunchShape s;
                s.block = block;
                s.slots = slots;
                v.push_back(s);
            }
        return v;
    }();
    return c;
}

TuneResult autotune_system(int gpu, const SystemLayout& L, uint32_t latticeKind, uint64_t seed, uint32_t mcs) {
    if (L.nMonomers == 0) throw std::invalid_argument("autotune: empty system");
    const Key key = system_key(0, L, latticeKind, 1);
    {
        std::lock_guard<std::mutex> lock(g_cacheMutex);
        auto it = cache().find(key);
        if (it != cache().end()) {
            TuneResult r = it->second;
            r.cached = true;
            return r;
        }
    }
    hip_check(hipSetDevice(gpu), "hipSetDevice");
    hipStream_t st = nullptr;
    hip_check(hipStreamCreateWithFlags(&st, hipStreamNonBlocking), "hipStreamCreate");
    std::vector<TuneTrial> trials;
    try {
        for (const LaunchShape& s : tune_candidates()) trials.push_back({s, time_system(L, latticeKind, seed, s, mcs, st)});
    } catch (...) {
        (void)hipStreamDestroy(st);
        throw;
    }
    (void)hipStreamDestroy(st);
    TuneResult r = pick(std::move(trials));
    std::lock_guard<std::mutex> lock(g_cacheMutex);
    cache()[key] = r;
    return r;
}

TuneResult autotune_batch(int gpu, const std::vector<SystemLayout>& sample, const std::vector<uint64_t>& seeds,
                          uint32_t latticeKind, uint32_t mcs) {
    if (sample.empty() || sample.size() != seeds.size()) throw std::invalid_argument("autotune: empty sample");
    uint64_t monomers = 0;
    for (const SystemLayout& L : sample) monomers += L.nMonomers;
    Key key = system_key(1, sample.front(), latticeKind, uint32_t(sample.size()));
    std::get<5>(key) = log2_ceil(monomers);
    {
        std::lock_guard<std::mutex> lock(g_cacheMutex);
        auto it = cache().find(key);
        if (it != cache().end()) {
            TuneResult r = it->second;
            r.cached = true;
            return r;
        }
    }
    std::vector<TuneTrial> trials;
    for (const LaunchShape& s : tune_candidates()) {
        uint64_t tiles = 0;
        for (const SystemLayout& L : sample)
            tiles += std::max<uint32_t>(1u, tiles_for(L, s.block * s.slots));
        if (tiles > (uint64_t(1) << 26)) continue;
        Batch b(gpu, latticeKind, uint32_t(tiles), uint32_t(sample.size()), s.block, s.slots);
        for (size_t i = 0; i < sample.size(); ++i) b.add(sample[i], seeds[i]);
        // The warm-up has the timed run's length, so the graphs the timed runs
        // replay are captured outside them; the faster of two runs is kept.
        b.run(mcs);
        const double ms = std::min(b.run(mcs), b.run(mcs));
        trials.push_back({s, ms / std::max<uint32_t>(mcs, 1u)});
    }
    if (trials.empty()) throw std::runtime_error("autotune: no candidate fits");
    TuneResult r = pick(std::move(trials));
    std::lock_guard<std::mutex> lock(g_cacheMutex);
    cache()[key] = r;
    return r;
}

}  // namespace pscbfm
