// Host code of the library on the runtime of fake_hip.h: the order of work
// and memory on error paths, and what is launched where.  One case per call.
//
//   host_rt CASE
#include <cstdio>
#include <cstring>
#include <functional>
#include <map>
#include <memory>
#include <stdexcept>
#include <string>
#include <vector>

#include "batch.h"
#include "fake_hip.h"
#include "generators.h"
#include "updater.h"

using namespace pscbfm;

namespace {

int failures = 0;

void expect(bool ok, const std::string& what) {
    if (!ok) {
        std::fprintf(stderr, "FAIL: %s\n", what.c_str());
        ++failures;
    }
}
void expect_clean(const std::string& when) {
    for (const std::string& v : fake::runtime().violations) expect(false, when + ": " + v);
    fake::runtime().violations.clear();
}

// The 108 allowed bond vectors (standard set), indexed as copyBondSet takes them.
bool allowed(int x, int y, int z) {
    const int d = x * x + y * y + z * z;
    return d == 4 || d == 5 || d == 6 || d == 9 || d == 10;
}

// A system in a cubic box; bonds by pairs of monomers.
void stage(Updater& u, uint32_t edge, const std::vector<int32_t>& xyz, const std::vector<uint32_t>& bonds) {
    u.setGpu(0);
    u.setNrOfAllMonomers(uint32_t(xyz.size() / 3));
    u.setMonomerCoordinatesBulk(xyz.data(), uint32_t(xyz.size() / 3));
    for (size_t i = 0; i + 1 < bonds.size(); i += 2) {
        u.setConnectivity(bonds[i], bonds[i + 1]);
        u.setConnectivity(bonds[i + 1], bonds[i]);
    }
    u.setLatticeSize(edge, edge, edge);
    for (int x = -4; x < 4; ++x)
        for (int y = -4; y < 4; ++y)
            for (int z = -4; z < 4; ++z) u.copyBondSet(x, y, z, !allowed(x, y, z));
    u.setSeed(7);
}

// Stars of `arms` arms of 9 (6 for more than four), ends crosslinked.
void stage_stars(Updater& u, uint32_t edge, uint32_t stars, uint32_t arms) {
    const uint32_t box[3] = {edge, edge, edge};
    std::vector<int32_t> xyz;
    std::vector<uint32_t> bonds;
    if (!build_star_network(box, stars, arms, arms > 4 ? 6 : 9, 1, xyz, bonds)) throw std::runtime_error("box too small");
    stage(u, edge, xyz, bonds);
}

uint32_t add_stars(Batch& b, uint32_t edge, uint32_t stars, uint32_t arms) {
    Updater u;
    stage_stars(u, edge, stars, arms);
    const StagedSystem s = u.staged();
    return b.add(layout_of(s), s.seed, 0);
}

// n ordered dimers: two species of n members.
void stage_dimers(Updater& u, uint32_t edge, uint32_t n) {
    const uint32_t box[3] = {edge, edge, edge};
    std::vector<int32_t> xyz;
    if (!place_linear_chains_ordered(box, n, 2, xyz)) throw std::runtime_error("box too small");
    std::vector<uint32_t> bonds(2 * n);
    for (uint32_t i = 0; i < 2 * n; ++i) bonds[i] = i;
    stage(u, edge, xyz, bonds);
}

uint32_t add_dimers(Batch& b, uint32_t edge, uint32_t n) {
    Updater u;
    stage_dimers(u, edge, n);
    const StagedSystem s = u.staged();
    return b.add(layout_of(s), s.seed, 0);
}

// A launch that fails behind the resident launches of its batch: what the
// caller does next must not meet their workgroups still running.
void failed_launch_joins_the_side_stream() {
    for (const bool first : {true, false}) {
        Batch b(0, kLatticeBit, 0, 4, 256, 2);
        const uint32_t resident = add_dimers(b, 32, 100), large = add_dimers(b, 128, 20000);
        b.setTarget(resident, 50);
        b.setTarget(large, 50);
        b.launch(64);
        b.synchronize();
        expect_clean("a launch that succeeds");
        if (first)
            fake::runtime().failGraphLaunch = 1;
        else
            fake::runtime().failGraphLaunch = 2;  // 100 = a bulk graph and others
        bool threw = false;
        try {
            b.launch(100);
        } catch (const std::runtime_error&) {
            threw = true;
        }
        expect(threw, "the failed graph launch is reported");
        b.remove(resident);
        expect_clean("a replica removed after the failed launch");
        add_dimers(b, 64, 4000);
        b.synchronize();
        expect_clean("a replica added after the failed launch");
    }
    expect_clean("batches ended");
}

// Streams are handed on between owners, but none outlives the device's state:
// neither past the last owner nor past a reset under a live one.
void no_stream_outlives_a_device_reset() {
    auto use_updater = [] {
        Updater u;
        stage_dimers(u, 64, 4000);
        u.initialize();
        u.runSimulationOnGPU(3);
    };
    auto use_batch = [] {
        Batch b(0, kLatticeBit, 0, 2, 256, 2);
        b.setTarget(add_dimers(b, 32, 100), 5);
        b.launch(10);
        b.synchronize();
    };
    use_updater();
    use_batch();
    expect(fake::live_streams() == 0, "no owner, no stream");
    fake::device_reset();
    use_updater();
    use_batch();
    expect_clean("new owners after a reset");
    {
        Updater owner;
        stage_dimers(owner, 32, 100);
        owner.initialize();
        use_updater();
        use_batch();
        expect(fake::live_streams() == 4, "sets of one and of two wait for their next owner");
        const uint64_t made = fake::runtime().streamsCreated;
        use_updater();
        use_batch();
        expect(fake::runtime().streamsCreated == made, "and are handed on");
        fake::device_reset();
        use_updater();
        use_batch();
        expect_clean("new owners after a reset under a live one");
    }
    fake::runtime().violations.clear();  // the owner's own stream went with the reset
    expect(fake::live_streams() == 0, "no owner, no stream");
}

// A set of streams belongs to the device it was made on, whatever device its
// owner is told to use next.
void streams_stay_with_their_device() {
    Updater other, u;
    stage_dimers(other, 32, 100);
    other.setGpu(1);
    other.initialize();
    stage_dimers(u, 32, 100);
    u.initialize();
    u.runSimulationOnGPU(3);
    u.setGpu(1);
    u.destruct();
    stage_dimers(u, 64, 4000);
    u.setGpu(1);
    u.initialize();
    u.runSimulationOnGPU(3);
    u.cleanup();
    expect_clean("an updater moved to the other device");
}

// prepareGraphs builds what a run of that many sweeps replays, logged or not.
void prepared_graphs_serve_logged_runs() {
    for (const bool logged : {false, true}) {
        Updater u;
        stage_dimers(u, 128, 20000);
        u.initialize();
        u.prepareGraphs(150);  // 300 substeps: the bulk graph and the rest's
        const uint64_t built = fake::runtime().graphsBuilt;
        std::vector<uint32_t> log(300);
        u.run(150, logged ? log.data() : nullptr, false, true);
        expect(fake::runtime().graphsBuilt == built, logged ? "a logged run builds nothing" : "a run builds nothing");
    }
}

// Launches of a kernel by a batch of the replicas that `add` puts in.
struct Paths {
    bool resident = false, twoPass = false;
};
Paths paths(const std::function<void(Batch&)>& add) {
    Batch b(0, kLatticeBit, 0, 64, 256, 2);
    add(b);
    for (uint32_t i = 0; i < b.liveReplicas(); ++i) b.setTarget(i, 1);
    fake::runtime().launches.clear();
    b.launch(2);
    b.synchronize();
    Paths p;
    for (const fake::Launch& l : fake::runtime().launches) {
        p.resident = p.resident || l.kernel.find("k_resident") != std::string::npos;
        p.twoPass = p.twoPass || l.kernel.find("k_check_batch") != std::string::npos;
    }
    return p;
}

// Bonds cost the resident sweep more than the two-pass kernels: 5304 members of
// up to four bonds take 8.0 us per substep resident, where four such replicas
// take 6.5 on two passes.
void branched_replicas_take_the_faster_path() {
    const Paths few = paths([](Batch& b) { add_stars(b, 64, 430, 4); });
    expect(!few.resident && few.twoPass, "5304 members of up to four bonds: two passes");
    const Paths beside = paths([](Batch& b) {
        add_stars(b, 64, 430, 4);
        for (int k = 0; k < 4; ++k) add_dimers(b, 128, 40000);
    });
    expect(beside.resident && beside.twoPass, "beside longer two-pass work: resident");
    const Paths chains = paths([](Batch& b) { add_dimers(b, 64, 5120); });
    expect(chains.resident && !chains.twoPass, "5120 members of chains: resident");
    const Paths small = paths([](Batch& b) { add_stars(b, 64, 300, 4); });
    expect(small.resident && !small.twoPass, "3700 members of up to four bonds: resident");
}

// The same of a system on its own: three species, 37 members a star of four arms
// and 49 of eight.
void branched_systems_take_the_faster_path() {
    struct {
        uint32_t stars, arms, lattice;
        bool resident;
    } const cases[] = {{350, 4, kLatticeBit, true},  {380, 4, kLatticeBit, false}, {390, 4, kLatticeU8, true},
                       {160, 8, kLatticeBit, true},  {220, 8, kLatticeBit, false}, {220, 8, kLatticeU8, true},
                       {250, 8, kLatticeU8, false}};
    for (const auto& c : cases) {
        Updater u;
        stage_stars(u, 64, c.stars, c.arms);
        u.setLatticeKind(c.lattice);
        u.initialize();
        fake::runtime().launches.clear();
        u.runSimulationOnGPU(2);
        bool resident = false;
        for (const fake::Launch& l : fake::runtime().launches)
            resident = resident || l.kernel.find("k_resident") != std::string::npos;
        expect(resident == c.resident, std::to_string(c.stars) + " stars of " + std::to_string(c.arms) + " arms, lattice " +
                                           std::to_string(c.lattice));
    }
}

// Kernels take a state's buffers as they are: what they could not read whole
// entries from never reaches the device.
void misaligned_buffers_are_refused() {
    Updater u;
    stage_dimers(u, 32, 100);
    hipStream_t st = nullptr;
    hip_check(hipStreamCreateWithFlags(&st, hipStreamNonBlocking), "hipStreamCreate");
    DeviceSystem dev;
    dev.allocate(layout_of(u.staged()), kLatticeBit, 7, true, 64, st);
    const DevState good = dev.readState(st);
    alignas(8) static uint32_t buffer[8];
    const auto at = [](size_t bytes) { return reinterpret_cast<char*>(buffer) + bytes; };
    for (int field = 0; field < 3; ++field)
        for (const size_t bytes : {0, 1, 2, 4, 6}) {
            DevState s = good;
            if (field == 0) s.drawTable = reinterpret_cast<uint32_t*>(at(bytes));
            if (field == 1) s.log = reinterpret_cast<uint32_t*>(at(bytes));
            if (field == 2) s.acceptedByBlock = reinterpret_cast<uint64_t*>(at(bytes));
            bool refused = false;
            try {
                dev.writeState(s, st);
            } catch (const std::invalid_argument&) {
                refused = true;
            }
            expect(refused == (bytes % (field == 1 ? 4 : 8) != 0),
                   "field " + std::to_string(field) + " at " + std::to_string(bytes));
            dev.writeState(good, st);
        }
    dev.release();
    (void)hipStreamDestroy(st);
}

const std::map<std::string, std::function<void()>> cases = {
    {"failed_launch_joins_the_side_stream", failed_launch_joins_the_side_stream},
    {"no_stream_outlives_a_device_reset", no_stream_outlives_a_device_reset},
    {"streams_stay_with_their_device", streams_stay_with_their_device},
    {"prepared_graphs_serve_logged_runs", prepared_graphs_serve_logged_runs},
    {"branched_replicas_take_the_faster_path", branched_replicas_take_the_faster_path},
    {"branched_systems_take_the_faster_path", branched_systems_take_the_faster_path},
    {"misaligned_buffers_are_refused", misaligned_buffers_are_refused},
};

}  // namespace

int main(int argc, char** argv) {
    if (argc != 2 || !cases.count(argv[1])) return 2;
    try {
        cases.at(argv[1])();
    } catch (const std::exception& e) {
        std::fprintf(stderr, "FAIL: exception: %s\n", e.what());
        return 1;
    }
    if (failures) return 1;
    std::printf("%s: passed\n", argv[1]);
    return 0;
}
