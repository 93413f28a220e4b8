// See fake_hip.h.  Order is kept as vector clocks: a stream's clock counts the
// work given to it, events and waits carry clocks from stream to stream, and
// the host's clock holds what it has waited for.
#include "fake_hip.h"

#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>

#include "common.h"

namespace {

using Clock = std::map<const void*, uint64_t>;
void merge(Clock& into, const Clock& from) {
    for (const auto& [s, v] : from) into[s] = std::max(into[s], v);
}

struct Work {
    fake::Launch launch;
    // k_advance and the resident sweep count substeps in the state
    pscbfm::DevState* state = nullptr;
    uint64_t substeps = 0;
};
struct Graph {
    std::vector<Work> work;
};
struct Stream {
    Clock clock;
    int device = 0;
    std::unique_ptr<Graph> capture;
};
struct Event {
    Clock clock;
};
struct Global {
    fake::Runtime rt;
    std::map<void*, std::unique_ptr<Stream>> streams;
    std::map<void*, std::unique_ptr<Event>> events;
    std::map<void*, std::unique_ptr<Graph>> graphs;
    std::set<void*> device, pinned;
    std::map<const void*, std::string> kernels;
    Clock host;
    int current = 0;
    struct {
        dim3 grid, block;
        size_t lds;
        hipStream_t stream;
    } config;
};
Global& g() {
    static Global* p = new Global();  // kernels register themselves before main
    return *p;
}

Stream* find(hipStream_t s, const char* who) {
    const auto it = g().streams.find(s);
    if (it != g().streams.end()) return it->second.get();
    g().rt.violations.push_back(std::string(who) + ": no such stream");
    return nullptr;
}
// The stream to give work to.
Stream* target(hipStream_t s, const char* who) {
    Stream* st = find(s, who);
    if (st && st->device != g().current) g().rt.violations.push_back(std::string(who) + " on another device's stream");
    return st;
}
// Whether the host has waited for all work of all streams.
void host_touches(const char* who) {
    for (const auto& [s, st] : g().streams)
        for (const auto& [q, v] : st->clock)
            if (g().host[q] < v) {
                g().rt.violations.push_back(std::string(who) + " while work is running");
                return;
            }
}
void issue(hipStream_t s, Stream* st, const Work& w) {
    g().rt.launches.push_back(w.launch);
    g().rt.launches.back().stream = s;
    ++st->clock[s];
    if (w.state) w.state->substep += std::min<uint64_t>(w.substeps, w.state->stopAt - w.state->substep);
}
bool countdown(int& n) { return n > 0 && --n == 0; }

}  // namespace

namespace fake {
Runtime& runtime() { return g().rt; }
void device_reset() {
    g().streams.clear();
    g().events.clear();
    g().graphs.clear();
    for (void* p : g().device) std::free(p);
    for (void* p : g().pinned) std::free(p);
    g().device.clear();
    g().pinned.clear();
}
size_t live_streams() { return g().streams.size(); }
}  // namespace fake

extern "C" {

// the device code that the host objects name; there is none
uint64_t __hip_fatbin;
void** __hipRegisterFatBinary(const void*) { return reinterpret_cast<void**>(&__hip_fatbin); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, dim3*, dim3*, int*) {
    g().kernels[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s) {
    g().config = {grid, block, lds, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* s) {
    *grid = g().config.grid;
    *block = g().config.block;
    *lds = g().config.lds;
    *s = g().config.stream;
    return hipSuccess;
}

hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t, hipStream_t s) {
    Stream* st = target(s, "hipLaunchKernel");
    if (!st) return hipErrorInvalidHandle;
    Work w;
    w.launch.kernel = g().kernels[f];
    w.launch.grid = grid.x;
    w.launch.block = block.x;
    const std::string& name = w.launch.kernel;
    if (name.find("k_advance_batch") == std::string::npos && name.find("k_advance") != std::string::npos) {
        w.state = *static_cast<pscbfm::DevState**>(args[0]);
        w.substeps = *static_cast<uint32_t*>(args[1]);
    } else if (name.find("k_resident") != std::string::npos && name.find("batch") == std::string::npos) {
        w.state = static_cast<pscbfm::SysDesc*>(args[0])->state;
        w.substeps = *static_cast<uint32_t*>(args[1]);
    }
    if (st->capture) {
        st->capture->work.push_back(w);
        return hipSuccess;
    }
    if (countdown(g().rt.failLaunch)) return hipErrorLaunchFailure;
    issue(s, st, w);
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void* f, hipFuncAttribute, int) {
    return g().kernels.count(f) ? hipSuccess : hipErrorInvalidDeviceFunction;
}

hipError_t hipGetDeviceCount(int* n) { return *n = 2, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = g().current, hipSuccess; }
hipError_t hipSetDevice(int d) { return g().current = d, hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorName(hipError_t) { return "hipErrorFake"; }
const char* hipGetErrorString(hipError_t) { return "made by the test"; }

hipError_t hipMalloc(void** p, size_t n) {
    *p = std::calloc(n ? n : 1, 1);
    g().device.insert(*p);
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    host_touches("hipFree");
    if (g().device.erase(p) == 0) return hipErrorInvalidValue;
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = std::calloc(n ? n : 1, 1);
    g().pinned.insert(*p);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    if (g().pinned.erase(p) == 0) return hipErrorInvalidValue;
    std::free(p);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
    static void* scratch = std::calloc(4 << 20, 1);
    return *p = scratch, hipSuccess;
}
hipError_t hipMemcpy(void* dst, const void* src, size_t n, hipMemcpyKind) { return std::memcpy(dst, src, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t s) {
    if (!find(s, "hipMemcpyAsync")) return hipErrorInvalidHandle;
    std::memcpy(dst, src, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* dst, int v, size_t n, hipStream_t s) {
    if (!find(s, "hipMemsetAsync")) return hipErrorInvalidHandle;
    std::memset(dst, v, n);
    return hipSuccess;
}
hipError_t hipDeviceSynchronize(void) {
    for (const auto& kv : g().streams) merge(g().host, kv.second->clock);
    return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    auto st = std::make_unique<Stream>();
    st->device = g().current;
    *s = reinterpret_cast<hipStream_t>(std::calloc(1, 1));  // never freed: a handle is not given twice
    g().streams[*s] = std::move(st);
    ++g().rt.streamsCreated;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { return g().streams.erase(s) ? hipSuccess : hipErrorInvalidHandle; }
hipError_t hipStreamQuery(hipStream_t s) { return g().streams.count(s) ? hipSuccess : hipErrorInvalidHandle; }
hipError_t hipStreamSynchronize(hipStream_t s) {
    Stream* st = find(s, "hipStreamSynchronize");
    if (!st) return hipErrorInvalidHandle;
    merge(g().host, st->clock);
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    Stream* st = find(s, "hipStreamWaitEvent");
    if (!st || !g().events.count(e)) return hipErrorInvalidHandle;
    merge(st->clock, g().events[e]->clock);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    auto ev = std::make_unique<Event>();
    *e = reinterpret_cast<hipEvent_t>(ev.get());
    g().events[*e] = std::move(ev);
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { return g().events.erase(e) ? hipSuccess : hipErrorInvalidHandle; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    Stream* st = find(s, "hipEventRecord");
    if (!st || !g().events.count(e)) return hipErrorInvalidHandle;
    g().events[e]->clock = st->clock;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    if (!g().events.count(e)) return hipErrorInvalidHandle;
    merge(g().host, g().events[e]->clock);
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1.0f, hipSuccess; }

hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
    Stream* st = find(s, "hipStreamBeginCapture");
    if (!st) return hipErrorInvalidHandle;
    st->capture = std::make_unique<Graph>();
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* out) {
    Stream* st = find(s, "hipStreamEndCapture");
    if (!st || !st->capture) return hipErrorInvalidHandle;
    *out = reinterpret_cast<hipGraph_t>(st->capture.get());
    g().graphs[*out] = std::move(st->capture);
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* exec, hipGraph_t graph, hipGraphNode_t*, char*, size_t) {
    auto copy = std::make_unique<Graph>(*g().graphs[graph]);
    *exec = reinterpret_cast<hipGraphExec_t>(copy.get());
    g().graphs[*exec] = std::move(copy);
    ++g().rt.graphsBuilt;
    return hipSuccess;
}
hipError_t hipGraphUpload(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t graph) { return g().graphs.erase(graph) ? hipSuccess : hipErrorInvalidHandle; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { return g().graphs.erase(e) ? hipSuccess : hipErrorInvalidHandle; }
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t s) {
    Stream* st = target(s, "hipGraphLaunch");
    if (!st || !g().graphs.count(e)) return hipErrorInvalidHandle;
    if (countdown(g().rt.failGraphLaunch)) return hipErrorLaunchFailure;
    for (const Work& w : g().graphs[e]->work) issue(s, st, w);
    return hipSuccess;
}

}  // extern "C"
