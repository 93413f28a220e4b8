// A HIP runtime of host memory for CPU tests of the library's host code: it
// runs no kernel, but it keeps what a caller has to keep too: which handles
// are alive, what was launched where, and which work is known to be done.
#pragma once

#include <cstdint>
#include <set>
#include <string>
#include <vector>

namespace fake {

struct Launch {
    std::string kernel;  // mangled name
    uint32_t grid = 0, block = 0;
    void* stream = nullptr;
};

struct Runtime {
    // Launches in order, those of a replayed graph among them.
    std::vector<Launch> launches;
    // Memory freed, or written by the host, while work the caller had not
    // waited for could still use it; uses of handles that do not exist; work for
    // a stream of another than the current device.
    std::vector<std::string> violations;
    int failGraphLaunch = 0;  // fail the n-th graph launch from now on (1: the next)
    int failLaunch = 0;       // the same for kernels outside a capture
    uint64_t graphsBuilt = 0, streamsCreated = 0;
};
Runtime& runtime();
// All streams, events, graphs and memory of the devices (two) are gone.
void device_reset();
size_t live_streams();

}  // namespace fake
