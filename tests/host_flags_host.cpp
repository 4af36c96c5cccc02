// Host-only checks of the status slots (torchproteinlibrary_amd/csrc/host_flags.h),
// linked against the few runtime functions below instead of the HIP runtime:
// what a call leaves behind when its launch or its wait fails.  Exits 0, or with
// the number of the check that failed.
#include <cstdlib>

#include "host_flags.h"

static int waits = 0;
static bool failing = false;
static uint32_t* late = nullptr;  // written when the stream is waited for, as by a kernel in flight

extern "C" {
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = std::calloc(1, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    ++waits;
    if (failing) return hipErrorUnknown;
    if (late) *late = 1;
    late = nullptr;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipErrorUnknown; }
const char* hipGetErrorString(hipError_t) { return "made to fail"; }
}

template <typename Call>
static bool throws(Call call) {
    try {
        call();
    } catch (const std::exception&) {
        return true;
    }
    return false;
}

int main() {
    using host_flags::run;
    if (run(nullptr, [](uint32_t* f) { f[2] = 1; }) != 4u || waits != 1) return 1;
    if (run(nullptr, [](uint32_t*) {}) != 0u || waits != 2) return 2;
    // the second of two launches fails while the first still runs
    if (!throws([&] { run(nullptr, [&](uint32_t* f) { late = f; throw std::runtime_error("launch"); }); })) return 3;
    if (waits != 3 || late) return 4;  // it was waited for before the slot went back
    if (run(nullptr, [](uint32_t*) {}) != 0u) return 5;
    // a slot whose wait failed is not given out again
    failing = true;
    uint32_t* lost[host_flags::kSlots] = {};
    for (int k = 0; k < host_flags::kSlots; ++k) {
        if (!throws([&] { run(nullptr, [&](uint32_t* f) { lost[k] = f; }); })) return 6;
        for (int j = 0; j < k; ++j)
            if (lost[j] == lost[k]) return 7;
    }
    failing = false;
    if (!throws([&] { run(nullptr, [](uint32_t*) {}); })) return 8;  // none is left: an error, no wait for ever
    return 0;
}
