// HIP entry points put in front of the runtime's for the builder's host-side
// tests: loaded with RTLD_GLOBAL before libsvo_hip.so, whose calls then come
// here first. All of them go on to the runtime.
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <chrono>
#include <condition_variable>
#include <map>
#include <mutex>
#include <set>

namespace {

std::mutex mu;
std::condition_variable cv;
std::map<hipEvent_t, std::set<hipStream_t>> recorded;
std::set<hipStream_t> streams;

int expected = 0, arrived = 0;
bool late = false;
thread_local bool met = false;

bool pinning = true;

template <typename F>
F real(const char *name) {
    void *h = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
    return reinterpret_cast<F>(dlsym(h, name));
}

}  // namespace

extern "C" {

// the most streams one event was recorded in; *distinct = streams recorded in
int shim_streams_per_event(int *distinct) {
    std::lock_guard<std::mutex> lock(mu);
    size_t most = 0;
    for (const auto &e : recorded) most = std::max(most, e.second.size());
    *distinct = int(streams.size());
    return int(most);
}

hipError_t hipEventRecord(hipEvent_t event, hipStream_t stream) {
    {
        std::lock_guard<std::mutex> lock(mu);
        recorded[event].insert(stream);
        streams.insert(stream);
    }
    return real<decltype(&hipEventRecord)>("hipEventRecord")(event, stream);
}

// From now on the first hipStreamSynchronize of each thread waits until
// `threads` threads have come to theirs, 5 s at most.
void shim_meet(int threads) {
    std::lock_guard<std::mutex> lock(mu);
    expected = threads;
    arrived = 0;
    late = false;
}

// whether they all came in time
int shim_met() {
    std::lock_guard<std::mutex> lock(mu);
    return arrived == expected && !late;
}

hipError_t hipStreamSynchronize(hipStream_t stream) {
    {
        std::unique_lock<std::mutex> lock(mu);
        if (expected && !met) {
            met = true;
            if (++arrived == expected) cv.notify_all();
            else if (!cv.wait_for(lock, std::chrono::seconds(5), [] { return arrived == expected; })) late = true;
        }
    }
    return real<decltype(&hipStreamSynchronize)>("hipStreamSynchronize")(stream);
}

// whether pinned memory can be had
void shim_pinning(int on) { pinning = on; }

hipError_t hipHostMalloc(void **ptr, size_t size, unsigned int flags) {
    if (!pinning) return hipErrorOutOfMemory;
    return real<hipError_t (*)(void **, size_t, unsigned int)>("hipHostMalloc")(ptr, size, flags);
}

}  // extern "C"
