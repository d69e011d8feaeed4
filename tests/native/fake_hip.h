// A HIP runtime of host memory for tests without a GPU: one queue per stream whose
// copies run when something waits for them, and calls that fail on request.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <vector>

namespace fake {
inline std::recursive_mutex m;
inline std::map<hipStream_t, std::vector<std::function<void()>>> queue;
inline std::map<void *, size_t> allocated;                // live hipMalloc blocks
inline size_t memory = size_t(1) << 40, used = 0;         // device memory, and what is allocated of it
inline int record_fails_at = -1, sync_fails_at = -1;      // this call of hipEventRecord / hipEventSynchronize fails
inline int records = 0, syncs = 0;

inline void drain(hipStream_t st) {
    std::lock_guard<std::recursive_mutex> lock(m);
    auto work = std::move(queue[st]);
    queue[st].clear();
    for (auto &w : work) w();
}
inline size_t pending() {
    std::lock_guard<std::recursive_mutex> lock(m);
    size_t n = 0;
    for (auto &q : queue) n += q.second.size();
    return n;
}
}  // namespace fake

extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t bytes) {
    std::lock_guard<std::recursive_mutex> lock(fake::m);
    if (fake::used + bytes > fake::memory) return hipErrorOutOfMemory;
    *p = std::malloc(1);  // an address; device memory is never touched here
    fake::allocated[*p] = bytes;
    fake::used += bytes;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    std::lock_guard<std::recursive_mutex> lock(fake::m);
    if (!p) return hipSuccess;
    fake::used -= fake::allocated.at(p);
    fake::allocated.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) { return *p = std::malloc(bytes), hipSuccess; }
hipError_t hipHostFree(void *p) { return std::free(p), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return *e = reinterpret_cast<hipEvent_t>(new hipStream_t{}), hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { return delete reinterpret_cast<hipStream_t *>(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t st) {
    std::lock_guard<std::recursive_mutex> lock(fake::m);
    if (fake::records++ == fake::record_fails_at) return hipErrorUnknown;
    *reinterpret_cast<hipStream_t *>(e) = st;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    std::lock_guard<std::recursive_mutex> lock(fake::m);
    if (fake::syncs++ == fake::sync_fails_at) return hipErrorUnknown;
    fake::drain(*reinterpret_cast<hipStream_t *>(e));
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t st) { return fake::drain(st), hipSuccess; }
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes, hipMemcpyKind, hipStream_t st) {
    std::lock_guard<std::recursive_mutex> lock(fake::m);
    fake::queue[st].push_back([=] { std::memcpy(dst, src, bytes); });
    return hipSuccess;
}
}
