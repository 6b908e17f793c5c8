/* A stream that a test drives, in place of the HIP runtime: copies are carried out when an event recorded after
   them, or the stream, is waited for, and the first wait lasts as long as the kernels queued before them would. */
#pragma once
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <thread>
#include <vector>

enum hipError_t { hipSuccess = 0, hipErrorUnknown = 999 };
enum hipMemcpyKind { hipMemcpyDeviceToHost = 2 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1 };
struct hipPointerAttribute_t {
    hipMemoryType type;
};
typedef int* hipStream_t;
struct StubEvent {
    size_t after = 0;   // copies queued before it
};
typedef StubEvent* hipEvent_t;
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;

namespace stub {
struct Copy {
    void* dst;
    const void* src;
    size_t n;
};
inline std::vector<Copy> queue;
inline size_t done = 0, copies = 0;
inline int busy_ms = 0;       // the stream's work before the next wait ends
inline long fail_at = -1;     // the copy that fails
inline void run(size_t upto) {
    std::this_thread::sleep_for(std::chrono::milliseconds(busy_ms));
    busy_ms = 0;
    for (; done < upto; ++done) std::memcpy(queue[done].dst, queue[done].src, queue[done].n);
}
}  // namespace stub

inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    if ((long)stub::copies++ == stub::fail_at) return hipErrorUnknown;
    stub::queue.push_back({d, s, n});
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { return e->after = stub::queue.size(), hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t e) { return stub::run(e->after), hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return stub::run(stub::queue.size()), hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = new StubEvent, hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { return delete e, hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return *p = std::malloc(n), hipSuccess; }
inline hipError_t hipHostFree(void* p) { return std::free(p), hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) {
    return a->type = hipMemoryTypeUnregistered, hipSuccess;
}
