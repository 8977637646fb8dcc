// The few runtime calls of lbm_amd/csrc/staging.h on the host, for
// staging_check.cpp: a stream is a queue whose copies and kernels (every thread of
// every block in turn) run only when something waits for them, as late as the real runtime may run them, so that a chunk
// refilled or read without a wait gives wrong bytes.
#pragma once

#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <vector>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1, hipMemoryTypeDevice = 2 };
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2, hipEventBlockingSync = 1;

struct hipPointerAttribute_t {
    hipMemoryType type;
};

struct FakeStream {
    std::vector<std::function<void()>> ops;
    size_t done = 0;
    void run(size_t upto) {
        for (; done < upto; ++done) ops[done]();
    }
};
struct FakeEvent {
    FakeStream *on = nullptr;
    size_t at = 0;
};
typedef FakeStream *hipStream_t;
typedef FakeEvent *hipEvent_t;

struct FakeHip {
    std::recursive_mutex lock;
    std::map<const char *, size_t> pinned;  // host allocations
    int host_mallocs = 0, copies = 0, launches = 0, fail_launch = -1, device = -1;
};
inline thread_local hipError_t fake_last = hipSuccess;
inline FakeHip &fake() {
    static FakeHip f;
    return f;
}
#define FAKE_LOCK std::lock_guard<std::recursive_mutex> guard_(fake().lock)

inline hipError_t fake_error(hipError_t e) {
    if (e != hipSuccess) fake_last = e;
    return e;
}
inline hipError_t hipGetLastError() {
    const hipError_t e = fake_last;
    fake_last = hipSuccess;
    return e;
}
inline hipError_t hipSetDevice(int dev) {
    FAKE_LOCK;
    fake().device = dev;
    return hipSuccess;
}
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    FAKE_LOCK;
    ++fake().host_mallocs;
    *p = std::malloc(n);
    fake().pinned[(const char *)*p] = n;
    return hipSuccess;
}
inline hipError_t hipHostFree(void *p) {
    FAKE_LOCK;
    fake().pinned.erase((const char *)p);
    std::free(p);
    return hipSuccess;
}
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
    FAKE_LOCK;
    auto it = fake().pinned.upper_bound((const char *)p);
    const bool known = it != fake().pinned.begin() && (--it, (const char *)p < it->first + it->second);
    if (!known) return fake_error(hipErrorInvalidValue);
    a->type = hipMemoryTypeHost;
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    *e = new FakeEvent;
    return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
    delete e;
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    FAKE_LOCK;
    e->on = s;
    e->at = s->ops.size();
    return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
    FAKE_LOCK;
    if (e->on) e->on->run(e->at);
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) {
    FAKE_LOCK;
    s->run(s->ops.size());
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind, hipStream_t s) {
    FAKE_LOCK;
    ++fake().copies;
    s->ops.push_back([=] { std::memcpy(dst, src, n); });
    return hipSuccess;
}

#define __global__
struct dim3 {
    unsigned x, y, z;
    dim3(unsigned x_ = 1, unsigned y_ = 1, unsigned z_ = 1) : x(x_), y(y_), z(z_) {}
};
inline thread_local dim3 blockIdx, threadIdx;
template <class... P, class... A>
void fake_launch(void (*kernel)(P...), dim3 grid, dim3 block, size_t, hipStream_t s, A... args) {
    FAKE_LOCK;
    if (fake().launches++ == fake().fail_launch) {
        fake_error(hipErrorUnknown);
        return;
    }
    s->ops.push_back([=] {
        for (blockIdx.x = 0; blockIdx.x < grid.x; ++blockIdx.x)
            for (threadIdx.x = 0; threadIdx.x < block.x; ++threadIdx.x) kernel(args...);
    });
}
#define hipLaunchKernelGGL fake_launch
