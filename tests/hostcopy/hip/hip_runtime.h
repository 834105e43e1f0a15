// The runtime calls of st_hostcopy.hip on the CPU, for a build without a GPU.  A stream is a
// queue that runs only when something waits for it, so that a transfer is as late as it can
// be; fail_record makes one event record fail, and copies counts the runtime's own copies.
#pragma once
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>

#define __global__
#define __launch_bounds__(n)

struct dim3 {
    unsigned x;
    dim3(unsigned v = 0) : x(v) {}
};
inline thread_local dim3 blockIdx, threadIdx;

enum hipError_t { hipSuccess, hipErrorUnknown, hipErrorNotReady };
enum { hipMemcpyHostToDevice, hipMemcpyDeviceToHost, hipHostMallocDefault = 0, hipEventDisableTiming = 0 };

struct SimStream {
    std::deque<std::function<void()>> ops;
    long queued = 0, done = 0;
    void run(long upto)
    {
        while (done < upto) {
            ops.front()();
            ops.pop_front();
            done++;
        }
    }
    void add(std::function<void()> f)
    {
        ops.push_back(f);
        queued++;
    }
};
typedef SimStream *hipStream_t;
typedef struct SimEvent {
    SimStream *s;
    long at;
} *hipEvent_t;

inline int fail_record = 0, copies = 0;  // fail_record: the how many-th record from now on
inline const void *pinned = nullptr;     // start of the one array that the runtime knows

enum hipMemoryType { hipMemoryTypeUnregistered, hipMemoryTypeHost, hipMemoryTypeDevice, hipMemoryTypeManaged };
struct hipPointerAttribute_t {
    hipMemoryType type;
};
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{
    if (p != pinned) return hipErrorUnknown;
    a->type = hipMemoryTypeHost;
    return hipSuccess;
}

inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    *p = aligned_alloc(4096, (n + 4095) / 4096 * 4096);
    return *p ? hipSuccess : hipErrorUnknown;
}
inline hipError_t hipHostFree(void *p)
{
    free(p);
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    *e = new SimEvent{nullptr, 0};
    return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e)
{
    delete e;
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    if (fail_record > 0 && --fail_record == 0) return hipErrorUnknown;
    e->s = s;
    e->at = s->queued;
    return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e)
{
    if (e->s) e->s->run(e->at);
    return hipSuccess;
}
inline hipError_t hipEventQuery(hipEvent_t e) { return e->s && e->s->done < e->at ? hipErrorNotReady : hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t s)
{
    s->run(s->queued);
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void *d, const void *src, size_t n, int, hipStream_t s)
{
    copies++;
    s->run(s->queued);
    memcpy(d, src, n);
    return hipSuccess;
}
#define hipLaunchKernelGGL(kernel, grid, block, lds, stream, ...)             \
    do {                                                                      \
        const unsigned g_ = (grid).x, b_ = (block).x;                         \
        (stream)->add([=] {                                                   \
            for (blockIdx.x = 0; blockIdx.x < g_; blockIdx.x++)               \
                for (threadIdx.x = 0; threadIdx.x < b_; threadIdx.x++) kernel(__VA_ARGS__); \
        });                                                                   \
    } while (0)
