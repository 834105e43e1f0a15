// Copies between the caller's arrays and the device (st_hostcopy.h).
//
// The runtime copies pageable memory through its own staging with one host thread: it is
// bound by that thread's copy and by the page faults of a fresh array.  Here an array goes
// through a ring of pinned slots: the calling thread issues the transfers, each a kernel
// that writes or reads the slot over the bus, and threads of the context copy between the
// slots and the array.  Device to host, 8.6 / 68 / 540 MB: 0.50 / 4.0 / 32 -> 0.27 / 1.5 /
// 11.4 ms (50 GB/s), into a fresh array of 540 MB in large pages 55 -> 14 ms.  Host to
// device, where the runtime is faster, 0.26 / 2.4 / 19 -> 0.33 / 2.1 / 15 ms, so only
// large arrays go this way.  With the copy engine instead of the kernel: 14 ms out and 14
// in, and 1 ms more on a stream's first use.  Slots of 1 MB: 31 GB/s instead of 41 with
// the engine; 4 threads take a fresh array twice as long as 8, 12 gain nothing; 32 MB of
// slots instead of 16 gain 2%.
#include "st_hostcopy.h"

#include <algorithm>
#include <cstring>

namespace st {

namespace {
typedef unsigned int w4 __attribute__((ext_vector_type(4)));
// one slot, written or read over the bus by the kernel itself
__global__ void __launch_bounds__(256) k_slot(w4 *__restrict__ d, const w4 *__restrict__ s, unsigned n16, unsigned tail)
{
    const unsigned i = blockIdx.x * 256u + threadIdx.x;
    if (i < n16) d[i] = s[i];
    if (i < tail) reinterpret_cast<char *>(d + n16)[i] = reinterpret_cast<const char *>(s + n16)[i];
}
hipError_t slot_copy(void *d, const void *s, size_t n, hipStream_t st)
{
    const unsigned n16 = (unsigned)(n / 16), tail = (unsigned)(n % 16);
    hipLaunchKernelGGL(k_slot, dim3(n16 / 256 + 1), dim3(256), 0, st, (w4 *)d, (const w4 *)s, n16, tail);
    return hipGetLastError();
}
bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }
// memory that the runtime knows (pinned, managed, of a device): it copies that itself, pinned
// memory at the rate of the bus (256^3, operator on pinned arrays: 19.8 ms, 25.7 by the slots)
// and memory that threads may not touch at all
bool known(const void *p)
{
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
    (void)hipGetLastError();
    return false;
}
}  // namespace

// slots and threads for an array of n bytes, made on first need (0.25 ms, 0.5 ms for the
// second half); false: use the runtime's copy
bool HostCopy::ready(size_t n)
{
    if (broken_) return false;
    const int half = n < BIG ? 1 : 2;
    for (int b = nslot_ / (NSLOT / 2); b < half; b++) {
        void *p = nullptr;
        bool ok = hipHostMalloc(&p, SLOT * (NSLOT / 2), hipHostMallocDefault) == hipSuccess;
        for (int k = b * (NSLOT / 2); ok && k < (b + 1) * (NSLOT / 2); k++)
            ok = ev_[k] || hipEventCreateWithFlags(&ev_[k], hipEventDisableTiming) == hipSuccess;
        if (!ok) {
            (void)hipGetLastError();
            if (p) hipHostFree(p);
            break;
        }
        pin_[b] = (char *)p;
        nslot_ += NSLOT / 2;
    }
    const unsigned hc = std::thread::hardware_concurrency();
    const size_t nt = std::min<size_t>(half * (NTHREAD / 2), hc > 1 ? hc : 1);
    try {
        while (th_.size() < nt) th_.emplace_back([this] { worker(); });
    } catch (...) {  // as many as there are
    }
    return nslot_ > 0 && !th_.empty();
}

HostCopy::~HostCopy()
{
    {
        std::lock_guard<std::mutex> l(m_);
        stop_ = true;
    }
    go_.notify_all();
    for (auto &t : th_) t.join();
    for (int k = 0; k < NSLOT; k++) {
        if (used_[k]) hipEventSynchronize(ev_[k]);
        if (ev_[k]) hipEventDestroy(ev_[k]);
    }
    for (char *p : pin_)
        if (p) hipHostFree(p);
}

void HostCopy::worker()
{
    std::unique_lock<std::mutex> l(m_);
    while (true) {
        go_.wait(l, [this] { return stop_ || (open_ && next_.load(std::memory_order_relaxed) < nchunk_); });
        if (stop_) return;
        in_job_++;
        l.unlock();
        work();
        l.lock();
        if (--in_job_ == 0) idle_.notify_all();
    }
}

void HostCopy::work()
{
    for (long k; (k = next_.fetch_add(1, std::memory_order_relaxed)) < nchunk_;) {
        while (ready_.load(std::memory_order_acquire) <= k) std::this_thread::yield();
        if (!drop_) {
            if (to_host_) memcpy(h_ + (size_t)k * SLOT, slot(k), len(k));
            else memcpy(slot(k), h_ + (size_t)k * SLOT, len(k));
        }
        done_[sl(k)].store(k + 1, std::memory_order_release);
    }
}

void HostCopy::open(bool to_host, char *h, size_t n)
{
    {
        std::lock_guard<std::mutex> l(m_);
        to_host_ = to_host;
        drop_ = false;
        h_ = h;
        n_ = n;
        nchunk_ = (long)((n + SLOT - 1) / SLOT);
        next_.store(0);
        ready_.store(0);
        for (auto &d : done_) d.store(0);
        open_ = true;
    }
    go_.notify_all();
}

void HostCopy::close()
{
    work();  // what no thread has taken yet
    std::unique_lock<std::mutex> l(m_);
    open_ = false;
    idle_.wait(l, [this] { return in_job_ == 0; });
}

// after a failed transfer: the threads copy no more, and what is queued on s has left the
// slots before they are used again
void HostCopy::give_up(hipStream_t s)
{
    drop_ = true;
    ready_.store(nchunk_, std::memory_order_release);
    if (hipStreamSynchronize(s) != hipSuccess) broken_ = true;
    for (bool &u : used_) u = false;
}

hipError_t HostCopy::out(void *h, const void *d, size_t n, hipStream_t s)
{
    if (n < MIN_OUT || !aligned16(d) || known(h) || !ready(n)) {
        const hipError_t e = hipMemcpyAsync(h, d, n, hipMemcpyDeviceToHost, s);
        return e != hipSuccess ? e : hipStreamSynchronize(s);
    }
    open(true, (char *)h, n);
    hipError_t e = hipSuccess;
    long issued = 0;
    for (long j = 0; j < nchunk_ && e == hipSuccess; j++) {
        // transfers ahead, as far as the slots are free (chunk j itself has to be issued)
        for (; issued < nchunk_ && issued < j + nslot_ && e == hipSuccess; issued++) {
            const long old = issued - nslot_;
            const int q = sl(issued);
            if (old >= 0 && done_[q].load(std::memory_order_acquire) != old + 1) {
                if (issued > j) break;
                while (done_[q].load(std::memory_order_acquire) != old + 1) std::this_thread::yield();
            }
            if (old < 0 && used_[q]) e = hipEventSynchronize(ev_[q]);  // an earlier in()
            if (e == hipSuccess)
                e = slot_copy(slot(issued), (const char *)d + (size_t)issued * SLOT, len(issued), s);
            if (e == hipSuccess) e = hipEventRecord(ev_[q], s);
            used_[q] = false;
        }
        if (e == hipSuccess) e = hipEventSynchronize(ev_[sl(j)]);
        if (e == hipSuccess) ready_.store(j + 1, std::memory_order_release);
    }
    if (e != hipSuccess) give_up(s);
    close();
    return e;
}

hipError_t HostCopy::in(void *d, const void *h, size_t n, hipStream_t s)
{
    if (n < MIN_IN || !aligned16(d) || known(h) || !ready(n)) return hipMemcpyAsync(d, h, n, hipMemcpyHostToDevice, s);
    open(false, (char *)const_cast<void *>(h), n);
    hipError_t e = hipSuccess;
    long freed = 0;
    for (long j = 0; j < nchunk_ && e == hipSuccess; j++) {
        // slots whose last transfer is over may be filled (chunk j's has to be)
        for (; freed < nchunk_ && freed < j + nslot_ && e == hipSuccess; freed++) {
            const int q = sl(freed);
            if (used_[q]) {
                if (freed > j && hipEventQuery(ev_[q]) == hipErrorNotReady) break;
                e = hipEventSynchronize(ev_[q]);
            }
            if (e == hipSuccess) {
                used_[q] = false;
                ready_.store(freed + 1, std::memory_order_release);
            }
        }
        const int q = sl(j);
        while (e == hipSuccess && done_[q].load(std::memory_order_acquire) != j + 1) std::this_thread::yield();
        if (e == hipSuccess) e = slot_copy((char *)d + (size_t)j * SLOT, slot(j), len(j), s);
        if (e == hipSuccess) e = hipEventRecord(ev_[q], s);
        if (e == hipSuccess) used_[q] = true;
    }
    if (e != hipSuccess) give_up(s);
    close();
    return e;
}

}  // namespace st
