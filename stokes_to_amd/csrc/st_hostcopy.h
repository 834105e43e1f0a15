// Copies between the caller's (pageable) arrays and the device through pinned slots.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <condition_variable>
#include <mutex>
#include <thread>
#include <vector>

namespace st {

class HostCopy {
public:
    HostCopy() = default;
    ~HostCopy();
    // the first half of the slots and threads now, for a context whose arrays have n bytes (the
    // second half, and without this call the first, are made on the first copy that needs them)
    void prepare(size_t n) { if (n >= MIN_OUT) ready(MIN_OUT); }
    // h may be read (out) or, unless it is memory that the runtime knows, changed (in) by the
    // caller when these return; the transfer of in() may still run on s
    hipError_t out(void *h, const void *d, size_t n, hipStream_t s);
    hipError_t in(void *d, const void *h, size_t n, hipStream_t s);

private:
    static constexpr size_t SLOT = 2u << 20;  // a slot of the ring
    static constexpr int NSLOT = 8, NTHREAD = 8;
    // smaller arrays than MIN_*: the runtime's own copy; from BIG on all slots and threads,
    // below it half of them
    static constexpr size_t MIN_OUT = 4u << 20, MIN_IN = 32u << 20, BIG = 32u << 20;

    bool ready(size_t n);
    void worker();
    void work();
    void open(bool to_host, char *h, size_t n);
    void close();
    void give_up(hipStream_t s);
    int sl(long k) const { return (int)(k % nslot_); }
    char *slot(long k) const { return pin_[sl(k) / (NSLOT / 2)] + (size_t)(sl(k) % (NSLOT / 2)) * SLOT; }
    size_t len(long k) const { return (size_t)(k + 1) * SLOT < n_ ? SLOT : n_ - (size_t)k * SLOT; }

    char *pin_[2] = {};  // half of the slots each
    int nslot_ = 0;
    hipEvent_t ev_[NSLOT] = {};
    bool used_[NSLOT] = {};  // ev_ recorded behind a transfer out of the slot
    bool broken_ = false;    // the stream could not be waited for after a failure: slots stay unused
    std::vector<std::thread> th_;
    std::mutex m_;
    std::condition_variable go_, idle_;
    bool open_ = false, stop_ = false;
    int in_job_ = 0;
    // the job: chunk k of h_ lies in slot sl(k); the threads copy the chunks below ready_
    // (drop_: a transfer failed, copy no more; set while threads copy)
    bool to_host_ = false;
    std::atomic<bool> drop_{false};
    char *h_ = nullptr;
    size_t n_ = 0;
    long nchunk_ = 0;
    std::atomic<long> next_{0}, ready_{0}, done_[NSLOT] = {};  // done_: 1 + last chunk copied
};

}  // namespace st
