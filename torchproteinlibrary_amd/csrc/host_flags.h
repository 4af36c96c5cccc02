// host_flags.h -- the host side of report.h's `flags`: words of pinned host
// memory that a kernel writes its status bits to, and the wait for them.
//
// The pool holds kSlots slots of one cache line each, allocated once per
// process and module.  A call takes a slot, launches, waits for its stream
// and gives the slot back, so a slot is never written by two calls; a call
// that finds none free waits for one (they are held only across a launch and
// its wait, by threads that need no lock of this one's).  A call whose launch
// fails waits too, since it may have put a first kernel on the stream; a slot
// whose wait fails may still be written and is never given out again.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <condition_variable>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

namespace host_flags {

constexpr int kSlots = 64, kWords = 16;  // words per slot: one 64-byte line
constexpr int kFlags = 8;                // of these, the words a kernel may write

class Pool {
  public:
    static Pool& get() {
        static Pool* p = new Pool;  // lives as long as the process: kernels may hold its memory
        return *p;
    }
    uint32_t* take() {
        std::unique_lock<std::mutex> lock(mu_);
        if (!base_) {
            void* m = nullptr;
            if (hipHostMalloc(&m, (size_t)kSlots * kWords * sizeof(uint32_t),
                              hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess)
                throw std::runtime_error("hipHostMalloc failed (status flags)");
            base_ = static_cast<uint32_t*>(m);
            for (int k = 0; k < kSlots; ++k) free_.push_back(k);
        }
        cv_.wait(lock, [this] { return !free_.empty() || lost_ == kSlots; });
        if (free_.empty()) throw std::runtime_error("no status flags left: the waits for them failed");
        const int k = free_.back();
        free_.pop_back();
        return base_ + (size_t)k * kWords;
    }
    void give(uint32_t* p) {
        {
            std::lock_guard<std::mutex> lock(mu_);
            free_.push_back((int)((p - base_) / kWords));
        }
        cv_.notify_one();
    }
    void lose() {
        {
            std::lock_guard<std::mutex> lock(mu_);
            ++lost_;
        }
        cv_.notify_all();
    }

  private:
    std::mutex mu_;
    std::condition_variable cv_;
    uint32_t* base_ = nullptr;
    std::vector<int> free_;
    int lost_ = 0;
};

// Calls launch(flags), which puts kernels on `stream`, waits for the stream
// and returns the bits they reported.
template <typename Launch>
uint32_t run(hipStream_t stream, Launch launch) {
    struct Slot {
        hipStream_t stream;
        uint32_t* p = Pool::get().take();
        bool waited = false;
        hipError_t wait() {
            const hipError_t e = hipStreamSynchronize(stream);
            waited = e == hipSuccess;
            return e;
        }
        ~Slot() {
            if (waited || wait() == hipSuccess)
                Pool::get().give(p);
            else
                Pool::get().lose();
        }
    } slot{stream};
    for (int k = 0; k < kFlags; ++k) __atomic_store_n(slot.p + k, 0u, __ATOMIC_RELEASE);
    launch(slot.p);
    if (slot.wait() != hipSuccess)
        throw std::runtime_error(std::string("hipStreamSynchronize failed: ") + hipGetErrorString(hipGetLastError()));
    uint32_t bits = 0;
    for (int k = 0; k < kFlags; ++k)
        if (__atomic_load_n(slot.p + k, __ATOMIC_ACQUIRE)) bits |= 1u << k;
    return bits;
}

}  // namespace host_flags
