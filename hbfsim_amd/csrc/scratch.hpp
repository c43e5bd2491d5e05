// scratch.hpp -- device scratch that calls borrow from a per-device pool.
//
// hipMalloc and hipFree cost 0.1-0.3 ms each here (hipFree waits for the
// device), more than many a call's kernels: an unordered 8.4M-record run spent
// 2.5 of its 4.0 ms in them.  A call takes one block for all its scratch and
// gives it back once its stream has been synchronised, so a block never has
// two users, whatever threads and streams they are on.  The pool keeps at
// most kScratchKeep bytes of idle blocks per device; they are freed when the
// last engine or sampler is destroyed, and before an allocation that failed
// is tried again.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace hbfamd {

constexpr std::size_t kScratchKeep = std::size_t{512} << 20;

// A block of at least `bytes` on the current device, nullptr when there is
// no memory; its contents are unspecified.
void* scratch_take(std::size_t bytes);
// Returns a block that no queued work uses any more.
void scratch_give(void* block);
// Frees the idle blocks of the current device.
void scratch_trim();
// Engines and samplers hold the pool for as long as they live; the last one
// to drop it frees the idle blocks of every device.
void scratch_hold();
void scratch_drop();

// Holds the pool for the scope of a call that needs no engine or sampler: with
// none alive its blocks are freed when it returns.
class ScratchHold {
public:
    ScratchHold() { scratch_hold(); }
    ~ScratchHold() { scratch_drop(); }
    ScratchHold(const ScratchHold&) = delete;
    ScratchHold& operator=(const ScratchHold&) = delete;
};

// Lays out several arrays in one block, each 256-byte aligned.
struct ScratchPlan {
    std::size_t bytes = 0;
    template <typename T>
    std::size_t add(std::size_t count)
    {
        const std::size_t at = (bytes + 255) & ~std::size_t{255};
        bytes = at + sizeof(T) * (count == 0 ? 1 : count);
        return at;
    }
};

// One block for the scope of a call.  The destructor waits for the stream
// first, unless synced() was given a success: the result of a wait made after
// the last work queued on the block (an error instead of it, also one that
// kept the wait from being made, leaves the wait to the destructor).
class ScratchLease {
public:
    ScratchLease(std::size_t bytes, hipStream_t stream)
        : ptr_(scratch_take(bytes)), stream_(stream)
    {
    }
    ~ScratchLease() { release(); }
    ScratchLease(const ScratchLease&) = delete;
    ScratchLease& operator=(const ScratchLease&) = delete;
    bool ok() const { return ptr_ != nullptr; }
    template <typename T>
    T* at(std::size_t offset) const
    {
        return reinterpret_cast<T*>(static_cast<unsigned char*>(ptr_) + offset);
    }
    void synced(hipError_t waited) { idle_ = waited == hipSuccess; }
    void release()
    {
        if (ptr_ != nullptr) {
            if (!idle_) {
                (void)hipStreamSynchronize(stream_);
            }
            scratch_give(ptr_);
            ptr_ = nullptr;
        }
    }

private:
    void* ptr_;
    hipStream_t stream_;
    bool idle_ = false;
};

}  // namespace hbfamd
