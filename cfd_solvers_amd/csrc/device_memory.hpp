// device_memory.hpp -- device allocation, and workspaces handed from call to call.
//
// hipMalloc and hipFree of a large block cost far more than the kernels that use it: mapping and
// clearing run at about 40 GB/s, so the 16.8 GB of checkpoint states of a 200-step two-level adjoint
// on 128^3 took 410 ms of a 457 ms call.  A call that needs such a block for its own duration takes it
// from WorkspacePool, which keeps the blocks of finished calls for the next one, of whichever solver:
// at most kKeptFraction of the device's memory, given back when the last solver goes and before any
// allocation of this library fails.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

namespace cfd_hip {

class WorkspacePool {
  public:
    // The idle blocks together hold at most this fraction of a device's memory (the adjoint's
    // automatic snapshot count leaves the same fraction of the free memory unused).
    static constexpr size_t kKeptFraction = 16;

    static WorkspacePool& instance() {
        static WorkspacePool* p = new WorkspacePool;  // outlives every user
        return *p;
    }

    // A block of at least `bytes` on the current device, for the caller alone until put().
    unsigned char* take(size_t bytes, size_t* got);
    // Ends the use of a block of the current device; no work that uses it is pending.
    void put(unsigned char* ptr, size_t bytes, bool keep);
    // Bytes of the idle blocks on the current device.
    size_t idle_bytes() {
        const std::lock_guard<std::mutex> lock(mutex_);
        return idle_bytes_locked(current_device());
    }
    // Gives back the idle blocks of the current device; false if there were none.
    bool trim() {
        const std::lock_guard<std::mutex> lock(mutex_);
        return trim_locked(current_device(), 0);
    }
    // Users (solvers) alive; the last one to leave gives back every idle block.
    void enter() {
        const std::lock_guard<std::mutex> lock(mutex_);
        ++users_;
    }
    void leave() {
        const std::lock_guard<std::mutex> lock(mutex_);
        if (--users_ == 0) {
            for (const Block& b : idle_) (void)hipFree(b.ptr);
            idle_.clear();
        }
    }

  private:
    struct Block {
        unsigned char* ptr;
        size_t bytes;
        int device;
    };
    static int current_device() {
        int d = 0;
        (void)hipGetDevice(&d);
        return d;
    }
    size_t idle_bytes_locked(int device) const {
        size_t sum = 0;
        for (const Block& b : idle_)
            if (b.device == device) sum += b.bytes;
        return sum;
    }
    // Frees the oldest idle blocks of the device until at most `limit` bytes are idle.
    bool trim_locked(int device, size_t limit) {
        bool any = false;
        for (size_t k = 0; k < idle_.size() && idle_bytes_locked(device) > limit;) {
            if (idle_[k].device != device) {
                ++k;
                continue;
            }
            (void)hipFree(idle_[k].ptr);
            idle_.erase(idle_.begin() + static_cast<std::ptrdiff_t>(k));
            any = true;
        }
        return any;
    }

    std::mutex mutex_;
    std::vector<Block> idle_;  // oldest first
    size_t users_ = 0;
};

// hipMalloc on the current device; when that finds the device full, once more after the idle
// workspaces have been given back.
inline hipError_t device_malloc(void** p, size_t bytes) {
    const hipError_t e = hipMalloc(p, bytes);
    if (e != hipErrorOutOfMemory || !WorkspacePool::instance().trim()) return e;
    (void)hipGetLastError();
    return hipMalloc(p, bytes);
}

inline unsigned char* WorkspacePool::take(size_t bytes, size_t* got) {
    {
        // The smallest idle block that holds the request, unless it would waste more than half of it.
        const std::lock_guard<std::mutex> lock(mutex_);
        const int device = current_device();
        size_t best = idle_.size();
        for (size_t k = 0; k < idle_.size(); ++k)
            if (idle_[k].device == device && idle_[k].bytes >= bytes && idle_[k].bytes / 2 <= bytes &&
                (best == idle_.size() || idle_[k].bytes < idle_[best].bytes))
                best = k;
        if (best < idle_.size()) {
            unsigned char* const p = idle_[best].ptr;
            *got = idle_[best].bytes;
            idle_.erase(idle_.begin() + static_cast<std::ptrdiff_t>(best));
            return p;
        }
    }
    void* p = nullptr;
    if (const hipError_t e = device_malloc(&p, bytes); e != hipSuccess)
        throw std::runtime_error(std::string("hipMalloc: ") + hipGetErrorString(e));
    *got = bytes;
    return static_cast<unsigned char*>(p);
}

inline void WorkspacePool::put(unsigned char* ptr, size_t bytes, bool keep) {
    const std::lock_guard<std::mutex> lock(mutex_);
    size_t free_b = 0, total = 0;
    if (keep && users_ > 0 && hipMemGetInfo(&free_b, &total) == hipSuccess && bytes <= total / kKeptFraction) {
        const int device = current_device();
        try {
            trim_locked(device, total / kKeptFraction - bytes);
            idle_.push_back(Block{ptr, bytes, device});
            return;
        } catch (...) {  // no host memory for the list: give the block back
        }
    }
    (void)hipFree(ptr);
}

// One block of the pool for the duration of a scope.  On the way out of a failed call the block is
// freed, which waits for whatever was launched on it.
class Workspace {
  public:
    explicit Workspace(size_t bytes) { ptr_ = WorkspacePool::instance().take(bytes, &bytes_); }
    ~Workspace() { WorkspacePool::instance().put(ptr_, bytes_, keep_); }
    Workspace(const Workspace&) = delete;
    Workspace& operator=(const Workspace&) = delete;
    unsigned char* get() const { return ptr_; }
    // The work on the block has completed: it may serve the next call.
    void finished() { keep_ = true; }

  private:
    unsigned char* ptr_ = nullptr;
    size_t bytes_ = 0;
    bool keep_ = false;
};

}  // namespace cfd_hip
