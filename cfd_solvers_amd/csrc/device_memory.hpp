// device_memory.hpp -- device allocation, and workspaces handed from call to call.
//
// hipMalloc and hipFree of a large block cost far more than the kernels that use it: mapping and
// clearing run at about 40 GB/s, so the 16.8 GB of checkpoint states of a 200-step two-level adjoint
// on 128^3 took 410 ms of a 457 ms call.  A call that needs such a block for its own duration takes it
// from WorkspacePool (Workspace), which keeps the blocks of finished calls for the next one, of
// whichever solver; a block that one object wants at every call it holds itself (HeldBlock).  Neither
// holds a state between calls.  Idle and held blocks are each bounded to 1 / kKeptFraction of the
// device's memory, and both are given back before any allocation of this library fails, with the last
// solver, or at cfd_lbm_release_workspaces: other allocators cannot reclaim them.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

namespace cfd_hip {

class HeldBlock;

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
    // What trim() would give back: the current device's idle blocks and the held ones that no call is
    // using.  A budget of the device's memory counts them as free.
    size_t reclaimable_bytes() {
        const std::lock_guard<std::mutex> lock(mutex_);
        const int device = current_device();
        return idle_bytes_locked(device) + held_bytes_locked(device, false);
    }
    // Gives back the current device's idle blocks and the held ones that no call is using; false if
    // there were none.
    bool trim();
    // trim() on every device that has blocks.
    void release();
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
    friend class HeldBlock;
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
    size_t held_bytes_locked(int device, bool busy_too) const;
    // The smallest idle block of the device with `bytes` to `most` bytes, no longer idle; null if none.
    unsigned char* take_idle_locked(int device, size_t bytes, size_t most, size_t* got);
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

    static size_t bound() {
        size_t total = 0;
        return hipDeviceTotalMem(&total, current_device()) == hipSuccess ? total / kKeptFraction : 0;
    }

    std::mutex mutex_;
    std::vector<Block> idle_;  // oldest first
    std::vector<HeldBlock*> held_;
    size_t users_ = 0;
};

// For its lifetime the calling thread may allocate although some stream, of whichever thread, is being
// captured: hipMalloc records nothing, but under a capture in global mode (torch's default) it fails
// and ends that capture.
class AllocationDuringCapture {
  public:
    AllocationDuringCapture() { set_ = hipThreadExchangeStreamCaptureMode(&mode_) == hipSuccess; }
    ~AllocationDuringCapture() {
        if (set_) (void)hipThreadExchangeStreamCaptureMode(&mode_);
    }
    AllocationDuringCapture(const AllocationDuringCapture&) = delete;
    AllocationDuringCapture& operator=(const AllocationDuringCapture&) = delete;

  private:
    hipStreamCaptureMode mode_ = hipStreamCaptureModeRelaxed;
    bool set_ = false;
};

// A block that its owner keeps from call to call: take() before its use, done() once the work on it
// has been launched (on one stream, which the owner waits for before it goes).  Between the two calls
// a full device may take it away, after waiting for that work.
class HeldBlock {
  public:
    HeldBlock() = default;
    HeldBlock(const HeldBlock&) = delete;
    HeldBlock& operator=(const HeldBlock&) = delete;
    ~HeldBlock() {
        WorkspacePool& pool = WorkspacePool::instance();
        {
            const std::lock_guard<std::mutex> lock(pool.mutex_);
            forget(pool);
        }
        if (ptr_) pool.put(ptr_, bytes_, true);
    }
    // The block, of `bytes` bytes at every call; null if there is no room for it.
    unsigned char* take(size_t bytes);
    void done() {
        const std::lock_guard<std::mutex> lock(WorkspacePool::instance().mutex_);
        busy_ = false;
    }
    size_t bytes() const {
        const std::lock_guard<std::mutex> lock(WorkspacePool::instance().mutex_);
        return bytes_;
    }

  private:
    friend class WorkspacePool;
    void forget(WorkspacePool& pool) {  // with the pool locked
        for (size_t k = 0; k < pool.held_.size(); ++k)
            if (pool.held_[k] == this) {
                pool.held_.erase(pool.held_.begin() + static_cast<std::ptrdiff_t>(k));
                return;
            }
    }
    unsigned char* ptr_ = nullptr;
    size_t bytes_ = 0;
    int device_ = 0;
    bool busy_ = false;
    // Takes still to pass before a device that was full is asked again: another owner may have freed
    // memory by then, and a failing hipMalloc at every call is not worth its time.
    static constexpr unsigned kPause = 255;
    unsigned pause_ = 0;
};

inline bool WorkspacePool::trim() {
    const std::lock_guard<std::mutex> lock(mutex_);
    const int device = current_device();
    bool any = trim_locked(device, 0);
    for (size_t k = held_.size(); k-- > 0;) {
        HeldBlock* const h = held_[k];
        if (h->busy_ || h->device_ != device) continue;
        (void)hipFree(h->ptr_);  // waits for the device, and with it for the block's last use
        h->ptr_ = nullptr;
        h->bytes_ = 0;
        held_.erase(held_.begin() + static_cast<std::ptrdiff_t>(k));
        any = true;
    }
    return any;
}

inline void WorkspacePool::release() {
    std::vector<int> devices;
    {
        const std::lock_guard<std::mutex> lock(mutex_);
        for (const Block& b : idle_) devices.push_back(b.device);
        for (const HeldBlock* h : held_) devices.push_back(h->device_);
    }
    std::sort(devices.begin(), devices.end());
    devices.erase(std::unique(devices.begin(), devices.end()), devices.end());
    const int before = current_device();
    for (const int d : devices)
        if (hipSetDevice(d) == hipSuccess) (void)trim();
    if (!devices.empty()) (void)hipSetDevice(before);
}

// hipMalloc on the current device; when that finds the device full, once more after the idle
// workspaces have been given back.
inline hipError_t device_malloc(void** p, size_t bytes) {
    const hipError_t e = hipMalloc(p, bytes);
    if (e != hipErrorOutOfMemory || !WorkspacePool::instance().trim()) return e;
    (void)hipGetLastError();
    return hipMalloc(p, bytes);
}

inline size_t WorkspacePool::held_bytes_locked(int device, bool busy_too) const {
    size_t sum = 0;
    for (const HeldBlock* h : held_)
        if (h->device_ == device && (busy_too || !h->busy_)) sum += h->bytes_;
    return sum;
}

inline unsigned char* WorkspacePool::take_idle_locked(int device, size_t bytes, size_t most, size_t* got) {
    size_t best = idle_.size();
    for (size_t k = 0; k < idle_.size(); ++k)
        if (idle_[k].device == device && idle_[k].bytes >= bytes && idle_[k].bytes <= most &&
            (best == idle_.size() || idle_[k].bytes < idle_[best].bytes))
            best = k;
    if (best == idle_.size()) return nullptr;
    unsigned char* const p = idle_[best].ptr;
    *got = idle_[best].bytes;
    idle_.erase(idle_.begin() + static_cast<std::ptrdiff_t>(best));
    return p;
}

inline unsigned char* WorkspacePool::take(size_t bytes, size_t* got) {
    {  // an idle block, unless it would waste more than half of it
        const std::lock_guard<std::mutex> lock(mutex_);
        if (unsigned char* const p = take_idle_locked(current_device(), bytes, 2 * bytes + 1, got)) return p;
    }
    void* p = nullptr;
    if (const hipError_t e = device_malloc(&p, bytes); e != hipSuccess)
        throw std::runtime_error(std::string("hipMalloc: ") + hipGetErrorString(e));
    *got = bytes;
    return static_cast<unsigned char*>(p);
}

inline void WorkspacePool::put(unsigned char* ptr, size_t bytes, bool keep) {
    const std::lock_guard<std::mutex> lock(mutex_);
    if (const size_t most = bound(); keep && users_ > 0 && bytes <= most) {
        const int device = current_device();
        try {
            trim_locked(device, most - bytes);
            idle_.push_back(Block{ptr, bytes, device});
            return;
        } catch (...) {  // no host memory for the list: give the block back
        }
    }
    (void)hipFree(ptr);
}

inline unsigned char* HeldBlock::take(size_t bytes) {
    WorkspacePool& pool = WorkspacePool::instance();
    {
        const std::lock_guard<std::mutex> lock(pool.mutex_);
        if (ptr_) {
            busy_ = true;
            return ptr_;
        }
        if (pause_ > 0) {
            --pause_;
            return nullptr;
        }
        const int device = WorkspacePool::current_device();
        const size_t held = pool.held_bytes_locked(device, true), bound = WorkspacePool::bound();
        if (held > bound || bytes > bound - held) return nullptr;
        try {
            pool.held_.push_back(this);
        } catch (...) {  // no host memory for the list
            return nullptr;
        }
        // Entered before the allocation, so that the next one to ask counts it.  An idle block is held
        // whole: only one of nearly the size that fits the bound too.
        device_ = device;
        bytes_ = bytes;
        busy_ = true;
        size_t got = 0;
        if (unsigned char* const p =
                pool.take_idle_locked(device, bytes, std::min(bytes + bytes / 8, bound - held), &got)) {
            ptr_ = p;
            bytes_ = got;
            return ptr_;
        }
    }
    // A plain hipMalloc: what the caller can do without takes no block from another owner.
    void* fresh = nullptr;
    hipError_t e;
    {
        const AllocationDuringCapture permit;  // a caller that steps expects no allocation
        e = hipMalloc(&fresh, bytes);
    }
    const std::lock_guard<std::mutex> lock(pool.mutex_);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        if (e == hipErrorOutOfMemory) pause_ = kPause;
        forget(pool);
        bytes_ = 0;
        busy_ = false;
        return nullptr;
    }
    ptr_ = static_cast<unsigned char*>(fresh);
    return ptr_;
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
