// Scenarios of the workspace pool on the stand-in device: 1600 bytes, so 100 may stay idle and 100 held.
#include "device_memory.hpp"

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <optional>

using cfd_hip::HeldBlock;
using cfd_hip::Workspace;
using cfd_hip::WorkspacePool;

#define EXPECT(c)                                                            \
    do {                                                                     \
        if (!(c)) {                                                          \
            std::fprintf(stderr, "line %d: %s does not hold\n", __LINE__, #c); \
            std::exit(1);                                                    \
        }                                                                    \
    } while (0)

namespace {

WorkspacePool& pool = WorkspacePool::instance();

// A block that a finished call leaves idle.
unsigned char* leave_idle(size_t bytes) {
    Workspace w(bytes);
    w.finished();
    return w.get();
}

void reuse() {
    pool.enter();
    unsigned char* const first = leave_idle(80);
    EXPECT(pool.idle_bytes() == 80);
    EXPECT(leave_idle(60) == first && stub::mallocs == 1);  // reused, and idle again
    EXPECT(leave_idle(30) != first);                        // more than half of it would be wasted: a block of its own
    EXPECT(pool.idle_bytes() == 30);                        // 110 is over the bound: the oldest goes
    { Workspace failed(30); }                               // never finished: given back
    EXPECT(pool.idle_bytes() == 0);
    leave_idle(101);                                        // over the bound
    EXPECT(pool.idle_bytes() == 0 && stub::used == 0);
    leave_idle(50);
    pool.leave();
    EXPECT(stub::used == 0);
}

void full_device() {
    pool.enter();
    HeldBlock busy, rests;
    EXPECT(busy.take(40) && rests.take(40));
    rests.done();
    leave_idle(90);
    void* p = nullptr;
    EXPECT(cfd_hip::device_malloc(&p, stub::capacity - 40) == hipSuccess);  // all but the block in use
    EXPECT(pool.idle_bytes() == 0 && rests.bytes() == 0 && busy.bytes() == 40);
    EXPECT(cfd_hip::device_malloc(&p, 1) == hipErrorOutOfMemory);
    busy.done();
    EXPECT(cfd_hip::device_malloc(&p, 40) == hipSuccess);
    EXPECT(busy.bytes() == 0);
    EXPECT(!rests.take(40));  // full: the caller does without
    pool.leave();
}

void foreign_capture() {
    pool.enter();
    stub::capturing = true;
    HeldBlock h;
    EXPECT(h.take(40));
    EXPECT(!stub::broken && stub::mode == hipStreamCaptureModeGlobal);
    h.done();
    pool.leave();
}

void held_bound() {
    pool.enter();
    leave_idle(90);
    HeldBlock small;
    EXPECT(small.take(60));  // not the idle block: half as much again would be held
    EXPECT(small.bytes() == 60 && pool.idle_bytes() == 90);
    HeldBlock near, over;
    EXPECT(near.take(38));  // 98 of 100 held
    EXPECT(!over.take(3));
    near.done();
    pool.leave();
}

void held_close_fit() {
    pool.enter();
    unsigned char* const idle = leave_idle(88);
    HeldBlock h;
    EXPECT(h.take(80) == idle && h.bytes() == 88 && pool.idle_bytes() == 0);
    pool.leave();
}

void held_close_fit_over_the_bound() {
    pool.enter();
    leave_idle(54);
    HeldBlock first, second;
    EXPECT(first.take(48) && first.bytes() == 54);
    leave_idle(54);
    EXPECT(second.take(46) && second.bytes() == 46);  // 54 + 54 is more than 100
    EXPECT(pool.idle_bytes() == 54);
    pool.leave();
}

void held_bound_two_threads() {
    pool.enter();
    HeldBlock a, b;
    unsigned char* other = nullptr;
    stub::during_malloc = [&] { other = b.take(60); };  // what a second thread does meanwhile
    EXPECT(a.take(60));
    EXPECT(!other && stub::used == 60);
    pool.leave();
}

void held_again_after_a_full_device() {
    pool.enter();
    void* all = nullptr;
    EXPECT(hipMalloc(&all, stub::capacity) == hipSuccess);
    HeldBlock h;
    const size_t before = stub::mallocs;
    for (int k = 0; k < 10; ++k) EXPECT(!h.take(60));
    EXPECT(stub::mallocs == before + 1);  // a full device is not asked at every call
    (void)hipFree(all);
    int calls = 0;
    while (!h.take(60) && calls < 1000) ++calls;
    EXPECT(calls < 300 && h.bytes() == 60);
    pool.leave();
}

void held_again_after_a_failed_call() {
    pool.enter();
    HeldBlock h;
    stub::fail_next = true;
    EXPECT(!h.take(60));
    EXPECT(h.take(60));  // not a full device: asked again at the next call
    pool.leave();
}

void reclaimable() {
    pool.enter();
    HeldBlock busy, rests;
    EXPECT(busy.take(30) && rests.take(50));
    rests.done();
    leave_idle(90);
    EXPECT(pool.reclaimable_bytes() == 140);
    // What a caller counts on is there: free memory and the reclaimable bytes in one block.
    void* p = nullptr;
    EXPECT(cfd_hip::device_malloc(&p, stub::capacity - stub::used + 140) == hipSuccess);
    EXPECT(pool.reclaimable_bytes() == 0);
    pool.leave();
}

void release() {
    pool.enter();
    HeldBlock busy, rests;
    EXPECT(busy.take(30) && rests.take(40));
    rests.done();
    leave_idle(50);
    stub::device = 1;
    leave_idle(60);
    stub::device = 2;
    EXPECT(stub::used == 180);
    pool.release();
    EXPECT(stub::used == 30 && stub::device == 2);  // the block in use stays
    stub::device = 0;
    EXPECT(rests.take(40) && leave_idle(50));
    pool.leave();
}

}  // namespace

int main(int, char** argv) {
    const struct {
        const char* name;
        void (*run)();
    } all[] = {{"reuse", reuse}, {"full_device", full_device}, {"foreign_capture", foreign_capture},
                 {"held_bound", held_bound}, {"held_close_fit", held_close_fit},
                 {"held_close_fit_over_the_bound", held_close_fit_over_the_bound},
                 {"held_bound_two_threads", held_bound_two_threads},
                 {"held_again_after_a_full_device", held_again_after_a_full_device},
                 {"held_again_after_a_failed_call", held_again_after_a_failed_call},
                 {"reclaimable", reclaimable},
                 {"release", release}};
    for (const auto& s : all)
        if (std::strcmp(argv[1], s.name) == 0) return s.run(), 0;
    return 2;
}
