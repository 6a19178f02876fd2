// Growth of an executor's device buffers.  It makes no device call of its own
// (mem.alloc / mem.release / mem.sync do), so that host tests can have an
// allocation fail.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <algorithm>

namespace srq {

struct DevBuf {
    void *p = nullptr;
    size_t n = 0;
};

// Grows b to at least `bytes`; false: mem.failed() says why, and b is empty or
// as it was.  A buffer that has to grow again takes half as much again as it
// held, so steps whose shapes creep up (the attention scratch gains a split
// every 64 positions) reallocate -- a stream synchronisation, a free and an
// allocation -- a logarithmic number of times.
template <class Mem>
bool grow(DevBuf &b, size_t bytes, Mem &mem) {
    if (bytes <= b.n) return true;
    size_t want = std::max(bytes, (size_t)256);
    if (b.p) {
        want = std::max(want, b.n + b.n / 2);
        if (!mem.sync() || !mem.release(b.p)) return false;
        b = DevBuf();
    }
    if (!mem.alloc(&b.p, want)) {
        b.p = nullptr;
        return false;
    }
    b.n = want;
    return true;
}

// A buffer that a call can do without.
struct OptionalBuf : DevBuf {
    size_t refused = SIZE_MAX;  // smallest size that could not be had
};

// Grows b to `bytes` and no more.  The old buffer stays until the new one is
// there, and a size once refused is not tried again: a failing allocation
// waits for the device, and every later call would pay for it.
template <class Mem>
bool grow_optional(OptionalBuf &b, size_t bytes, Mem &mem) {
    if (bytes <= b.n) return true;
    if (bytes >= b.refused) return false;
    void *p = nullptr;
    if (!mem.alloc(&p, bytes)) {
        b.refused = bytes;
        return false;
    }
    if (b.p && (!mem.sync() || !mem.release(b.p))) {
        (void)mem.release(p);
        return false;
    }
    b.p = p;
    b.n = bytes;
    return true;
}

// Frees b for a buffer that is needed; its size counts as refused from now
// on, so that the two do not take it from each other in turn.  False: nothing
// was freed.
template <class Mem>
bool give_back(OptionalBuf &b, Mem &mem) {
    if (!b.p || !mem.sync() || !mem.release(b.p)) return false;
    b.refused = std::min(b.refused, b.n);
    b.p = nullptr;
    b.n = 0;
    return true;
}

// grow() of a needed buffer, at the cost of the optional one where memory is
// short.
template <class Mem>
bool grow_or_give_back(DevBuf &b, size_t bytes, OptionalBuf &spare, Mem &mem) {
    return grow(b, bytes, mem) || (mem.out_of_memory() && give_back(spare, mem) && grow(b, bytes, mem));
}

}  // namespace srq
