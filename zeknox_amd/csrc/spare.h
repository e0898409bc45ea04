// Working memory that its user can do without: it grows on demand, keeps what
// it has when it cannot grow, does not ask again on each call once it has been
// refused, and can be dropped at any time that nothing runs on it.
// Host-only; not synchronised (Device::spare_mu guards the device's).
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <algorithm>

namespace zkx {

class SpareMemory {
public:
    using Alloc = void *(*)(size_t);  // null when there is none
    using Free = void (*)(void *);    // waits for what still runs on it

    // After a refusal, this many calls that need as much or more make do with
    // what is there: a refused allocation costs a call more than the memory
    // saves it.
    static constexpr uint32_t kRefusedCalls = 64;

    SpareMemory(Alloc alloc, Free free) : alloc_(alloc), free_(free) {}
    ~SpareMemory() { drop(); }
    SpareMemory(const SpareMemory &) = delete;
    SpareMemory &operator=(const SpareMemory &) = delete;

    void *get() const { return p_; }
    size_t bytes() const { return bytes_; }

    // Makes room for `want` units of `unit` bytes if it can; returns how many
    // of them (at most `want`, possibly none) there is room for.
    uint64_t hold(uint64_t want, size_t unit)
    {
        const size_t need = (size_t)want * unit;
        if (bytes_ < need) {
            if (skip_ && need >= refused_) {
                skip_--;
            } else if (void *p = alloc_(need)) {
                drop();
                p_ = p;
                bytes_ = need;
            } else {
                refused_ = need;
                skip_ = kRefusedCalls;
            }
        }
        return std::min<uint64_t>(want, bytes_ / unit);
    }

    // Whether there was anything to give back.
    bool drop()
    {
        skip_ = 0;
        if (!p_) return false;
        free_(p_);
        p_ = nullptr;
        bytes_ = 0;
        return true;
    }

private:
    Alloc alloc_;
    Free free_;
    void *p_ = nullptr;
    size_t bytes_ = 0;
    size_t refused_ = 0;  // size of the last refusal
    uint32_t skip_ = 0;   // calls that still take it for an answer
};

}  // namespace zkx
