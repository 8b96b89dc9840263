// sp_slots.h -- equal slots of memory, lent for the length of a call.
//
// Pinned host memory costs about 0.15 ms a slot to get and to touch, and 1 ms
// and more to give back (the runtime waits for the whole device), many times
// what a small call takes.  So contexts and networks hold none of their own:
// they borrow slots and return them when the call ends.  Host code only.
#pragma once

#include <cstddef>
#include <mutex>

namespace sp {

constexpr size_t kSlotBytes = 256 << 10;

// Mem::get(void** p, size_t bytes) returns 0 or an error code, Mem::drop(void*)
// frees.  Between calls the pool keeps at most Keep slots; what comes back
// beyond them is freed.  Any number of threads may take and give at once.
template <class Mem, int Keep>
class SlotPool {
public:
    SlotPool() = default;
    SlotPool(const SlotPool&) = delete;
    SlotPool& operator=(const SlotPool&) = delete;

    // n slots into out, or none and Mem's error
    int take(void** out, int n) {
        int got = 0;
        {
            std::lock_guard<std::mutex> lk(mu_);
            while (got < n && idle_ > 0) out[got++] = slot_[--idle_];
        }
        int e = 0;
        for (; got < n && e == 0; ++got) e = Mem::get(&out[got], kSlotBytes);
        if (e != 0) give(out, got - 1);
        return e;
    }

    void give(void* const* s, int n) {
        int kept = 0;
        {
            std::lock_guard<std::mutex> lk(mu_);
            while (kept < n && idle_ < Keep) slot_[idle_++] = s[kept++];
        }
        for (; kept < n; ++kept) Mem::drop(s[kept]);
    }

private:
    std::mutex mu_;
    void* slot_[Keep] = {};
    int idle_ = 0;               // of them, the first are filled
};

}  // namespace sp
