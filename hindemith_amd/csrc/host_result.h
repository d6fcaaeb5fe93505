// Host copies of a program's results, kept with its record.
#pragma once

#include <atomic>
#include <cstdint>
#include <cstdlib>

namespace hmx {

// A result's host copy.  Pinned, and kept while the record lives: a fresh pageable one per
// run costs a page fault and a clearing pass per page besides a staged copy (the
// canonical program at 1920x1080, two planes: 5.24 ms a call, 4.59 with these).
// Pageable where the system refuses pinned memory or all records together hold
// PinnedBudget's limit of it.
struct HostResult {
    char *p = nullptr;
    int64_t cap = 0, bytes = 0;
    bool pinned = false;
};

// What all records may pin together (bytes).
class PinnedBudget {
public:
    explicit PinnedBudget(int64_t limit) : left_(limit) {}
    bool take(int64_t n) {
        int64_t left = left_.load();
        while (left >= n)
            if (left_.compare_exchange_weak(left, left - n)) return true;
        return false;
    }
    void give(int64_t n) { left_ += n; }

private:
    std::atomic<int64_t> left_;
};

// pin(size): pinned memory, or null where there is none; unpin frees it.
template <typename Unpin>
void host_result_free(HostResult &h, PinnedBudget &budget, Unpin &&unpin) {
    if (h.pinned) {
        unpin(h.p);
        budget.give(h.cap);
    } else {
        std::free(h.p);
    }
    h = HostResult();
}

// Room for `bytes` in h; false if there is no host memory left.
template <typename Pin, typename Unpin>
bool host_result_reserve(HostResult &h, int64_t bytes, PinnedBudget &budget, Pin &&pin,
                         Unpin &&unpin) {
    if (h.cap >= bytes) return true;
    host_result_free(h, budget, unpin);
    if (budget.take(bytes)) {
        h.p = static_cast<char *>(pin((size_t)bytes));
        h.pinned = h.p != nullptr;
        if (!h.pinned) budget.give(bytes);
    }
    if (!h.p) h.p = static_cast<char *>(std::malloc((size_t)bytes));
    if (h.p) h.cap = bytes;
    return h.p != nullptr;
}

}  // namespace hmx
