// Host copies of results: pinned within the budget, pageable beyond it or where pinned
// memory is refused, and the budget given back.  Prints "ok".
#include <cstdio>
#include <cstring>
#include <vector>

#include "../hindemith_amd/csrc/host_result.h"

using namespace hmx;

static bool refuse = false;
static int pins = 0, unpins = 0;
static void *pin(size_t n) {
    if (refuse) return nullptr;
    ++pins;
    return std::malloc(n);
}
static void unpin(void *p) {
    ++unpins;
    std::free(p);
}
#define CHECK(x)                                     \
    do {                                             \
        if (!(x)) {                                  \
            std::printf("line %d: %s\n", __LINE__, #x); \
            return 1;                                \
        }                                            \
    } while (0)

int main() {
    PinnedBudget budget(1000);
    HostResult a, b, c, z;
    auto reserve = [&](HostResult &h, int64_t n) {
        return host_result_reserve(h, n, budget, pin, unpin);
    };
    auto release = [&](HostResult &h) { host_result_free(h, budget, unpin); };
    CHECK(reserve(z, 0) && !z.p && !z.pinned);  // an empty result takes nothing
    CHECK(reserve(a, 600) && a.pinned && a.cap == 600);
    char *const p = a.p;
    CHECK(reserve(a, 500) && a.p == p && pins == 1);  // room already
    CHECK(reserve(b, 600) && !b.pinned && b.cap == 600 && pins == 1);  // beyond the budget
    std::memset(b.p, 1, 600);
    CHECK(reserve(c, 400) && c.pinned);  // the rest of it
    release(c);
    CHECK(!c.p && c.cap == 0 && unpins == 1);
    CHECK(reserve(a, 1000) && a.pinned && unpins == 2);  // grown: its own 600 given back first
    release(a);
    refuse = true;  // the system refuses: pageable, and the budget is whole again
    CHECK(reserve(a, 1000) && !a.pinned && a.cap == 1000);
    std::memset(a.p, 1, 1000);
    refuse = false;
    CHECK(reserve(c, 1000) && c.pinned);
    release(a);
    release(b);
    release(c);
    release(z);
    CHECK(budget.take(1000) && !budget.take(1) && pins == unpins);
    std::printf("ok\n");
    return 0;
}
