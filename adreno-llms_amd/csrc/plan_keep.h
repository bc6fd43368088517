// Plans of the GEMM that a thread keeps.  Plain C++.
#pragma once
#include <cstddef>

namespace mi {

// All that a plan follows from; cus: of the device that mi_init set up last.
struct PlanKey {
    int mode = -1, cus = 0, kind = 0, M = 0, N = 0, K = 0;
    size_t bytes = 0;                                    // of workspace
    bool operator==(const PlanKey& o) const {
        return mode == o.mode && cus == o.cus && kind == o.kind && M == o.M && N == o.N && K == o.K && bytes == o.bytes;
    }
};

// make(), or what it gave this thread for the same key: the last 64 are kept, one per slot.  A plan takes a host 1 to 2 us to make, most
// of it estimates, where a layer's calls come again and again.
template <typename Plan, typename Make>
const Plan& kept_plan(const PlanKey& key, Make&& make) {
    struct Slot { PlanKey key; Plan plan; };
    constexpr unsigned kSlots = 64;
    thread_local Slot slots[kSlots];
    const unsigned h = (static_cast<unsigned>(key.N) * 2654435761u + static_cast<unsigned>(key.K) * 40503u +
                        static_cast<unsigned>(key.M) * 97u + static_cast<unsigned>(key.kind)) >> 7;
    Slot& s = slots[h % kSlots];
    if (!(s.key == key)) s = Slot{key, make()};
    return s.plan;
}

}  // namespace mi
