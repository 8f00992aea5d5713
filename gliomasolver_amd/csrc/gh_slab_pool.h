// gh_slab_pool.h -- the free staging slabs between transfers (gh_stage.hip).
#pragma once
#include <cstddef>
#include <vector>

namespace gh {

// Free slabs of all devices, not locked.  A Slab has a `device` and its size
// `bytes`; the sizes are few.  At most kPerSize slabs of a size are kept per
// device -- a limit over both sizes together let small slabs, which no large
// transfer can use, keep the large ones out: each was pinned and freed again per
// transfer (0.5 ms a MiB).
template <typename Slab>
struct SlabPool {
    static constexpr size_t kPerSize = 8;
    std::vector<Slab> slabs;

    // the smallest slab of `device` with at least `need` bytes
    bool take(int device, size_t need, Slab& s) {
        size_t best = slabs.size();
        for (size_t i = 0; i < slabs.size(); ++i)
            if (slabs[i].device == device && slabs[i].bytes >= need &&
                (best == slabs.size() || slabs[i].bytes < slabs[best].bytes))
                best = i;
        if (best == slabs.size()) return false;
        s = slabs[best];
        slabs.erase(slabs.begin() + best);
        return true;
    }
    // false: enough of its size are here
    bool give(const Slab& s) {
        if (ready(s.device, s.bytes) >= kPerSize) return false;
        slabs.push_back(s);
        return true;
    }
    size_t ready(int device, size_t bytes) const {
        size_t n = 0;
        for (const Slab& f : slabs) n += f.device == device && f.bytes == bytes;
        return n;
    }
};

}  // namespace gh
