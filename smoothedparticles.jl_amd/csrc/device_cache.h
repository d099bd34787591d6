// A value looked up once per device; plain C++, so that a host program can run
// it.
#pragma once

#include <atomic>

namespace sph {

// The values (> 0) of the devices with ids below N.  Safe with several threads:
// two that miss at once ask twice and store the same value.  A failed query
// (a result <= 0) gives `fallback` for this time and is made again the next.
template <int N>
class DeviceCache {
public:
    template <class Query>
    int get(int device, int fallback, Query query)
    {
        const bool slot = device >= 0 && device < N;
        int v = slot ? value_[device].load(std::memory_order_relaxed) : 0;
        if (v > 0) return v;
        v = query(device);
        if (v <= 0) return fallback;
        if (slot) value_[device].store(v, std::memory_order_relaxed);
        return v;
    }

private:
    std::atomic<int> value_[N] = {};
};

}  // namespace sph
