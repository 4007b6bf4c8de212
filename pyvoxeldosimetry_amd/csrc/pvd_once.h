// Something that is set up once per device of a process, at the first call on each: a
// kernel's LDS limit belongs to the device it was set on.
#ifndef PVD_ONCE_H
#define PVD_ONCE_H

#include <atomic>

struct pvd_device_once {
    std::atomic<unsigned long long> done{0};       // devices 0..63; any other runs every time

    // f() returns an error code whose value 0 is success; a failed run is not remembered.  Two
    // threads may both run f() at a device's first call.
    template <typename F>
    auto run(int dev, F f) -> decltype(f()) {
        const unsigned long long bit = dev >= 0 && dev < 64 ? 1ull << dev : 0ull;
        if (done.load(std::memory_order_acquire) & bit) return decltype(f()){};
        const auto e = f();
        if (e == decltype(f()){}) done.fetch_or(bit, std::memory_order_release);
        return e;
    }
};

#endif
