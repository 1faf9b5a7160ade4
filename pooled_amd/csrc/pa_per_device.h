// Host state kept per device (no HIP types: host tests build it alone).
#pragma once
#include <atomic>

#define PA_MAX_DEVICES 64

// Something to be done once on every device, by contexts of any thread.  Threads that meet on one device may do it twice, so it must
// bear repeating; it counts as done on a device only after it succeeded there.
struct PaPerDevice {
  std::atomic<bool> done[PA_MAX_DEVICES] = {};
  template <class F> auto once(int device, F f) -> decltype(f()) {
    typedef decltype(f()) E;
    const bool known = device >= 0 && device < PA_MAX_DEVICES;
    if (known && done[device].load(std::memory_order_acquire)) return E(0);
    const E e = f();
    if (known && e == E(0)) done[device].store(true, std::memory_order_release);
    return e;
  }
};
