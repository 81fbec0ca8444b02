// Which of a caller's memory a kernel writes in place of a copy (host code).
#pragma once
#include <cstddef>
#include <cstdint>

namespace vk {

// what the runtime says of an address
struct Target {
    bool device;      // device memory (not managed, not host memory it can reach)
    int dev;          // the device it was allocated on
    uintptr_t base;   // its allocation
    size_t size;
};

// `bytes` at p as 16-byte values, by a kernel of a handle made on device dev:
// memory of that device, whichever device is current (another device's may not
// be mapped there; a copy handles it), and the whole range inside one allocation.
inline bool kernel_writable(uintptr_t p, size_t bytes, const Target& t, int dev)
{
    return p % 16 == 0 && t.device && t.dev == dev && p >= t.base && p - t.base <= t.size &&
           bytes <= t.size - (p - t.base);
}

}  // namespace vk
