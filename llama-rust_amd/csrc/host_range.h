// Whether a kernel can use a buffer of the caller's in host memory in place.
#ifndef NATIVE_HIP_HOST_RANGE_H
#define NATIVE_HIP_HOST_RANGE_H

#include <cstddef>
#include <cstdint>

namespace nh {

// What the runtime knows of a host address: where the device sees it, and the one mapping around that place.
struct HostMapping {
    const void *device = nullptr;
    const void *base = nullptr;
    size_t size = 0;
};

// Where the device sees [p, p + bytes), null if it does not see the whole of it: a caller may have pinned a part of an
// allocation only, and beyond that part a kernel must not go.  find(p, &mapping) is false for memory that is not pinned.
template <typename Find> void *device_view(const void *p, size_t bytes, Find &&find) {
    HostMapping m;
    if (!find(p, &m) || !m.device) return nullptr;
    const uintptr_t at = reinterpret_cast<uintptr_t>(m.device), base = reinterpret_cast<uintptr_t>(m.base);
    if (at < base || at - base > m.size || bytes > m.size - (at - base)) return nullptr;
    return const_cast<void *>(m.device);
}

}  // namespace nh
#endif
