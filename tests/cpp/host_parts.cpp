// Checks of the library's host-only parts (llama-rust_amd/csrc/*.h that need no device), for the host compiler alone.
// Prints "OK" and returns 0, or says what failed and returns 1.
#include <cstdio>

#include "../../llama-rust_amd/csrc/host_range.h"

static int failures = 0;
#define CHECK(cond)                                                         \
    do {                                                                    \
        if (!(cond)) {                                                      \
            std::printf("%s:%d: %s\n", __FILE__, __LINE__, #cond);          \
            failures++;                                                     \
        }                                                                   \
    } while (0)

// A buffer is used in place only where one mapping holds all of it.
static void host_range() {
    char *const host = reinterpret_cast<char *>(0x10000), *const device = reinterpret_cast<char *>(0x7000000);
    // [host + 4096, host + 12288) is pinned, and so is, on its own, what follows directly
    auto find = [&](const void *p, nh::HostMapping *m) {
        const size_t at = (size_t)(static_cast<const char *>(p) - host);
        if (at < 4096 || at >= 16384) return false;
        m->device = device + at;
        m->base = device + (at < 12288 ? 4096 : 12288);
        m->size = at < 12288 ? 8192 : 4096;
        return true;
    };
    CHECK(nh::device_view(host + 4096, 8192, find) == device + 4096);
    CHECK(nh::device_view(host + 5000, 7288, find) == device + 5000);
    CHECK(nh::device_view(host + 12287, 1, find) == device + 12287);
    CHECK(nh::device_view(host + 4096, 8193, find) == nullptr);   // the first part is pinned only
    CHECK(nh::device_view(host + 5000, 7289, find) == nullptr);
    CHECK(nh::device_view(host + 4096, 12288, find) == nullptr);  // two mappings
    CHECK(nh::device_view(host, 8192, find) == nullptr);          // the last part is pinned only
    CHECK(nh::device_view(host + 4096, SIZE_MAX, find) == nullptr);
    CHECK(nh::device_view(host + 4096, 16, [](const void *, nh::HostMapping *) { return true; }) == nullptr);
}

int main() {
    host_range();
    if (failures == 0) std::printf("OK\n");
    return failures != 0;
}
