// Which of a host call's buffers its kernels read and write in pinned memory.
#ifndef NATIVE_HIP_HOST_ROUTE_H
#define NATIVE_HIP_HOST_ROUTE_H

#include <cstddef>
#include <cstdint>

namespace nh {

struct HostProduct {
    size_t tokens, rows, cols;
    uint32_t type;
};

// Whether products go out as one launch: single tokens of one input (q, k, v; gate, up).  at(g): product g.
template <typename At> bool launched_together(size_t n, bool shared_x, At &&at) {
    const HostProduct first = at(0);
    bool together = n > 1 && n <= 8 && shared_x;
    for (size_t g = 0; g < n && together; g++) {
        const HostProduct p = at(g);
        together = p.tokens == 1 && p.rows != 0 && p.type == first.type && p.cols == first.cols;
    }
    return together;
}

struct HostRoute {
    bool x = false, y = false;  // the kernels read x, write y in pinned memory: no launches that copy them
};

// A decode step's products, called one by one, spend more time on the copies around them than on their weights: their kernels
// read a short x from pinned memory as they stage it and write y there, in one launch instead of three (host calls, us: Q4_K
// 4096x4096 22.1 -> 17.0, 14336x4096 27.6 -> 21.0, Q6_K 32000x4096 42.7 -> 36.1, Q5_0 4864x896 21.2 -> 15.3).  Rows of more
// than 16384 columns are summed in y by several launches, and more than two tokens by kernels that write y in scattered pieces.
//
// Reading x that way costs a launch 2 us with 4096 columns, 3 with 8192 and 8 with 14336 (every workgroup stages all of it; the
// caches serve all but the first), where a launch that copies it first costs 4: longer rows are copied.  Two tokens of F32 /
// F16 go to a kernel that reads x again for every 16 rows, also from those caches (direct / copied first, us: F16 4096x4096 24.7
// / 26.4, 14336x4096 42.8 / 45.2, 32000x4096 69.7 / 71.6, F32 32000x4096 115.4 / 117.4); two tokens of blocks are two launches
// that each stage x (Q8_0 512x1024 20.5 / 21.3, 4096x4096 28.5 / 27.6, 14336x4096 43.7 / 44.6).
//
// y_in_place: y is the caller's own buffer, which a call that fails leaves as it was unless its only launch does.  So kernels write
// there only where one launch makes all of y, else it is copied there when all launches have gone out.
template <typename At> HostRoute host_route(size_t n, bool shared_x, size_t x_total, bool y_in_place, At &&at) {
    constexpr size_t TOKENS = 2, X_FLOATS = 8192, COLS = 16384;
    HostRoute r{true, true};
    for (size_t g = 0; g < n; g++) {
        const HostProduct p = at(g);
        r.y = r.y && p.tokens <= TOKENS && p.cols <= COLS;
    }
    r.y = r.y && (!y_in_place || (n == 1 && at(0).tokens == 1) || launched_together(n, shared_x, at));
    r.x = r.y && x_total <= X_FLOATS;
    return r;
}

}  // namespace nh
#endif
