// What the dispatch layer takes from the executor beyond the C ABI: its worker threads, and a product of host buffers in
// two halves - the layer begins the product of the matrix it expects to find and compares that matrix's bytes with the
// caller's while the product runs.
#ifndef NATIVE_HIP_EARLY_GEMM_H
#define NATIVE_HIP_EARLY_GEMM_H

#include <cstddef>

#include "../../include/native_hip.h"
#include "host_pool.h"

namespace nh {

// The executor's worker threads (confined, like the executor, to one caller at a time).
HostPool &host_pool(lnh_exec *e);

// Enqueues lnh_gemm(e, m, tokens, x, x_len, y, y_len) up to the copy of y into the executor's staging.  False (nothing
// in flight, nothing reported): the call has to go through lnh_gemm - its arguments are wrong, its buffers are larger
// than the staging, or the product would first make the matrix's multi-token layout, which is not to be done for a
// matrix that may turn out to be another one.
bool gemm_begin(lnh_exec *e, const lnh_matrix *m, size_t tokens, const float *x, size_t x_len, size_t y_len);
// Waits for it and writes y, or drops the result (y null).  Exactly one after each gemm_begin that returned true,
// before any other call on e.
int gemm_end(lnh_exec *e, float *y);

}  // namespace nh
#endif
