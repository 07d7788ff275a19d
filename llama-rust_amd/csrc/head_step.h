// What the device sessions and the routed layer take from the executor beyond the C ABI: the last product of a greedy step
// together with what stands around it, the router's product together with the copy of its input.
#ifndef NATIVE_HIP_HEAD_STEP_H
#define NATIVE_HIP_HEAD_STEP_H

#include <cstddef>
#include <cstdint>

#include "../../include/native_hip.h"

namespace nh {

// One token: dy = m rmsnorm(dx) * norm_w, and head_candidates(m) candidates for the largest output (value and row; a row of
// 0xffffffff where there is none).  0 candidates: m has no such launch.
size_t head_candidates(const lnh_matrix *m);
int head_device(lnh_exec *e, const lnh_matrix *m, const float *dx, const float *norm_w, float eps, float *dy, float *cand_v,
                uint32_t *cand_i, void *stream);
// Several tokens, from split activations: the rows of lnh_gemm_act_device and n_cand candidates of each.
int head_act_device(lnh_exec *e, const lnh_matrix *m, const lnh_act *x, size_t tokens, float *dy, float *cand_v, uint32_t *cand_i,
                    uint32_t n_cand, void *stream);

// A product by F32 / F16 weights of at most 16 rows whose input lies in pinned host memory: logits (pinned or device) = m x, and
// the rows of x to x_device.  LNH_ERR_UNSUPPORTED, nothing enqueued: m is another matrix.
int router_device(lnh_exec *e, const lnh_matrix *m, size_t tokens, const float *x, float *x_device, float *logits, void *stream);

}  // namespace nh
#endif
