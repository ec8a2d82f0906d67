/* C ABI of libek_hip.so, second part: the projections of a prompt's rows
 * (engine/ek_model.py:280-334 runs them as torch.matmul). Conventions as in
 * ek_hip.h: device pointers, element strides, a hipStream_t, the return value
 * a hipError_t, nothing allocated, nothing synchronised.
 *
 * x [m, k] and w [n, k] are bf16 rows (strides ldx, ldw; both and the
 * pointers multiples of 16 bytes), k a positive multiple of 64, sums fp32.
 * m >= 1; a few hundred rows at most is where these kernels are for. */
#ifndef EK_HIP_PROMPT_H
#define EK_HIP_PROMPT_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* y[m, n] = x w^T in bf16 */
int ek_linear(const void* x, const void* w, void* y, int64_t m, int64_t n, int64_t k, int64_t ldx, int64_t ldw,
              int64_t ldy, void* stream);

/* parts[sk, m, n] = the sk fp32 partial sums of x w^T over K (sk <= k / 64),
 * as ek_add_rms_norm_parts takes them */
int ek_linear_parts(const void* x, const void* w, float* parts, int64_t m, int64_t n, int64_t k, int64_t ldx,
                    int64_t ldw, int64_t sk, void* stream);

/* y[m, inter] = bf16(silu(bf16 gate)) (x) bf16(up) with w the fused [2 inter,
 * k] gate/up matrix: ek_linear and ek_silu_mul in one launch */
int ek_linear_swiglu(const void* x, const void* w, void* y, int64_t m, int64_t inter, int64_t k, int64_t ldx,
                     int64_t ldw, int64_t ldy, void* stream);

#ifdef __cplusplus
}
#endif
#endif
