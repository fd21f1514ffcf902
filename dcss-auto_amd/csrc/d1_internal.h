/* Entry points of libd1hip.so that only this package's Python surface calls; include/d1hip.h is
 * the library's public C ABI. Same conventions (device pointers, asynchronous on `stream`,
 * 0 / hipError_t / D1_E_*). */
#ifndef D1_INTERNAL_H
#define D1_INTERNAL_H
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* d1_gae followed by adv = (adv - mean) / (std + eps) over the whole [T, n] buffer with the
 * unbiased standard deviation (gpu-d1/scripts/run_ring_ablations.py:354-362): two launches,
 * moments in fp64. `work` holds d1_gae_norm_work_bytes(n) bytes, 8-byte aligned. */
int64_t d1_gae_norm_work_bytes(int n);
int d1_gae_norm(const float *reward, const uint8_t *done, const float *value, const float *bootstrap, int T, int n,
                float gamma, float gamma_lambda, float eps, float *adv, float *returns, void *work, int64_t work_bytes,
                void *stream);

#ifdef __cplusplus
}
#endif
#endif
