/* Entry points of libd1hip.so that only this package's Python surface calls; include/d1hip.h is
 * the library's public C ABI. Same conventions (device pointers, asynchronous on `stream`,
 * 0 / hipError_t / D1_E_*). */
#ifndef D1_INTERNAL_H
#define D1_INTERNAL_H
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* adv[0..count) = (adv - *mean) / (*std + eps) in fp32, in place (the whole-buffer advantage
 * normalisation of gpu-d1/scripts/run_ring_ablations.py:362; mean and std are device scalars). */
int d1_adv_norm(float *adv, int64_t count, const float *mean, const float *std, float eps, void *stream);

#ifdef __cplusplus
}
#endif
#endif
