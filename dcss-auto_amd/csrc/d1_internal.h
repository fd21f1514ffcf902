/* Entry points of libd1hip.so that only this package's Python surface calls; include/d1hip.h is
 * the library's public C ABI. Same conventions (device pointers, asynchronous on `stream`,
 * 0 / hipError_t / D1_E_*). */
#ifndef D1_INTERNAL_H
#define D1_INTERNAL_H
#include <stdint.h>

#include "../../include/d1hip.h"

#ifdef __cplusplus
extern "C" {
#endif

/* d1_step (every world active) that also writes reward[i] = out[i][0] and done[i] =
 * out[i][1], the rows a rollout buffer keeps of the step. */
int d1_step_into(void *state, int n, int max_monsters, const D1Config *cfg, const D1Tables *tab, const int64_t *actions,
                 uint8_t *obs, float *out, uint32_t *hash, float *reward, uint8_t *done, void *stream);

/* adv[0..count) = (adv - *mean) / (*std + eps) in fp32, in place (the whole-buffer advantage
 * normalisation of gpu-d1/scripts/run_ring_ablations.py:362; mean and std are device scalars). */
int d1_adv_norm(float *adv, int64_t count, const float *mean, const float *std, float eps, void *stream);

#ifdef __cplusplus
}
#endif
#endif
