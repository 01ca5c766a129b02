/* C ABI of the kernels behind the Transformer-XL client, in liborion_kernels.so
 * beside the co-location kernels (orion_kernels.h, whose status codes and rules
 * hold here too: device pointers, `stream` a hipStream_t, every call only
 * enqueues work).
 */
#ifndef ORION_MODEL_KERNELS_H_
#define ORION_MODEL_KERNELS_H_

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* One LAMB step over `count` fp32 tensors of n contiguous elements each: weight,
 * gradient and the two moments, all 4-byte aligned (16-byte aligned ones take
 * wider accesses).  Moments without bias correction; the update of a tensor is
 * scaled by min(|w|, 10) / (|update| + eps), by 1 where either norm is zero
 * (related/baselines/transformer/lamb.py:108-144 of the reference).  `workspace`
 * is 8-byte aligned device memory of at least orion_lamb_workspace_bytes(...)
 * that the call's kernels alone use until they have run.  `tensors` is host
 * memory and may go as soon as the call has returned. */
typedef struct orion_lamb_tensor {
  float* w;
  const float* g;
  float* m;
  float* v;
  uint64_t n;
} orion_lamb_tensor;
size_t orion_lamb_workspace_bytes(const orion_lamb_tensor* tensors, int count);
int orion_lamb_step(const orion_lamb_tensor* tensors, int count, double lr,
                    double b1, double b2, double eps, double decay,
                    void* workspace, size_t workspace_bytes, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* ORION_MODEL_KERNELS_H_ */
