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

/* Hidden states of a Transformer-XL segment in bf16 (relative attention of heads
 * 64 wide, model width 512, post-layer-norm blocks): x0 [q_len, batch, 512] are the
 * embedded tokens, mems [layers][m_len, batch, 512] with mem_stride elements from
 * one layer to the next (unused for m_len 0), hidden [q_len, batch, 512].  The last
 * mem_rows_out positions of every layer's input are written to new_mems + layer *
 * new_mem_stride (none if it is null).  u, v [heads * 64] are the biases of the
 * content and position queries.  A layer's weights are [out, in] row-major: qkv
 * [3 * heads * 64, 512], pos [heads * 64, 512], out [512, heads * 64], ff1 [inner,
 * 512], ff2 [512, inner].  heads is even and inner a multiple of 128
 * (ORION_ERR_SHAPE); every address is 16-byte aligned, the strides a multiple of 8.
 * `workspace` is device memory of at least orion_txl_workspace_bytes(dims), 0 for
 * dims that are refused, that the call's kernels alone use until they have run;
 * `dims` and `layers` are host memory and may go as soon as the call has returned. */
typedef struct orion_txl_dims {
  int layers, heads, inner, q_len, m_len, batch;
  float eps;
} orion_txl_dims;
typedef struct orion_txl_layer {
  const void *qkv, *pos, *out, *norm1_w, *norm1_b;
  const void *ff1_w, *ff1_b, *ff2_w, *ff2_b, *norm2_w, *norm2_b;
} orion_txl_layer;
size_t orion_txl_workspace_bytes(const orion_txl_dims* dims);
int orion_txl_hidden(const orion_txl_dims* dims, const orion_txl_layer* layers,
                     const void* u, const void* v, const void* x0, const void* mems,
                     size_t mem_stride, void* new_mems, size_t new_mem_stride,
                     int mem_rows_out, void* hidden, void* workspace,
                     size_t workspace_bytes, void* stream);

/* Negative log-likelihoods nll [rows] (bf16) of target [rows] (int64) under an
 * adaptive softmax over hidden [rows, 512] (bf16): edges 0, cutoffs, vocabulary
 * size; weight and bias of every token; tail_weight [tails, 512] and tail_bias are
 * the head's entries for the tails (at most 7).  A target outside the vocabulary
 * gives 0.  Workspace as above. */
typedef struct orion_nll {
  const void *hidden, *weight, *bias, *tail_weight, *tail_bias, *target;
  int rows, tails;
  int edges[9];
} orion_nll;
size_t orion_nll_workspace_bytes(const orion_nll* args);
int orion_nll_bf16(const orion_nll* args, void* nll, void* workspace,
                   size_t workspace_bytes, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* ORION_MODEL_KERNELS_H_ */
