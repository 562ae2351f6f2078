/*
 * C ABI of libmi_model.so: the projections of a decode step's few tokens on MI355X (gfx950), each
 * with the steps either side of it in the same launch.
 *
 * They replace, for up to 64 tokens, the reference's nn.Linear calls (model.py:81-84,112-120,
 * 204-207) together with its RMSNorm (model.py:49-55), rotary embedding and cache write
 * (model.py:58-65,92, kv_cache.py:108-115), SwiGLU and residual adds (model.py:128-138).
 *
 * Common rules.  dtype: 0 bf16, 1 fp16 (tensors and weights alike); sums are fp32, and every value
 * is rounded to the dtype where the reference's separate tensor ops round it.  Row strides are in
 * elements, multiples of 8; pointers are 16-byte aligned device pointers.  Weights are row-major
 * [out features][in features], contiguous, as nn.Linear holds them.  norm_weight: NULL, or the
 * weight of an RMSNorm applied to x first (at most 16 rows; in features at most 2048).  All launches
 * are asynchronous on `stream`, allocate nothing and may be captured in a graph.
 *
 * Status codes as in mi_fa2.h: 0 ok, 1 invalid argument, 2 unsupported, 3 workspace too small,
 * 4 launch failed; mi_model_last_error() gives the calling thread's last message.
 */
#ifndef MI_MODEL_H
#define MI_MODEL_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define MI_MODEL_API __attribute__((visibility("default")))

MI_MODEL_API const char* mi_model_last_error(void);

/*
 * out = [residual +] ([rmsnorm] x W^T + bias): x [rows, in], w [out_features, in], bias
 * [out_features] or NULL, residual [rows, out_features] or NULL (may be `out`).
 * rows <= 64; in: a multiple of 32, at most 2048; out_features: a multiple of 16.
 */
MI_MODEL_API int mi_model_linear(int32_t dtype, const void* x, int64_t x_stride,
                                 const void* norm_weight, float eps, const void* w,
                                 const void* bias, const void* residual, int64_t residual_stride,
                                 void* out, int64_t out_stride, int32_t rows,
                                 int32_t out_features, int32_t in_features, void* stream);

/*
 * Rotary tables (model.py:151-155): cos/sin [rows * tokens_per_row, 128] of
 * float(starts[row] + t) * float(inv_freq[d % 64]), taken in fp32 and rounded; inv_freq [64].
 */
MI_MODEL_API int mi_model_rope_table(int32_t dtype, const int32_t* starts, const void* inv_freq,
                                     void* cos, void* sin, int32_t rows, int32_t tokens_per_row,
                                     void* stream);

/*
 * The MLP of one layer, out = [residual +] (silu(g) * u) Wd^T with (g | u) = [rmsnorm] x Wgu^T:
 * x, out, residual [rows, hidden], gate_up_w [2 * inter, hidden] (gate rows first), down_w
 * [hidden, inter].  rows <= 64; hidden: a multiple of 32, at most 2048; inter: a multiple of 32.
 * workspace: mi_model_mlp_workspace_size(rows, hidden, inter) bytes, 16-byte aligned, contents
 * arbitrary; not shared by calls that may overlap in time.  out may be residual and x.
 */
MI_MODEL_API size_t mi_model_mlp_workspace_size(int32_t rows, int32_t hidden, int32_t inter);
MI_MODEL_API int mi_model_mlp(int32_t dtype, const void* x, int64_t x_stride,
                              const void* norm_weight, float eps, const void* gate_up_w,
                              const void* down_w, const void* residual, int64_t residual_stride,
                              void* out, int64_t out_stride, int32_t rows, int32_t hidden,
                              int32_t inter, void* workspace, size_t workspace_bytes,
                              void* stream);

/*
 * The q/k/v projection with what follows it, mi_fa2_rope_kv_write's contract for the second half:
 * (q | k | v) = rmsnorm(x) W^T + bias, w [(heads_q + 2 heads_kv) * 128, hidden]; rotated q to q_out
 * [rows, heads_q * 128], rotated k and v to the cache slot of each token (a slot outside
 * [0, num_slots) writes nothing).  rows <= 16; hidden: a multiple of 32, at most 2048.
 */
MI_MODEL_API int mi_model_qkv_rope(int32_t dtype, const void* x, int64_t x_stride,
                                   const void* norm_weight, float eps, const void* w,
                                   const void* bias, const void* cos, const void* sin,
                                   int64_t cs_stride, const int32_t* slot_mapping, void* q_out,
                                   int64_t q_stride, void* k_pool, void* v_pool,
                                   const int64_t* pool_strides, int32_t num_slots, int32_t rows,
                                   int32_t hidden, int32_t heads_q, int32_t heads_kv,
                                   void* stream);

#ifdef __cplusplus
}
#endif

#endif /* MI_MODEL_H */
