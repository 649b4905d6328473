/* Entry points of libmdattn.so for this package's own host side (ops.py), beside the C ABI of mdattn.h: sizes that pick a
 * faster form of an ABI call, and fused forms of several ABI calls.  Same conventions as mdattn.h. */
#pragma once
#include <stdint.h>

#include "mdattn.h"

#ifdef __cplusplus
extern "C" {
#endif

/* Workspace of mdattn_bwd_bf16 / mdattn_bwd_bf16_bias with which a pass that has too few rows of its own to fill the chip
 * (cross-attention: dk / dv of a few hundred keys) is split over the other sequence: mdattn_bwd_workspace_floats plus the
 * f32 partial gradients.  With less, it is split as far as the partials fit. */
int64_t mdattn_bwd_split_workspace_floats(int B, int H, int Sq, int Skv, int D);

/* A [B, Skv] keep-mask (bytes) -> the additive bias of mdattn_key_mask_bias (-inf for excluded keys; bias_stride a multiple of
 * 32) and, in `tiles` (mdattn_host_key_tiles_ints ints), per batch element the lists of key tiles that hold a kept key. */
int64_t mdattn_host_key_tiles_ints(int B, int Skv);
int mdattn_host_key_tiles(void* stream, const void* keep, float* bias, int* tiles, int B, int Skv, int64_t bias_stride);

/* Dense copies of one buffer, or of two (src1 and dst1 not null) of the same size, in one launch.  16-byte aligned, bytes a multiple
 * of 16. */
int mdattn_host_copy(void* stream, const void* src0, void* dst0, const void* src1, void* dst1, int64_t bytes);

/* mdattn_quant_e4m3 of an attention call's q (premul q_premul, power-of-two scale), k (power-of-two scale) and v in two
 * launches.  ws: mdattn_host_quant3_floats floats, 16-byte aligned, of which [2 t] and [2 t + 1] become scale and absmax of
 * tensor t. */
int64_t mdattn_host_quant3_floats(void);
int mdattn_host_quant3_e4m3(void* stream, const void* q, const void* k, const void* v, void* q8, void* k8, void* v8, float* ws, int64_t nq,
                            int64_t nkv, float q_premul);

/* Whether mdattn_host_fwd_bf16 and mdattn_host_bwd_bf16 take head dim D. */
int mdattn_host_head_dim(int D);

/* mdattn_fwd_bf16, or (key_bias and tiles of mdattn_host_key_tiles) the same under a key mask, at head dims 64, 128 and the multiples
 * of 8 up to 48 and from 72 to 96.  workspace: mdattn_host_fwd_workspace_floats floats, 16-byte aligned, with which a call without a bias whose query
 * tiles leave the chip idle is split over its keys; 0: it would not be.  With less, the call runs unsplit. */
int64_t mdattn_host_fwd_workspace_floats(int B, int H, int Sq, int Skv, int D);
int mdattn_host_fwd_bf16(void* stream, const void* q, const void* k, const void* v, void* out, float* lse, int B, int H, int Sq, int Skv, int D,
                         const mdattn_strides* q_strides, const mdattn_strides* k_strides, const mdattn_strides* v_strides,
                         const mdattn_strides* o_strides, float scale, const float* key_bias, int64_t bias_stride, const int* tiles,
                         float* workspace, int64_t workspace_floats);

/* The schedule (of mdattn_set_fwd_schedule) of a forward without a bias whose keys are not cut, as mdattn_fwd_bf16 and
 * mdattn_fwd_bf16_merge choose it. */
int mdattn_host_fwd_schedule(int B, int H, int Sq, int Skv, int D, float scale);

/* How a backward call launches its passes, dq and dk with dv: waves per workgroup, pieces of the other sequence and 32-row tiles in each,
 * floats of one tensor's partial gradients (0: one piece). */
typedef struct {
  int waves, pieces, tiles;
  int64_t floats;
} mdattn_host_bwd_pass;
typedef struct {
  mdattn_host_bwd_pass dq, dkv;
} mdattn_host_bwd_plan;
/* The plan (or null) of a call, with a key bias or mask or without, and with a workspace of so many floats, at least mdattn_bwd_workspace_floats; negative: as many as it asks for.
 * Returns how many it uses, 0 for sizes that are refused. */
int64_t mdattn_host_bwd_plan_floats(int B, int H, int Sq, int Skv, int D, int key_bias, int64_t workspace_floats, mdattn_host_bwd_plan* plan);

/* mdattn_bwd_bf16 / mdattn_bwd_bf16_bias (key_bias with or without tiles) at the head dims of mdattn_host_fwd_bf16.  plan: of these
 * sizes; null: made from the workspace. */
int mdattn_host_bwd_bf16(void* stream, const void* q, const void* k, const void* v, const void* out, const void* dout, const float* lse, void* dq,
                         void* dk, void* dv, float* workspace, int64_t workspace_floats, int B, int H, int Sq, int Skv, int D,
                         const mdattn_strides* q_strides, const mdattn_strides* k_strides, const mdattn_strides* v_strides,
                         const mdattn_strides* o_strides, float scale, const float* key_bias, int64_t bias_stride, const int* tiles,
                         const mdattn_host_bwd_plan* plan);

/* The prologue and its backward with the rotary table in the layout the model made it in:
 *   PLANES    cos, sin f32 [S, D/2] (the layout of mdattn.h's entry points)
 *   COMPLEX   cos = complex64 [S, D/2], sin null
 *   REPEATED  cos, sin f32 [S, D], each angle for both members of its pair      (per-head forms only)
 *   MATRIX    cos = f32 [S, D/2, 2, 2] = [[cos, -sin], [sin, cos]], sin null     (per-head forms only)
 * No table: cos null, sin null, PLANES.
 * The backward forms write the weight (and bias) gradients as f32, or (dw_bf16) rounded to bf16.  gv, dv_in (the fused form
 * with biases; or null): the value block's output gradient, strided like gq, and its place in the fused gradient buffer;
 * dbias then has 3*H*D entries and the workspace 5*H*D columns. */
#define MDATTN_TABLE_PLANES 0
#define MDATTN_TABLE_COMPLEX 1
#define MDATTN_TABLE_REPEATED 2
#define MDATTN_TABLE_MATRIX 3
int mdattn_host_norm_rope_fullrow(void* stream, const void* q_in, const void* k_in, void* q_out, void* k_out, const void* wq,
                                  const void* wk, const float* cos, const float* sin, int table, int B, int S, int H, int D,
                                  float eps, float q_mul, int64_t in_stride_batch, int64_t in_stride_seq, const mdattn_strides* out_strides);
int mdattn_host_norm_rope_qkv(void* stream, const void* qkv, const void* bias, void* q_out, void* k_out, void* v_out, const void* wq,
                              const void* wk, const float* cos, const float* sin, int table, int B, int S, int H, int D, float eps,
                              float q_mul, int64_t qkv_stride_batch, int64_t qkv_stride_seq, const mdattn_strides* out_strides);
int mdattn_host_norm_rope_perhead(void* stream, const void* q_in, const void* k_in, void* q_out, void* k_out, const void* wq,
                                  const void* wk, const void* wq_txt, const void* wk_txt, int n_txt, const float* cos, const float* sin,
                                  int table, int B, int S, int H, int D, float eps, float q_mul, const mdattn_strides* in_strides,
                                  const mdattn_strides* out_strides);
int mdattn_host_norm_rope_fullrow_bwd(void* stream, const void* q_in, const void* k_in, const void* bias, const void* gq, const void* gk,
                                      void* dq_in, void* dk_in, const void* wq, const void* wk, void* dwq, void* dwk, void* dbias,
                                      int dw_bf16, const void* gv, void* dv_in,
                                      const float* cos, const float* sin, int table, int B, int S, int H, int D, float eps, float q_mul,
                                      int64_t in_stride_batch, int64_t in_stride_seq, int64_t dx_stride_batch, int64_t dx_stride_seq,
                                      const mdattn_strides* g_strides, float* workspace, int64_t workspace_floats);
int mdattn_host_norm_rope_perhead_bwd(void* stream, const void* q_in, const void* k_in, const void* gq, const void* gk, void* dq_in,
                                      void* dk_in, const void* wq, const void* wk, const void* wq_txt, const void* wk_txt, int n_txt,
                                      void* dwq, void* dwk, void* dwq_txt, void* dwk_txt, int dw_bf16, const float* cos, const float* sin,
                                      int table, int B, int S, int H, int D, float eps, float q_mul, const mdattn_strides* in_strides,
                                      const mdattn_strides* dx_strides, const mdattn_strides* g_strides, float* workspace,
                                      int64_t workspace_floats);

/* mdattn_norm_rope_rows and its backward over q and k of one shape at once, the tables shared (k null: one tensor; with k at
 * most 4,096 channels), the factor w_mul multiplied into q's weight (dwq is the gradient of the weight without it).
 * workspace: mdattn_norm_rope_bwd_workspace_floats(B*S, H*D times the number of tensors). */
int mdattn_host_norm_rope_rows(void* stream, const void* q_in, const void* k_in, int x_is_f32, void* q_out, void* k_out, const float* wq,
                               const float* wk, const float* cos, const float* sin, int rope_mode, int B, int S, int H, int D, float eps,
                               float w_mul, int64_t in_stride_batch, int64_t in_stride_seq, const mdattn_strides* out_strides);
int mdattn_host_norm_rope_rows_bwd(void* stream, const void* q_in, const void* k_in, int x_is_f32, const void* gq, const void* gk, void* dq, void* dk,
                                   const float* wq, const float* wk, float* dwq, float* dwk, const float* cos, const float* sin, int rope_mode,
                                   int B, int S, int H, int D, float eps, float w_mul, int64_t in_stride_batch, int64_t in_stride_seq,
                                   int64_t dx_stride_batch, int64_t dx_stride_seq, const mdattn_strides* g_strides, float* workspace,
                                   int64_t workspace_floats);

#ifdef __cplusplus
}
#endif
