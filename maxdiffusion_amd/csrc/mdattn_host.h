/* Entry points of libmdattn.so for this package's own host side (ops.py), beside the C ABI of mdattn.h: sizes that pick a
 * faster form of an ABI call, and fused forms of several ABI calls.  Same conventions as mdattn.h. */
#pragma once
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Workspace of mdattn_bwd_bf16 / mdattn_bwd_bf16_bias with which a pass that has too few rows of its own to fill the chip
 * (cross-attention: dk / dv of a few hundred keys) is split over the other sequence: mdattn_bwd_workspace_floats plus the
 * f32 partial gradients.  With less, the call runs unsplit. */
int64_t mdattn_bwd_split_workspace_floats(int B, int H, int Sq, int Skv, int D);

#ifdef __cplusplus
}
#endif
