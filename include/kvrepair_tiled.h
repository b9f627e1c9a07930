/*
 * kvrepair_tiled.h — projections and decoder layers of more than 64 packed
 * refresh rows. Conventions, descriptors and statuses are kvrepair.h's.
 */
#ifndef KVREPAIR_TILED_H
#define KVREPAIR_TILED_H

#include "kvrepair.h"

#ifdef __cplusplus
extern "C" {
#endif

/*
 * The projections of kvr_linear_multi for more rows (any m up to 2^20), by a
 * kernel that tiles x and the weights through LDS: same operands, epilogues and
 * rounding, the same bits from call to call. The order of a sum over k depends on m
 * and on all the weights of the call (tile, K split and the start of the walk over
 * k follow from them): other calls over the same row, kvr_linear_multi's, and for
 * the gated epilogue two separate projections with kvr_silu_mul, agree up to the
 * order of their fp32 sums. k is a multiple of 64 and every weight's row count
 * a multiple of 8; ldx and ldw are multiples of 8 elements (at most 2^21) on
 * 16-byte aligned bases, ldy and ldr multiples of 4 on 8-byte aligned ones;
 * `workspace` (16-byte aligned) has kvr_tiled_linear_workspace_bytes(m, rows
 * over the call's weights, k) bytes, which the gated epilogue does not use.
 * Replaces the same nn.Linear calls (transformers 5.15.0
 * models/llama/modeling_llama.py:165-175, 243-252); no reference counterpart of
 * its own.
 */
int64_t kvr_tiled_linear_workspace_bytes(int32_t m, int32_t rows, int32_t k);
int kvr_tiled_linear_multi(const void* x, int32_t n_weights, const void* const* w, const int32_t* rows,
                           const int64_t* ldw, void* y, int32_t m, int32_t k, int64_t ldx, int64_t ldy,
                           int32_t epilogue, const void* residual, int64_t ldr, void* workspace,
                           int64_t workspace_bytes, int32_t dtype, void* stream);

/*
 * kvr_decoder_forward over those projections, for any number of rows up to
 * 2^20; hidden, q_heads * head_dim and intermediate are multiples of 64.
 * Scratch and GEMM workspace have their own sizes.
 */
int64_t kvr_decoder_tiled_scratch_bytes(const kvr_refresh_desc* d);
int64_t kvr_decoder_tiled_gemm_workspace_bytes(const kvr_refresh_desc* d);
int kvr_decoder_tiled_forward(const kvr_layer_desc* layers, int32_t n_layers, const kvr_refresh_desc* d,
                              void* hidden, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* KVREPAIR_TILED_H */
