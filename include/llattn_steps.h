/* Entry points that this package's own Python side calls beside those of
 * llattn.h: fused steps of its language model and block.  Same conventions
 * (status codes, llattn_last_error, explicit stream, caller-supplied memory). */
#ifndef LLATTN_STEPS_H
#define LLATTN_STEPS_H

#include "llattn.h"

#ifdef __cplusplus
extern "C" {
#endif

/* llattn_rmsnorm_bwd with dx also written in bf16 (dx16, may be null; needs
 * dres): the gradient of a bf16 residual addend, which autograd holds apart
 * from dx. */
int32_t llattn_rmsnorm_bwd_residual(const void* dy, int32_t dy_dtype, int64_t lddy, const void* x, int32_t x_dtype,
                                    int64_t ldx, const float* rstd, const float* weight, int32_t M, int32_t D,
                                    void* dx, int64_t lddx, float* dweight, const void* dres, int64_t lddres,
                                    void* dx16, int64_t lddx16, void* workspace, size_t workspace_bytes,
                                    void* stream);

/* Two bf16 products that do not depend on each other: in one launch where that
 * is expected to pay (d0: x W^T or dy W into bf16; d1: dy^T x into fp32, or
 * another x W^T after x W^T), else one after the other.  The k order of the
 * sums can then differ from the single products'. */
size_t llattn_gemm_pair_workspace_size(const llattn_gemm_desc* d0, const llattn_gemm_desc* d1);
int32_t llattn_gemm_pair(const llattn_gemm_desc* d0, const llattn_gemm_desc* d1, void* workspace,
                         size_t workspace_bytes, void* stream);

/* ---- whole steps ---------------------------------------------------------
 * The attention block, its core and the feed-forward as one call per
 * direction: the launches of the entry points of llattn.h in a row, without a
 * host language between them.  The caller passes memory: `kept` holds what the
 * forward leaves for the backward (llattn_*_bytes, which = 0; without a
 * backward it is the forward's scratch), `ws` the scratch of one call
 * (which = 1: forward, 2: backward, 3: backward without dx; may be NULL where
 * that is 0 bytes).  Outputs also serve as scratch before they are written:
 * out and dx overlap no input.  Everything is 16-byte aligned. */

/* The block: x [B][T][d_model] in shape.dtype, fp32 parameters.  `saved`: a
 * backward will follow.  The layout flags choose split-head storage
 * (llattn_heads_layout) for the projection output, r_out's output, the core's
 * output gradient and the latent output's gradient. */
typedef struct llattn_block_cfg {
  llattn_shape shape;
  int32_t d_model;
  int32_t macro;    /* pooled query blocks and a projection of their own (reference models.py:343-353) */
  int32_t has_bias;
  int32_t saved;
  int32_t heads, remote_heads, dy_heads, lat_heads;
} llattn_block_cfg;

typedef struct llattn_block_params {
  const float *w_qkv, *b_qkv, *w_rq, *b_rq, *w_rkv, *b_rkv, *w_r, *b_r, *w_out, *b_out; /* biases NULL without */
  const float *gate_l, *gate_r;
} llattn_block_params;

/* Gradients, fp32: qkv is [3 d_model (+ Ld)][d_model], its rq rows last when
 * token-wise (then rq is NULL), and likewise its bias. */
typedef struct llattn_block_grads {
  float *w_qkv, *b_qkv, *w_rq, *b_rq, *w_rkv, *b_rkv, *w_r, *b_r, *w_out, *b_out;
  float *gate_l, *gate_r;
} llattn_block_grads;

size_t llattn_block_bytes(const llattn_block_cfg* c, int32_t which);
int32_t llattn_block_fwd(const llattn_block_cfg* c, const llattn_block_params* p, const void* x, void* kept, void* ws,
                         size_t ws_bytes, void* out, void* stream);
/* dy [B][T][d_model]; dx may be NULL. */
int32_t llattn_block_bwd(const llattn_block_cfg* c, const llattn_block_params* p, const void* x, const void* kept,
                         const void* dy, void* dx, const llattn_block_grads* g, void* ws, size_t ws_bytes,
                         void* stream);

/* The core on head tensors: latent attention, r_out, local attention with the
 * gate; r_w / r_b fp32 (r_b may be NULL), y written through its view. */
typedef struct llattn_core_views {
  llattn_tensor q, k, v, gq, gk, gv;
} llattn_core_views;
size_t llattn_core_bytes(const llattn_block_cfg* c, int32_t which);
int32_t llattn_core_fwd(const llattn_block_cfg* c, const llattn_core_views* in, const float* gate_l,
                        const float* gate_r, const float* r_w, const float* r_b, void* kept, void* ws,
                        size_t ws_bytes, const llattn_tensor* y, void* stream);
int32_t llattn_core_bwd(const llattn_block_cfg* c, const llattn_core_views* in, const float* gate_l,
                        const float* gate_r, const float* r_w, const void* kept, const llattn_tensor* dy,
                        const llattn_core_views* d, float* dgate_l, float* dgate_r, float* dr_w, float* dr_b,
                        void* ws, size_t ws_bytes, void* stream);

/* The feed-forward w2(gelu(w1 x)) in bf16 on x [rows][d]: reference
 * models.py:50-58 under bf16 autocast.  Biases may be NULL. */
typedef struct llattn_ffn_cfg {
  int32_t rows, d, d_ff, d_out, saved;
} llattn_ffn_cfg;
size_t llattn_ffn_bytes(const llattn_ffn_cfg* c, int32_t which);
int32_t llattn_ffn_fwd(const llattn_ffn_cfg* c, const void* x, const float* w1, const float* b1, const float* w2,
                       const float* b2, void* kept, void* ws, size_t ws_bytes, void* y, void* stream);
int32_t llattn_ffn_bwd(const llattn_ffn_cfg* c, const void* x, const void* kept, const void* dy, void* dx, float* dw1,
                       float* db1, float* dw2, float* db2, void* ws, size_t ws_bytes, void* stream);

#ifdef __cplusplus
}
#endif

#endif
