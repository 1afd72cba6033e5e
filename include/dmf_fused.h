/*
 * Fused entry points beyond the operator boundary of dmf_attn.h / dmf_block.h: combinations of those operators that run as
 * fewer passes.  Same conventions as there (plain pointers, element strides, return codes, a hipStream_t as void*; nothing
 * allocates, frees or synchronises); each is optional for a caller, who can always compose the basic entry points.
 */
#ifndef DMF_FUSED_H
#define DMF_FUSED_H

#include "dmf_attn.h"

#ifdef __cplusplus
extern "C" {
#endif

/*
 * dmf_attn_bwd behind per-head RMS norms of q and k (dmf_attn_fwd_qknorm): q_hat, k_hat are the normalised rows the forward
 * handed out, q, k the raw ones; dq, dk are the gradients of the RAW rows and dq_gain, dk_gain (D) fp32 those of the gains --
 * dmf_attn_bwd followed by dmf_rmsnorm_bwd for q and for k, with the norm's backward applied where the rows of dq_hat,
 * dk_hat are stored.  strides: 10 tensors {dout, q_hat, k_hat, v, o, dq, dk, dv, q, k}.  workspace:
 * dmf_attn_bwd_qknorm_workspace_floats() floats.  Deterministic (no atomics).  bf16 shapes the tuned kernels cover;
 * DMF_ATTN_ENOKERNEL otherwise (nothing launched).
 */
DMF_ATTN_API int64_t dmf_attn_bwd_qknorm_workspace_floats(int B, int H, int Lq, int Lkv, int D);
DMF_ATTN_API int dmf_attn_bwd_qknorm(const void* dout, const void* q_hat, const void* k_hat, const void* v,
                        const void* o, const float* lse, const void* q, const void* k,
                        const float* q_gain, const float* k_gain, float eps,
                        void* dq, void* dk, void* dv, float* dq_gain, float* dk_gain,
                        float* delta, float* workspace, const int64_t* strides,
                        int B, int H, int Lq, int Lkv, int D, float scale, int dtype, void* stream);

/*
 * The adaLN projections of a stack in one launch, bf16: out[g] = s[cond[g]] w[g]^T + bias[g] for `groups` (1 .. 64) groups, w[g]
 * (n, K) row-major -- (n_last, K) for the last one --, bias[g] (n) or NULL, s[0 .. 1] the (B, K) activated conditioning vectors
 * (s[1] may be NULL if no group uses it).  jvp: s[.] holds B more rows, the tangents, and out[g] takes B more rows, t w^T.  B up
 * to 128, K a multiple of 128, n a multiple of 32; w and s 16-byte, bias and out 8-byte aligned.
 */
DMF_ATTN_API int dmf_modulation_fwd(const void* const* s, const void* const* w, const void* const* bias, void* const* out, const int* cond,
                        int groups, int B, int K, int n, int n_last, int jvp, void* stream);

/*
 * y = x w^T + bias (gelu: with the tanh form of gelu applied), bf16 with fp32 accumulation: x (M, K), w (N, K), bias (N) or NULL,
 * y (M, N), all dense; tx / ty (both or neither): ty = tx w^T besides, in the same grid (gelu: times the activation's derivative).
 * K a multiple of 64, N of 8, at most 2^30 elements in x, w and y; 16-byte aligned, bias 8-byte.  dmf_linear_plan: 1 where this
 * kernel is the better choice (and covers the shape), 0 where a library product is; host-only.  dmf_linear_fwd_plan: the name of the kernel
 * that dmf_linear_fwd launches for the shape on the current device, as profilers print it; host-only.
 */
DMF_ATTN_API int dmf_linear_plan(int64_t M, int N, int K, int jvp, int gelu);
DMF_ATTN_API int dmf_linear_fwd_plan(int64_t M, int N, int K, int jvp, int gelu, char* buf, int buflen);
DMF_ATTN_API int dmf_linear_fwd(const void* x, const void* tx, const void* w, const void* bias, void* y, void* ty, int M, int N, int K,
                        int gelu, void* stream);

/*
 * The first half of an MLP whose backward pass follows: pre = x w^T + bias, y = gelu(pre) and ty, the tangent of y along tx, activated from the fp32 sums
 * (of which pre is the rounding).  Types, sizes and alignment of dmf_linear_fwd; the shapes for which dmf_linear_gelu_plan says 1, DMF_ATTN_ESHAPE
 * otherwise (dmf_linear_fwd and dmf_gelu_tanh_fwd do those).
 */
DMF_ATTN_API int dmf_linear_gelu_plan(int64_t M, int N, int K);
DMF_ATTN_API int dmf_linear_gelu_fwd(const void* x, const void* tx, const void* w, const void* bias, void* pre, void* y, void* ty, int M, int N, int K, void* stream);

/*
 * gx = g w, the gradient of a linear layer's input: g (M, N), w (N, K), gx (M, K), bf16 and dense, fp32 accumulation.  N a multiple of 64, K
 * of 8, both up to 65536, at most 2^30 elements in each; 16-byte aligned.  dmf_linear_dgrad_plan: as dmf_linear_plan.
 */
DMF_ATTN_API int dmf_linear_dgrad_plan(int64_t M, int N, int K);
DMF_ATTN_API int dmf_linear_dgrad(const void* g, const void* w, void* gx, int M, int N, int K, void* stream);

/*
 * gw = g^T x, contracted over the M rows: g (M, N), x (M, K), bf16 and dense, gw (N, K) fp32, fp32 accumulation in a fixed order;
 * gbias (N, fp32) or NULL: the column sums of g besides.
 * N and K multiples of 8, fewer than 2^30 elements in each; 16-byte aligned.  workspace: dmf_linear_wgrad_workspace_floats(M, N, K)
 * floats (0: none is needed and NULL will do; -1: shape not covered), not cleared.  dmf_linear_wgrad_plan: as dmf_linear_plan;
 * dmf_linear_wgrad_sums_plan: the same for calls that want the column sums, which a library product does not give.
 */
DMF_ATTN_API int64_t dmf_linear_wgrad_workspace_floats(int64_t M, int N, int K);
DMF_ATTN_API int dmf_linear_wgrad_plan(int64_t M, int N, int K);
DMF_ATTN_API int dmf_linear_wgrad_sums_plan(int64_t M, int N, int K);
/* As dmf_linear_fwd_plan, for a layer's training: which 0 dmf_linear_gelu_fwd, 1 dmf_linear_dgrad, 2 dmf_linear_wgrad (with its splits of the rows). */
DMF_ATTN_API int dmf_linear_train_plan(int which, int64_t M, int N, int K, char* buf, int buflen);
DMF_ATTN_API int dmf_linear_wgrad(const void* g, const void* x, float* gw, float* gbias, float* workspace, int M, int N, int K, void* stream);

/*
 * dst[k] = src[k] rounded to bf16 (nearest, ties to even), k < count <= 4: dense fp32 arrays of n[k] elements, a multiple of 8.
 * The casts of a linear layer's operands under autocast.
 */
DMF_ATTN_API int dmf_cast_bf16(const void* const* src, void* const* dst, const int64_t* n, int count, void* stream);

/*
 * Sinusoidal embedding of n times: y[b] = [cos(t[b] f) | sin(t[b] f)] over the frequencies f[i] = exp(neg_log_period i / (dim / 2)),
 * i < dim / 2, a zero behind them where dim is odd, and when `ty` is given its tangent, [-sin(t f) f tt | cos(t f) f tt].
 * Replaces timestep_embedding (models/layers.py:46-55) and the cast behind it (:71).  t, tt: (n) of dtype; y, ty: (n, dim) of dtype;
 * computed in fp32.
 */
DMF_ATTN_API int dmf_timestep_embedding_fwd(const void* t, const void* tt, void* y, void* ty, int64_t n, int dim,
                                            float neg_log_period, int dtype, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* DMF_FUSED_H */
