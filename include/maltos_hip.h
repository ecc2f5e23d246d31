/*
 * maltos_hip.h -- C ABI of libmaltos_hip.so, the MI355X (gfx950) kernels for the per-GPU
 * training-step hot path of MALTOS: causal / document-masked attention forward and backward,
 * ring block attention with log-sum-exp merge, RMSNorm, interleaved RoPE, SwiGLU, causal
 * cross-entropy, global-norm clipping and fused AdamW over flat fp32 buffers.
 *
 * The reference (xing7code/maltos) is pure Python and has no FFI; each entry point below names
 * the reference call site (file:line under the reference tree) whose native work it replaces.
 *
 * Conventions
 *  - Every pointer is a DEVICE pointer unless stated otherwise.  Nothing here allocates or frees
 *    device memory: outputs and workspaces are caller-allocated.
 *  - `stream` is a hipStream_t passed as void*; NULL is the default stream.  All work is enqueued
 *    asynchronously on it; no entry point synchronises the host.
 *  - Return value: MLTS_OK (0) or an MLTS_ERR_* code; mlts_last_error() gives the message of the
 *    last failure on the calling thread.  Argument checks happen on the host before any launch.
 *  - dtype codes: MLTS_F32 = 0, MLTS_BF16 = 1.
 *  - Tensors are described by element strides where noted; the innermost (head_dim / hidden)
 *    dimension is always contiguous.
 */
#ifndef MALTOS_HIP_H
#define MALTOS_HIP_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define MLTS_OK 0
#define MLTS_ERR_INVALID 1     /* bad shape / pointer / alignment / dtype */
#define MLTS_ERR_UNSUPPORTED 2 /* valid request this build has no kernel for (see mlts_attn_supports) */
#define MLTS_ERR_LAUNCH 3      /* HIP runtime reported an error at launch */

#define MLTS_F32 0
#define MLTS_BF16 1

/* attention mask modes */
#define MLTS_MASK_NONE 0   /* every key visible (ring off-diagonal blocks) */
#define MLTS_MASK_CAUSAL 1 /* key j visible to query i iff j <= i + (Sk - Sq) */
#define MLTS_MASK_DOC 2    /* visible iff k_pos[j] <= q_pos[i] && q_seq[i] == k_seq[j] && q_seq[i] >= 0 */

typedef void* mlts_stream_t;

int mlts_abi_version(void);
const char* mlts_last_error(void);

/* Measurement aid with no counterpart in the reference (it times whole steps with a device
 * synchronise, tools/profile_train_perf.py:900-919): when enabled, the main kernel of each entry
 * point is bracketed by HIP events on its launch stream.  Names: "attn_fwd", "attn_bwd_dkdv",
 * "attn_bwd_dq", "attn_delta", "attn_doc_prepass", "attn_merge", "adamw", "ce", "rmsnorm_fwd",
 * "rmsnorm_bwd", "rope", "swiglu_fwd", "swiglu_bwd", "grad_to_f32", "grad_sum_slices".
 * mlts_kernel_timing_read synchronises on the recorded events and returns the summed kernel time
 * and the number of launches since timing was enabled.  Enabling or disabling clears the records. */
void mlts_kernel_timing_enable(int enable);
int mlts_kernel_timing_read(const char* name, double* total_ms, int64_t* launches);

/* ------------------------------------------------------------------------------------------ */
/* Attention                                                                                  */
/* ------------------------------------------------------------------------------------------ */

/* Layout of one attention call.  q/o/do/dq are [B, Hq, Sq, D]; k/v/dk/dv are [B, Hkv, Sk, D];
 * strides are in elements for (batch, head, seq); D is contiguous.  Query head h reads KV head
 * h / (Hq / Hkv) (the reference's repeat_interleave, models/llama.py:97-100). */
typedef struct mlts_attn_shape {
  int32_t B, Hq, Hkv, Sq, Sk, D;
  int32_t dtype;     /* MLTS_BF16 (MFMA path) or MLTS_F32 */
  int32_t mask_mode; /* MLTS_MASK_* */
  float scale;       /* softmax scale, the reference uses D^-0.5 (utils/attention_backend.py:128) */
  int64_t q_stride[3], k_stride[3], v_stride[3], o_stride[3];
  /* MLTS_MASK_DOC only: int32 [B, Sq] / [B, Sk] contiguous position and sequence ids
   * (runtime/layers/attn_masking_utils.py:54-87).  seq id < 0 marks padding
   * (utils/constants.py:4); padded queries produce zeros and lse = -inf. */
  const int32_t* q_pos;
  const int32_t* k_pos;
  const int32_t* q_seq;
  const int32_t* k_seq;
  /* MLTS_MASK_DOC only, optional: a plan built by mlts_attn_doc_plan for the same B, Hq, Hkv, Sq, Sk and the same
   * contents of the four id arrays.  NULL: the call builds its own at the front of its workspace. */
  const void* doc_plan;
} mlts_attn_shape;

/* NULL if (dtype, D, mask_mode, strides) is served by a kernel, else a static reason string.
 * Mirrors flash_attn_fallback_reason / flash_attn_dense_block_fallback_reason
 * (runtime/layers/flash_utils.py:105-135). */
const char* mlts_attn_supports(const mlts_attn_shape* s);

/* Bytes of device workspace mlts_attn_fwd / mlts_attn_bwd need for this shape: the per-row statistics the kernels
 * share (delta, LSE in base 2): O(B * Hq * Sq), the workspace class of the flash backward the reference calls
 * (runtime/layers/flash_utils.py:239-258).  With MLTS_MASK_DOC also the per-tile position / sequence-id ranges and
 * the visibility bits of the (64 queries, 64 keys) pairs that a document boundary or the causal diagonal cuts, which a
 * pre-pass forms once per call for all heads: B * Sq * Sk / 8 bytes (forward), twice that (backward). */
int64_t mlts_attn_fwd_workspace_bytes(const mlts_attn_shape* s);
int64_t mlts_attn_bwd_workspace_bytes(const mlts_attn_shape* s, int accumulate_f32);

/* Document-mask plan: what mlts_attn_fwd and mlts_attn_bwd derive from the ids in front of their kernels (tile
 * statistics, visibility bits of the tile pairs a document boundary or the diagonal cuts, the order in which the
 * kernels walk their blocks).  It depends on B, Hq / Hkv, Sq, Sk and the ids only, not on q, k, v: every layer of a
 * model, forward and backward, attends under the same mask, so a caller can build the plan once per batch into a
 * buffer of mlts_attn_doc_plan_bytes (16-byte aligned, B * Sq * Sk / 4 bytes and a little) and pass it in
 * mlts_attn_shape::doc_plan; the calls then skip their pre-pass (three small launches, 28 us at B=2, S=8192) and
 * mlts_attn_*_workspace_bytes no longer include it.  The plan must not be rewritten while a call that uses it is in
 * flight.  No counterpart in the reference, whose callers rebuild the varlen metadata per call
 * (runtime/layers/flash_utils.py:566-640).  Returns 0 bytes / does nothing for shapes the 16-row kernels serve. */
int64_t mlts_attn_doc_plan_bytes(const mlts_attn_shape* s);
int mlts_attn_doc_plan(const mlts_attn_shape* s, void* plan, int64_t plan_bytes, mlts_stream_t stream);

/* O = softmax(scale * Q K^T + mask) V and LSE = logsumexp (natural log, fp32, [B, Hq, Sq]).
 * Replaces F.scaled_dot_product_attention (utils/attention_backend.py:60-64,109-116),
 * flash_attn_dense / flash_attn_dense_with_lse / flash_attn_varlen
 * (runtime/layers/flash_utils.py:180-215,266-276,493-520).
 *
 * Bits (this call and mlts_attn_bwd): the same call gives the same bits every time.  A batch row in a call on more rows has
 * the bits of a call on that row alone only for MLTS_BF16 at D 64 and 128 whose walk is shorter than 512 rows (O, LSE and dQ: Sk < 512;
 * dK and dV: Sq < 512).  Otherwise the kernel, or how many wavefronts share a row's walk, follows the size of the whole
 * call, and a row's last bits may change with B; so they may with the linear layers' products below. */
int mlts_attn_fwd(const mlts_attn_shape* s, const void* q, const void* k, const void* v, void* o,
                  float* lse, void* workspace, int64_t workspace_bytes, mlts_stream_t stream);

/* dQ, dK, dV by recompute from (Q, K, V, O, LSE, dO); O and LSE may be the GLOBAL ones of a ring
 * schedule, which is what makes per-block calls compose.  Replaces flash_attn_dense_backward
 * (runtime/layers/flash_utils.py:218-263) and the autograd of SDPA.
 * accumulate_f32 (strides dq_stride etc are in elements of the respective type):
 *   MLTS_BWD_OVERWRITE (0)     dq/dk/dv have the input dtype and are overwritten.
 *   MLTS_BWD_ACCUMULATE (1)    dq/dk/dv are fp32 and are ADDED to (the `dq += block_dq.float()` form of
 *                              runtime/layers/functional.py:1121-1146).
 *   MLTS_BWD_DQ_ACCUMULATE (2) dq is fp32 and added to; dk/dv have the input dtype and are overwritten: a block of a
 *                              ring step on the rank that owns the queries, where a K/V chunk meets the local queries
 *                              exactly once (functional.py:1104-1146: one `dk += ...` per chunk and rank).
 *   MLTS_BWD_DQ_STORE (3)      as 2, but dq (fp32) is overwritten: the first block of such an accumulation, which
 *                              saves clearing the fp32 buffer beforehand. */
#define MLTS_BWD_OVERWRITE 0
#define MLTS_BWD_ACCUMULATE 1
#define MLTS_BWD_DQ_ACCUMULATE 2
#define MLTS_BWD_DQ_STORE 3
int mlts_attn_bwd(const mlts_attn_shape* s, const void* dout, const int64_t do_stride[3], const void* q,
                  const void* k, const void* v, const void* o, const float* lse, void* dq,
                  const int64_t dq_stride[3], void* dk, const int64_t dk_stride[3], void* dv,
                  const int64_t dv_stride[3], int accumulate_f32, void* workspace, int64_t workspace_bytes,
                  mlts_stream_t stream);

/* mlts_attn_bwd with MLTS_BWD_OVERWRITE of queries and keys that were rotated (mlts_rope_pair, mlts_gemm_rope), and mlts_rope_pair with `inverse` over dq
 * and dk in place: the same values (bf16: the same bits), where a kernel of this shape can without a pass of its own.  Sq and Sk are equal.  cos, sin, max_pos,
 * positions and position_offset as mlts_rope takes them, and refused as there. */
typedef struct {
  const void *cos, *sin;
  const int32_t* positions;
  int32_t max_pos, position_offset;
} mlts_attn_rotation;
int mlts_attn_bwd_rope(const mlts_attn_shape* s, const void* dout, const int64_t do_stride[3], const void* q,
                       const void* k, const void* v, const void* o, const float* lse, void* dq,
                       const int64_t dq_stride[3], void* dk, const int64_t dk_stride[3], void* dv,
                       const int64_t dv_stride[3], const mlts_attn_rotation* rotation, void* workspace,
                       int64_t workspace_bytes, mlts_stream_t stream);

/* mlts_attn_bwd for callers that cannot allocate device memory or bring a workspace (code under HIP graph capture,
 * tight serving loops, harnesses that forbid hipMalloc).  It has no counterpart in the reference.  Same arguments and
 * results as mlts_attn_bwd with a workspace of exactly mlts_attn_bwd_workspace_bytes (the recomputing backward); the
 * workspace is a buffer of MLTS_ATTN_BWD_NOALLOC_MAX_WORKSPACE bytes inside the library image, one copy per GPU, held
 * until the process ends.  Shapes whose workspace is larger (about B * Hq * Sq > 1 M query rows; with MLTS_MASK_DOC
 * also B * Sq * Sk / 4 bytes of visibility bits, e.g. B * S * S beyond about 28 M) are rejected with MLTS_ERR_INVALID.  No hipMalloc / hipFree is made.  All calls on one GPU share that buffer.  Calls on
 * different streams of one GPU are made to take turns (each waits for an event recorded behind the last), except calls
 * recorded into a HIP graph: graphs that hold this call and may run at the same time on one GPU race on the buffer and
 * must be ordered by the caller, or use mlts_attn_bwd with one workspace per graph. */
#define MLTS_ATTN_BWD_NOALLOC_MAX_WORKSPACE (8 << 20)
int mlts_attn_bwd_noalloc(const mlts_attn_shape* s, const void* dout, const int64_t do_stride[3], const void* q,
                          const void* k, const void* v, const void* o, const float* lse, void* dq,
                          const int64_t dq_stride[3], void* dk, const int64_t dk_stride[3], void* dv,
                          const int64_t dv_stride[3], int accumulate_f32, mlts_stream_t stream);

/* Which splits a pass of bf16 attention takes over wavefronts with two blocks of 16 rows each; host only.  pass: 0 forward, 1 dQ, 2 dK/dV;
   blocks: pairs of row blocks, of all heads; units: of 32 rows, that each walks. */
int32_t mlts_attn_small_splits(int32_t pass, int32_t head_dim, int64_t blocks, int64_t units);

/* Log-sum-exp merge of one block into the running fp32 state, rows [q_off, q_off + q_len):
 *   lse' = logaddexp(lse, lse_b); out' = out * exp(lse - lse') + out_b * exp(lse_b - lse'),
 * with exp(-inf - x) := 0 (a row where both are -inf becomes 0 with lse -inf).  Replaces
 * _merge_attention_blocks / _exp_delta_or_zero (runtime/layers/functional.py:717-748).
 * out_acc fp32 [B, H, S, D] contiguous; lse_acc fp32 [B, H, S]; o_blk [B, H, q_len, D] of
 * blk_dtype with strides; lse_blk fp32 [B, H, q_len] contiguous. */
int mlts_attn_merge(float* out_acc, float* lse_acc, const void* o_blk, const int64_t o_blk_stride[3],
                    int32_t blk_dtype, const float* lse_blk, int32_t B, int32_t H, int32_t S, int32_t D,
                    int32_t q_off, int32_t q_len, mlts_stream_t stream);

/* ------------------------------------------------------------------------------------------ */
/* Layer kernels                                                                              */
/* ------------------------------------------------------------------------------------------ */

/* y = w * round(x * rsqrt(mean(x^2) + eps)) with fp32 statistics and the reference's two
 * roundings (models/llama.py:55-57).  x, y [rows, hidden] contiguous; rstd_out fp32 [rows]. */
int mlts_rmsnorm_fwd(const void* x, const void* w, void* y, float* rstd_out, int64_t rows, int32_t hidden,
                     float eps, int32_t dtype, mlts_stream_t stream);
/* dx [rows, hidden]; dw [hidden] (same dtype).  dw_partial: fp32 workspace of
 * mlts_rmsnorm_bwd_workspace_bytes(rows, hidden) bytes. */
int64_t mlts_rmsnorm_bwd_workspace_bytes(int64_t rows, int32_t hidden);
int mlts_rmsnorm_bwd(const void* dy, const void* x, const void* w, const float* rstd, void* dx, void* dw,
                     void* workspace, int64_t workspace_bytes, int64_t rows, int32_t hidden, int32_t dtype,
                     mlts_stream_t stream);
/* The residual add in front of a norm fused into it (models/llama.py:224-230 `x = x + sublayer(...)` followed by the
 * next RMSNorm, :55-57): sum_out = round(x + res), y = RMSNorm(sum_out) with the roundings of the two separate ops.
 * sum_out and y are different buffers; sum_out may alias x or res. */
int mlts_add_rmsnorm_fwd(const void* x, const void* res, void* sum_out, const void* w, void* y, float* rstd_out,
                         int64_t rows, int32_t hidden, float eps, int32_t dtype, mlts_stream_t stream);
/* Backward of the pair: x is the summed row (sum_out above), dres the gradient reaching it by the residual path;
 * dx = round(dx of the norm) + dres, the gradient of both addends.  Other arguments as mlts_rmsnorm_bwd. */
int mlts_add_rmsnorm_bwd(const void* dy, const void* x, const void* w, const float* rstd, const void* dres, void* dx,
                         void* dw, void* workspace, int64_t workspace_bytes, int64_t rows, int32_t hidden, int32_t dtype,
                         mlts_stream_t stream);
/* Both (dres NULL: no residual path), with the weight gradient added onto dw in fp32 and rounded once. */
int mlts_rmsnorm_bwd_accumulate(const void* dy, const void* x, const void* w, const float* rstd, const void* dres, void* dx,
                                void* dw, void* workspace, int64_t workspace_bytes, int64_t rows, int32_t hidden,
                                int32_t dtype, mlts_stream_t stream);


/* Token-embedding gradient (nn.Embedding, models/llama.py:238): dw[ids[t]] += dy[t].  ids int64 [n] (ids outside
 * [0, vocab) are skipped: the forward lookup rejects them), dy [n, hidden], dw [vocab, hidden]; equal ids are summed in fp32 in a fixed order and added onto dw with one rounding.
 * mlts_embedding_bwd_supports: NULL, or why these sizes are not taken. */
const char* mlts_embedding_bwd_supports(int64_t n, int64_t hidden, int64_t vocab, int32_t dtype);
int mlts_embedding_bwd(const int64_t* ids, const void* dy, void* dw, int64_t n, int64_t hidden, int64_t vocab, int32_t dtype,
                       mlts_stream_t stream);

/* Interleaved-pair rotary embedding (models/llama.py:89-94,134-144):
 *   (x[2i], x[2i+1]) -> (x[2i] c - x[2i+1] s, x[2i] s + x[2i+1] c), c/s = cos/sin[pos, i],
 * every product and the sum rounded to `dtype` as the reference's eager ops do.
 * x, y: [B, H, S, D] with element strides (batch, head, seq); cos/sin: [max_pos, D/2] of `dtype`.
 * positions: int32 [B, S] or NULL (then pos = position_offset + s).  inverse != 0 rotates by
 * -theta, which is the backward pass.  y may be x with the same strides (rotation in place); any other overlap of the
 * two is undefined. */
int mlts_rope(const void* x, const int64_t x_stride[3], void* y, const int64_t y_stride[3], const void* cos_tab,
              const void* sin_tab, int32_t max_pos, const int32_t* positions, int32_t position_offset,
              int32_t B, int32_t H, int32_t S, int32_t D, int32_t dtype, int32_t inverse,
              mlts_stream_t stream);

/* The two rotations of one attention layer, q = rotary(q) and k = rotary(k) (models/llama.py:143-144), in one launch:
 * operand a is [B, Ha, S, D], operand b [B, Hb, S, D]; everything else as mlts_rope, whose results it equals bit for
 * bit.  Each operand must hold fewer than 2^31 16-byte vectors. */
int mlts_rope_pair(const void* xa, const int64_t xa_stride[3], void* ya, const int64_t ya_stride[3], int32_t Ha,
                   const void* xb, const int64_t xb_stride[3], void* yb, const int64_t yb_stride[3], int32_t Hb,
                   const void* cos_tab, const void* sin_tab, int32_t max_pos, const int32_t* positions,
                   int32_t position_offset, int32_t B, int32_t S, int32_t D, int32_t dtype, int32_t inverse,
                   mlts_stream_t stream);

/* h = round(silu(gate)) * up (models/llama.py:205-206); n = number of elements, contiguous. */
int mlts_swiglu_fwd(const void* gate, const void* up, void* h, int64_t n, int32_t dtype, mlts_stream_t stream);
int mlts_swiglu_bwd(const void* dh, const void* gate, const void* up, void* dgate, void* dup, int64_t n,
                    int32_t dtype, mlts_stream_t stream);

/* The same over [rows, cols] matrices with row strides in elements (multiples of 16 bytes): gate and up are the two
 * column halves of ONE projection output (gate_proj and up_proj of models/llama.py:196-206 run as one GEMM over their
 * adjacent weights), dgate and dup the halves of one gradient buffer, so that the next GEMM reads them without a copy. */
int mlts_swiglu_fwd_rows(const void* gate, const void* up, int64_t ld_in, void* h, int64_t ld_h, int64_t rows, int64_t cols,
                         int32_t dtype, mlts_stream_t stream);
int mlts_swiglu_bwd_rows(const void* dh, int64_t ld_dh, const void* gate, const void* up, int64_t ld_in, void* dgate, void* dup,
                         int64_t ld_out, int64_t rows, int64_t cols, int32_t dtype, mlts_stream_t stream);

/* Causal cross-entropy, forward and gradient in one pass over the logits (utils/losses.py:9-15):
 *   loss = sum_{t: label_t != ignore_index} (logsumexp(z_t) - z_t[label_t]) / max(1, #targets)
 *   dlogits_t = (softmax(z_t) - onehot(label_t)) / max(1, #targets) for supervised rows, else 0.
 * logits, dlogits: [rows, vocab] contiguous of `dtype` (dlogits may alias logits); labels int64
 * [rows]; loss_out fp32 [1]; count_out int32 [1]; workspace: fp32 [rows] + 64 bytes. */
int64_t mlts_ce_workspace_bytes(int64_t rows);
int mlts_ce_fwd_bwd(const void* logits, const int64_t* labels, void* dlogits, float* loss_out,
                    int32_t* count_out, void* workspace, int64_t workspace_bytes, int64_t rows, int32_t vocab,
                    int64_t ignore_index, int32_t dtype, mlts_stream_t stream);
/* x *= *scale (device fp32 scalar) unless *scale == 1: applies the upstream d(loss) to the
 * gradient that mlts_ce_fwd_bwd stored. */
int mlts_scale_by_device_scalar(void* x, const float* scale, int64_t n, int32_t dtype, mlts_stream_t stream);

/* ------------------------------------------------------------------------------------------ */
/* Optimizer step over flat buffers                                                           */
/* ------------------------------------------------------------------------------------------ */

#define MLTS_SQNORM_WS_BYTES 16384

/* dst_f32[i] (=|+=) float(src[i]); optional fused sum of squares of the RESULT in fp64.
 * Replaces the per-parameter grad upcast of MasterWeightsOptimizer.copy_master_params
 * (runtime/optim.py:43-56).  sq_out (fp64 [1]) and workspace (MLTS_SQNORM_WS_BYTES) may be NULL. */
int mlts_grad_to_f32(float* dst, const void* src, int32_t src_dtype, int64_t n, int accumulate, double* sq_out,
                     void* workspace, mlts_stream_t stream);

/* out[i] = (accumulate ? out[i] : 0) + sum over s < slices of parts[s * n + i], added in fp32 and rounded once to
 * `dtype` (bf16 or fp32; out and parts share it).  Finishes a weight gradient dW = dY^T X of nn.Linear
 * (models/llama.py:69-75,196-198) that was computed as `slices` row-slice products, and with accumulate != 0 adds it
 * onto the gradient already held in a view of the flat gradient buffer (runtime/plugins/zero1.py:117-121), which is
 * what autograd's `param.grad += dW` does there in a second pass. */
int mlts_grad_sum_slices(void* out, const void* parts, int32_t dtype, int32_t slices, int64_t n, int accumulate,
                         mlts_stream_t stream);

/* *sq_out = sum x[i]^2 accumulated in fp64 (runtime/plugins/grad_clip.py:62-77,
 * runtime/plugins/zero_common.py:324-329).  workspace: MLTS_SQNORM_WS_BYTES. */
int mlts_sq_norm(const float* x, int64_t n, double* sq_out, void* workspace, mlts_stream_t stream);

/* Matrix products of the linear layers (models/llama.py:69-75,134-142,196-206 and their gradients, which the reference leaves to
 * the vendor library through torch): C[M, N] = A B, row major, fp32 accumulation, one rounding.
 *   MLTS_GEMM_NT  A[M, K] B[N, K]   y = x W^T
 *   MLTS_GEMM_NN  A[M, K] B[K, N]   dx = dy W
 *   MLTS_GEMM_TN  A[K, M] B[K, N]   dW = dy^T x; C dense
 * ld*: elements between rows.  accumulate != 0: added onto C in fp32 before the rounding.  mlts_gemm_supports: NULL, or why a
 * product is not served (alignment of 16 bytes along rows, operands below 2 GiB).  Workspace: mlts_gemm_workspace_bytes (the
 * fp32 parts of a contraction that is split over workgroups; 0 for most). */
#define MLTS_GEMM_NT 0
#define MLTS_GEMM_NN 1
#define MLTS_GEMM_TN 2
const char* mlts_gemm_supports(int32_t form, int32_t dtype, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc);
int64_t mlts_gemm_workspace_bytes(int32_t form, int32_t dtype, int64_t M, int64_t N, int64_t K);
int mlts_gemm(int32_t form, int32_t dtype, int64_t M, int64_t N, int64_t K, const void* a, int64_t lda, const void* b, int64_t ldb,
              void* c, int64_t ldc, int32_t accumulate, void* workspace, int64_t workspace_bytes, mlts_stream_t stream);
/* Up to four products in one call, small ones in one launch.  A product of the NN form may be the sum over up to three
 * segments a[i] b[i] (the input gradient of layers that share their input), in bf16 with the roundings of separate products.
 * A launch takes the segments of one product: a call with more of them takes more launches.  The outputs of a call must not
 * overlap (MLTS_ERR_INVALID).  Bits: the same call gives the same every time.  An element's depend on its own row and column, the sizes of the product, and in MLTS_F32
 * also on what shares the call, which the tile is chosen for: small tiles multiply fp32 numbers whole, larger ones in three bf16 parts (24 bits, exact for every fp32
 * number), with a third of the error.  An MLTS_BF16 weight gradient keeps the split it has alone. */
typedef struct {
  int32_t form, segments, accumulate;
  int64_t M, N;
  int64_t k[3];
  const void *a[3], *b[3];
  int64_t lda[3], ldb[3];
  void* c;
  int64_t ldc;
} mlts_gemm_product;
int64_t mlts_gemm_multi_workspace_bytes(const mlts_gemm_product* products, int32_t count, int32_t dtype);
int mlts_gemm_multi(const mlts_gemm_product* products, int32_t count, int32_t dtype, void* workspace, int64_t workspace_bytes,
                    mlts_stream_t stream);
/* What a call would launch, decided on the host (nothing runs, no GPU is asked for): each product's tile, into how many slices its contraction is
 * split, and whether it shares a launch with the others.  with: the products by themselves, or what mlts_gemm_rope, mlts_gemm_swiglu_bwd (dW and dh) or
 * mlts_gemm_swiglu (one product, N of each of the two) makes of them. */
#define MLTS_GEMM_WITH_NOTHING 0
#define MLTS_GEMM_WITH_ROTATION 1
#define MLTS_GEMM_WITH_ACTIVATION 2
#define MLTS_GEMM_WITH_GATE_UP 3
typedef struct {
  int32_t tile_m, tile_n, slices, together;
  int32_t busiest; /* tiles of the launch that the XCD with the most of them gets */
} mlts_gemm_tiles;
int mlts_gemm_plan(const mlts_gemm_product* products, int32_t count, int32_t dtype, int32_t with, mlts_gemm_tiles* tiles);
/* The backward pass of h W^T (W [K, N], h = round(silu(gate)) * up) in one launch: dW (+)= dy^T h (dense; null: not wanted), and d gate,
 * d up of dh = dy W, which is not written: the values of two products and mlts_swiglu_bwd_rows.  supports: NULL and the workspace it takes, or why not. */
const char* mlts_gemm_swiglu_bwd_supports(int32_t dtype, int32_t weight, int64_t M, int64_t N, int64_t K, int64_t ldy, int64_t ldw, int64_t ldh,
                                          int64_t ldg, int64_t ldd, int64_t* workspace_bytes);
int mlts_gemm_swiglu_bwd(int32_t dtype, int64_t M, int64_t N, int64_t K, const void* dy, int64_t ldy, const void* w, int64_t ldw, const void* h,
                         int64_t ldh, void* dw, int32_t accumulate, const void* gate, const void* up, int64_t ldg, void* dgate, void* dup,
                         int64_t ldd, void* workspace, int64_t workspace_bytes, mlts_stream_t stream);
/* NT products of one call, some of whose columns are heads that are rotated to their positions as they are written
 * (models/llama.py:143-146): the values of mlts_gemm_multi followed by mlts_rope over them.  Row r is token r % seq of its batch row, at
 * positions[r], or at position_offset + r % seq.  columns[i]: two ranges [begin, end) of whole heads of product i (empty: begin = end).
 * Products that would be split are not served: mlts_gemm_rope_supports says NULL, or why. */
typedef struct {
  const void *cos, *sin; /* [max_pos, head_dim / 2], the products' dtype, 8-byte aligned */
  const int32_t* positions;
  int32_t max_pos, position_offset, seq, head_dim;
  int64_t columns[4][4];
} mlts_gemm_rotation;
const char* mlts_gemm_rope_supports(const mlts_gemm_product* products, int32_t count, int32_t dtype, const mlts_gemm_rotation* rotation);
int mlts_gemm_rope(const mlts_gemm_product* products, int32_t count, int32_t dtype, const mlts_gemm_rotation* rotation, mlts_stream_t stream);
/* gate = x W_gate^T, up = x W_up^T (W [N, K], x [M, K]) and h = round(silu(gate)) * up of the rounded gate and up (models/llama.py:205-206)
 * in one launch: the values of two products and mlts_swiglu_fwd_rows.  gate and up may be null (nobody reads them).  Sizes whose products
 * would be split (fp32: or are faster with a pass behind them) are not served: mlts_gemm_swiglu_supports says NULL, or why. */
const char* mlts_gemm_swiglu_supports(int32_t dtype, int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int64_t ldc, int64_t ldh);
int mlts_gemm_swiglu(int32_t dtype, int64_t M, int64_t N, int64_t K, const void* x, int64_t ldx, const void* w_gate, const void* w_up,
                     int64_t ldw, void* gate, void* up, int64_t ldc, void* h, int64_t ldh, mlts_stream_t stream);


/* The norm, scaling and AdamW passes over a list of fp32 tensors (host arrays of device pointers and element counts) in one
 * launch per 48 tensors, for parameters that do not share a flat buffer: what the reference's optimizer does per parameter
 * (torch's multi-tensor AdamW, train/cli.py:420-443; runtime/plugins/grad_clip.py:30-77).  Workspace of the norm:
 * mlts_list_sq_norm_workspace_bytes. */
int64_t mlts_list_sq_norm_workspace_bytes(const int64_t* sizes, int32_t count);
int mlts_list_sq_norm(const float* const* tensors, const int64_t* sizes, int32_t count, double* sq_out, void* workspace,
                      int64_t workspace_bytes, mlts_stream_t stream);
int mlts_list_scale(float* const* tensors, const int64_t* sizes, int32_t count, float scale, mlts_stream_t stream);
int mlts_list_adamw_step(float* const* p, const float* const* g, float* const* m, float* const* v, const int64_t* sizes,
                         int32_t count, float lr, float beta1, float beta2, float eps, float weight_decay, int64_t step,
                         float grad_scale, const double* sq_norm, float max_norm, mlts_stream_t stream);

/* x *= scale (runtime/plugins/grad_clip.py:55-58). */
int mlts_scale(float* x, float scale, int64_t n, mlts_stream_t stream);

/* Decoupled-weight-decay Adam on flat fp32 p/g/m/v (torch.optim.AdamW as built by
 * train/cli.py:432-441, stepped inside runtime/optim.py:65-71):
 *   g' = g * c;  p *= 1 - lr*wd;  m = lerp(m, g', 1-b1);  v = b2 v + (1-b2) g'^2;
 *   p -= (lr / (1-b1^t)) * m / (sqrt(v)/sqrt(1-b2^t) + eps)
 * c = grad_scale, further multiplied by the clip coefficient max_norm / (sqrt(*sq_norm) + 1e-6)
 * when sq_norm != NULL and that coefficient is < 1 (runtime/plugins/grad_clip.py:54-58).
 * p_lowp, if not NULL, receives bf16(p) in the same pass (the write-back of
 * runtime/optim.py:68-70).  step is the 1-based step count t. */
int mlts_adamw_step(float* p, const float* g, float* m, float* v, void* p_lowp, int64_t n, float lr, float beta1,
                    float beta2, float eps, float weight_decay, int64_t step, float grad_scale,
                    const double* sq_norm, float max_norm, mlts_stream_t stream);

#ifdef __cplusplus
}
#endif
#endif /* MALTOS_HIP_H */
