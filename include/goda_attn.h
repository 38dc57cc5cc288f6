/*
 * goda_attn.h -- C-ABI of the MI355X (gfx950) attention hot path.
 *
 * The library (libgoda_attn.so) replaces the attention kernels that goda calls
 * from Python. Every entry point takes plain device pointers, element strides
 * and sizes; nothing here names a framework type. Work is enqueued on the HIP
 * stream passed in `stream` (a hipStream_t; NULL = the default stream) and the
 * call returns without synchronising. The library never allocates device
 * memory: outputs and the workspace are owned by the caller.
 *
 * Logical layouts (strides are in ELEMENTS, the head dimension must be
 * contiguous, i.e. stride 1):
 *   dense  q/o : [batch, seqlen_q, heads_q,  head_dim]   any (b, t, h) strides
 *   dense  k/v : [batch, seqlen_k, heads_kv, head_dim]   any (b, t, h) strides
 *   varlen q/o : [total_q, heads_q,  head_dim], rows of sequence b are
 *                cu_seqlens_q[b] .. cu_seqlens_q[b+1]-1  (stride_b ignored)
 *   varlen k/v : same with cu_seqlens_k
 * so both goda's module layout [B,T,H,D] (mint/nn/attn.py:53-55) and the kernel
 * layout [B,H,T,D] (kernels_/flash_attn_gqa/cuda.py:358-363) are accepted as
 * strided views without copies.
 *
 * Semantics follow goda's eager attention (mint/nn/flashattn.py:221-273):
 *   - query head h reads key/value head h / (heads_q / heads_kv);
 *   - causal alignment is bottom-right: query row i of a sequence with Lq
 *     queries and Lk keys sees key j iff j <= (Lk - Lq) + i;
 *   - left window W >= 0 additionally requires (Lk - Lq + i) - j <= W;
 *   - ALiBi adds slope[h] * (j - (Lk - Lq + i)) to the scaled score
 *     (mint/nn/pos.py:186-207);
 *   - RoPE is the half-split rotation of mint/nn/pos.py:90-98 with caller
 *     supplied fp32 cos/sin tables [rope_len, head_dim/2]; query row i is
 *     rotated at position rope_q_offset + (Lk - Lq) + i (rope_pos_abs = 0)
 *     or rope_q_offset + i (rope_pos_abs = 1), key row j at
 *     rope_k_offset + j;
 *   - an optional boolean mask (goda's base_attn_mask,
 *     mint/nn/flashattn.py:242-243) further hides keys: bit-packed, see
 *     goda_prefill_args.mask_bits;
 *   - the optional fused QK-RMSNorm is goda's RMSNorm (mint/nn/norm.py:17-27)
 *     as applied to q and k before RoPE (mint/nn/attn.py:57-60): a head row
 *     x becomes x * rsqrt(mean(x^2) + norm_eps) * (1 + w) in fp32, with a
 *     caller supplied fp32 weight w [head_dim] (the module's `scale`);
 *   - lse = ln(sum_j exp(score_ij)) over the scaled, biased scores of the
 *     visible keys
 *     (kernels_/flash_attn_gqa/cuda.py:496-499). A row with no visible key
 *     produces o = 0 and lse = -inf.
 *
 * Every entry point returns GODA_OK (0) or a negative status; the message of
 * the last failure on the calling thread is returned by goda_attn_last_error.
 */
#ifndef GODA_ATTN_H
#define GODA_ATTN_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define GODA_ATTN_ABI_VERSION 6

/* element types */
#define GODA_DTYPE_F32 0
#define GODA_DTYPE_F16 1
#define GODA_DTYPE_BF16 2

/* status codes */
#define GODA_OK 0
#define GODA_ERR_INVALID_ARG (-1)
#define GODA_ERR_UNSUPPORTED (-2)
#define GODA_ERR_WORKSPACE (-3)
#define GODA_ERR_HIP (-4)

typedef struct goda_prefill_args {
  int32_t dtype;       /* GODA_DTYPE_* of q, k, v and o */
  int32_t batch;       /* number of sequences */
  int32_t heads_q;
  int32_t heads_kv;    /* must divide heads_q */
  int32_t head_dim;
  int32_t seqlen_q;    /* dense: T_q; varlen: max over sequences */
  int32_t seqlen_k;    /* dense: T_k; varlen: max over sequences */
  int32_t causal;      /* 0 / 1 */
  int32_t window_left; /* -1: unlimited */
  float softmax_scale; /* goda uses 1/sqrt(head_dim) (mint/nn/flashattn.py:143) */

  const void* q;
  const void* k;
  const void* v;
  void* o;
  int64_t q_stride_b, q_stride_t, q_stride_h;
  int64_t k_stride_b, k_stride_t, k_stride_h;
  int64_t v_stride_b, v_stride_t, v_stride_h;
  int64_t o_stride_b, o_stride_t, o_stride_h;

  /* fp32 log-sum-exp, dense [B, Hq, T_q] / varlen [Hq, total_q]; row stride 1.
   * NULL: not written. */
  float* lse;
  int64_t lse_stride_b, lse_stride_h;

  const int32_t* cu_seqlens_q; /* [batch+1] or NULL (dense) */
  const int32_t* cu_seqlens_k; /* [batch+1] or NULL (dense) */
  const int32_t* seqused_k;    /* [batch] keys used per sequence, or NULL */

  const float* alibi_slopes;   /* [heads_q] or NULL */

  const float* rope_cos;       /* [rope_len, head_dim/2] fp32, or NULL */
  const float* rope_sin;
  int32_t rope_len;
  int32_t rope_q;              /* rotate q rows */
  int32_t rope_k;              /* rotate k rows */
  int32_t rope_q_offset;
  int32_t rope_k_offset;
  float norm_eps;              /* epsilon of the fused RMSNorm (goda: 1e-6) */
  int32_t rope_pos_abs;        /* 1: query row i rotates at rope_q_offset + i
                                  (a caller-given start position, as goda's
                                  RoPE(q, k, start_pos), mint/nn/pos.py:100-112);
                                  0: at rope_q_offset + (Lk - Lq) + i */
  int32_t rope_packed_rows;    /* 1 (packed rows, cu_seqlens): query and key
                                  rows rotate at their packed row index modulo
                                  rope_len (at least 64), the offsets and
                                  rope_pos_abs unused: documents packed from
                                  rows of rope_len tokens keep their positions
                                  in the row (shorter rows: tables that
                                  repeat). ABI 6: what was padding before. */

  /* Fused QK-RMSNorm weights, fp32 [head_dim] each, or NULL (no norm on
   * that side; goda's q_norm / k_norm, mint/nn/norm.py:17-27, weight
   * 1 + w, before RoPE). goda_attn_prefill_bwd differentiates through them:
   * its dq / dk are the gradients of the rows before the norm, and
   * goda_prefill_grads.dq_norm_weight / dk_norm_weight receive dL/dw. */
  const float* q_norm_weight;
  const float* k_norm_weight;

  /* Optional boolean mask composed with causal / window / ALiBi, goda's
   * base_attn_mask (mint/nn/flashattn.py:242-243, broadcastable to
   * [B, Hq, Lq, Lk]): key j is visible to query row i (0-based within its
   * sequence) of query head h in sequence b only if bit j % 32 of word
   *   mask_bits[b*mask_stride_b + h*mask_stride_h + i*mask_stride_q + j/32]
   * is 1. Strides are in 32-bit words (0 broadcasts that dimension) and must
   * be even, the pointer 8-byte aligned, and every row must hold
   * 2*ceil(seqlen_k/64) readable words (bits past the keys are ignored).
   * Dense launches only (cu_seqlens NULL). NULL: no mask. A row that sees no
   * key produces o = 0 and lse = -inf. */
  const uint32_t* mask_bits;
  int64_t mask_stride_b, mask_stride_h, mask_stride_q;

  void* workspace;             /* size from goda_attn_prefill_workspace_size */
  int64_t workspace_bytes;

  /* Optional hipEvent_t pair recorded on `stream` right before and right
   * after the attention kernel itself (not the K/V pre-pass), so a caller
   * can time that kernel alone. NULL: not recorded. */
  void* timing_begin;
  void* timing_end;
} goda_prefill_args;

typedef struct goda_decode_args {
  int32_t dtype;
  int32_t batch;
  int32_t heads_q;
  int32_t heads_kv;
  int32_t head_dim;
  int32_t max_seqlen;   /* rows of the cache (Lmax) */
  int32_t window_left;  /* -1: unlimited */
  int32_t split_size;   /* keys per work range (multiple of 64); 0 = the visible
                           keys of all sequences spread evenly over the GPU */
  float softmax_scale;
  int32_t rope_pos_abs; /* 1: q rotates at rope_q_offset (a caller-given
                           position); 0: at cache_seqlens[b] - 1 + rope_q_offset */

  const void* q;        /* [batch, heads_q, head_dim]: one new token per sequence */
  int64_t q_stride_b, q_stride_h;
  const void* k_cache;  /* [batch, Lmax, heads_kv, D] or [batch, heads_kv, Lmax, D] via strides */
  int64_t k_stride_b, k_stride_t, k_stride_h;
  const void* v_cache;
  int64_t v_stride_b, v_stride_t, v_stride_h;
  const int32_t* cache_seqlens; /* [batch] valid keys per sequence (new token included) */
  void* o;              /* [batch, heads_q, head_dim] */
  int64_t o_stride_b, o_stride_h;
  float* lse;           /* [batch, heads_q] fp32 or NULL */
  int64_t lse_stride_b;

  const float* alibi_slopes; /* [heads_q] or NULL */
  const float* rope_cos;     /* rotate q (position: see rope_pos_abs) */
  const float* rope_sin;
  int32_t rope_len;
  int32_t rope_q;
  int32_t rope_q_offset;
  float norm_eps;
  const float* q_norm_weight; /* fused RMSNorm of q before RoPE, fp32 [head_dim], or NULL */

  void* workspace;           /* size from goda_attn_decode_workspace_size */
  int64_t workspace_bytes;

  /* Optional hipEvent_t pair recorded on `stream` right before and right
   * after the split-K kernel (not the merge). NULL: not recorded. */
  void* timing_begin;
  void* timing_end;
} goda_decode_args;

typedef struct goda_kv_append_args {
  int32_t dtype;
  int32_t batch;
  int32_t heads_kv;
  int32_t head_dim;
  int32_t max_seqlen;   /* rows of the cache (Lmax) */
  int32_t seqlen_new;   /* rows appended to every sequence */
  const void* k_new;    /* [batch, seqlen_new, heads_kv, D] via strides */
  int64_t kn_stride_b, kn_stride_t, kn_stride_h;
  const void* v_new;
  int64_t vn_stride_b, vn_stride_t, vn_stride_h;
  void* k_cache;
  int64_t k_stride_b, k_stride_t, k_stride_h;
  void* v_cache;
  int64_t v_stride_b, v_stride_t, v_stride_h;
  int32_t* cache_seqlens; /* [batch]: in = write position, out = position + seqlen_new,
                             clamped to max_seqlen */
  const float* rope_cos;  /* rotate new k row t at (cache position + rope_k_offset), or
                             at rope_k_offset + t with rope_pos_abs */
  const float* rope_sin;
  int32_t rope_len;
  int32_t rope_k;
  int32_t rope_k_offset;
  float norm_eps;
  const float* k_norm_weight; /* fused RMSNorm of new k rows before RoPE, fp32 [head_dim], or NULL */
  int32_t rope_pos_abs;
  int32_t reserved0;
  /* Overflow report, or NULL: a sequence whose rows would pass max_seqlen
   * keeps only the rows that fit, its length stops at max_seqlen, and the
   * launch stores 1 here (never 0: the caller clears it). goda's
   * KVCache.update fails on the same input (mint/kvcache/base.py:40-43). */
  int32_t* status;
} goda_kv_append_args;

/* Gradients for goda_attn_prefill_bwd. Every tensor uses the (b, t, h)
 * element-stride convention of goda_prefill_args (b strides unused for
 * varlen); the dtype is the forward's. */
typedef struct goda_prefill_grads {
  const void* d_o;      /* dL/dO, laid out like o */
  int64_t do_stride_b, do_stride_t, do_stride_h;
  void* dq;             /* dL/dq for the caller's (unrotated) q, like q */
  int64_t dq_stride_b, dq_stride_t, dq_stride_h;
  void* dk;             /* dL/dk, like k: heads_kv heads, each the sum over
                           its query-head group; rows past a sequence's keys
                           (seqused_k) are written as 0 */
  int64_t dk_stride_b, dk_stride_t, dk_stride_h;
  void* dv;             /* dL/dv, like v */
  int64_t dv_stride_b, dv_stride_t, dv_stride_h;
  /* With the fused QK-RMSNorm (fwd->q_norm_weight / k_norm_weight set), dq and
   * dk are the gradients of the caller's rows before the norm, and these
   * receive dL/dw of each norm weight, fp32 [head_dim] (NULL: not computed;
   * ignored without the norm; zeros for an empty problem, batch 0 or no rows
   * and no keys). Deterministic: no atomics. */
  float* dq_norm_weight;
  float* dk_norm_weight;

  void* workspace;      /* size from goda_attn_prefill_bwd_workspace_size */
  int64_t workspace_bytes;

  /* Optional hipEvent_t pair recorded around the gradient kernels (after the
   * row-statistics pre-pass). NULL: not recorded. */
  void* timing_begin;
  void* timing_end;
} goda_prefill_grads;

/* ABI version and struct sizes, so that a binding can check its mirror. */
int32_t goda_attn_abi_version(void);
int64_t goda_attn_sizeof_prefill_args(void);
int64_t goda_attn_sizeof_decode_args(void);
int64_t goda_attn_sizeof_kv_append_args(void);
int64_t goda_attn_sizeof_prefill_grads(void);

/* Message of the last failed call on this thread ("" if none). */
const char* goda_attn_last_error(void);

/* Workspace needed by goda_attn_prefill_fwd for these arguments (bytes, >= 0),
 * or a negative status if the arguments are rejected. */
int64_t goda_attn_prefill_workspace_size(const goda_prefill_args* args);

/* Causal / non-causal GQA-MQA prefill forward: o = softmax(q k^T * scale + bias) v,
 * plus the optional lse. Replaces FlashAttentionGQAKernel.forward
 * (kernels_/flash_attn_gqa/cuda.py:515-575), FlashAttentionMQAKernel.forward
 * (kernels_/flash_attn_mqa/cuda.py:470-527) and the SDPA branch of
 * FlashAttention._attention (mint/nn/flashattn.py:156-172, 221-273), including
 * the packed varlen call of mint/nn/flashattn.py:123-133 (cu_seqlens). */
int32_t goda_attn_prefill_fwd(const goda_prefill_args* args, void* stream);

/* Workspace of goda_attn_prefill_bwd for these forward arguments (bytes, >= 0),
 * or a negative status if they are rejected. fp32 calls also run, somewhat
 * slower, in a smaller one that holds their operand images (the status
 * GODA_ERR_WORKSPACE names that size): one workspace sized for a program's
 * largest batch serves its smaller ones. */
int64_t goda_attn_prefill_bwd_workspace_size(const goda_prefill_args* fwd);

/* Backward of goda_attn_prefill_fwd: dq, dk, dv from d_o and the forward's
 * saved o and lse (fwd->o and fwd->lse must hold the forward's outputs for
 * the same q, k, v and options; fwd->workspace is not used). With Hkv < Hq,
 * dk/dv of a KV head sum its query heads' contributions. With RoPE the
 * gradients are taken back through the rotation (dq, dk refer to the
 * unrotated inputs). Replaces FlashAttentionGQAKernel.backward
 * (kernels_/flash_attn_gqa/cuda.py:577-658: D = rowsum(dO * O), then
 * dK/dV and dQ from P = exp(scale * q k^T - M)). */
int32_t goda_attn_prefill_bwd(const goda_prefill_args* fwd, const goda_prefill_grads* grads, void* stream);

/* Workspace needed by goda_attn_decode for these arguments (bytes, >= 0). */
int64_t goda_attn_decode_workspace_size(const goda_decode_args* args);

/* One-token decode over a contiguous KV cache with per-sequence lengths:
 * the visible keys of all sequences and KV heads are cut into equal ranges
 * for a persistent grid (split-K), partial softmax results of a sequence that
 * spans several ranges are merged by log-sum-exp.
 * Replaces FlashAttention._attention_with_kvcache for q_len == 1
 * (mint/nn/flashattn.py:174-219); its argument set mirrors the
 * flash_attn_with_kvcache call at mint/nn/flashattn.py:191-200. */
int32_t goda_attn_decode(const goda_decode_args* args, void* stream);

/* goda_attn_decode that allocates nothing and takes no workspace
 * (args->workspace / workspace_bytes are ignored). No counterpart in the
 * reference: it is for callers that cannot allocate device memory (code under
 * HIP graph capture, tight serving loops, harnesses that forbid hipMalloc).
 * The split-K partials live in a fixed device-resident array of 36 MiB
 * (GODA_DECODE_NOALLOC_SCRATCH_BYTES) that each GPU holds until the process
 * ends; every decode with split_size 0 (the balanced default) fits, and a
 * call whose partials would not fit fails with GODA_ERR_WORKSPACE. All calls
 * on one GPU share that array: calls that overlap on one GPU (concurrent
 * streams or threads) race and must be serialised by the caller. Results
 * equal goda_attn_decode's for the same arguments. */
#define GODA_DECODE_NOALLOC_SCRATCH_BYTES (36ll << 20)
int32_t goda_attn_decode_noalloc(const goda_decode_args* args, void* stream);

/* Append seqlen_new rows of k/v to every sequence at its own position
 * cache_seqlens[b] (optionally rotating k), then advance cache_seqlens.
 * Replaces KVCache.update (mint/kvcache/base.py:35-50) without the
 * device-to-host read of mint/nn/flashattn.py:202. */
int32_t goda_attn_kv_append(const goda_kv_append_args* args, void* stream);

/* Bit-packs a boolean mask (one byte a key, any nonzero byte visible) of any
 * byte strides into the words of goda_prefill_args.mask_bits: bits receives
 * [batch][heads][rows][2 * ceil(keys / 64)] contiguous words; key j >= mask_keys
 * is hidden (mask_keys 0: every key, and mask may be NULL). stride_k 0 with
 * mask_keys = keys broadcasts one byte to every key. */
typedef struct goda_pack_mask_args {
  const void* mask;
  int64_t stride_b, stride_h, stride_q, stride_k; /* bytes */
  int32_t batch, heads, rows, keys, mask_keys;
  int32_t reserved0;
  void* bits;
} goda_pack_mask_args;
int64_t goda_attn_sizeof_pack_mask_args(void);
int32_t goda_attn_pack_mask(const goda_pack_mask_args* args, void* stream);

/* Document segments of goda's doc_ids [rows, cols] (row stride in elements,
 * 4- or 8-byte integers): cu receives the rows * cols + 1 or fewer cumulative
 * starts of the maximal runs of equal ids inside each row (a run never crosses a
 * row), then rows * cols; result (3 words, device) = {number of runs, longest
 * run, 1 if an id occupies more than one run of its row, 2 if that was not
 * determined (over 1024 runs of ids in no order), else 0}. Replaces the
 * doc_ids -> cu_seqlens conversion of mint/nn/flashattn.py:98-137. */
int64_t goda_attn_doc_segments_scratch_bytes(int32_t rows, int32_t cols);
int32_t goda_attn_doc_segments(const void* ids, int32_t id_bytes, int64_t stride_row, int32_t rows, int32_t cols,
                               int32_t* cu, int32_t* result, void* scratch, int64_t scratch_bytes, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* GODA_ATTN_H */
