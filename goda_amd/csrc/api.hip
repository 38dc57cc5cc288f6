// C-ABI entry points of libgoda_attn.so: argument validation on the host,
// then dispatch to the kernels. Nothing here allocates or synchronises.

#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <string>

#include "goda_attn.h"
#include "launch.h"

namespace {

thread_local std::string g_last_error;

int32_t fail(int32_t code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
int32_t fail(int32_t code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_last_error = buf;
  return code;
}

int32_t ok() {
  g_last_error.clear();
  return GODA_OK;
}

int32_t hip_status(hipError_t e, const char* what) {
  if (e == hipSuccess) return ok();
  if (e == hipErrorNotSupported) return fail(GODA_ERR_UNSUPPORTED, "%s: no kernel instance for these arguments", what);
  return fail(GODA_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
}

bool dtype_ok(int32_t d) { return d == GODA_DTYPE_F32 || d == GODA_DTYPE_F16 || d == GODA_DTYPE_BF16; }

bool head_dim_ok(int32_t d) { return d == 64 || d == 128 || d == 256; }

// Checks shared by prefill; returns GODA_OK or a failure status. The
// workspace query passes need_ptrs = false: it depends on the sizes and options
// (of the pointers only on which are set and, in the backward, on whether both
// cu_seqlens are one array).
int32_t check_prefill(const goda_prefill_args* a, bool need_ptrs) {
  if (!a) return fail(GODA_ERR_INVALID_ARG, "prefill: args is NULL");
  if (!dtype_ok(a->dtype)) return fail(GODA_ERR_INVALID_ARG, "prefill: unknown dtype %d", a->dtype);
  if (a->batch < 0 || a->seqlen_q < 0 || a->seqlen_k < 0)
    return fail(GODA_ERR_INVALID_ARG, "prefill: negative size (batch %d, seqlen_q %d, seqlen_k %d)",
                a->batch, a->seqlen_q, a->seqlen_k);
  if (a->heads_q <= 0 || a->heads_kv <= 0)
    return fail(GODA_ERR_INVALID_ARG, "prefill: heads_q %d / heads_kv %d must be positive", a->heads_q,
                a->heads_kv);
  if (a->heads_q % a->heads_kv != 0)
    return fail(GODA_ERR_INVALID_ARG, "prefill: heads_q %d is not a multiple of heads_kv %d", a->heads_q,
                a->heads_kv);
  if (!head_dim_ok(a->head_dim))
    return fail(GODA_ERR_UNSUPPORTED,
                "prefill: head_dim %d not in {64, 128, 256} (goda_amd's Python layers zero-pad other head dims)",
                a->head_dim);
  if ((a->cu_seqlens_q == nullptr) != (a->cu_seqlens_k == nullptr))
    return fail(GODA_ERR_INVALID_ARG, "prefill: cu_seqlens_q and cu_seqlens_k must both be set or both NULL");
  if (!(a->softmax_scale > 0.f))
    return fail(GODA_ERR_INVALID_ARG, "prefill: softmax_scale must be positive (got %g)", (double)a->softmax_scale);
  if ((a->q_norm_weight || a->k_norm_weight) && !(a->norm_eps >= 0.f))
    return fail(GODA_ERR_INVALID_ARG, "prefill: norm_eps must be >= 0 (got %g)", (double)a->norm_eps);
  if (a->batch == 0 || a->seqlen_q == 0) return GODA_OK;
  if (need_ptrs && (!a->q || !a->k || !a->v || !a->o))
    return fail(GODA_ERR_INVALID_ARG, "prefill: NULL tensor pointer");
  if (a->rope_q || a->rope_k) {
    if (!a->rope_cos || !a->rope_sin || a->rope_len <= 0)
      return fail(GODA_ERR_INVALID_ARG, "prefill: RoPE requested without cos/sin tables");
    // Highest position touched: q rows sit at rope_q_offset + (Lk - Lq) + i <=
    // rope_q_offset + seqlen_k - 1 when Lq >= 1 (rope_pos_abs: at
    // rope_q_offset + i); k rows at rope_k_offset + j.
    const int64_t qmax = (int64_t)a->rope_q_offset + (a->rope_pos_abs ? a->seqlen_q : a->seqlen_k) - 1;
    const int64_t kmax = (int64_t)a->rope_k_offset + a->seqlen_k - 1;
    if (a->rope_packed_rows) {  // packed row index modulo rope_len: always inside the table
      if (!a->cu_seqlens_q)
        return fail(GODA_ERR_INVALID_ARG, "prefill: rope_packed_rows needs packed rows (cu_seqlens)");
      if (a->rope_len < 64)
        return fail(GODA_ERR_INVALID_ARG, "prefill: rope_packed_rows needs tables of at least 64 positions (got %d)", a->rope_len);
    } else if (a->rope_q && (a->rope_q_offset < 0 || qmax >= a->rope_len))
      return fail(GODA_ERR_INVALID_ARG, "prefill: q positions up to %lld exceed rope_len %d",
                  (long long)qmax, a->rope_len);
    if (!a->rope_packed_rows && a->rope_k && (a->rope_k_offset < 0 || kmax >= a->rope_len))
      return fail(GODA_ERR_INVALID_ARG, "prefill: k positions up to %lld exceed rope_len %d",
                  (long long)kmax, a->rope_len);
    if (a->rope_q && !a->rope_pos_abs && !a->cu_seqlens_q && a->seqlen_q > a->seqlen_k && !a->seqused_k)
      return fail(GODA_ERR_INVALID_ARG, "prefill: RoPE on q needs seqlen_q <= seqlen_k");
  }
  if (a->mask_bits) {
    if (a->cu_seqlens_q)
      return fail(GODA_ERR_UNSUPPORTED, "prefill: a mask needs a dense launch (cu_seqlens NULL)");
    if ((reinterpret_cast<uintptr_t>(a->mask_bits) & 7) != 0 || (a->mask_stride_b & 1) || (a->mask_stride_h & 1) ||
        (a->mask_stride_q & 1) || a->mask_stride_b < 0 || a->mask_stride_h < 0 || a->mask_stride_q < 0)
      return fail(GODA_ERR_INVALID_ARG,
                  "prefill: mask_bits must be 8-byte aligned with even, non-negative word strides");
  }
  return GODA_OK;
}

goda::PrefillParams make_prefill_params(const goda_prefill_args* a) {
  goda::PrefillParams p;
  memset(&p, 0, sizeof(p));
  p.a = *a;
  p.group = a->heads_q / a->heads_kv;
  p.scale_log2 = a->softmax_scale * 1.4426950408889634f;
  return p;
}

int64_t prefill_workspace_bytes(const goda_prefill_args& a) {
  if (goda::prefill_f32_streams(a)) return goda::prefill_f32_workspace_bytes(a);
  return goda::prefill_mfma_supported(a) ? goda::prefill_mfma_workspace_bytes(a) : 0;
}

// Checks of goda_attn_decode / goda_attn_decode_noalloc (everything but the
// workspace); returns GODA_OK or a failure status.
int32_t check_decode(const goda_decode_args* a) {
  if (!a) return fail(GODA_ERR_INVALID_ARG, "decode: args is NULL");
  if (!dtype_ok(a->dtype)) return fail(GODA_ERR_INVALID_ARG, "decode: unknown dtype %d", a->dtype);
  if (a->batch < 0 || a->max_seqlen < 0)
    return fail(GODA_ERR_INVALID_ARG, "decode: negative size (batch %d, max_seqlen %d)", a->batch,
                a->max_seqlen);
  if (a->heads_q <= 0 || a->heads_kv <= 0 || a->heads_q % a->heads_kv != 0)
    return fail(GODA_ERR_INVALID_ARG, "decode: heads_q %d must be a positive multiple of heads_kv %d",
                a->heads_q, a->heads_kv);
  if (!head_dim_ok(a->head_dim))
    return fail(GODA_ERR_UNSUPPORTED, "decode: head_dim %d not in {64, 128, 256}", a->head_dim);
  if (a->split_size < 0 || (a->split_size > 0 && a->split_size % 64 != 0))
    return fail(GODA_ERR_INVALID_ARG, "decode: split_size %d must be 0 or a positive multiple of 64",
                a->split_size);
  if (!(a->softmax_scale > 0.f))
    return fail(GODA_ERR_INVALID_ARG, "decode: softmax_scale must be positive (got %g)", (double)a->softmax_scale);
  if (a->q_norm_weight && !(a->norm_eps >= 0.f))
    return fail(GODA_ERR_INVALID_ARG, "decode: norm_eps must be >= 0 (got %g)", (double)a->norm_eps);
  if (a->batch == 0) return GODA_OK;
  if (!a->q || !a->k_cache || !a->v_cache || !a->o || !a->cache_seqlens)
    return fail(GODA_ERR_INVALID_ARG, "decode: NULL tensor pointer");
  if (a->rope_q) {
    if (!a->rope_cos || !a->rope_sin || a->rope_len <= 0)
      return fail(GODA_ERR_INVALID_ARG, "decode: RoPE requested without cos/sin tables");
    const int64_t qmax = (int64_t)a->rope_q_offset + (a->rope_pos_abs ? 0 : a->max_seqlen - 1);
    if (a->rope_q_offset < 0 || qmax >= a->rope_len)
      return fail(GODA_ERR_INVALID_ARG, "decode: q positions up to %lld exceed rope_len %d", (long long)qmax,
                  a->rope_len);
  }
  return GODA_OK;
}

goda::DecodeParams make_decode_params(const goda_decode_args& a) {
  goda::DecodeParams p;
  memset(&p, 0, sizeof(p));
  p.a = a;
  p.group = a.heads_q / a.heads_kv;
  p.scale_log2 = a.softmax_scale * 1.4426950408889634f;
  p.split = a.split_size;
  p.nslots = goda::decode_slots(a);
  return p;
}

}  // namespace

extern "C" {

int32_t goda_attn_abi_version(void) { return GODA_ATTN_ABI_VERSION; }
int64_t goda_attn_sizeof_prefill_args(void) { return sizeof(goda_prefill_args); }
int64_t goda_attn_sizeof_decode_args(void) { return sizeof(goda_decode_args); }
int64_t goda_attn_sizeof_kv_append_args(void) { return sizeof(goda_kv_append_args); }
int64_t goda_attn_sizeof_prefill_grads(void) { return sizeof(goda_prefill_grads); }

const char* goda_attn_last_error(void) { return g_last_error.c_str(); }

int64_t goda_attn_prefill_workspace_size(const goda_prefill_args* a) {
  const int32_t st = check_prefill(a, false);
  if (st != GODA_OK) return st;
  return prefill_workspace_bytes(*a);
}

int32_t goda_attn_prefill_fwd(const goda_prefill_args* a, void* stream) {
  const int32_t st = check_prefill(a, true);
  if (st != GODA_OK) return st;
  if (a->batch == 0 || a->seqlen_q == 0) return ok();
  goda::PrefillParams p = make_prefill_params(a);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const bool streams = goda::prefill_f32_streams(*a), mfma = goda::prefill_mfma_supported(*a);
  const int64_t need = mfma && !streams ? goda::prefill_mfma_least_bytes(*a) : prefill_workspace_bytes(*a);
  if (need > 0 && (!a->workspace || a->workspace_bytes < need)) {
    // (fp32 at head_dim 256 also runs without a workspace, on the vector ALUs)
    if (!mfma) return hip_status(goda::launch_prefill_generic(p, s), "prefill_fwd");
    return fail(GODA_ERR_WORKSPACE, "prefill: workspace of %lld bytes needed, %lld given",
                (long long)need, (long long)a->workspace_bytes);
  }
  if (streams) return hip_status(goda::launch_prefill_f32(p, s), "prefill_fwd");
  if (mfma) return hip_status(goda::launch_prefill_mfma(p, s), "prefill_fwd");
  return hip_status(goda::launch_prefill_generic(p, s), "prefill_fwd");
}

int64_t goda_attn_prefill_bwd_workspace_size(const goda_prefill_args* a) {
  const int32_t st = check_prefill(a, false);
  if (st != GODA_OK) return st;
  return goda::prefill_bwd_workspace_bytes(*a);
}

int32_t goda_attn_prefill_bwd(const goda_prefill_args* a, const goda_prefill_grads* g, void* stream) {
  const int32_t st = check_prefill(a, false);
  if (st != GODA_OK) return st;
  if (!g) return fail(GODA_ERR_INVALID_ARG, "prefill_bwd: grads is NULL");
  if (a->batch == 0 || (a->seqlen_q == 0 && a->seqlen_k == 0))  // nothing to differentiate: dL/dw = 0
    return hip_status(goda::zero_norm_dw(*a, *g, reinterpret_cast<hipStream_t>(stream)), "prefill_bwd");
  if (!a->q || !a->k || !a->v || !a->o || !g->d_o || !g->dq || !g->dk || !g->dv)
    return fail(GODA_ERR_INVALID_ARG, "prefill_bwd: NULL tensor pointer");
  if (!a->lse) return fail(GODA_ERR_INVALID_ARG, "prefill_bwd: the forward's lse is required");
  const int64_t need = goda::prefill_bwd_least_bytes(*a);
  if (need > 0 && (!g->workspace || g->workspace_bytes < need))
    return fail(GODA_ERR_WORKSPACE, "prefill_bwd: workspace of %lld bytes needed, %lld given", (long long)need,
                (long long)g->workspace_bytes);
  goda::BwdParams p;
  memset(&p, 0, sizeof(p));
  p.a = *a;
  p.g = *g;
  p.group = a->heads_q / a->heads_kv;
  p.scale_log2 = a->softmax_scale * 1.4426950408889634f;
  return hip_status(goda::launch_prefill_bwd(p, reinterpret_cast<hipStream_t>(stream)), "prefill_bwd");
}

int64_t goda_attn_decode_workspace_size(const goda_decode_args* a) {
  if (!a) return fail(GODA_ERR_INVALID_ARG, "decode: args is NULL");
  if (a->heads_q <= 0 || a->heads_kv <= 0 || a->heads_q % a->heads_kv != 0)
    return fail(GODA_ERR_INVALID_ARG, "decode: heads_q %d must be a positive multiple of heads_kv %d",
                a->heads_q, a->heads_kv);
  if (!head_dim_ok(a->head_dim))
    return fail(GODA_ERR_UNSUPPORTED, "decode: head_dim %d not in {64, 128, 256}", a->head_dim);
  return goda::decode_workspace_bytes(*a);
}

int32_t goda_attn_decode(const goda_decode_args* a, void* stream) {
  const int32_t st = check_decode(a);
  if (st != GODA_OK) return st;
  if (a->batch == 0) return ok();
  const int64_t need = goda::decode_workspace_bytes(*a);
  if (need > 0 && (!a->workspace || a->workspace_bytes < need))
    return fail(GODA_ERR_WORKSPACE, "decode: workspace of %lld bytes needed, %lld given", (long long)need,
                (long long)a->workspace_bytes);
  return hip_status(goda::launch_decode(make_decode_params(*a), reinterpret_cast<hipStream_t>(stream)), "decode");
}

int32_t goda_attn_decode_noalloc(const goda_decode_args* a, void* stream) {
  const int32_t st = check_decode(a);
  if (st != GODA_OK) return st;
  if (a->batch == 0) return ok();
  const int64_t need = goda::decode_workspace_bytes(*a);
  if (need > goda::kDecodeScratchBytes)
    return fail(GODA_ERR_WORKSPACE,
                "decode_noalloc: the split-K partials need %lld bytes, more than the %lld-byte scratch array "
                "(use split_size 0 or a larger split, or goda_attn_decode with a workspace)",
                (long long)need, (long long)goda::kDecodeScratchBytes);
  goda_decode_args b = *a;
  void* ptr = nullptr;
  hipError_t e = goda::decode_scratch(&ptr);
  if (e != hipSuccess) return hip_status(e, "decode_noalloc: scratch lookup");
  b.workspace = ptr;
  b.workspace_bytes = goda::kDecodeScratchBytes;
  return hip_status(goda::launch_decode(make_decode_params(b), reinterpret_cast<hipStream_t>(stream)),
                    "decode_noalloc");
}

int32_t goda_attn_kv_append(const goda_kv_append_args* a, void* stream) {
  if (!a) return fail(GODA_ERR_INVALID_ARG, "kv_append: args is NULL");
  if (!dtype_ok(a->dtype)) return fail(GODA_ERR_INVALID_ARG, "kv_append: unknown dtype %d", a->dtype);
  if (a->batch < 0 || a->seqlen_new < 0 || a->heads_kv <= 0 || a->head_dim <= 0 || a->head_dim % 2 != 0)
    return fail(GODA_ERR_INVALID_ARG, "kv_append: bad sizes (batch %d, seqlen_new %d, heads_kv %d, head_dim %d)",
                a->batch, a->seqlen_new, a->heads_kv, a->head_dim);
  if (!head_dim_ok(a->head_dim))
    return fail(GODA_ERR_UNSUPPORTED, "kv_append: head_dim %d not in {64, 128, 256}", a->head_dim);
  if (a->k_norm_weight && !(a->norm_eps >= 0.f))
    return fail(GODA_ERR_INVALID_ARG, "kv_append: norm_eps must be >= 0 (got %g)", (double)a->norm_eps);
  if (a->batch == 0) return ok();
  if (!a->k_new || !a->v_new || !a->k_cache || !a->v_cache || !a->cache_seqlens)
    return fail(GODA_ERR_INVALID_ARG, "kv_append: NULL tensor pointer");
  if (a->rope_k) {
    if (!a->rope_cos || !a->rope_sin || a->rope_len <= 0)
      return fail(GODA_ERR_INVALID_ARG, "kv_append: RoPE requested without cos/sin tables");
    const int64_t kmax = (int64_t)a->rope_k_offset + (a->rope_pos_abs ? a->seqlen_new : a->max_seqlen) - 1;
    if (a->rope_k_offset < 0 || kmax >= a->rope_len)
      return fail(GODA_ERR_INVALID_ARG, "kv_append: positions up to %lld exceed rope_len %d", (long long)kmax,
                  a->rope_len);
  }
  return hip_status(goda::launch_kv_append(*a, reinterpret_cast<hipStream_t>(stream)), "kv_append");
}

int64_t goda_attn_sizeof_pack_mask_args(void) { return sizeof(goda_pack_mask_args); }

int32_t goda_attn_pack_mask(const goda_pack_mask_args* a, void* stream) {
  if (!a) return fail(GODA_ERR_INVALID_ARG, "pack_mask: args is NULL");
  if (a->batch < 0 || a->heads < 0 || a->rows < 0 || a->keys < 0 || a->mask_keys < 0 || a->mask_keys > a->keys)
    return fail(GODA_ERR_INVALID_ARG, "pack_mask: bad sizes (batch %d, heads %d, rows %d, keys %d, mask_keys %d)", a->batch,
                a->heads, a->rows, a->keys, a->mask_keys);
  if ((int64_t)a->batch * a->heads * a->rows * a->keys == 0) return ok();
  // (a mask of no keys is not read: it hides every key)
  if ((!a->mask && a->mask_keys > 0) || !a->bits || (reinterpret_cast<uintptr_t>(a->bits) & 7) != 0)
    return fail(GODA_ERR_INVALID_ARG, "pack_mask: mask is NULL or bits not an 8-byte aligned pointer");
  return hip_status(goda::launch_pack_mask(*a, reinterpret_cast<hipStream_t>(stream)), "pack_mask");
}

int64_t goda_attn_doc_segments_scratch_bytes(int32_t rows, int32_t cols) {
  if (rows < 0 || cols < 0) return fail(GODA_ERR_INVALID_ARG, "doc_segments: negative size");
  return ((int64_t)rows * cols + 3 * (int64_t)rows) * 4;
}

int32_t goda_attn_doc_segments(const void* ids, int32_t id_bytes, int64_t stride_row, int32_t rows, int32_t cols,
                               int32_t* cu, int32_t* result, void* scratch, int64_t scratch_bytes, void* stream) {
  if (rows <= 0 || cols <= 0 || (int64_t)rows * cols > 0x7fffffff)
    return fail(GODA_ERR_INVALID_ARG, "doc_segments: bad sizes (rows %d, cols %d)", rows, cols);
  if (id_bytes != 4 && id_bytes != 8) return fail(GODA_ERR_INVALID_ARG, "doc_segments: ids of %d bytes", id_bytes);
  if (!ids || !cu || !result || !scratch) return fail(GODA_ERR_INVALID_ARG, "doc_segments: NULL pointer");
  if (scratch_bytes < goda_attn_doc_segments_scratch_bytes(rows, cols))
    return fail(GODA_ERR_WORKSPACE, "doc_segments: scratch of %lld bytes needed, %lld given",
                (long long)goda_attn_doc_segments_scratch_bytes(rows, cols), (long long)scratch_bytes);
  return hip_status(goda::launch_doc_segments(ids, id_bytes, stride_row, rows, cols, reinterpret_cast<int32_t*>(scratch), cu,
                                              result, reinterpret_cast<hipStream_t>(stream)),
                    "doc_segments");
}

}  // extern "C"
