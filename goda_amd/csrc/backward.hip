// Backward of prefill attention: dq, dk, dv from dO and the forward's saved o
// and log-sum-exp (kernels_/flash_attn_gqa/cuda.py:577-658 computes the same
// quantities: D = rowsum(dO * O), P = exp(scale * q k^T - M),
// dV = P^T dO, dS = P * (dO V^T - D), dQ = scale * dS K, dK = scale * dS^T Q).
// This file chooses between the 16-bit kernels (backward_mfma.hip) and the fp32
// ones (backward_f32.hip) and adds the fused QK-RMSNorm's backward, which
// turns their dq / dk (gradients of the normalized rows) into dx and dw.

#include <cstdint>

#include "common.h"
#include "launch.h"

namespace goda {
namespace {

int64_t align_up(int64_t x) { return (x + 255) / 256 * 256; }

bool normed(const goda_prefill_args& a) { return a.q_norm_weight || a.k_norm_weight; }

// The gradient kernels' own region, rounded up, then with the fused norm its
// dw partials. In a workspace of `bytes`, the region's share of it:
int64_t kernel_room(const goda_prefill_args& a, int64_t bytes) {
  return normed(a) ? (bytes - norm_bwd_part_bytes(a)) / 256 * 256 : bytes;
}
int64_t kernel_bytes(const goda_prefill_args& a, int64_t room) {
  return a.dtype == GODA_DTYPE_F32 ? prefill_bwd_f32_workspace_bytes(a, room) : prefill_bwd_mfma_workspace_bytes(a);
}
int64_t all_bytes(const goda_prefill_args& a, int64_t room) {
  const int64_t bytes = kernel_bytes(a, room);
  return normed(a) ? align_up(bytes) + norm_bwd_part_bytes(a) : bytes;
}

}  // namespace

int64_t prefill_bwd_workspace_bytes(const goda_prefill_args& a) { return all_bytes(a, INT64_MAX); }
int64_t prefill_bwd_least_bytes(const goda_prefill_args& a) { return all_bytes(a, 0); }

hipError_t launch_prefill_bwd(const BwdParams& p, hipStream_t s) {
  const goda_prefill_args& a = p.a;
  const int64_t room = kernel_room(a, p.g.workspace_bytes);
  const hipError_t e = a.dtype == GODA_DTYPE_F32 ? launch_prefill_bwd_f32(p, room, s) : launch_prefill_bwd_mfma(p, s);
  if (e != hipSuccess || !normed(a)) return e;
  unsigned char* part = reinterpret_cast<unsigned char*>(p.g.workspace) + align_up(kernel_bytes(a, room));
  return launch_norm_bwd(a, p.g, reinterpret_cast<float*>(part), s);
}

}  // namespace goda
