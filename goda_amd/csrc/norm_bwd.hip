// Backward of the fused QK-RMSNorm (goda's RMSNorm, mint/nn/norm.py:17-27,
// applied to every q and k head row before RoPE, mint/nn/attn.py:57-60):
//   y = x r g,  r = rsqrt(mean(x^2) + eps),  g = 1 + w   (fp32),
//   dx = r (g dy - x^ mean(x^ g dy)),  x^ = x r,  dw = sum over rows of x^ dy.
// The attention backward leaves dy (the gradient of the normalized, unrotated
// rows, in the caller's dq / dk buffer and dtype, as the unfused path holds
// it); norm_bwd_kernel turns it into dx in place and writes one fp32 partial
// of dw per workgroup; norm_dw_reduce_kernel sums the partials of both sides
// in a fixed order (no atomics: the result does not depend on scheduling).
//
// Row layout: a group of D/8 lanes holds one row, 8 elements per lane
// (16-byte loads at 16-bit dtypes); a wave covers 512/D rows at a time and a
// workgroup of 4 waves kNormRows rows of one (sequence, head), all of whose
// loads are issued before the first row's reductions. The kernel is bound by
// HBM where the grid fills the GPU and by one round trip to it where it does
// not: 256 rows one after the other took 28.6 us for the k rows of B=2, T=4096,
// 8 heads, D=128 bf16 (256 workgroups, 50 MB) whatever their number.

#include "common.h"
#include "launch.h"
#include "mfma_common.h"

namespace goda {
namespace {

constexpr int kNormRows = 64;  // rows per workgroup

template <typename T, int D>
struct NormGeom {
  static constexpr int LPR = D / 8;        // lanes per row
  static constexpr int RPW = 64 / LPR;     // rows per wave step
  static constexpr int SLOTS = 4 * RPW;    // row groups of a workgroup
};

struct NormRows {
  const void* x;  // rows before the norm (the caller's q or k)
  int64_t x_sb, x_st, x_sh;
  void* y;        // dy in, dx out
  int64_t y_sb, y_st, y_sh;
  const float* w;
  float eps;
  float* part;    // fp32 [gridDim.z][gridDim.y][gridDim.x][D]
  int heads;
  bool q_side;    // rows of q (lengths lq) or of k (lengths lk)
};

__device__ __forceinline__ int norm_len(const goda_prefill_args& a, int b, bool q_side, int64_t* row0) {
  const SeqGeom g = seq_geom(b, a.seqlen_q, a.seqlen_k, a.cu_seqlens_q, a.cu_seqlens_k, a.seqused_k);
  *row0 = q_side ? g.q_row0 : g.k_row0;
  if (q_side) return g.lq;
  // padded batches: the rows past seqused_k are zero in dk and stay zero
  return g.lk;
}

template <typename T, int D>
__global__ void __launch_bounds__(256) norm_bwd_kernel(const goda_prefill_args a, const NormRows n) {
  typedef typename Vec<T>::v8 v8;
  typedef NormGeom<T, D> NG;
  const int b = blockIdx.z, h = blockIdx.y;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int sub = lane / NG::LPR, c = (lane % NG::LPR) * 8;
  int64_t row0;
  const int len = norm_len(a, b, n.q_side, &row0);
  const bool varlen = (n.q_side ? a.cu_seqlens_q : a.cu_seqlens_k) != nullptr;
  float g[8], acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    g[e] = 1.f + n.w[c + e];
    acc[e] = 0.f;
  }
  // Every lane of a row group takes part in its reductions (rows past the
  // sequence load zeros).
  constexpr int STEPS = kNormRows / NG::SLOTS;
  static_assert(kNormRows % NG::SLOTS == 0, "whole rounds of the row groups");
  const int first = blockIdx.x * kNormRows + wave * NG::RPW + sub;
  const T* xb = reinterpret_cast<const T*>(n.x) + (varlen ? 0 : (int64_t)b * n.x_sb) + (int64_t)h * n.x_sh + c;
  T* yb = reinterpret_cast<T*>(n.y) + (varlen ? 0 : (int64_t)b * n.y_sb) + (int64_t)h * n.y_sh + c;
  v8 xv[STEPS], dv[STEPS];
#pragma unroll
  for (int k = 0; k < STEPS; ++k) {
    const int r = first + k * NG::SLOTS;
    xv[k] = dv[k] = v8{};
    if (r < len) {
      xv[k] = ld_stream<v8>(xb + (row0 + r) * n.x_st);
      dv[k] = ld_stream<v8>(yb + (row0 + r) * n.y_st);
    }
  }
#pragma unroll
  for (int k = 0; k < STEPS; ++k) {
    const int r = first + k * NG::SLOTS;
    T* yp = yb + (row0 + r) * n.y_st;
    float x[8];
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      x[e] = (float)xv[k][e];
      ss = fmaf(x[e], x[e], ss);
    }
    const float rs = rms_scale(lane_group_sum<NG::LPR>(ss), D, n.eps);
    v8 out;
    float dy[8], t = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      dy[e] = (float)dv[k][e];
      x[e] *= rs;  // x^
      t = fmaf(x[e] * g[e], dy[e], t);
      acc[e] = fmaf(x[e], dy[e], acc[e]);
    }
    const float m = lane_group_sum<NG::LPR>(t) / (float)D;
#pragma unroll
    for (int e = 0; e < 8; ++e) out[e] = (T)(rs * (g[e] * dy[e] - x[e] * m));
    if (r < len) st_vec<v8>(yp, out);
  }
  // dw partial of this workgroup: row groups in slots, summed in slot order.
  __shared__ float sdw[NG::SLOTS][D];
#pragma unroll
  for (int e = 0; e < 8; ++e) sdw[wave * NG::RPW + sub][c + e] = acc[e];
  __syncthreads();
  for (int d = threadIdx.x; d < D; d += 256) {
    float s = 0.f;
#pragma unroll 4
    for (int k = 0; k < NG::SLOTS; ++k) s += sdw[k][d];
    const int64_t blk = ((int64_t)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
    n.part[blk * D + d] = s;
  }
}

// The partials of one norm weight: dw[d] = sum over k < n of part[k][d].
struct DwSum {
  const float* part;
  int64_t n;
  float* dw;  // nullptr: this side is not wanted
};

// A workgroup sums 16 columns of one side (blockIdx.y): 64 rows of 4 lanes
// take every 64th partial, four in flight, and meet in LDS in row order. One
// thread per column over all partials was a serial chain of loads in a single
// workgroup: 232 us for the 1024 partials of B=2, T=4096, 32 heads, D=128
// (a training pass at that size, 8 KV heads, bf16, with this reduction and 64
// rows per workgroup above: 1558 -> 1256 us).
constexpr int kDwCols = 16, kDwRows = 64;
__global__ void __launch_bounds__(256) norm_dw_reduce_kernel(const DwSum q, const DwSum k, int head_dim) {
  const DwSum u = blockIdx.y == 0 ? q : k;
  if (!u.dw) return;  // (the whole workgroup)
  const int row = threadIdx.x >> 2, c = 4 * (threadIdx.x & 3);
  const int d = blockIdx.x * kDwCols + c;
  f32x4 s = {};
#pragma unroll 4
  for (int64_t i = row; i < u.n; i += kDwRows) s += ld_vec<f32x4>(u.part + i * head_dim + d);
  __shared__ __align__(16) float sums[kDwRows][kDwCols];
  st_vec<f32x4>(&sums[row][c], s);
  __syncthreads();
  if (threadIdx.x < kDwCols) {
    float t = 0.f;
#pragma unroll 8
    for (int r = 0; r < kDwRows; ++r) t += sums[r][threadIdx.x];
    u.dw[blockIdx.x * kDwCols + threadIdx.x] = t;
  }
}

hipError_t launch_dw_reduce(const DwSum& q, const DwSum& k, int head_dim, hipStream_t s) {
  if (!q.dw && !k.dw) return hipSuccess;
  // head_dim is 64, 128 or 256: whole column blocks
  norm_dw_reduce_kernel<<<dim3(head_dim / kDwCols, 2), 256, 0, s>>>(q, k, head_dim);
  return hipGetLastError();
}

template <typename T, int D>
hipError_t launch_rows(const goda_prefill_args& a, const NormRows& n, int64_t seqlen, hipStream_t s) {
  const dim3 grid((unsigned)((seqlen + kNormRows - 1) / kNormRows), (unsigned)n.heads, (unsigned)a.batch);
  if (grid.x == 0 || grid.y == 0 || grid.z == 0) return hipSuccess;
  norm_bwd_kernel<T, D><<<grid, 256, 0, s>>>(a, n);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_rows_t(const goda_prefill_args& a, const NormRows& n, int64_t seqlen, hipStream_t s) {
  switch (a.head_dim) {
    case 64:
      return launch_rows<T, 64>(a, n, seqlen, s);
    case 128:
      return launch_rows<T, 128>(a, n, seqlen, s);
    case 256:
      return launch_rows<T, 256>(a, n, seqlen, s);
    default:
      return hipErrorNotSupported;
  }
}

hipError_t launch_rows_any(const goda_prefill_args& a, const NormRows& n, int64_t seqlen, hipStream_t s) {
  if (a.dtype == GODA_DTYPE_BF16) return launch_rows_t<bf16>(a, n, seqlen, s);
  if (a.dtype == GODA_DTYPE_F16) return launch_rows_t<f16>(a, n, seqlen, s);
  if (a.dtype == GODA_DTYPE_F32) return launch_rows_t<float>(a, n, seqlen, s);
  return hipErrorNotSupported;
}

int64_t parts(int64_t seqlen, int heads, int batch) {
  return (seqlen + kNormRows - 1) / kNormRows * heads * batch;
}

}  // namespace

int64_t norm_bwd_part_bytes(const goda_prefill_args& a) {
  int64_t n = 0;
  if (a.q_norm_weight) n += parts(a.seqlen_q, a.heads_q, a.batch);
  if (a.k_norm_weight) n += parts(a.seqlen_k, a.heads_kv, a.batch);
  return n * a.head_dim * (int64_t)sizeof(float);
}

hipError_t zero_norm_dw(const goda_prefill_args& a, const goda_prefill_grads& g, hipStream_t s) {
  // sums of nothing: 0
  const DwSum q{nullptr, 0, a.q_norm_weight ? g.dq_norm_weight : nullptr};
  const DwSum k{nullptr, 0, a.k_norm_weight ? g.dk_norm_weight : nullptr};
  return launch_dw_reduce(q, k, a.head_dim, s);
}

hipError_t launch_norm_bwd(const goda_prefill_args& a, const goda_prefill_grads& g, float* part, hipStream_t s) {
  hipError_t e;
  DwSum sum[2] = {};
  for (int side = 0; side < 2; ++side) {
    const bool q_side = side == 0;
    const float* w = q_side ? a.q_norm_weight : a.k_norm_weight;
    if (!w) continue;
    NormRows n{};
    const int heads = q_side ? a.heads_q : a.heads_kv;
    const int64_t seqlen = q_side ? a.seqlen_q : a.seqlen_k;
    n.x = q_side ? a.q : a.k;
    n.x_sb = q_side ? a.q_stride_b : a.k_stride_b;
    n.x_st = q_side ? a.q_stride_t : a.k_stride_t;
    n.x_sh = q_side ? a.q_stride_h : a.k_stride_h;
    n.y = q_side ? g.dq : g.dk;
    n.y_sb = q_side ? g.dq_stride_b : g.dk_stride_b;
    n.y_st = q_side ? g.dq_stride_t : g.dk_stride_t;
    n.y_sh = q_side ? g.dq_stride_h : g.dk_stride_h;
    n.w = w;
    n.eps = a.norm_eps;
    n.part = part;
    n.heads = heads;
    n.q_side = q_side;
    if ((e = launch_rows_any(a, n, seqlen, s)) != hipSuccess) return e;
    const int64_t np = parts(seqlen, heads, a.batch);
    sum[side] = DwSum{part, np, q_side ? g.dq_norm_weight : g.dk_norm_weight};
    part += np * a.head_dim;
  }
  return launch_dw_reduce(sum[0], sum[1], a.head_dim, s);
}

}  // namespace goda
