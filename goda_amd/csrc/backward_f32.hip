// Backward of fp32 prefill attention on gfx950 matrix cores, head_dim 64, 128
// and 256 (quantities as in backward_mfma.hip). As in the fp32 forward, the
// operands are 1 KB chunks (f32_tile.h) that every wave streams from L2 into
// registers at its own pace; the only barriers are around the sums at the end.
//
//   1. pack_q_f32_kernel: per (32-row query tile, head, sequence) the chunks of
//      q * scale * log2(e), dO, dO^T and q^T in the order the dk/dv kernel
//      reads them, and the row statistics lse * log2(e) and delta;
//   2. pack_kv_bwd_f32_kernel: per (key tile, KV head, sequence) the row images
//      of k and v and the transposed image of k;
//   3. bwd_dkv_f32_kernel: a workgroup owns 32 keys of a KV head, their k and v
//      operands in LDS; its four waves take every fourth (query tile, head) that
//      sees them, each accumulating dK^T and dV^T in registers (D), and add up
//      at the end:
//        S [rows][keys]  = Q K^T            dP = dO V^T     A = image, B = LDS
//        dV^T [d][keys] += dO^T P           dK^T += Q^T dS  A = image, B = S, dP in place
//      Each dS tile also goes to memory (4 KB, as the next kernel's B operand);
//   4. bwd_dq_f32_kernel: a wave owns 32 query rows of a head (or shares them
//      with others of its workgroup, which take every split-th key tile):
//        dQ^T [d][rows] += K^T dS^T         A = k^T image, B = stored dS
//      3 and 4 run in turn for as many (sequence, KV head) pairs as the buffer of
//      dS tiles holds. Where those of one pair pass kDsMaxBytes, or the workspace
//      has no room for them, 4 forms S and dP again (RECOMPUTE: three products
//      per tile instead of one).
//
// Bound by the fp32 products (154 TFLOP/s reached by a large matrix product).
// Whole backward, us, before (LDS rings with one wave per SIMD at head_dim 64
// and 128, vector ALUs at 256) and now, causal, RoPE:
//   B=1 T=4096 32/8 D=128    4475 / 3524      B=16 T=512 4/4 D=128 window 128   281 / 135
//   B=2 T=4096 16/16 D=64    2640 / 1844      B=2 T=512 6/2 D=128               196 /  76
//   B=1 T=2048 16/1 D=256   29082 /  867      B=8 T=4096 16/1 D=256 ALiBi    140576 / 22704

#include <algorithm>

#include "common.h"
#include "f32_tile.h"
#include "launch.h"
#include "mfma_common.h"

namespace goda {
namespace {

constexpr int kWaves = 4;
constexpr int kRing = 8;  // chunks in flight, as in the forward
// dS tiles held at a time: all up to kDsMaxBytes, else as many (sequence, KV
// head) pairs as kDsChunkBytes hold, or one pair up to kDsMaxBytes. Whole
// backward, ms, with S and dP formed again / with the tiles of a part at a time:
//   B=8 T=4096 32/8 D=128 causal   32.6 / 25.3     B=1 T=16384 32/8 D=128   63.1 / 49.1
//   B=2 T=16384 8/8 D=64 causal    17.6 / 13.6     the same, window 128     1.82 / 1.46
//   packed 8192 + 16 x 200 rows, 16/4 D=128                                 15.8 / 7.9
// Every run ends with its longest workgroups: B=1 T=11264 32/8 D=128 23.4 at
// once, 24.1 in two runs, hence the larger limit for all. (Past both, the dq
// kernel that forms S and dP again is 3% slower than the LDS-ring kernels that
// it replaced at head_dim 128 and 9% at 64.)
constexpr int64_t kDsMaxBytes = 8ll << 30;
constexpr int64_t kDsChunkBytes = 4ll << 30;
constexpr int kDsTile = kF32Rows * kF32Rows * 4;
template <int D>
constexpr int kWavesPerSimd = D <= 128 ? 2 : 1;

// A query tile: 4 D/8 chunks (q, dO by turns, then dO^T, q^T by turns), then
// lse2[32] and delta[32].
template <int D>
struct QTile {
  static constexpr int STAT = 4 * kF32Img<D>;
  static constexpr int BYTES = STAT + 256;
};
// A key tile: k and v row images, k transposed.
template <int D>
struct KTile {
  static constexpr int V = kF32Img<D>, KT = 2 * kF32Img<D>, BYTES = 3 * kF32Img<D>;
};

template <int D>
__device__ __forceinline__ const unsigned char* q_tile(const BwdParams& p, int b, int qt, int hq) {
  return p.qimg + (((int64_t)b * p.ntq + qt) * p.a.heads_q + hq) * QTile<D>::BYTES;
}
template <int D>
__device__ __forceinline__ const unsigned char* k_tile(const BwdParams& p, int b, int kt, int hk) {
  return p.kvimg + (((int64_t)b * p.ntk + kt) * p.a.heads_kv + hk) * KTile<D>::BYTES;
}
// dS tile of query head h of a pair's group (pair: of this launch; diag = Lk -
// Lq of the sequence): for key group g and lane half l / 32, row l % 32's keys
// 8 g + 4 (l / 32) + e at (64 g + l) 16 + 4 e.
__device__ __forceinline__ unsigned char* ds_tile(const BwdParams& p, int pair, int diag, int qt, int kt, int h) {
  int64_t at;
  if (p.ds_band > 0)
    at = (int64_t)qt * p.ds_band + kt - max(0, diag + qt * kF32Rows - p.a.window_left) / kF32Rows;
  else
    at = ds_row_off(qt, p.ntk, p.ds_c, p.ds_tri != 0) + kt;
  return p.ds + ((pair * p.ds_per_pair + at) * p.group + h) * kDsTile;
}

__device__ __forceinline__ const float* row_of(const void* base, int64_t sb, int64_t st, int64_t sh, bool varlen, int b,
                                               int64_t row, int h) {
  return reinterpret_cast<const float*>(base) + (varlen ? 0 : (int64_t)b * sb) + row * st + (int64_t)h * sh;
}
__device__ __forceinline__ float* row_of(void* base, int64_t sb, int64_t st, int64_t sh, bool varlen, int b, int64_t row,
                                         int h) {
  return reinterpret_cast<float*>(base) + (varlen ? 0 : (int64_t)b * sb) + row * st + (int64_t)h * sh;
}

template <int D>
__global__ void __launch_bounds__(256) pack_q_f32_kernel(const BwdParams p) {
  const goda_prefill_args& a = p.a;
  const int qt = blockIdx.x, hq = blockIdx.y, b = blockIdx.z;
  const SeqGeom g = seq_geom(b, a.seqlen_q, a.seqlen_k, a.cu_seqlens_q, a.cu_seqlens_k, a.seqused_k);
  const int i0 = qt * kF32Rows;
  if (i0 >= g.lq) return;
  const bool varlen = a.cu_seqlens_q != nullptr;
  __shared__ __align__(16) float qrows[kF32Rows][D + 4], grows[kF32Rows][D + 4];
  __shared__ float delta[kF32Rows];
  const int tid = threadIdx.x;
  constexpr int TPR = D / 8;
  const int c = (tid % TPR) * 4;
  const RopePos rope = rope_qrows(a, g, i0);
#pragma unroll
  for (int r = tid / TPR; r < kF32Rows; r += 256 / TPR) {
    const int i = i0 + r;
    f32x4 q1 = {}, q2 = {}, g1 = {}, g2 = {}, o1 = {}, o2 = {};
    if (i < g.lq) {
      const float* qr = row_of(a.q, a.q_stride_b, a.q_stride_t, a.q_stride_h, varlen, b, g.q_row0 + i, hq) + c;
      const float* gr = row_of(p.g.d_o, p.g.do_stride_b, p.g.do_stride_t, p.g.do_stride_h, varlen, b, g.q_row0 + i, hq) + c;
      const float* orow = row_of((const void*)a.o, a.o_stride_b, a.o_stride_t, a.o_stride_h, varlen, b, g.q_row0 + i, hq) + c;
      q1 = ld_stream<f32x4>(qr);
      q2 = ld_stream<f32x4>(qr + D / 2);
      g1 = ld_stream<f32x4>(gr);
      g2 = ld_stream<f32x4>(gr + D / 2);
      o1 = ld_stream<f32x4>(orow);
      o2 = ld_stream<f32x4>(orow + D / 2);
    }
    norm_rope_f32<D>(q1, q2, c, a.q_norm_weight, a.norm_eps, i < g.lq && a.rope_q, rope.at(r),
                     a.rope_cos, a.rope_sin);
    st_vec<f32x4>(&qrows[r][c], q1);
    st_vec<f32x4>(&qrows[r][c + D / 2], q2);
    st_vec<f32x4>(&grows[r][c], g1);
    st_vec<f32x4>(&grows[r][c + D / 2], g2);
    const f32x4 og = o1 * g1 + o2 * g2;
    const float dl = lane_group_sum<TPR>((og[0] + og[1]) + (og[2] + og[3]));
    if (tid % TPR == 0) delta[r] = dl;
  }
  __syncthreads();
  unsigned char* img = const_cast<unsigned char*>(q_tile<D>(p, b, qt, hq));
  write_row_image<D, 2>(qrows, img, tid, p.scale_log2);
  write_row_image<D, 2>(grows, img + 1024, tid);
  write_tr_image<D, 2>(grows, img + 2 * kF32Img<D>, tid);
  write_tr_image<D, 2>(qrows, img + 2 * kF32Img<D> + 1024, tid);
  if (tid < kF32Rows) {
    const int i = i0 + tid;
    float l2 = kNegInf;
    if (i < g.lq) {
      const int64_t li = varlen ? (int64_t)hq * a.lse_stride_h + g.q_row0 + i
                                : (int64_t)b * a.lse_stride_b + (int64_t)hq * a.lse_stride_h + i;
      l2 = a.lse[li] * kLog2e;
    }
    float* st = reinterpret_cast<float*>(img + QTile<D>::STAT);
    st[tid] = l2;
    st[kF32Rows + tid] = delta[tid];
  }
}

template <int D>
__global__ void __launch_bounds__(256) pack_kv_bwd_f32_kernel(const BwdParams p) {
  const goda_prefill_args& a = p.a;
  const int kt = blockIdx.x, hk = blockIdx.y, b = blockIdx.z;
  const SeqGeom g = seq_geom(b, a.seqlen_q, a.seqlen_k, a.cu_seqlens_q, a.cu_seqlens_k, a.seqused_k);
  const int kv0 = kt * kF32Rows;
  if (kv0 >= g.lk) return;
  const bool varlen = a.cu_seqlens_k != nullptr;
  __shared__ __align__(16) float krows[kF32Rows][D + 4], vrows[kF32Rows][D + 4];
  const int tid = threadIdx.x;
  constexpr int TPR = D / 8;
  const int c = (tid % TPR) * 4;
  const RopePos rope = rope_krows(a, g, kv0);
#pragma unroll
  for (int r = tid / TPR; r < kF32Rows; r += 256 / TPR) {
    const int row = kv0 + r;
    f32x4 k1 = {}, k2 = {}, v1 = {}, v2 = {};
    if (row < g.lk) {
      const float* kr = row_of(a.k, a.k_stride_b, a.k_stride_t, a.k_stride_h, varlen, b, g.k_row0 + row, hk) + c;
      const float* vr = row_of(a.v, a.v_stride_b, a.v_stride_t, a.v_stride_h, varlen, b, g.k_row0 + row, hk) + c;
      k1 = ld_stream<f32x4>(kr);
      k2 = ld_stream<f32x4>(kr + D / 2);
      v1 = ld_stream<f32x4>(vr);
      v2 = ld_stream<f32x4>(vr + D / 2);
    }
    norm_rope_f32<D>(k1, k2, c, a.k_norm_weight, a.norm_eps, row < g.lk && a.rope_k, rope.at(r), a.rope_cos,
                     a.rope_sin);
    st_vec<f32x4>(&krows[r][c], k1);
    st_vec<f32x4>(&krows[r][c + D / 2], k2);
    st_vec<f32x4>(&vrows[r][c], v1);
    st_vec<f32x4>(&vrows[r][c + D / 2], v2);
  }
  __syncthreads();
  unsigned char* img = const_cast<unsigned char*>(k_tile<D>(p, b, kt, hk));
  write_row_image<D>(krows, img, tid);
  write_row_image<D>(vrows, img + KTile<D>::V, tid);
  write_tr_image<D>(krows, img + KTile<D>::KT, tid);
}

// The waves' [32 rows][D] sums of one gradient, and the pair (d, d + D/2) of a
// row's elements rotated back by the transpose of the half-split rotation.
template <int D>
struct SumSmem {
  float x[kWaves][kF32Rows][D + 4];
};
template <int D>
__device__ __forceinline__ void put_acc(float (*rows)[D + 4], const f32x16 (&x)[D / 32], int lane) {
#pragma unroll
  for (int md = 0; md < D / 32; ++md)
#pragma unroll
    for (int gq = 0; gq < 4; ++gq)
      st_vec<f32x4>(&rows[lane & 31][32 * md + 8 * gq + 4 * (lane >> 5)], acc_chunk(x[md], gq));
}
__device__ __forceinline__ void rotate_back(f32x4& x1, f32x4& x2, const float* cos_row, const float* sin_row) {
  const f32x4 cs = ld_vec<f32x4>(cos_row), sn = ld_vec<f32x4>(sin_row);
  const f32x4 y1 = x1 * cs + x2 * sn;
  x2 = x2 * cs - x1 * sn;
  x1 = y1;
}

// ---------------------------------------------------------------------------
// 3. dk, dv
// ---------------------------------------------------------------------------
template <int D, bool ALIBI, bool MASK>
__global__ void __launch_bounds__(kWaves * 64, kWavesPerSimd<D>) bwd_dkv_f32_kernel(const BwdParams p) {
  constexpr int KS = D / 8, MD = D / 32;
  static_assert(2 * KS % kRing == 0, "a ring slot is a compile-time constant of the chunk");
  extern __shared__ __align__(16) unsigned char smem[];
  const goda_prefill_args& a = p.a;
  // Workgroup order of backward_mfma.hip: units (sequence, KV head, share of the
  // walk) in chunks, the key tile most rows see first.
  int unit, kt;
  chunked_order((int)blockIdx.x, p.ntk, p.npairs * p.nsplit, unit, kt);
  const int pair = unit / p.nsplit, split = unit % p.nsplit;  // (pair: of this launch)
  const int b = (p.pair0 + pair) / a.heads_kv, hk = (p.pair0 + pair) % a.heads_kv;
  const SeqGeom g = seq_geom(b, a.seqlen_q, a.seqlen_k, a.cu_seqlens_q, a.cu_seqlens_k, a.seqused_k);
  const bool varlen = a.cu_seqlens_k != nullptr;
  const int kend = varlen ? g.lk : a.seqlen_k;  // rows this launch writes
  const int kv0 = kt * kF32Rows;
  if (kv0 >= kend) return;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, l32 = lane & 31, hi = lane >> 5;
  const unsigned lane16 = lane * 16;
  const int key = kv0 + l32;
  const int diag = g.lk - g.lq;
  const bool causal = a.causal != 0;
  const int window_left = a.window_left;
  const bool use_window = window_left >= 0 && (causal || g.lq == 1);

  // Query tiles that see a key of the workgroup, and this share of the walk:
  // step it is head it % group of tile qt_lo + nq - 1 - it / group (all the key
  // tiles of a head walk down from the last query tile together).
  const int kv_last = min(kv0 + kF32Rows, g.lk) - 1;
  int i_lo = 0, i_hi = g.lq;
  if (causal) i_lo = max(0, kv0 - diag);
  if (use_window) i_hi = min(g.lq, kv_last + window_left - diag + 1);
  if (kv0 >= g.lk) i_hi = i_lo;
  const int qt_lo = i_lo / kF32Rows;
  const int nq = i_hi > i_lo ? (i_hi - 1) / kF32Rows + 1 - qt_lo : 0;
  const int n = p.group * nq;
  const int it0 = (int)((int64_t)n * split / p.nsplit) + wave;
  const int it1 = (int)((int64_t)n * (split + 1) / p.nsplit);
  auto head_of = [&](int it) { return hk * p.group + it % p.group; };
  auto tile_of = [&](int it) { return qt_lo + nq - 1 - it / p.group; };

  f32x4 ring[kRing];
  const unsigned char* cur = p.qimg;
  if (it0 < it1) {
    cur = q_tile<D>(p, b, tile_of(it0), head_of(it0));
#pragma unroll
    for (int i = 0; i < kRing; ++i) ring[i] = img_chunk(cur, i, lane16);
  }
  if (n > 0) {
    // k and v row images into LDS
    const unsigned char* img = k_tile<D>(p, b, kt, hk);
#pragma unroll 4
    for (int i = tid; i < 2 * kF32Img<D> / 16; i += kWaves * 64)
      *reinterpret_cast<f32x4*>(smem + i * 16) = *reinterpret_cast<const f32x4*>(img + i * 16);
  }
  __syncthreads();
  const unsigned char* kl = smem;
  const unsigned char* vl = smem + kF32Img<D>;

  f32x16 dv[MD], dk[MD];
#pragma unroll
  for (int md = 0; md < MD; ++md) dv[md] = dk[md] = f32x16{};
  const bool key_ok = key < g.lk;
  const unsigned ds_lane = ((l32 >> 3) * 64 + ((l32 >> 2) & 1) * 32 + 4 * hi) * 16 + (l32 & 3) * 4;

  for (int it = it0; it < it1; it += kWaves) {
    const int hq = head_of(it), qt = tile_of(it);
    const int q0 = qt * kF32Rows;
    const unsigned char* next = it + kWaves < it1 ? q_tile<D>(p, b, tile_of(it + kWaves), head_of(it + kWaves)) : cur;
    auto refill = [&](int i) {
      ring[i % kRing] = i + kRing < 4 * KS ? img_chunk(cur, i + kRing, lane16) : img_chunk(next, i + kRing - 4 * KS, lane16);
    };
    const float* stat = reinterpret_cast<const float*>(cur + QTile<D>::STAT) + 4 * hi;
    f32x4 l2[4], dl[4];
#pragma unroll
    for (int gq = 0; gq < 4; ++gq) {
      l2[gq] = ld_vec<f32x4>(stat + 8 * gq);
      dl[gq] = ld_vec<f32x4>(stat + kF32Rows + 8 * gq);
    }
    uint32_t mword = ~0u;
    if (MASK && key_ok) mword = p.mask_t[b * p.mt_stride_b + hq * p.mt_stride_h + (int64_t)key * p.ntq + qt] >> (4 * hi);
    // S and dP, by turns; register r is row 8 (r/4) + r%4 past q0 + 4 hi
    f32x16 s = {}, dp = {};
    f32x4 kb = img_chunk(kl, 0, lane16), vb = img_chunk(vl, 0, lane16);
#pragma unroll
    for (int c = 0; c < KS; ++c) {
      const f32x4 k1 = kb, v1 = vb;
      if (c + 1 < KS) {
        kb = img_chunk(kl, c + 1, lane16);
        vb = img_chunk(vl, c + 1, lane16);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s = __builtin_amdgcn_mfma_f32_32x32x2f32(ring[(2 * c) % kRing][e], k1[e], s, 0, 0, 0);
        dp = __builtin_amdgcn_mfma_f32_32x32x2f32(ring[(2 * c + 1) % kRing][e], v1[e], dp, 0, 0, 0);
      }
      refill(2 * c);
      refill(2 * c + 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    // P and dS; hidden entries replaced (exp2 of a hidden score may overflow)
    const int rel = q0 + 4 * hi;
    int lo_lim = -1, hi_lim = g.lq - 1 - rel;
    if (causal) lo_lim = key - diag - rel;
    if (use_window) hi_lim = min(hi_lim, key + window_left - diag - rel);
    uint32_t vis = key_ok ? range_bits(lo_lim, hi_lim) : 0u;
    if (MASK) vis &= mword;
    const float slope2 = ALIBI ? a.alibi_slopes[hq] * kLog2e : 0.f;
    const float base = ALIBI ? slope2 * (float)(key - diag - rel) : 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      // (bias - lse2 first: both may be large where their sum is not)
      const float bias = ALIBI ? base - slope2 * (float)(8 * (r >> 2) + (r & 3)) : 0.f;
      s[r] = fast_exp2(s[r] + (bias - l2[r >> 2][r & 3]));
      dp[r] = s[r] * (dp[r] - dl[r >> 2][r & 3]);
    }
    if (__builtin_amdgcn_ballot_w64(vis != ~0u) != 0) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[r] = keep_if_bit(s[r], vis, 8 * (r >> 2) + (r & 3), 0.f);
        dp[r] = keep_if_bit(dp[r], vis, 8 * (r >> 2) + (r & 3), 0.f);
      }
    }
    if (p.ds) {
      unsigned char* dst = ds_tile(p, pair, diag, qt, kt, hq - hk * p.group) + ds_lane;
#pragma unroll
      for (int r = 0; r < 16; ++r) *reinterpret_cast<float*>(dst + (8 * (r >> 2) + (r & 3)) * 16) = dp[r];
    }
#pragma unroll
    for (int c = 0; c < KS; ++c) {
      const int i = 2 * KS + 2 * c;
      const f32x4 pb = acc_chunk(s, c / MD), db = acc_chunk(dp, c / MD);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        dv[c % MD] = __builtin_amdgcn_mfma_f32_32x32x2f32(ring[i % kRing][e], pb[e], dv[c % MD], 0, 0, 0);
        dk[c % MD] = __builtin_amdgcn_mfma_f32_32x32x2f32(ring[(i + 1) % kRing][e], db[e], dk[c % MD], 0, 0, 0);
      }
      refill(i);
      refill(i + 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    cur = next;
  }

  // ---- the workgroup's sums, whole rows out --------------------------------
  SumSmem<D>& sm = *reinterpret_cast<SumSmem<D>*>(smem);
  const int64_t prow = ((int64_t)b * a.seqlen_k + kv0);
  const int64_t rows = (int64_t)a.batch * a.seqlen_k;
  const RopePos rope = rope_krows(a, g, kv0);
  auto write = [&](bool is_k) {
    constexpr int PAIRS = D / 8;  // 16-byte pieces of half a row
    for (int i = tid; i < kF32Rows * PAIRS; i += kWaves * 64) {
      const int r = i / PAIRS, d0 = 4 * (i % PAIRS);
      const int kr = kv0 + r;
      if (kr >= kend) continue;
      f32x4 x1 = {}, x2 = {};
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        x1 += ld_vec<f32x4>(&sm.x[w][r][d0]);
        x2 += ld_vec<f32x4>(&sm.x[w][r][d0 + D / 2]);
      }
      if (p.nsplit > 1) {
        float* out = p.part + (((int64_t)(2 * split + (is_k ? 0 : 1)) * rows + prow + r) * a.heads_kv + hk) * D + d0;
        st_vec<f32x4>(out, x1);
        st_vec<f32x4>(out + D / 2, x2);
        continue;
      }
      float* out;
      if (is_k) {
        x1 *= a.softmax_scale;
        x2 *= a.softmax_scale;
        const int64_t at = (int64_t)rope.at(r) * (D / 2) + d0;
        if (a.rope_k && kr < g.lk) rotate_back(x1, x2, a.rope_cos + at, a.rope_sin + at);
        out = row_of(p.g.dk, p.g.dk_stride_b, p.g.dk_stride_t, p.g.dk_stride_h, varlen, b, g.k_row0 + kr, hk);
      } else {
        out = row_of(p.g.dv, p.g.dv_stride_b, p.g.dv_stride_t, p.g.dv_stride_h, varlen, b, g.k_row0 + kr, hk);
      }
      st_vec<f32x4>(out + d0, x1);
      st_vec<f32x4>(out + d0 + D / 2, x2);
    }
  };
  __syncthreads();  // every wave is past its last read of k and v
  put_acc<D>(sm.x[wave], dv, lane);
  __syncthreads();
  write(false);
  __syncthreads();
  put_acc<D>(sm.x[wave], dk, lane);
  __syncthreads();
  write(true);
}

// Sum of the nsplit partials of dk and dv; dk scaled and rotated back.
template <int D>
__global__ void __launch_bounds__(256) bwd_dkv_reduce_f32_kernel(const BwdParams p) {
  const goda_prefill_args& a = p.a;
  const int b = blockIdx.z, hk = blockIdx.y;
  const SeqGeom g = seq_geom(b, a.seqlen_q, a.seqlen_k, a.cu_seqlens_q, a.cu_seqlens_k, a.seqused_k);
  const bool varlen = a.cu_seqlens_k != nullptr;
  const int kend = varlen ? g.lk : a.seqlen_k;
  constexpr int PAIRS = D / 8;
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int key = (int)(idx / PAIRS), d0 = 4 * (int)(idx % PAIRS);
  if (key >= kend) return;
  const int64_t rows = (int64_t)a.batch * a.seqlen_k;
  const float* part = p.part + (((int64_t)b * a.seqlen_k + key) * a.heads_kv + hk) * D + d0;
  const int64_t step = rows * a.heads_kv * D;
  f32x4 k1 = {}, k2 = {}, v1 = {}, v2 = {};
#pragma unroll 2
  for (int s = 0; s < p.nsplit; ++s) {
    k1 += ld_vec<f32x4>(part + 2 * s * step);
    k2 += ld_vec<f32x4>(part + 2 * s * step + D / 2);
    v1 += ld_vec<f32x4>(part + (2 * s + 1) * step);
    v2 += ld_vec<f32x4>(part + (2 * s + 1) * step + D / 2);
  }
  k1 *= a.softmax_scale;
  k2 *= a.softmax_scale;
  const int key0 = (int)((int64_t)blockIdx.x * 256 / PAIRS);  // of the workgroup
  const int64_t at = (int64_t)rope_krows(a, g, key0).at(key - key0) * (D / 2) + d0;
  if (a.rope_k && key < g.lk) rotate_back(k1, k2, a.rope_cos + at, a.rope_sin + at);
  float* krow = row_of(p.g.dk, p.g.dk_stride_b, p.g.dk_stride_t, p.g.dk_stride_h, varlen, b, g.k_row0 + key, hk) + d0;
  float* vrow = row_of(p.g.dv, p.g.dv_stride_b, p.g.dv_stride_t, p.g.dv_stride_h, varlen, b, g.k_row0 + key, hk) + d0;
  st_vec<f32x4>(krow, k1);
  st_vec<f32x4>(krow + D / 2, k2);
  st_vec<f32x4>(vrow, v1);
  st_vec<f32x4>(vrow + D / 2, v2);
}

// ---------------------------------------------------------------------------
// 4. dq
// ---------------------------------------------------------------------------
template <int D, bool RECOMPUTE, bool ALIBI, bool MASK>
__global__ void __launch_bounds__(kWaves * 64, (RECOMPUTE && D == 128 ? 1 : kWavesPerSimd<D>)) bwd_dq_f32_kernel(const BwdParams p) {
  constexpr int KS = D / 8, MD = D / 32;
  // chunks of a key tile: (k, v by turns and) k^T
  constexpr int NC = RECOMPUTE ? 3 * KS : KS;
  constexpr int NT = RECOMPUTE ? 2 * KS : 0;  // first of k^T
  static_assert(NC % kRing == 0, "a ring slot is a compile-time constant of the chunk");
  extern __shared__ __align__(16) unsigned char smem[];
  const goda_prefill_args& a = p.a;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, l32 = lane & 31, hi = lane >> 5;
  const unsigned lane16 = lane * 16;
  // items as in the forward: heads innermost, the last query tile first
  const int split = p.key_split;  // waves sharing an item's key tiles
  const int per_wg = kWaves / split;
  const int nblk = (p.ntq * p.group + per_wg - 1) / per_wg;
  int pair, blk;  // (pair: of this launch)
  chunked_order((int)blockIdx.x, nblk, p.npairs, pair, blk);
  const int b = (p.pair0 + pair) / a.heads_kv, hk = (p.pair0 + pair) % a.heads_kv;
  const int item = blk * per_wg + wave / split;
  const int part = wave % split;
  const int qt = p.ntq - 1 - item / p.group;
  const int hq = hk * p.group + item % p.group;
  const SeqGeom g = seq_geom(b, a.seqlen_q, a.seqlen_k, a.cu_seqlens_q, a.cu_seqlens_k, a.seqused_k);
  const int qr0 = qt * kF32Rows;
  const bool live = qt >= 0 && qr0 < g.lq;  // an idle wave still takes the barriers below
  const bool varlen = a.cu_seqlens_q != nullptr;
  const int diag = g.lk - g.lq;
  const bool causal = a.causal != 0;
  const int window_left = a.window_left;
  const bool use_window = window_left >= 0 && (causal || g.lq == 1);
  const int i = qr0 + l32;
  const int iabs = diag + i;

  // key tiles some row sees (exactly the stored dS tiles of this query tile)
  const int q_last = min(qr0 + kF32Rows, g.lq) - 1;
  int kv_hi = g.lk;
  if (causal) kv_hi = min(kv_hi, diag + q_last + 1);
  const int kv_lo = use_window ? max(0, diag + qr0 - window_left) : 0;
  const int j_lo = kv_lo / kF32Rows;
  const int j_hi = kv_hi > 0 ? (kv_hi + kF32Rows - 1) / kF32Rows : 0;
  const int n = live ? max(0, j_hi - j_lo) : 0;

  auto chunk = [&](const unsigned char* tile, int c) {
    return c < NT ? img_chunk(tile + (c & 1) * KTile<D>::V, c >> 1, lane16) : img_chunk(tile + KTile<D>::KT, c - NT, lane16);
  };
  f32x4 ring[kRing];
  f32x4 dsb[4];
  const unsigned char* cur = p.kvimg;
  if (part < n) {
    cur = k_tile<D>(p, b, j_lo + part, hk);
#pragma unroll
    for (int c = 0; c < kRing; ++c) ring[c] = chunk(cur, c);
    if constexpr (!RECOMPUTE) {
      const unsigned char* t = ds_tile(p, pair, diag, qt, j_lo + part, item % p.group);
#pragma unroll
      for (int k = 0; k < 4; ++k) dsb[k] = img_chunk(t, k, lane16);
    }
  }
  f32x4 qf[RECOMPUTE ? KS : 1], gf[RECOMPUTE ? KS : 1];
  float l2 = kNegInf, dl = 0.f;
  if constexpr (RECOMPUTE) {
    if (n > 0) {
      const unsigned char* img = q_tile<D>(p, b, qt, hq);
#pragma unroll
      for (int c = 0; c < KS; ++c) {
        qf[c] = img_chunk(img, 2 * c, lane16);
        gf[c] = img_chunk(img, 2 * c + 1, lane16);
      }
      const float* stat = reinterpret_cast<const float*>(img + QTile<D>::STAT);
      l2 = stat[l32];
      dl = stat[kF32Rows + l32];
    }
#pragma unroll
    for (int c = 0; c < KS; ++c) {
      asm volatile("" : "+v"(qf[c]));
      asm volatile("" : "+v"(gf[c]));
    }
  }
  const float slope2 = ALIBI ? a.alibi_slopes[hq] * kLog2e : 0.f;
  const uint32_t* mrow = MASK ? mask_row(a, b, hq, max(0, min(i, g.lq - 1))) : nullptr;
  f32x16 dq[MD];
#pragma unroll
  for (int md = 0; md < MD; ++md) dq[md] = f32x16{};

  for (int t = part; t < n; t += split) {
    const int kt = j_lo + t;
    const bool more = t + split < n;
    const unsigned char* next = more ? k_tile<D>(p, b, kt + split, hk) : cur;
    auto refill = [&](int c) { ring[c % kRing] = c + kRing < NC ? chunk(cur, c + kRing) : chunk(next, c + kRing - NC); };
    f32x4 db[4];
    if constexpr (RECOMPUTE) {
      const uint32_t mword = MASK ? mrow[kt] >> (4 * hi) : ~0u;
      f32x16 s = {}, dp = {};
#pragma unroll
      for (int c = 0; c < KS; ++c) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s = __builtin_amdgcn_mfma_f32_32x32x2f32(ring[(2 * c) % kRing][e], qf[c][e], s, 0, 0, 0);
          dp = __builtin_amdgcn_mfma_f32_32x32x2f32(ring[(2 * c + 1) % kRing][e], gf[c][e], dp, 0, 0, 0);
        }
        refill(2 * c);
        refill(2 * c + 1);
        __builtin_amdgcn_sched_barrier(0);
      }
      // register r is key 8 (r/4) + r%4 past rel
      const int rel = kt * kF32Rows + 4 * hi;
      int hi_lim = g.lk - 1 - rel;
      if (causal) hi_lim = min(hi_lim, iabs - rel);
      const int lo_lim = use_window ? iabs - window_left - rel : 0;
      const uint32_t vis = (i < g.lq ? range_bits(lo_lim, hi_lim) : 0u) & mword;
      const float base = (ALIBI ? slope2 * (float)(rel - iabs) : 0.f) - l2;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float x = ALIBI ? base + slope2 * (float)(8 * (r >> 2) + (r & 3)) : base;  // bias - lse2
        dp[r] = keep_if_bit(fast_exp2(s[r] + x) * (dp[r] - dl), vis, 8 * (r >> 2) + (r & 3), 0.f);
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) db[k] = acc_chunk(dp, k);
    } else {
      const unsigned char* tn = ds_tile(p, pair, diag, qt, more ? kt + split : kt, item % p.group);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        db[k] = dsb[k];
        dsb[k] = img_chunk(tn, k, lane16);
      }
    }
#pragma unroll
    for (int c = 0; c < KS; ++c) {
      dq[c % MD] = mfma_chunk(ring[(NT + c) % kRing], db[c / MD], dq[c % MD]);
      refill(NT + c);
      __builtin_amdgcn_sched_barrier(0);
    }
    cur = next;
  }

  // ---- the item's sums, whole rows out ---------------------------------------
  SumSmem<D>& sm = *reinterpret_cast<SumSmem<D>*>(smem);
  put_acc<D>(sm.x[wave], dq, lane);
  __syncthreads();
  if (!live) return;
  constexpr int PAIRS = D / 8;
  constexpr int RPS = 64 / PAIRS;  // rows a wave writes at once
  const int rows = kF32Rows / split, w0 = wave - part;
  const int d0 = 4 * (lane % PAIRS);
  const RopePos rope = rope_qrows(a, g, qr0);
  for (int r = part * rows + lane / PAIRS; r < (part + 1) * rows; r += RPS) {
    if (qr0 + r >= g.lq) break;
    f32x4 x1 = {}, x2 = {};
    for (int w = 0; w < split; ++w) {
      x1 += ld_vec<f32x4>(&sm.x[w0 + w][r][d0]);
      x2 += ld_vec<f32x4>(&sm.x[w0 + w][r][d0 + D / 2]);
    }
    x1 *= a.softmax_scale;
    x2 *= a.softmax_scale;
    if (a.rope_q) {
      const int64_t at = (int64_t)rope.at(r) * (D / 2) + d0;
      rotate_back(x1, x2, a.rope_cos + at, a.rope_sin + at);
    }
    float* out = row_of(p.g.dq, p.g.dq_stride_b, p.g.dq_stride_t, p.g.dq_stride_h, varlen, b, g.q_row0 + qr0 + r, hq) + d0;
    st_vec<f32x4>(out, x1);
    st_vec<f32x4>(out + D / 2, x2);
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// Workgroups per key tile of the dk/dv kernel: enough that the grid over `pairs`
// (sequence, KV head) pairs holds ~1024, at most 8, and four steps of the walk
// (one per wave) each.
int dkv_splits(const goda_prefill_args& a, int64_t pairs) {
  const int64_t wgs = (int64_t)((a.seqlen_k + kF32Rows - 1) / kF32Rows) * pairs;
  if (wgs <= 0) return 1;
  const int64_t steps = (int64_t)(a.heads_q / a.heads_kv) * ((a.seqlen_q + kF32Rows - 1) / kF32Rows);
  const int64_t ns = std::min<int64_t>((1024 + wgs - 1) / wgs, steps / kWaves);
  return (int)std::max<int64_t>(1, std::min<int64_t>(ns, 8));
}

int64_t align256(int64_t x) { return (x + 255) / 256 * 256; }

// Workspace: query tiles, key tiles, dk/dv partials, key-major mask words, dS
// tiles of ds_pairs pairs (ds < 0: none).
struct Layout {
  int ntq, ntk, nsplit, ds_c, ds_tri, ds_band;
  int64_t kvimg, part, mask, ds, ds_per_pair, ds_pairs, total;
};
int64_t ds_pair_bytes(const goda_prefill_args& a, const Layout& l) {
  return l.ds_per_pair * (a.heads_q / a.heads_kv) * kDsTile;
}
// The layout with dS tiles of `pairs` pairs (0: none).
template <int D>
Layout layout_with(const goda_prefill_args& a, int nsplit, int64_t pairs) {
  Layout l{};
  l.ntq = (a.seqlen_q + kF32Rows - 1) / kF32Rows;
  l.ntk = (a.seqlen_k + kF32Rows - 1) / kF32Rows;
  l.nsplit = nsplit;
  l.kvimg = (int64_t)a.batch * l.ntq * a.heads_q * QTile<D>::BYTES;
  l.part = l.kvimg + (int64_t)a.batch * l.ntk * a.heads_kv * KTile<D>::BYTES;
  l.mask = l.part;
  if (l.nsplit > 1) l.mask += (int64_t)l.nsplit * 2 * a.batch * a.seqlen_k * a.heads_kv * D * 4;
  l.mask = align256(l.mask);
  l.total = l.mask + 4 * bwd_mask_t_words(a);
  // A causal batch keeps only the key tiles that a query tile can see: up to the
  // diagonal where every sequence's keys run the same way past its queries (equal
  // lengths, or the same packed rows: then past them only as far as the clamp to
  // the launch's sizes leaves), and those of the left window.
  l.ds_tri = a.causal && (!a.cu_seqlens_q || a.cu_seqlens_q == a.cu_seqlens_k);
  l.ds_c = l.ds_tri ? (std::max(0, a.seqlen_k - a.seqlen_q) + kF32Rows - 1) / kF32Rows : 0;
  l.ds_per_pair = ds_row_off(l.ntq, l.ntk, l.ds_c, l.ds_tri != 0);
  if (a.window_left >= 0 && (a.causal || a.seqlen_q == 1)) {
    // keys from W before a tile's first row to its last row: W + 32 positions
    const int64_t band = ((int64_t)a.window_left + 2 * (kF32Rows - 1)) / kF32Rows + 1;
    if (band < l.ntk && l.ntq * band < l.ds_per_pair) {
      l.ds_band = (int)band;
      l.ds_per_pair = l.ntq * band;
    }
  }
  l.ds_pairs = pairs;
  l.ds = -1;
  if (pairs > 0) {
    l.ds = align256(l.total);
    l.total = l.ds + pairs * ds_pair_bytes(a, l);
  }
  return l;
}
// The layout for a workspace of `room` bytes. Where it does not hold the dS tiles
// wanted, those of fewer pairs (a grid of 512 key tiles at least: fewer leave the
// GPU idle), then none, then no split walk of dk/dv. The last is the least that a
// launch runs with, and grows with every size.
template <int D>
Layout layout(const goda_prefill_args& a, int64_t room) {
  const int64_t pairs = (int64_t)a.batch * a.heads_kv;
  const int nsplit = dkv_splits(a, pairs);
  const Layout none = layout_with<D>(a, nsplit, 0);
  const int64_t bytes = ds_pair_bytes(a, none);
  int64_t n = pairs;
  if (bytes * pairs > kDsMaxBytes) n = bytes > kDsMaxBytes ? 0 : std::max<int64_t>(1, kDsChunkBytes / bytes);
  if (n > 0) {
    Layout l = layout_with<D>(a, dkv_splits(a, n), n);
    if (l.total <= room) return l;
    for (n = std::min(n, (room - none.total) / std::max<int64_t>(bytes, 1)); n > 0 && n * l.ntk >= 512; n = n * 7 / 8) {
      l = layout_with<D>(a, dkv_splits(a, n), n);
      if (l.total <= room) return l;
    }
  }
  return none.total <= room ? none : layout_with<D>(a, 1, 0);
}

template <int D, bool ALIBI, bool MASK>
hipError_t launch_main(BwdParams p, hipStream_t s) {
  const goda_prefill_args& a = p.a;
  hipError_t e;
  constexpr int lds = (int)std::max<size_t>(sizeof(SumSmem<D>), 2 * kF32Img<D>);
  if ((e = record_timing(p.g.timing_begin, s)) != hipSuccess) return e;
  auto dkv = bwd_dkv_f32_kernel<D, ALIBI, MASK>;
  auto dq = p.ds ? bwd_dq_f32_kernel<D, false, false, false> : bwd_dq_f32_kernel<D, true, ALIBI, MASK>;
  constexpr int sums = (int)sizeof(SumSmem<D>);
  if ((e = hipFuncSetAttribute((const void*)dkv, hipFuncAttributeMaxDynamicSharedMemorySize, lds)) != hipSuccess) return e;
  if ((e = hipFuncSetAttribute((const void*)dq, hipFuncAttributeMaxDynamicSharedMemorySize, sums)) != hipSuccess) return e;
  // Equal runs of pairs, no more than the dS tiles have room for, in whole
  // rounds over the XCDs (chunked_order) where that allows.
  const int pairs = a.batch * a.heads_kv;
  int most = p.npairs;
  if (most < pairs && most >= kOrderChunk) most = most / kOrderChunk * kOrderChunk;
  const int runs = (pairs + most - 1) / most;
  int run = (pairs + runs - 1) / runs;
  if (run < pairs && run >= kOrderChunk) run = (run + kOrderChunk - 1) / kOrderChunk * kOrderChunk;
  for (p.pair0 = 0; p.pair0 < pairs; p.pair0 += run) {
    p.npairs = std::min(run, pairs - p.pair0);
    if (p.ntk > 0) {
      const int64_t nblk = (int64_t)p.ntk * p.npairs * p.nsplit;
      if (nblk > 0x7fffffff) return hipErrorInvalidValue;
      dkv<<<dim3((unsigned)nblk), kWaves * 64, lds, s>>>(p);
      if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    if (p.ntq > 0) {
      p.key_split = f32_key_split(a, (int64_t)p.ntq * p.group * p.npairs);
      const int per_wg = kWaves / p.key_split;
      const int64_t nblk = ((int64_t)p.ntq * p.group + per_wg - 1) / per_wg * p.npairs;
      if (nblk > 0x7fffffff) return hipErrorInvalidValue;
      dq<<<dim3((unsigned)nblk), kWaves * 64, sums, s>>>(p);
      if ((e = hipGetLastError()) != hipSuccess) return e;
    }
  }
  if (p.ntk > 0 && p.nsplit > 1) {
    const int64_t threads = (int64_t)a.seqlen_k * (D / 8);
    bwd_dkv_reduce_f32_kernel<D><<<dim3((unsigned)((threads + 255) / 256), a.heads_kv, a.batch), 256, 0, s>>>(p);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  return record_timing(p.g.timing_end, s);
}

template <int D>
hipError_t launch_d(BwdParams p, int64_t room, hipStream_t s) {
  const goda_prefill_args& a = p.a;
  const Layout l = layout<D>(a, room);
  p.ntq = l.ntq;
  p.ntk = l.ntk;
  p.nsplit = l.nsplit;
  p.qimg = reinterpret_cast<unsigned char*>(p.g.workspace);
  p.kvimg = p.qimg + l.kvimg;
  p.part = reinterpret_cast<float*>(p.qimg + l.part);
  p.ds = l.ds >= 0 ? p.qimg + l.ds : nullptr;
  p.ds_per_pair = l.ds_per_pair;
  p.ds_c = l.ds_c;
  p.ds_tri = l.ds_tri;
  p.ds_band = l.ds_band;
  p.npairs = p.ds ? (int)l.ds_pairs : a.batch * a.heads_kv;
  hipError_t e;
  if (a.mask_bits) {
    p.mask_t = reinterpret_cast<uint32_t*>(p.qimg + l.mask);
    if ((e = launch_bwd_mask_t(p, s)) != hipSuccess) return e;
  }
  if (p.ntq > 0) {
    pack_q_f32_kernel<D><<<dim3(p.ntq, a.heads_q, a.batch), 256, 0, s>>>(p);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  if (p.ntk > 0) {
    pack_kv_bwd_f32_kernel<D><<<dim3(p.ntk, a.heads_kv, a.batch), 256, 0, s>>>(p);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  if (a.mask_bits) return a.alibi_slopes ? launch_main<D, true, true>(p, s) : launch_main<D, false, true>(p, s);
  return a.alibi_slopes ? launch_main<D, true, false>(p, s) : launch_main<D, false, false>(p, s);
}

}  // namespace

int64_t prefill_bwd_f32_workspace_bytes(const goda_prefill_args& a, int64_t room) {
  return a.head_dim == 64 ? layout<64>(a, room).total : a.head_dim == 128 ? layout<128>(a, room).total : layout<256>(a, room).total;
}

hipError_t launch_prefill_bwd_f32(const BwdParams& p, int64_t room, hipStream_t s) {
  switch (p.a.head_dim) {
    case 64:
      return launch_d<64>(p, room, s);
    case 128:
      return launch_d<128>(p, room, s);
    case 256:
      return launch_d<256>(p, room, s);
    default:
      return hipErrorNotSupported;
  }
}

}  // namespace goda
