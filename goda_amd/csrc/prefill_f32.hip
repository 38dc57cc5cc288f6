// fp32 prefill attention on gfx950 matrix cores, head_dim 64, 128 and 256.
//
// An fp32 product needs one 256-byte operand per 64 clocks and wave, 4 bytes a
// clock, which L1 and L2 supply directly. So unlike the 16-bit kernel there is
// no LDS ring and no barrier in the key loop: every wave streams the key
// tiles' operand chunks (the workspace images of f32_tile.h, written by
// pack_kv_f32_kernel) into registers, kRing chunks ahead of their use, at its
// own pace.
//
// A wave owns 32 query rows of one head, Q^T and O^T in registers (D/2 each):
// two waves per SIMD up to head_dim 128, one at 256. Per 32-key tile, with the
// softmax of the 16-bit kernel (exponents out of the products, lazy rescale):
//   S^T[kv][q] = K[kv][d] . Q^T[d][q] - m[q] + bias     A = k image, B = q
//   O^T[d][q] += V^T[d][kv] . P^T[kv][q]                A = v^T image, B = S^T in place
//
// An item (32 query rows of one head) is walked by key_split waves of a
// workgroup of four, wave w taking every key_split-th key tile; they add up in
// LDS at the end (f32_key_split, launch.h, chooses).

#include "common.h"
#include "f32_tile.h"
#include "launch.h"
#include "mfma_common.h"

namespace goda {
namespace {

constexpr int kWaves = 4;
// Chunks in flight (4 registers and 256 clocks of products each, times the
// waves of a SIMD): 2048 clocks and more cover a load that misses L2.
constexpr int kRing = 8;
// Rescale margin in log2 units: at head_dim 64 and 128 that of the LDS-ring
// kernel, which larger calls run on (fp32 accumulators hold rows of 2^20 keys at
// 2^60). At 256 the vector-ALU kernel runs beside this one, whose probabilities
// are at most 1, so that values up to the type's largest over the number of keys
// stay finite: here they are at most 2^8 and the v image holds v * 2^-8, which
// the division by the row sum takes back. (A margin of 0 rescaled at most tiles:
// 315 -> 333 us at B=1, T=2048, 16/1 heads, causal.)
template <int D>
constexpr float kRescaleThresh = D == 256 ? 8.f : 60.f;
template <int D>
constexpr float kValueScale = D == 256 ? 1.f / 256.f : 1.f;

template <int D>
constexpr int kWavesPerSimd = D <= 128 ? 2 : 1;

template <int D>
constexpr int kTileBytes = 2 * kF32Img<D>;  // k row image, then v transposed

__device__ __forceinline__ int64_t kv_tile(int b, int j, int hk, int ntiles, int hkv) {
  return ((int64_t)b * ntiles + j) * hkv + hk;
}

// Per (key tile, KV head, sequence): the row image of k (normalized, rotated)
// and the transposed image of v (times kValueScale), rows past the sequence zero.
template <int D>
__global__ void __launch_bounds__(256) pack_kv_f32_kernel(const PrefillParams p) {
  const goda_prefill_args& a = p.a;
  const int j = blockIdx.x, hk = blockIdx.y, b = blockIdx.z;
  const SeqGeom g = seq_geom(b, a.seqlen_q, a.seqlen_k, a.cu_seqlens_q, a.cu_seqlens_k, a.seqused_k);
  const int kv0 = j * kF32Rows;
  if (kv0 >= g.lk) return;
  const float* kbase = reinterpret_cast<const float*>(a.k) + (a.cu_seqlens_k ? 0 : (int64_t)b * a.k_stride_b) +
                       (int64_t)hk * a.k_stride_h;
  const float* vbase = reinterpret_cast<const float*>(a.v) + (a.cu_seqlens_k ? 0 : (int64_t)b * a.v_stride_b) +
                       (int64_t)hk * a.v_stride_h;
  __shared__ __align__(16) float krows[kF32Rows][D + 4], vrows[kF32Rows][D + 4];
  const int tid = threadIdx.x;
  constexpr int TPR = D / 8;  // threads per row: consecutive lanes
  const int c = (tid % TPR) * 4;
  const RopePos rope = rope_krows(a, g, kv0);
#pragma unroll
  for (int r = tid / TPR; r < kF32Rows; r += 256 / TPR) {
    const int row = kv0 + r;
    f32x4 k1 = {}, k2 = {}, v1 = {}, v2 = {};
    if (row < g.lk) {
      const float* kr = kbase + (g.k_row0 + row) * a.k_stride_t + c;
      const float* vr = vbase + (g.k_row0 + row) * a.v_stride_t + c;
      k1 = ld_stream<f32x4>(kr);
      k2 = ld_stream<f32x4>(kr + D / 2);
      v1 = ld_stream<f32x4>(vr);
      v2 = ld_stream<f32x4>(vr + D / 2);
    }
    norm_rope_f32<D>(k1, k2, c, a.k_norm_weight, a.norm_eps, row < g.lk && a.rope_k, rope.at(r), a.rope_cos,
                     a.rope_sin);
    st_vec<f32x4>(&krows[r][c], k1);
    st_vec<f32x4>(&krows[r][c + D / 2], k2);
    st_vec<f32x4>(&vrows[r][c], v1 * kValueScale<D>);
    st_vec<f32x4>(&vrows[r][c + D / 2], v2 * kValueScale<D>);
  }
  __syncthreads();
  unsigned char* tile = reinterpret_cast<unsigned char*>(a.workspace) +
                        kv_tile(b, j, hk, p.ntiles_k, a.heads_kv) * kTileBytes<D>;
  write_row_image<D>(krows, tile, tid);
  write_tr_image<D>(vrows, tile + kF32Img<D>, tid);
}

// Max / sum over the two lanes l, l ^ 32 of a query row.
__device__ __forceinline__ float half_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <int D>
struct MergeSmem {
  float o[kWaves][kF32Rows][D + 4];
  float m[kWaves][kF32Rows];
  float l[kWaves][kF32Rows];
};

template <int D, bool ALIBI, bool MASK>
__global__ void __launch_bounds__(kWaves * 64, kWavesPerSimd<D>) prefill_f32_kernel(const PrefillParams p) {
  constexpr int KS = D / 8;    // chunks of a k image
  constexpr int MD = D / 32;   // 32-wide head-dim blocks of O^T
  constexpr int NC = 2 * KS;   // chunks of a tile: KS of k, then KS of v^T
  static_assert(KS % kRing == 0, "a ring slot is a compile-time constant of the chunk");
  extern __shared__ __align__(16) unsigned char smem[];

  const goda_prefill_args& a = p.a;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, l32 = lane & 31, hi = lane >> 5;
  const int split = p.key_split;
  // Items of a (sequence, KV head) pair, heads innermost (the waves of a
  // workgroup read the same key tiles), the last query tile first.
  const int per_wg = kWaves / split;
  const int nqt = p.qtiles;
  const int nblk = (nqt * p.group + per_wg - 1) / per_wg;
  int pair, blk;
  chunked_order((int)blockIdx.x, nblk, a.batch * a.heads_kv, pair, blk);
  const int b = pair / a.heads_kv, hk = pair % a.heads_kv;
  const int item = blk * per_wg + wave / split;
  const int part = wave % split;
  const int qt = nqt - 1 - item / p.group;
  const int hq = hk * p.group + item % p.group;

  const SeqGeom g = seq_geom(b, a.seqlen_q, a.seqlen_k, a.cu_seqlens_q, a.cu_seqlens_k, a.seqused_k);
  const int qr0 = qt * kF32Rows;
  // An idle wave (no item, or its rows past the sequence) walks no tile; in a
  // split workgroup it still takes the barriers.
  const bool live = qt >= 0 && qr0 < g.lq;
  if (!live && split == 1) return;
  const int diag = g.lk - g.lq;
  const bool causal = a.causal != 0;
  const int window_left = a.window_left;
  const bool use_window = window_left >= 0 && (causal || g.lq == 1);
  const int qi = qr0 + l32;
  const bool row_ok = live && qi < g.lq;

  // key tiles some row of the item sees; this wave's steps
  const int q_last = min(qr0 + kF32Rows, g.lq) - 1;
  int kv_hi = g.lk;
  if (causal) kv_hi = min(kv_hi, diag + q_last + 1);
  const int kv_lo = use_window ? max(0, diag + qr0 - window_left) : 0;
  const int j_lo = kv_lo / kF32Rows;
  const int j_hi = kv_hi > 0 ? (kv_hi + kF32Rows - 1) / kF32Rows : 0;
  const int ntile = live ? max(0, j_hi - j_lo) : 0;
  // With ALiBi the tiles are walked from the last down (nearly every row's max
  // is then met first).
  auto tile_of = [&](int t) { return ALIBI ? j_hi - 1 - t : j_lo + t; };
  const unsigned char* ws = reinterpret_cast<const unsigned char*>(a.workspace);
  auto tile_at = [&](int t) { return ws + kv_tile(b, tile_of(t), hk, p.ntiles_k, a.heads_kv) * kTileBytes<D>; };
  const unsigned lane16 = lane * 16;
  f32x4 ring[kRing];
  if (part < ntile) {
    const unsigned char* first = tile_at(part);
#pragma unroll
    for (int c = 0; c < kRing; ++c) ring[c] = img_chunk(first, c, lane16);
  }

  // ---- Q^T: lane half h holds elements 8 s + 4 h .. + 3 of its row -----------
  f32x4 qf[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) qf[s] = f32x4{};
  if (row_ok) {
    const float* qr = reinterpret_cast<const float*>(a.q) + (a.cu_seqlens_q ? 0 : (int64_t)b * a.q_stride_b) +
                      (int64_t)hq * a.q_stride_h + (g.q_row0 + qi) * a.q_stride_t + 4 * hi;
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s] = ld_vec<f32x4>(qr + 8 * s);
    if (a.q_norm_weight) {
      float ss = 0.f;
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int e = 0; e < 4; ++e) ss = fmaf(qf[s][e], qf[s][e], ss);
      const float inv = rms_scale(half_sum(ss), D, a.norm_eps);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const f32x4 w = ld_vec<f32x4>(a.q_norm_weight + 8 * s + 4 * hi);
        qf[s] *= inv * (1.f + w);
      }
    }
    if (a.rope_q) {
      const int pos = rope_qrows(a, g, qr0).at(l32);
#pragma unroll
      for (int s = 0; s < KS / 2; ++s) {
        const f32x4 cs = ld_vec<f32x4>(a.rope_cos + (int64_t)pos * (D / 2) + 8 * s + 4 * hi);
        const f32x4 sn = ld_vec<f32x4>(a.rope_sin + (int64_t)pos * (D / 2) + 8 * s + 4 * hi);
        const f32x4 y1 = qf[s] * cs - qf[s + KS / 2] * sn;
        qf[s + KS / 2] = qf[s] * sn + qf[s + KS / 2] * cs;
        qf[s] = y1;
      }
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s] *= p.scale_log2;
  }
  // (pinned: the read-only loads would otherwise be repeated inside the loop)
#pragma unroll
  for (int s = 0; s < KS; ++s) asm volatile("" : "+v"(qf[s]));

  f32x16 oacc[MD];
#pragma unroll
  for (int md = 0; md < MD; ++md) oacc[md] = f32x16{};
  float m_run = kNegInf, l_run = 0.f, gthr = kNegInf;
  const float slope2 = ALIBI ? a.alibi_slopes[hq] * kLog2e : 0.f;
  const uint32_t* mrow = MASK ? mask_row(a, b, hq, max(0, min(qi, g.lq - 1))) : nullptr;
  const int iabs = diag + qi;

  const bool together = split == 1 && p.group % kWaves == 0;
  // Without ALiBi a tile's scores start at -m of the lane's query row: minit
  // holds that block as the first product's C operand, so that no tile refills
  // its accumulators.
  f32x16 minit = {};
  uint32_t mword = MASK && part < ntile ? mrow[tile_of(part)] : 0u;
  for (int t = part; t < ntile; t += split) {
    const int kvb = tile_of(t) * kF32Rows;
    const unsigned char* cur = tile_at(t);
    // The tile's chunks in order, k then v^T: a chunk is replaced, when used,
    // by the one kRing further on, the last ones by the next tile's first (the
    // last tile: by its own first, unused).
    const unsigned char* next = t + split < ntile ? tile_at(t + split) : cur;
    auto refill = [&](int c) {
      ring[c % kRing] = c + kRing < NC ? img_chunk(cur, c + kRing, lane16) : img_chunk(next, c + kRing - NC, lane16);
    };
    // Waves of a workgroup that walk the same tiles keep together, so that one
    // read of a chunk serves them out of L1 (B=4, T=2048, 32/8 heads, D=128
    // full: 2125 -> 2012 us).
    if (together) __builtin_amdgcn_s_barrier();
    f32x16 s = minit;
    if constexpr (ALIBI) {
      const float m0 = (m_run == kNegInf) ? 0.f : -m_run;
      const float base = m0 + slope2 * (float)(kvb + 4 * hi - iabs);
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = base + slope2 * (float)(8 * (r >> 2) + (r & 3));
    }
#pragma unroll
    for (int c = 0; c < KS; ++c) {
      s = mfma_chunk(ring[c % kRing], qf[c], s);
      refill(c);
      __builtin_amdgcn_sched_barrier(0);
    }
    // hidden keys: a range of the register's key offset 8 (r/4) + r%4 past
    // kvb + 4 hi, and the caller's mask bits
    const bool need = (kvb + kF32Rows > g.lk) || (causal && kvb + kF32Rows - 1 > diag + qr0) ||
                      (use_window && kvb < diag + qr0 + kF32Rows - 1 - window_left) || MASK;
    if (need) {
      const int rel = kvb + 4 * hi;
      int hi_lim = g.lk - 1 - rel;
      if (causal) hi_lim = min(hi_lim, iabs - rel);
      const int lo_lim = use_window ? iabs - window_left - rel : 0;
      uint32_t vis = range_bits(lo_lim, hi_lim);
      if (MASK) {
        vis &= mword >> (4 * hi);
        // (loaded a tile ahead: a wait for it would take in the chunks behind it)
        if (t + split < ntile) mword = mrow[tile_of(t + split)];
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = keep_if_bit(s[r], vis, 8 * (r >> 2) + (r & 3), kNegInf);
    }
    float mx = kNegInf;
#pragma unroll
    for (int r = 0; r < 16; r += 2) mx = fmaxf(fmaxf(mx, s[r]), s[r + 1]);
    if (__builtin_amdgcn_ballot_w64(mx > gthr) != 0) {
      const float mq = (m_run == kNegInf) ? 0.f : m_run;
      const float mn = fmaxf(m_run, half_max(mx) + mq);
      const float alpha = (m_run == kNegInf) ? 0.f : fast_exp2(m_run - mn);
      const float shift = (mn == kNegInf) ? 0.f : mn - mq;
      m_run = mn;
      gthr = (mn == kNegInf) ? kNegInf : kRescaleThresh<D>;
      l_run *= alpha;
#pragma unroll
      for (int md = 0; md < MD; ++md) oacc[md] *= alpha;
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] -= shift;
      if constexpr (!ALIBI) {
        minit = f32x16{} - ((mn == kNegInf) ? 0.f : mn);
        asm volatile("" : "+v"(minit));
      }
    }
    float ls[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = fast_exp2(s[r]);
      ls[r & 3] += s[r];
    }
    l_run += (ls[0] + ls[1]) + (ls[2] + ls[3]);
#pragma unroll
    for (int c = 0; c < KS; ++c) {
      oacc[c % MD] = mfma_chunk(ring[(KS + c) % kRing], acc_chunk(s, c / MD), oacc[c % MD]);
      refill(KS + c);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // ---- epilogue: lane l32 owns query row qi; register (md, r) is head-dim
  // 32 md + 8 (r/4) + 4 hi + r%4
  float* obase = reinterpret_cast<float*>(a.o) + (a.cu_seqlens_q ? 0 : (int64_t)b * a.o_stride_b) +
                 (int64_t)hq * a.o_stride_h + g.q_row0 * a.o_stride_t;
  float* lse = a.lse;
  if (lse) lse += a.cu_seqlens_q ? (int64_t)hq * a.lse_stride_h + g.q_row0 : (int64_t)b * a.lse_stride_b + (int64_t)hq * a.lse_stride_h;
  float l = half_sum(l_run);
  if (split == 1) {
    if (!row_ok) return;
    const float inv = l > 0.f ? 1.f / (l * kValueScale<D>) : 0.f;
    float* orow = obase + qi * a.o_stride_t;
#pragma unroll
    for (int md = 0; md < MD; ++md)
#pragma unroll
      for (int gq = 0; gq < 4; ++gq) st_vec<f32x4>(orow + 32 * md + 8 * gq + 4 * hi, acc_chunk(oacc[md], gq) * inv);
    if (lse && hi == 0) lse[qi] = l > 0.f ? (m_run + log2f(l)) * kLn2 : kNegInf;
    return;
  }
  // The waves of an item: each scales its sums to the item's max; then the
  // item's waves add them, a share of the rows each, and store whole rows.
  MergeSmem<D>& sm = *reinterpret_cast<MergeSmem<D>*>(smem);
  const int w0 = wave - part;
  if (hi == 0) sm.m[wave][l32] = m_run;
  __syncthreads();
  float M = kNegInf;
  for (int w = 0; w < split; ++w) M = fmaxf(M, sm.m[w0 + w][l32]);
  const float f = (m_run == kNegInf) ? 0.f : fast_exp2(m_run - M);
  if (hi == 0) sm.l[wave][l32] = l * f;
#pragma unroll
  for (int md = 0; md < MD; ++md)
#pragma unroll
    for (int gq = 0; gq < 4; ++gq) st_vec<f32x4>(&sm.o[wave][l32][32 * md + 8 * gq + 4 * hi], acc_chunk(oacc[md], gq) * f);
  __syncthreads();
  constexpr int CPR = D / 4;         // 16-byte pieces of a row
  constexpr int RPS = 64 / CPR > 0 ? 64 / CPR : 1;  // rows a wave stores at once
  const int rows = kF32Rows / split;
  for (int r = part * rows + lane / CPR; r < (part + 1) * rows; r += RPS) {
    float ls = 0.f;
    f32x4 o = {};
    for (int w = 0; w < split; ++w) {
      ls += sm.l[w0 + w][r];
      o += ld_vec<f32x4>(&sm.o[w0 + w][r][4 * (lane % CPR)]);
    }
    if (live && qr0 + r < g.lq) {
      st_vec<f32x4>(obase + (int64_t)(qr0 + r) * a.o_stride_t + 4 * (lane % CPR), o * (ls > 0.f ? 1.f / (ls * kValueScale<D>) : 0.f));
      if (lse && lane % CPR == 0) {
        float mr = kNegInf;
        for (int w = 0; w < split; ++w) mr = fmaxf(mr, sm.m[w0 + w][r]);
        lse[qr0 + r] = ls > 0.f ? (mr + log2f(ls)) * kLn2 : kNegInf;
      }
    }
  }
}

template <int D, bool ALIBI, bool MASK>
hipError_t launch_attn(PrefillParams p, hipStream_t s) {
  const goda_prefill_args& a = p.a;
  p.qtiles = (a.seqlen_q + kF32Rows - 1) / kF32Rows;
  const int64_t items = (int64_t)p.qtiles * a.heads_q * a.batch;
  p.key_split = f32_key_split(a, items);
  const int per_wg = kWaves / p.key_split;
  const int64_t nblk = ((int64_t)p.qtiles * p.group + per_wg - 1) / per_wg * a.heads_kv * a.batch;
  if (nblk > 0x7fffffff) return hipErrorInvalidValue;
  auto kern = prefill_f32_kernel<D, ALIBI, MASK>;
  const size_t lds = p.key_split > 1 ? sizeof(MergeSmem<D>) : 0;
  hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(MergeSmem<D>));
  if (e != hipSuccess) return e;
  if ((e = record_timing(a.timing_begin, s)) != hipSuccess) return e;
  kern<<<dim3((unsigned)nblk), kWaves * 64, lds, s>>>(p);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  return record_timing(a.timing_end, s);
}

template <int D>
hipError_t launch_d(PrefillParams p, hipStream_t s) {
  const goda_prefill_args& a = p.a;
  p.ntiles_k = (a.seqlen_k + kF32Rows - 1) / kF32Rows;
  if (p.ntiles_k > 0) {
    pack_kv_f32_kernel<D><<<dim3(p.ntiles_k, a.heads_kv, a.batch), 256, 0, s>>>(p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (a.mask_bits) return a.alibi_slopes ? launch_attn<D, true, true>(p, s) : launch_attn<D, false, true>(p, s);
  return a.alibi_slopes ? launch_attn<D, true, false>(p, s) : launch_attn<D, false, false>(p, s);
}

}  // namespace

// Where the 16-bit kernel's LDS ring (fp32 instances at head_dim 64 and 128)
// has too few workgroups to fill the GPU, the independent waves here are
// faster: us a call, ring / here (pre-pass included), causal:
//   items 1536  B=16 T=512 6/2 D=128        145 /  98
//   items 2048  B=1 T=2048 32/8 D=128       515 / 346
//   items 2048  B=2 T=2048 16/16 D=64       275 / 193
//   items 3072  B=1 T=3072 32/8 D=128       770 / 667
//   items 3072  B=3 T=2048 16/16 D=64       319 / 299
//   items 4096  B=8 T=512 32/8 D=128        177 / 213
//   items 4096  B=8 T=1024 16/16 D=64       204 / 232
// Not so where the ring's workgroups are one whole round of equal work and an
// item's walk here is shared by its waves: full attention over 1024 keys or more
// (fewer: 148 / 148 at T=512 below, 87 / 84 at T=256):
//   B=1 T=2048 32/8 D=128    509 / 547        B=1 T=1856 32/8 D=128   461 / 498
//   B=2 T=8192 4/4 D=64     1021 / 1103       B=1 T=1792 32/8 D=128   445 / 424
//   B=2 T=1024 32/8 D=128    269 / 286        B=1 T=2304 32/8 D=128  1111 / 688
// At head_dim 256, which has no ring instance, they replace the vector-ALU
// kernel (B=8, T=4096, 16/1 heads, ALiBi: 38.0 -> 8.7 ms), which has no pre-pass
// and reads k and v once for 64 rows of a head. It stays for calls of at most
// two key tiles, and for at most 64 rows of heads with keys of their own, over
// walks too short to share, where it fills the GPU (512 workgroups at once) as
// well as this one; us, vector ALUs / here, 16/16 heads:
//   B=256, 4 rows on 70 keys    614 / 672     B=96, 1 row on 256 keys    1 / 1.06
//   B=256, 4 on 200            1415 / 1608    B=80, 64 on 896            1 / 0.96
//   B=64, 64 on 70              170 / 184     B=48, 64 on 256            1 / 0.86
//   B=64, 64 on 992             1 / 1.14      B=64, 33 on 1024           1 / 0.85
bool prefill_f32_streams(const goda_prefill_args& a) {
  if (a.dtype != GODA_DTYPE_F32) return false;
  const int64_t items = (int64_t)((a.seqlen_q + kF32Rows - 1) / kF32Rows) * a.heads_q * a.batch;
  const bool shared = f32_key_split(a, items) > 1;
  if (a.head_dim == 256) {
    if (a.seqlen_k <= 2 * kF32Rows) return false;
    if (a.heads_q != a.heads_kv || a.seqlen_q > 64 || shared) return true;
    const int64_t wgs = (int64_t)a.heads_q * a.batch, rounds = (wgs + 511) / 512;
    return 8 * wgs < 7 * 512 * rounds;
  }
  if (items > 3072) return false;
  const bool equal = !a.causal && !a.cu_seqlens_q && !a.seqused_k;
  return !(equal && shared && items > 7 * 256 && prefill_mfma_workgroups(a) <= 256);
}

int64_t prefill_f32_workspace_bytes(const goda_prefill_args& a) {
  const int64_t ntiles = (a.seqlen_k + kF32Rows - 1) / kF32Rows;
  return 2 * (int64_t)a.batch * ntiles * a.heads_kv * kF32Rows * a.head_dim * 4;
}

hipError_t launch_prefill_f32(const PrefillParams& p, hipStream_t s) {
  switch (p.a.head_dim) {
    case 64:
      return launch_d<64>(p, s);
    case 128:
      return launch_d<128>(p, s);
    case 256:
      return launch_d<256>(p, s);
    default:
      return hipErrorNotSupported;
  }
}

}  // namespace goda
