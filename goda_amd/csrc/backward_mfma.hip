// Backward of prefill attention on gfx950 matrix cores: bf16 / fp16 operands
// at head_dim 64, 128 or 256, fp32 accumulation (fp32 operands:
// backward_f32.hip).
// Same quantities as kernels_/flash_attn_gqa/cuda.py:6-246:
//   P = exp(scale q k^T + bias - lse), dV = P^T dO, dP = dO V^T,
//   dS = P * (dP - delta) with delta = rowsum(dO * O),
//   dQ = scale dS K, dK = scale dS^T Q.
//
// Four launches:
//   1. pack_q_bwd_kernel: per (32-row query tile, query head, sequence),
//      the row-major operand images of rotated q (prescaled) and of dO
//      ("chunk-column-major" [D/8][32] 16-byte chunks, the A operand of a
//      product over head_dim), plus the row statistics lse*log2(e) and delta.
//      The operands of products over rows are read out of the same images
//      with transposing LDS reads (ds_read_b64_tr_b16).
//   2. pack_kv_bwd_kernel: per (32-key tile, KV head, sequence), the
//      row-major images of rotated k and of v (k^T likewise by transposing
//      reads).
//   3. bwd_dkv_mfma_kernel: one workgroup of 8 waves per 128 keys of a KV
//      head, in pairs (two waves of one SIMD) that share 32 keys; the pair
//      pins the k and v operands of its keys and walks the query tiles of
//      every head of the group (GQA reduction in the accumulators, no
//      atomics), the tiles moving through a three-stage LDS ring. One wave
//      of a pair computes S, dP, P and dS and hands P and dS to the other
//      through LDS, which accumulates dV and dK one tile behind:
//        S    [rows][keys] = Q K^T        A = Q image,   B = k (registers)
//        dV^T [d][keys]   += dO^T P        A = dO^T (transposing reads), B = P (packed S)
//        dP   [rows][keys] = dO V^T        A = dO image,  B = v (registers)
//        dK^T [d][keys]   += Q^T dS        A = Q^T (transposing reads), B = dS (packed)
//      head_dim 256 (bwd_dkv_wide_kernel): a wave needs both operand sets and
//      both accumulators (~450 registers), so four waves, one per SIMD, each
//      owning 32 keys and doing all four products; with few key blocks the
//      walk is split over several workgroups whose fp32 partials
//      bwd_dkv_reduce_kernel sums.
//   4. bwd_dq_mfma_kernel: one workgroup of 8 waves (two per SIMD, so one
//      wave's products overlap the other's exp work; 4 waves, one per SIMD,
//      at head_dim 256) per (query tile, head slice); each wave pins the q and
//      dO operands of its 32 rows and walks the key tiles:
//        S^T  [keys][rows] = K Q^T         A = k image,   B = q (registers)
//        dP^T [keys][rows] = V dO^T        A = v image,   B = dO (registers)
//        dQ^T [d][rows]   += K^T dS^T      A = K^T (transposing reads), B = dS^T (packed)
// A packed accumulator becomes a B operand directly because the transposing
// reads hand out rows / keys in the accumulator's register order (kPermKey). With the
// log-sum-exp known there is no online softmax.

#include <algorithm>

#include "common.h"
#include "launch.h"
#include "mfma_common.h"

namespace goda {
namespace {

constexpr int kQRows = 32;   // rows per query tile
constexpr int kBKV = 32;     // keys per key tile
// dq workgroup: two waves per SIMD, or one at head_dim 256 (q and dO operands
// plus the dQ^T accumulator take ~350 registers there).
template <int D>
struct DqShape {
  static constexpr bool WIDE = D >= 256;
  static constexpr int WAVES = WIDE ? 4 : 8;
  static constexpr int OCC = WIDE ? 1 : 2;
};

// Images are counted in 8-element chunks of 16 bytes. The dK accumulators
// multiply the prescaled q image (q * scale * log2(e)): dk = ln(2) * dK^T.
template <typename T, int D>
struct QImg {
  static constexpr int CHB = (int)sizeof(typename Vec<T>::v8);
  static constexpr int CH = D / 8 * kQRows;  // chunks of one image
  static constexpr int NIMG = 2;
  static constexpr int QA = 0, GA = CH;
  // Row-major images: chunk (c, r) (head-dim 8c..8c+7 of row r) at
  // c*32 + (r ^ SWZ*(c%2)). A transposing read
  // of 16 lanes covers rows r..r+3 of two adjacent chunk columns, 512 bytes
  // apart (the same LDS banks); swapping the 4-row halves of every odd column
  // puts them on disjoint banks. A 32-row column read stays one contiguous
  // 512-byte block.
  static constexpr int SWZ = 4;
  static constexpr int STAT = NIMG * CH;     // lse2[32] then delta[32]: 256 bytes
  static constexpr int STAT_CH = 256 / CHB;
  static constexpr int CHUNKS = NIMG * CH + STAT_CH;
  static constexpr int64_t BYTES = (int64_t)CHUNKS * CHB;
};

// Key-side images: row-major k and v, with the query images' odd-column
// swizzle.
template <typename T, int D>
struct KVImg {
  static constexpr int CHB = (int)sizeof(typename Vec<T>::v8);
  static constexpr int CH = D / 8 * kBKV;
  static constexpr int NIMG = 2;
  static constexpr int SWZ = 4;
  static constexpr int KA = 0, VA = CH;
  static constexpr int CHUNKS = NIMG * CH;
  static constexpr int64_t BYTES = (int64_t)CHUNKS * CHB;
};

// A operand of a product over the 32 rows (or keys) of a row-major image
// tile, i.e. the transposed tile, for 16-bit images with the odd-column
// swizzle: lane l gets head-dim 32 md + l%32 over rows 16 half + 4 (l/32) +
// {0..3, 8..11}, the order of the packed accumulator registers of its lane
// half (kPermKey). Two ds_read_b64_tr_b16: that instruction hands lane j of a
// 16-lane group element j%4 of the 8-byte segments read by lanes j/4 + 4e,
// e = 0..3; lane s reads row 16 half + 8 k + 4 (l/32) + s/4 at head-dim
// 32 md + 16 ((l/16)%2) + 4 (s%4), so lane j receives rows
// 16 half + 8 k + 4 (l/32) + e at head-dim 32 md + l%32. Row r, head-dim d
// sits at byte ((d/8)*32 + (r ^ 4*((d/8)%2)))*16 + (d%8)*2 of the image.
template <typename V>
__device__ __forceinline__ V tr_operand(const unsigned char* img, int lane, int half, int md) {
  static_assert(sizeof(V) == 16, "16-bit operands");
  const int hi = lane >> 5;
  const int d = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  const int row = 4 * (hi ^ ((d >> 3) & 1)) + ((lane & 15) >> 2);  // odd-column swizzle
  const unsigned char* base = img + ((d >> 3) * 32 + row) * 16 + (d & 7) * 2 + md * (4 * 32 * 16) + half * 256;
  typedef short s4 __attribute__((ext_vector_type(4)));
  typedef short s8 __attribute__((ext_vector_type(8)));
  const s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4*)(base));
  const s4 up = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4*)(base + 128));
  return __builtin_bit_cast(V, (s8)__builtin_shufflevector(lo, up, 0, 1, 2, 3, 4, 5, 6, 7));
}

__device__ __forceinline__ int64_t q_tile_index(int b, int qt, int hq, int ntq, int heads_q) {
  return ((int64_t)b * ntq + qt) * heads_q + hq;
}
__device__ __forceinline__ int64_t kv_tile_index(int b, int j, int hk, int ntk, int heads_kv) {
  return ((int64_t)b * ntk + j) * heads_kv + hk;
}

// Byte offset of dS tile (sequence b, query tile qt, key tile kt, query head
// hq). A stored tile (32 query rows x 32 keys, 2 KB) holds the B operands of
// the dq product over its keys: 16 bytes per (k-step s, lane half h, row) at
// ((2 s + h) 32 + row) 16, element e = key 16 s + 4 h + (e & 3) + 8 (e >> 2)
// (the kPermKey order of tr_operand's K^T operand).
__device__ __forceinline__ int64_t ds_tile_offset(const BwdParams& p, int b, int qt, int kt, int hq) {
  return (((int64_t)b * p.ds_per_b + ds_row_off(qt, p.ntk, p.ds_c, p.ds_tri != 0) + kt) * p.a.heads_q + hq) * 2048;
}

// Step it = h * nq + q of a walk over (query head h of a KV group, query
// tile q of nq), advanced one step at a time: no division per tile.
struct QWalk {
  int h, q, nq;
  __device__ __forceinline__ QWalk(int it, int nq_) : h(nq_ > 0 ? it / nq_ : 0), q(it - h * nq_), nq(nq_) {}
  __device__ __forceinline__ void next() {
    if (++q == nq) {
      q = 0;
      ++h;
    }
  }
};

// The same steps in the order the dk/dv kernels walk them: query tile
// outermost, from the last tile down, the group's heads innermost (step it is
// head it % g of tile nq - 1 - it / g). Every key block of a KV head then
// reads the same tile images in the same order from the same starting tile,
// whatever its causal first tile, so the blocks running at once share them
// in L2.
struct QWalkDown {
  int h, q, g;
  __device__ __forceinline__ QWalkDown(int it, int nq, int g_) : h(it % g_), q(nq - 1 - it / g_), g(g_) {}
  __device__ __forceinline__ void next() {
    if (++h == g) {
      h = 0;
      --q;
    }
  }
};

template <typename T>
__device__ __forceinline__ const T* grow(const void* base, int64_t sb, int64_t st, int64_t sh, bool varlen, int b,
                                         int64_t row, int h) {
  return reinterpret_cast<const T*>(base) + (varlen ? 0 : (int64_t)b * sb) + row * st + (int64_t)h * sh;
}

// Elements c..c+7 and c+D/2..c+D/2+7 of a q or k row, held by one of the
// row's N consecutive lanes: goda's RMSNorm (weight w, or none) and then the
// half-split rotation at `pos` (when `rot`), in fp32 and rounded once, as
// the forward's pre-passes compute them. With `sc1`, `sc2` also the row times
// `scale`, rounded once from the same fp32 values (the forward's q operand).
// Every lane of the row's group must call it (the norm's sum of squares is a
// group reduction).
template <typename T, int D, int N>
__device__ __forceinline__ void norm_rope_row(typename Vec<T>::v8& h1, typename Vec<T>::v8& h2, int c, const float* w,
                                              float eps, bool rot, int pos, const goda_prefill_args& a,
                                              float scale = 0.f, typename Vec<T>::v8* sc1 = nullptr,
                                              typename Vec<T>::v8* sc2 = nullptr) {
  if (!w && !rot && !sc1) return;
  float x1[8], x2[8];
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    x1[e] = (float)h1[e];
    x2[e] = (float)h2[e];
    ss = fmaf(x1[e], x1[e], fmaf(x2[e], x2[e], ss));
  }
  if (w) {
    const float inv = rms_scale(lane_group_sum<N>(ss), D, eps);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      x1[e] *= inv * (1.f + w[c + e]);
      x2[e] *= inv * (1.f + w[c + D / 2 + e]);
    }
  }
  if (rot) {
    const float* cs = a.rope_cos + (int64_t)pos * (D / 2) + c;
    const float* sn = a.rope_sin + (int64_t)pos * (D / 2) + c;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float y1 = x1[e] * cs[e] - x2[e] * sn[e];
      x2[e] = x1[e] * sn[e] + x2[e] * cs[e];
      x1[e] = y1;
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    h1[e] = (T)x1[e];
    h2[e] = (T)x2[e];
    if (sc1) {
      (*sc1)[e] = (T)(x1[e] * scale);
      (*sc2)[e] = (T)(x2[e] * scale);
    }
  }
}

// ---------------------------------------------------------------------------
// 1. query-side images
// ---------------------------------------------------------------------------
template <typename T, int D>
__global__ void __launch_bounds__(256) pack_q_bwd_kernel(const BwdParams p) {
  typedef typename Vec<T>::v8 v8;
  typedef QImg<T, D> QI;
  const goda_prefill_args& a = p.a;
  const int qt = blockIdx.x, hq = blockIdx.y, b = blockIdx.z;
  const SeqGeom g = seq_geom(b, a.seqlen_q, a.seqlen_k, a.cu_seqlens_q, a.cu_seqlens_k, a.seqused_k);
  const int i0 = qt * kQRows;
  if (i0 >= g.lq) return;
  const bool varlen = a.cu_seqlens_q != nullptr;
  __shared__ __align__(16) T qsrows[kQRows][D + 8];  // q * scale * log2(e)
  __shared__ __align__(16) T grows[kQRows][D + 8];
  const int tid = threadIdx.x;
  constexpr int HALF8 = D / 16;
  const RopePos rope = rope_qrows(a, g, i0);

  // normalized, rotated q and dO rows (zero past the sequence); a row's
  // HALF8 threads are consecutive lanes (and the loop is uniform per wave)
  for (int idx = tid; idx < kQRows * HALF8; idx += 256) {
    const int r = idx / HALF8;
    const int c = (idx % HALF8) * 8;
    const int i = i0 + r;
    v8 q1 = {}, q2 = {}, g1 = {}, g2 = {};
    if (i < g.lq) {
      const T* qr = grow<T>(a.q, a.q_stride_b, a.q_stride_t, a.q_stride_h, varlen, b, g.q_row0 + i, hq);
      const T* gr = grow<T>(p.g.d_o, p.g.do_stride_b, p.g.do_stride_t, p.g.do_stride_h, varlen, b, g.q_row0 + i, hq);
      q1 = ld_stream<v8>(qr + c);
      q2 = ld_stream<v8>(qr + c + D / 2);
      g1 = ld_stream<v8>(gr + c);
      g2 = ld_stream<v8>(gr + c + D / 2);
    }
    v8 qs1, qs2;
    norm_rope_row<T, D, HALF8>(q1, q2, c, a.q_norm_weight, a.norm_eps, i < g.lq && a.rope_q,
                               rope.at(r), a, p.scale_log2, &qs1, &qs2);
    st_vec<v8>(&qsrows[r][c], qs1);
    st_vec<v8>(&qsrows[r][c + D / 2], qs2);
    st_vec<v8>(&grows[r][c], g1);
    st_vec<v8>(&grows[r][c + D / 2], g2);
  }
  __syncthreads();

  v8* img = reinterpret_cast<v8*>(p.qimg + q_tile_index(b, qt, hq, p.ntq, a.heads_q) * QI::BYTES);
  // row-major images: chunk (c, r) at c*32 + r (q prescaled: the scores leave
  // the matrix core in log2 units, as in the forward)
  for (int idx = tid; idx < QI::CH; idx += 256) {
    const int c = idx / kQRows, r = idx % kQRows;
    const int at = c * kQRows + (r ^ (QI::SWZ * (c & 1)));
    img[QI::QA + at] = ld_vec<v8>(&qsrows[r][8 * c]);
    img[QI::GA + at] = ld_vec<v8>(&grows[r][8 * c]);
  }
  // row statistics: 8 threads per row
  {
    const int r = tid >> 3, part = tid & 7;
    const int i = i0 + r;
    float dl = 0.f;
    if (i < g.lq) {
      const T* orow = grow<T>(a.o, a.o_stride_b, a.o_stride_t, a.o_stride_h, varlen, b, g.q_row0 + i, hq);
      // 16-byte loads: the row's 8 threads read 8 consecutive chunks at a time
#pragma unroll
      for (int c = 8 * part; c < D; c += 64) {
        const v8 ov = ld_stream<v8>(orow + c);
        const v8 gv = ld_vec<v8>(&grows[r][c]);
#pragma unroll
        for (int e = 0; e < 8; ++e) dl = fmaf((float)ov[e], (float)gv[e], dl);
      }
    }
    dl += shfl_xor_f(dl, 1);
    dl += shfl_xor_f(dl, 2);
    dl += shfl_xor_f(dl, 4);
    if (part == 0) {
      float l2 = kNegInf;
      if (i < g.lq) {
        const int64_t li = a.cu_seqlens_q ? (int64_t)hq * a.lse_stride_h + g.q_row0 + i
                                          : (int64_t)b * a.lse_stride_b + (int64_t)hq * a.lse_stride_h + i;
        l2 = a.lse[li] * kLog2e;
      }
      float* st = reinterpret_cast<float*>(img + QI::STAT);
      st[r] = l2;
      st[kQRows + r] = dl;
    }
  }
}

// ---------------------------------------------------------------------------
// 2. key-side images
// ---------------------------------------------------------------------------
template <typename T, int D>
__global__ void __launch_bounds__(256) pack_kv_bwd_kernel(const BwdParams p) {
  typedef typename Vec<T>::v8 v8;
  typedef KVImg<T, D> KI;
  const goda_prefill_args& a = p.a;
  const int j = blockIdx.x, hk = blockIdx.y, b = blockIdx.z;
  const SeqGeom g = seq_geom(b, a.seqlen_q, a.seqlen_k, a.cu_seqlens_q, a.cu_seqlens_k, a.seqused_k);
  const int kv0 = j * kBKV;
  if (kv0 >= g.lk) return;
  const bool varlen = a.cu_seqlens_k != nullptr;
  __shared__ __align__(16) T krows[kBKV][D + 8];
  __shared__ __align__(16) T vrows[kBKV][D + 8];
  const int tid = threadIdx.x;
  constexpr int HALF8 = D / 16;
  const RopePos rope = rope_krows(a, g, kv0);
  for (int idx = tid; idx < kBKV * HALF8; idx += 256) {
    const int r = idx / HALF8;
    const int c = (idx % HALF8) * 8;
    const int row = kv0 + r;
    v8 k1 = {}, k2 = {}, v1 = {}, v2 = {};
    if (row < g.lk) {
      const T* kr = grow<T>(a.k, a.k_stride_b, a.k_stride_t, a.k_stride_h, varlen, b, g.k_row0 + row, hk);
      const T* vr = grow<T>(a.v, a.v_stride_b, a.v_stride_t, a.v_stride_h, varlen, b, g.k_row0 + row, hk);
      k1 = ld_stream<v8>(kr + c);
      k2 = ld_stream<v8>(kr + c + D / 2);
      v1 = ld_stream<v8>(vr + c);
      v2 = ld_stream<v8>(vr + c + D / 2);
    }
    norm_rope_row<T, D, HALF8>(k1, k2, c, a.k_norm_weight, a.norm_eps, row < g.lk && a.rope_k, rope.at(r),
                               a);
    st_vec<v8>(&krows[r][c], k1);
    st_vec<v8>(&krows[r][c + D / 2], k2);
    st_vec<v8>(&vrows[r][c], v1);
    st_vec<v8>(&vrows[r][c + D / 2], v2);
  }
  __syncthreads();
  v8* img = reinterpret_cast<v8*>(p.kvimg + kv_tile_index(b, j, hk, p.ntk, a.heads_kv) * KI::BYTES);
  for (int idx = tid; idx < KI::CH; idx += 256) {
    const int c = idx / kBKV, r = idx % kBKV;
    const int at = c * kBKV + (r ^ (KI::SWZ * (c & 1)));
    img[KI::KA + at] = ld_vec<v8>(&krows[r][8 * c]);
    img[KI::VA + at] = ld_vec<v8>(&vrows[r][8 * c]);
  }
}

// Key-major copy of the caller's row-major mask bits, for the dk/dv kernels
// (a lane there holds one key and 16 query rows of a 32-row tile): word
// [b][h][key][query tile] bit r = row 32 * tile + r. A thread reads the 32
// row words of one (query tile, 32-key word), transposes the 32x32 bit block
// in registers and writes the 32 key words.
__global__ void __launch_bounds__(256) bwd_mask_t_kernel(const BwdParams p) {
  const goda_prefill_args& a = p.a;
  const int nkw = (a.seqlen_k + 31) / 32;
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (int64_t)p.ntq * nkw) return;
  const int qt = (int)(idx % p.ntq), kw = (int)(idx / p.ntq);
  const int hm = blockIdx.y, bm = blockIdx.z;
  uint32_t m[32];
#pragma unroll
  for (int r = 0; r < 32; ++r) {
    const int i = 32 * qt + r;
    m[r] = i < a.seqlen_q ? mask_row(a, bm, hm, i)[kw] : 0u;
  }
  uint32_t* out = p.mask_t + bm * p.mt_stride_b + hm * p.mt_stride_h;
#pragma unroll
  for (int c = 0; c < 32; ++c) {
    uint32_t w = 0;
#pragma unroll
    for (int r = 0; r < 32; ++r) w |= ((m[r] >> c) & 1u) << r;
    const int key = 32 * kw + c;
    if (key < a.seqlen_k) out[(int64_t)key * p.ntq + qt] = w;
  }
}

// A phase of NJ products, each with one LDS operand: the operands of the
// first L products are read first, each product's register is refilled with
// the operand L products later, and scheduling fences keep that order (left
// alone, the compiler moves every read next to its product, leaving about one
// in flight; `lead_schedule` asks for the order but is not always honoured).
// `after(j)` runs after product j, inside the same fence: independent VALU
// work placed there issues while the products execute.
template <int NJ, int L, typename V, typename Src, typename Prod, typename After>
__device__ __forceinline__ void prefetched_products(Src src, Prod prod, After after) {
  constexpr int P = L < NJ ? L : NJ;
  V op[P];
#pragma unroll
  for (int j = 0; j < P; ++j) op[j] = src(j);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    prod(j, op[j % P]);
    if (j + P < NJ) op[j % P] = src(j + P);
    after(j);
    __builtin_amdgcn_sched_barrier(0);
  }
}

template <int NJ, int L, typename V, typename Src, typename Prod>
__device__ __forceinline__ void prefetched_products(Src src, Prod prod) {
  prefetched_products<NJ, L, V>(src, prod, [](int) {});
}

// Schedule of a phase of NM MFMAs, each with one LDS operand read: the reads
// run LEAD MFMAs ahead (not all hoisted, which would hold 4 registers each).
template <typename T, int NM, int LEAD>
__device__ __forceinline__ void lead_schedule() {
  constexpr int M = kMfmaPerStep<T>;                            // MFMAs per step
  constexpr int R = (int)sizeof(typename Vec<T>::v8) / 16;      // 16-byte reads per operand
  __builtin_amdgcn_sched_group_barrier(0x100, LEAD * R, 0);
#pragma unroll
  for (int i = 0; i < NM - LEAD; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, M, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, R, 0);
  }
  __builtin_amdgcn_sched_group_barrier(0x008, LEAD * M, 0);
}

// Packs accumulator registers 8g..8g+7 of a 32x32 tile into an operand.
template <typename V, typename T>
__device__ __forceinline__ V pack8(const float* x) {
  V v;
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = (T)x[e];
  return v;
}

// ---------------------------------------------------------------------------
// 3. dk, dv
// ---------------------------------------------------------------------------
// Eight waves, two per SIMD, in pairs that share 32 keys. Wave w < 4 ("A",
// scores) pins the k and v operands of the keys and, per query tile, issues
// S = Q K^T and dP = dO V^T, then computes P and dS = P (dP - delta) and
// hands both, packed as operands, to its partner through LDS. Wave w + 4
// ("B", gradients, same SIMD) holds the dV^T and dK^T accumulators and, one
// tile behind, issues dV^T += dO^T P and dK^T += Q^T dS. Each iteration
// A wave's VALU instructions do not issue while the other wave of its SIMD
// has matrix instructions waiting, so A's VALU work cannot hide under B's
// products: A runs one tile ahead of itself instead, issuing the products of
// tile it + 1 with the VALU work of tile it (P, dS) placed between them, where
// it issues while A's own products execute. Query tiles move through a
// four-stage ring (A reads tiles it and it + 1, B tile it - 1, tile it + 2 is
// being copied); the P / dS exchange is double-buffered. (Copying two tiles
// ahead through a fifth stage is slower: the copies then land during the
// products, whose operand reads already saturate the LDS.)
constexpr int kWavesKv = 8;
constexpr int kKvStages = 4;

template <typename T, int D>
struct DkvSmem {
  static constexpr int64_t RING = kKvStages * QImg<T, D>::BYTES;
  // operand exchange: [parity][pair][P0, P1, dS0, dS1][lane] 16-byte chunks
  static constexpr int64_t XBUF = 2 * 4 * 4 * 64 * 16;
  static constexpr int64_t BYTES = RING + XBUF;
};

__device__ __forceinline__ void chunked_order_3d(int& bx, int& by, int& bz) {
  const int lin = (int)(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z));
  int unit;
  chunked_order(lin, (int)gridDim.x, (int)(gridDim.y * gridDim.z), unit, bx);
  by = unit % (int)gridDim.y;
  bz = unit / (int)gridDim.y;
}

template <typename T, int D, bool ALIBI, bool MASK>
__global__ void __launch_bounds__(kWavesKv * 64, 1) bwd_dkv_mfma_kernel(const BwdParams p) {
  typedef typename Vec<T>::v8 v8;
  typedef typename Vec<T>::v4 v4;
  typedef QImg<T, D> QI;
  typedef KVImg<T, D> KI;
  constexpr int KS = D / 16;  // k-steps over head_dim
  constexpr int MD = D / 32;  // 32-wide head_dim tiles of dK^T / dV^T
  static_assert(sizeof(T) == 2, "B's operands come from transposing reads of 16-bit images");
  constexpr int LOADS = QI::NIMG * QI::CH / (kWavesKv * 64);
  static_assert(QI::NIMG * QI::CH % (kWavesKv * 64) == 0, "tile must split over the waves");
  extern __shared__ __align__(16) unsigned char smem[];
  v8* xbuf = reinterpret_cast<v8*>(smem + DkvSmem<T, D>::RING);

  const goda_prefill_args& a = p.a;
  int bx, by, bz;
  chunked_order_3d(bx, by, bz);
  const int b = bz, hk = by;
  const SeqGeom g = seq_geom(b, a.seqlen_q, a.seqlen_k, a.cu_seqlens_q, a.cu_seqlens_k, a.seqused_k);
  const bool varlen = a.cu_seqlens_k != nullptr;
  const int kend = varlen ? g.lk : a.seqlen_k;  // rows this launch writes
  const int kv0 = bx * 128;
  if (kv0 >= kend) return;

  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63, l32 = lane & 31, hi = lane >> 5;
  const bool role_b = wave >= 4;  // wave-uniform
  const int pair = wave & 3;
  const int kw0 = kv0 + 32 * pair;
  const int key = kw0 + l32;
  const int diag = g.lk - g.lq;
  const bool use_window = a.window_left >= 0 && (a.causal || g.lq == 1);

  // Query tiles that can see a key of this workgroup.
  const int kv_last = min(kv0 + 128, g.lk) - 1;
  int i_lo = 0, i_hi = g.lq;
  if (a.causal) i_lo = max(0, kv0 - diag);
  if (use_window) i_hi = min(g.lq, kv_last + a.window_left - diag + 1);
  if (kv0 >= g.lk) i_hi = i_lo;
  const int qt_lo = i_lo / kQRows;
  const int nq = i_hi > i_lo ? (i_hi - 1) / kQRows + 1 - qt_lo : 0;
  const int n = p.group * nq;

  // Query tiles move into the ring by direct global->LDS loads (dma_blocks),
  // issued by the B waves only (A's scores are the critical path): B wave w's
  // share of a tile is 2 LOADS blocks of 64 consecutive 16-byte chunks at
  // the same offsets in the image and in the stage, and wave 4's lanes below
  // STAT_CH copy the row statistics. Tile it + 2 lands in stage
  // (it + 2) % kKvStages during interval it, when A reads stages it and
  // it + 1 and B stage it - 1 (all mod kKvStages); the barrier opening
  // interval it + 1 waits for it (vmcnt(0)).
  static_assert(2 * LOADS == 2 || 2 * LOADS == 4, "DMA share of 2 or 4 blocks");
  static_assert(QI::STAT_CH <= 64, "statistics fit one wave's copy");
  const int bw = __builtin_amdgcn_readfirstlane(wave) & 3;
  const unsigned lane_off = (unsigned)((bw * 2 * LOADS * 64 + lane) * 16);
  const unsigned stat_off = (unsigned)((QI::STAT + lane) * 16);
  QWalkDown ld(0, nq, p.group);  // the next tile to copy; copies come in walk order
  auto tile_dma = [&](int it) {
    const int64_t t = q_tile_index(b, qt_lo + ld.q, hk * p.group + ld.h, p.ntq, a.heads_q);
    ld.next();
    const unsigned long long base = (unsigned long long)(uintptr_t)(p.qimg + t * QI::BYTES);
    const unsigned lds = (unsigned)(uintptr_t)(smem + (it % kKvStages) * QI::BYTES);
    dma_blocks<2 * LOADS>(lds + (unsigned)(bw * 2 * LOADS * 64 * 16), lane_off, base);
    if (bw == 0 && lane < QI::STAT_CH) dma_blocks<1>(lds + QI::STAT * 16, stat_off, base);
  };
  auto stage = [&](int it) { return reinterpret_cast<const v8*>(smem + (it % kKvStages) * QI::BYTES); };
  auto xchg = [&](int it, int c) -> v8& { return xbuf[(((it & 1) * 4 + pair) * 4 + c) * 64 + lane]; };
  // Iterations 0..n of a role (B runs one tile behind A, so both take n + 1
  // barriers). `pre(it)` issues the role's own global loads; `copy(it)` the
  // tile copies of the role that makes them.
  auto walk = [&](auto&& copy, auto&& pre, auto&& step) {
    if (n > 0) copy(0);
    if (n > 1) copy(1);
    for (int it = 0; it <= n; ++it) {
      dma_ring_barrier<0>();
      if (it + 2 < n) copy(it + 2);
      pre(it);
      step(it);
    }
  };
  // The same intervals unrolled by two: `step(it, parity)` gets the parity as
  // a compile-time constant, so A's two accumulator sets keep fixed registers.
  auto walk2 = [&](auto&& pre, auto&& step) {
    auto interval = [&](int it, auto parity) {
      dma_ring_barrier<0>();
      pre(it);
      step(it, parity);
    };
    for (int it = 0;; it += 2) {
      interval(it, std::integral_constant<int, 0>{});
      if (it + 1 > n) break;
      interval(it + 1, std::integral_constant<int, 1>{});
      if (it + 2 > n) break;
    }
  };

  if (!role_b) {
    // ---- A: scores --------------------------------------------------------
    v8 kf[KS], vf[KS];
    if (kw0 < g.lk) {
      const v8* img = reinterpret_cast<const v8*>(p.kvimg + kv_tile_index(b, kw0 / kBKV, hk, p.ntk, a.heads_kv) * KI::BYTES);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        kf[ks] = img[KI::KA + (2 * ks + hi) * kBKV + (l32 ^ (KI::SWZ * hi))];
        vf[ks] = img[KI::VA + (2 * ks + hi) * kBKV + (l32 ^ (KI::SWZ * hi))];
      }
    } else {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) kf[ks] = vf[ks] = v8{};
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      asm volatile("" : "+v"(kf[ks]));
      asm volatile("" : "+v"(vf[ks]));
    }
    const bool key_ok = key < g.lk;
    QWalkDown cu(0, nq, p.group);
    uint32_t mword = 0;
    auto pre = [&](int it) {
      // the caller's mask bits of this key for the tile's 32 rows
      if (MASK && key_ok && it < n)
        mword = p.mask_t[b * p.mt_stride_b + (hk * p.group + cu.h) * p.mt_stride_h + (int64_t)key * p.ntq + qt_lo +
                         cu.q] >> (4 * hi);
    };
    // S [rows][keys] and dP of tile `it` into (sn, dpn): two interleaved
    // accumulation chains (the q image holds q * scale * log2(e): S leaves
    // the matrix core in log2 units); after(j) follows product j.
    auto products = [&](int it, f32x16& sn, f32x16& dpn, auto&& after) {
      const v8* st = stage(it);
      sn = f32x16{};
      dpn = f32x16{};
      prefetched_products<2 * KS, 4, v8>(
          [&](int j) { return st[((j & 1) ? QI::GA : QI::QA) + (2 * (j >> 1) + hi) * kQRows + (l32 ^ (QI::SWZ * hi))]; },
          [&](int j, const v8& o) {
            if (j & 1)
              dpn = mfma32(o, vf[j >> 1], dpn);
            else
              sn = mfma32(o, kf[j >> 1], sn);
          },
          after);
    };
    // P and dS of tile it from (s, dp), interleaved with the products of tile
    // it + 1 into (sn, dpn); RPS registers after each product.
    constexpr int RPS = 16 / (2 * KS);
    static_assert(16 % (2 * KS) == 0, "whole registers per product");
    auto scores = [&](int it, const f32x16& s, const f32x16& dp, f32x16& sn, f32x16& dpn) {
      const int hq = hk * p.group + cu.h;
      const int q0 = (qt_lo + cu.q) * kQRows;
      cu.next();
      const float* stat = reinterpret_cast<const float*>(stage(it) + QI::STAT);
      f32x4 l2[4], dl[4];
#pragma unroll
      for (int gq = 0; gq < 4; ++gq) {
        l2[gq] = ld_vec<f32x4>(stat + 8 * gq + 4 * hi);
        dl[gq] = ld_vec<f32x4>(stat + kQRows + 8 * gq + 4 * hi);
      }
      // Visibility as a range of the register's row offset
      // off = row - (q0 + 4 hi). (Starting the accumulators at -lse2 and
      // -delta, as the head_dim-256 and dq kernels do, saves two VALU
      // instructions per entry but makes the products wait for the row
      // statistics' LDS reads.)
      const float slope2 = ALIBI ? a.alibi_slopes[hq] * kLog2e : 0.f;
      const int rel = q0 + 4 * hi;
      int lo_lim = -1, hi_lim = g.lq - 1 - rel;
      if (a.causal) lo_lim = key - diag - rel;
      if (use_window) hi_lim = min(hi_lim, key + a.window_left - diag - rel);
      // Visible rows as one bit per register offset (bit off = 8 gq + e).
      uint32_t vis = key_ok ? range_bits(lo_lim, hi_lim) : 0u;
      if (MASK) vis &= mword;
      const float base = ALIBI ? slope2 * (float)(key - diag - rel) : 0.f;
      float pr[16], ds[16];
      auto slice = [&](int j) {
#pragma unroll
        for (int k = 0; k < RPS; ++k) {
          const int r = j * RPS + k, gq = r >> 2, e = r & 3;
          float t = s[r];
          if (ALIBI) t += base - slope2 * (float)(8 * gq + e);
          pr[r] = fast_exp2(t - l2[gq][e]);
          ds[r] = pr[r] * (dp[r] - dl[gq][e]);
        }
      };
      // (On the last tile the products re-read tile it; they go unused.)
      products(min(it + 1, n - 1), sn, dpn, slice);
      // Hidden entries are replaced (not scaled: exp2 of a hidden score may
      // overflow) on the tiles where some lane of the wave has one; a
      // wave-uniform branch, most tiles skip it.
      if (__builtin_amdgcn_ballot_w64(vis != ~0u) != 0) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int off = 8 * (r >> 2) + (r & 3);
          pr[r] = keep_if_bit(pr[r], vis, off, 0.f);
          ds[r] = keep_if_bit(ds[r], vis, off, 0.f);
        }
      }
      xchg(it, 0) = pack8<v8, T>(pr);
      xchg(it, 1) = pack8<v8, T>(pr + 8);
      xchg(it, 2) = pack8<v8, T>(ds);
      xchg(it, 3) = pack8<v8, T>(ds + 8);
    };
    // Two accumulator sets alternate by parity: tile it's products sit in
    // set it % 2.
    f32x16 s0, d0, s1, d1;
    walk2(pre, [&](int it, auto parity) {
      if constexpr (parity == 0) {
        if (it == 0 && n > 0) products(0, s0, d0, [](int) {});
        if (it < n) scores(it, s0, d0, s1, d1);
      } else {
        if (it < n) scores(it, s1, d1, s0, d0);
      }
    });
    return;
  }

  // ---- B: gradients ---------------------------------------------------------
  f32x16 dv[MD], dk[MD];
#pragma unroll
  for (int md = 0; md < MD; ++md) dv[md] = dk[md] = f32x16{};
  // B's A operands dO^T and q^T come out of the row-major images by
  // transposing reads (tr_operand).
  walk(tile_dma, [](int) {}, [&](int it) {
    if (it > 0) {
      const unsigned char* st = reinterpret_cast<const unsigned char*>(stage(it - 1));
      const v8 p0 = xchg(it - 1, 0), p1 = xchg(it - 1, 1);
      const v8 d0 = xchg(it - 1, 2), d1 = xchg(it - 1, 3);
      // Operand reads 8 products ahead (A's 4): with the matrix core shared
      // with A, B's products otherwise wait on LDS latency (phase
      // timestamps: B's 16 products spread over ~2100 clocks with about one
      // read in flight). j: half = j / (2 MD), md = (j / 2) % MD, odd: dK.
      prefetched_products<4 * MD, 8, v8>(
          [&](int j) {
            const int half = j / (2 * MD), md = (j >> 1) % MD;
            return tr_operand<v8>(st + ((j & 1) ? QI::QA : QI::GA) * QI::CHB, lane, half, md);
          },
          [&](int j, const v8& o) {
            const int half = j / (2 * MD), md = (j >> 1) % MD;
            if (j & 1)
              dk[md] = mfma32(o, half ? d1 : d0, dk[md]);
            else
              dv[md] = mfma32(o, half ? p1 : p0, dv[md]);
          });
    }
  });

  // ---- epilogue: lane l32 owns key row `key`; register (md, r) is head-dim
  // 32 md + 8 (r/4) + 4 hi + r%4.
  if (key >= kend) return;
  T* krow = reinterpret_cast<T*>(p.g.dk) + (varlen ? 0 : (int64_t)b * p.g.dk_stride_b) +
            (g.k_row0 + key) * p.g.dk_stride_t + (int64_t)hk * p.g.dk_stride_h;
  T* vrow = reinterpret_cast<T*>(p.g.dv) + (varlen ? 0 : (int64_t)b * p.g.dv_stride_b) +
            (g.k_row0 + key) * p.g.dv_stride_t + (int64_t)hk * p.g.dv_stride_h;
  auto put = [&](T* row, int md, const f32x16& x) {
#pragma unroll
    for (int gq = 0; gq < 4; ++gq)
      st_vec<v4>(row + 32 * md + 8 * gq + 4 * hi, v4{(T)x[4 * gq], (T)x[4 * gq + 1], (T)x[4 * gq + 2], (T)x[4 * gq + 3]});
  };
  const bool rot = a.rope_k && key < g.lk;
  const int pos = rope_krows(a, g, kw0).at(l32);
  // dk: pairs of head-dim blocks (md, md + MD/2: the rotation's partners),
  // scaled and rotated back. dK^T accumulated against the row-major q image,
  // which holds q * scale * log2(e): dk = scale * (dS^T q) = ln(2) * dK^T.
#pragma unroll
  for (int md = 0; md < MD / 2; ++md) {
    f32x16 x1 = dk[md] * kLn2, x2 = dk[md + MD / 2] * kLn2;
    if (rot) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int d = 32 * md + 8 * (r >> 2) + 4 * hi + (r & 3);
        const float cs = a.rope_cos[(int64_t)pos * (D / 2) + d], sn = a.rope_sin[(int64_t)pos * (D / 2) + d];
        const float y1 = x1[r] * cs + x2[r] * sn;
        x2[r] = x2[r] * cs - x1[r] * sn;
        x1[r] = y1;
      }
    }
    put(krow, md, x1);
    put(krow, md + MD / 2, x2);
  }
#pragma unroll
  for (int md = 0; md < MD; ++md) put(vrow, md, dv[md]);
}

// ---------------------------------------------------------------------------
// 3b. dk, dv at head_dim 256
// ---------------------------------------------------------------------------
// Four waves, one per SIMD: each owns 32 keys, pins their k and v operands
// (2 x 64 registers) and accumulates dK^T and dV^T (2 x 128 registers), and
// per query tile computes S, dP, P, dS and both products itself. Query tiles
// (64 KB of images each) move through a two-stage LDS ring, staged through
// registers in four parts issued between the four product phases. Workgroup
// (key block, hk * nsplit + split) walks its share of the (query head, query
// tile) pairs; with nsplit > 1 it writes fp32 partials.
constexpr int kWavesWide = 4;

template <typename T, int D, bool ALIBI, bool MASK, bool DS>
__global__ void __launch_bounds__(kWavesWide * 64, 1) bwd_dkv_wide_kernel(const BwdParams p) {
  // Operand reads in flight per product phase: one wave per SIMD, nothing
  // else hides their LDS latency (cfg3-shape dk/dv: 4.54 ms with about one in
  // flight, 3.04 with 4; 8 or more spill).
  constexpr int WL = 4;
  typedef typename Vec<T>::v8 v8;
  typedef typename Vec<T>::v4 v4;
  typedef QImg<T, D> QI;
  typedef KVImg<T, D> KI;
  constexpr int KS = D / 16;
  constexpr int MD = D / 32;
  constexpr int NTH = kWavesWide * 64;
  constexpr int LOADS = QI::NIMG * QI::CH / NTH;
  static_assert(QI::NIMG * QI::CH % NTH == 0, "tile must split over the threads");
  extern __shared__ __align__(16) unsigned char smem[];

  const goda_prefill_args& a = p.a;
  int bx, by, bz;
  chunked_order_3d(bx, by, bz);
  const int b = bz;
  const int hk = by / p.nsplit, split = by % p.nsplit;
  const SeqGeom g = seq_geom(b, a.seqlen_q, a.seqlen_k, a.cu_seqlens_q, a.cu_seqlens_k, a.seqused_k);
  const bool varlen = a.cu_seqlens_k != nullptr;
  const int kend = varlen ? g.lk : a.seqlen_k;  // rows this launch writes
  const int kv0 = bx * 32 * kWavesWide;
  if (kv0 >= kend) return;

  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63, l32 = lane & 31, hi = lane >> 5;
  const int kw0 = kv0 + 32 * wave;
  const int key = kw0 + l32;
  const int diag = g.lk - g.lq;
  const bool use_window = a.window_left >= 0 && (a.causal || g.lq == 1);

  v8 kf[KS], vf[KS];
  if (kw0 < g.lk) {
    const v8* img = reinterpret_cast<const v8*>(p.kvimg + kv_tile_index(b, kw0 / kBKV, hk, p.ntk, a.heads_kv) * KI::BYTES);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      kf[ks] = img[KI::KA + (2 * ks + hi) * kBKV + (l32 ^ (KI::SWZ * hi))];
      vf[ks] = img[KI::VA + (2 * ks + hi) * kBKV + (l32 ^ (KI::SWZ * hi))];
    }
  } else {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) kf[ks] = vf[ks] = v8{};
  }
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    asm volatile("" : "+v"(kf[ks]));
    asm volatile("" : "+v"(vf[ks]));
  }
  f32x16 dv[MD], dk[MD];
#pragma unroll
  for (int md = 0; md < MD; ++md) dv[md] = dk[md] = f32x16{};

  // Query tiles that can see a key of this workgroup, and this split's share.
  const int kv_last = min(kv0 + 32 * kWavesWide, g.lk) - 1;
  int i_lo = 0, i_hi = g.lq;
  if (a.causal) i_lo = max(0, kv0 - diag);
  if (use_window) i_hi = min(g.lq, kv_last + a.window_left - diag + 1);
  if (kv0 >= g.lk) i_hi = i_lo;
  const int qt_lo = i_lo / kQRows;
  const int nq = i_hi > i_lo ? (i_hi - 1) / kQRows + 1 - qt_lo : 0;
  const int n = p.group * nq;
  const int it0 = (int)((int64_t)n * split / p.nsplit);
  const int it1 = (int)((int64_t)n * (split + 1) / p.nsplit);

  auto src_of = [&](const QWalk& w) {
    const int64_t t = q_tile_index(b, qt_lo + w.q, hk * p.group + w.h, p.ntq, a.heads_q);
    return reinterpret_cast<const v8*>(p.qimg + t * QI::BYTES);
  };

  // Tiles move by direct global->LDS loads (dma_blocks): wave w
  // copies chunks [w LOADS 64, (w + 1) LOADS 64) of the image to the same
  // offsets of the stage, and wave 0's lanes below STAT_CH the statistics.
  // Tile it + 1 lands in stage (it + 1) % 2 during interval it (the barrier
  // opening the interval ends every read of tile it - 1 there), its blocks
  // issued between the score products; the barrier closing the interval
  // waits for the copies (vmcnt(0)).
  static_assert(QI::STAT_CH <= 64, "statistics fit one wave's copy");
  static_assert(2 * LOADS + 1 < 2 * KS, "every copy block issues between score products");
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  const unsigned lane_off = (unsigned)((wave_u * LOADS * 64 + lane) * 16);
  const unsigned stat_off = (unsigned)((QI::STAT + lane) * 16);
  auto tile_dma = [&](const QWalk& w, int it) {
    const unsigned long long base = (unsigned long long)(uintptr_t)src_of(w);
    const unsigned lds = (unsigned)(uintptr_t)(smem + (it % 2) * QI::BYTES);
    dma_span<LOADS>(lds + (unsigned)(wave_u * LOADS * 64 * 16), lane_off, base);
    if (wave_u == 0 && lane < QI::STAT_CH) dma_blocks<1>(lds + QI::STAT * 16, stat_off, base);
  };

  // dS tiles for the dq kernel that reads them (p.ds set): tile it's values
  // go out during tile it + 1's score products, one 2-byte store per register
  // after every other product, so the barrier closing an interval (which waits
  // for every access of the wave) does not wait on fresh stores; the last
  // tile's after the loop. A tile with no slot (no key visible to its rows)
  // goes to a sink nobody reads.
  constexpr bool kStoreDs = DS;
  static_assert(!kStoreDs || 2 * KS >= 32, "a store after every other score product");
  v8 dsp0{}, dsp1{};
  unsigned char* dsp_tile = kStoreDs ? p.ds + p.ds_sink : nullptr;
  const int ds_lane = (2 * (l32 >> 4) + ((l32 >> 2) & 1)) * 512 + 2 * ((l32 & 3) + 4 * ((l32 >> 3) & 1)) + 64 * hi;
  QWalk cu(it0, nq), nw(it0, nq);
  if (it0 < it1) tile_dma(cu, it0);
  dma_ring_barrier<0>();
  for (int it = it0; it < it1; ++it) {
    // The next tile is staged into the other stage (on the last tile: this
    // tile again, into a stage nobody reads), so the loop body is branch-free.
    if (it + 1 < it1) nw.next();
    const int hq = hk * p.group + cu.h;
    const int qt = qt_lo + cu.q;
    const int q0 = qt * kQRows;
    cu.next();
    const float slope2 = ALIBI ? a.alibi_slopes[hq] * kLog2e : 0.f;
    const v8* st = reinterpret_cast<const v8*>(smem + (it % 2) * QI::BYTES);
    const float* stat = reinterpret_cast<const float*>(st + QI::STAT);

    // The caller's mask bits of this key for the tile's 32 rows.
    uint32_t mword = 0;
    if (MASK && key < g.lk)
      mword = p.mask_t[b * p.mt_stride_b + hq * p.mt_stride_h + (int64_t)key * p.ntq + qt] >> (4 * hi);
    // S and dP: two independent accumulation chains, interleaved, starting
    // at -lse2 (+ the ALiBi bias) and -delta (the q image is prescaled, as in
    // the 8-wave kernel). Register r is row off = 8 (r/4) + r%4 past q0 + 4 hi.
    const int rel = q0 + 4 * hi;
    const float base = ALIBI ? slope2 * (float)(key - diag - rel) : 0.f;
    f32x16 s, dp;
#pragma unroll
    for (int gq = 0; gq < 4; ++gq) {
      const f32x4 l2 = ld_vec<f32x4>(stat + 8 * gq + 4 * hi);
      const f32x4 dl = ld_vec<f32x4>(stat + kQRows + 8 * gq + 4 * hi);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[4 * gq + e] = (ALIBI ? base - slope2 * (float)(8 * gq + e) : 0.f) - l2[e];
        dp[4 * gq + e] = -dl[e];
      }
    }
    // One wave per SIMD: nothing else hides a product's LDS operand latency,
    // so the reads run WL products ahead. S and dP stay in VGPRs
    // (mfma32_vgpr), where the VALU fills and reads them.
    mfma_vgpr_fill(s, dp);
    prefetched_products<2 * KS, WL, v8>(
        [&](int j) { return st[((j & 1) ? QI::GA : QI::QA) + (2 * (j >> 1) + hi) * kQRows + (l32 ^ (QI::SWZ * hi))]; },
        [&](int j, const v8& o) {
          if (j & 1)
            mfma32_vgpr(o, vf[j >> 1], dp);
          else
            mfma32_vgpr(o, kf[j >> 1], s);
        },
        [&](int j) {
          // The next tile's copies, one block after every other product, so
          // each issue (the copies of the CU's four waves queue at its
          // address unit) waits beside products already in flight rather
          // than in front of the phase (s_memtime probe: ~450 of ~5000
          // clocks a step; cfg3-shape backward kernels -9% in a same-box
          // A/B). On the last tile nw is this tile again: its copy lands in
          // the stage nobody reads, and the loop stays branch-free.
          if ((j & 1) && (j >> 1) < LOADS) {
            const int k = j >> 1;
            const unsigned lds = (unsigned)(uintptr_t)(smem + ((it + 1) % 2) * QI::BYTES);
            dma_blocks<1>(lds + (unsigned)((wave_u * LOADS + k) * 1024), lane_off,
                          (unsigned long long)(uintptr_t)src_of(nw) + k * 1024);
          }
          if (j == 2 * LOADS + 1 && wave_u == 0 && lane < QI::STAT_CH)
            dma_blocks<1>((unsigned)(uintptr_t)(smem + ((it + 1) % 2) * QI::BYTES) + QI::STAT * 16, stat_off,
                          (unsigned long long)(uintptr_t)src_of(nw));
          if constexpr (kStoreDs) {
            if (!(j & 1)) {
              const int r = j >> 1;
              *reinterpret_cast<T*>(dsp_tile + ds_lane + 128 * (r >> 2) + 16 * (r & 3)) = r < 8 ? dsp0[r] : dsp1[r - 8];
            }
          }
        });
    mfma_vgpr_drain(s, dp);

    // P and dS; visibility as a range of the register's row offset.
    int lo_lim = -1, hi_lim = g.lq - 1 - rel;
    if (a.causal) lo_lim = key - diag - rel;
    if (use_window) hi_lim = min(hi_lim, key + a.window_left - diag - rel);
    const bool key_ok = key < g.lk;
    // visible rows as bits; hidden entries replaced on the tiles that have
    // some (as in the 8-wave kernel)
    uint32_t vis = key_ok ? range_bits(lo_lim, hi_lim) : 0u;
    if (MASK) vis &= mword;
    float pr[16], ds[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      pr[r] = fast_exp2(s[r]);
      ds[r] = pr[r] * dp[r];
    }
    if (__builtin_amdgcn_ballot_w64(vis != ~0u) != 0) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int off = 8 * (r >> 2) + (r & 3);
        pr[r] = keep_if_bit(pr[r], vis, off, 0.f);
        ds[r] = keep_if_bit(ds[r], vis, off, 0.f);
      }
    }
    const v8 pp0 = pack8<v8, T>(pr), pp1 = pack8<v8, T>(pr + 8);
    const v8 d0 = pack8<v8, T>(ds), d1 = pack8<v8, T>(ds + 8);
    // this tile's dS and its slot (every tile a causal query tile can see;
    // the others are zero and have none)
    if constexpr (kStoreDs) {
      dsp0 = d0;
      dsp1 = d1;
      dsp_tile = kw0 < g.lk && (!a.causal || kw0 <= q0 + kQRows - 1 + diag) ? p.ds + ds_tile_offset(p, b, qt, kw0 / kBKV, hq)
                                                                               : p.ds + p.ds_sink;
    }
    prefetched_products<2 * MD, WL, v8>(
        [&](int j) {
          return tr_operand<v8>(reinterpret_cast<const unsigned char*>(st + QI::GA), lane, j & 1, j >> 1);
        },
        [&](int j, const v8& o) { dv[j >> 1] = mfma32(o, (j & 1) ? pp1 : pp0, dv[j >> 1]); });
    prefetched_products<2 * MD, WL, v8>(
        [&](int j) {
          return tr_operand<v8>(reinterpret_cast<const unsigned char*>(st + QI::QA), lane, j & 1, j >> 1);
        },
        [&](int j, const v8& o) { dk[j >> 1] = mfma32(o, (j & 1) ? d1 : d0, dk[j >> 1]); });
    dma_ring_barrier<0>();
  }

  if constexpr (kStoreDs) {
    if (it0 < it1) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        *reinterpret_cast<T*>(dsp_tile + ds_lane + 128 * (r >> 2) + 16 * (r & 3)) = r < 8 ? dsp0[r] : dsp1[r - 8];
    }
  }

  // ---- epilogue: lane l32 owns key row `key`; register (md, r) is head-dim
  // 32 md + 8 (r/4) + 4 hi + r%4.
  if (key >= kend) return;
  if (p.nsplit > 1) {
    const int64_t rows = (int64_t)a.batch * a.seqlen_k;
    const int64_t row = (int64_t)b * a.seqlen_k + key;
    float* pk = p.part + (((int64_t)(2 * split) * rows + row) * a.heads_kv + hk) * D;
    float* pv = p.part + (((int64_t)(2 * split + 1) * rows + row) * a.heads_kv + hk) * D;
#pragma unroll
    for (int md = 0; md < MD; ++md)
#pragma unroll
      for (int gq = 0; gq < 4; ++gq) {
        const int d0 = 32 * md + 8 * gq + 4 * hi;
        st_vec<f32x4>(pk + d0, f32x4{dk[md][4 * gq], dk[md][4 * gq + 1], dk[md][4 * gq + 2], dk[md][4 * gq + 3]});
        st_vec<f32x4>(pv + d0, f32x4{dv[md][4 * gq], dv[md][4 * gq + 1], dv[md][4 * gq + 2], dv[md][4 * gq + 3]});
      }
    return;
  }
  T* krow = reinterpret_cast<T*>(p.g.dk) + (varlen ? 0 : (int64_t)b * p.g.dk_stride_b) +
            (g.k_row0 + key) * p.g.dk_stride_t + (int64_t)hk * p.g.dk_stride_h;
  T* vrow = reinterpret_cast<T*>(p.g.dv) + (varlen ? 0 : (int64_t)b * p.g.dv_stride_b) +
            (g.k_row0 + key) * p.g.dv_stride_t + (int64_t)hk * p.g.dv_stride_h;
  auto put = [&](T* row, int md, const f32x16& x) {
#pragma unroll
    for (int gq = 0; gq < 4; ++gq)
      st_vec<v4>(row + 32 * md + 8 * gq + 4 * hi, v4{(T)x[4 * gq], (T)x[4 * gq + 1], (T)x[4 * gq + 2], (T)x[4 * gq + 3]});
  };
  const bool rot = a.rope_k && key < g.lk;
  const int pos = rope_krows(a, g, kw0).at(l32);
  // dk: one pair of head-dim blocks (md, md + MD/2: the rotation's partners)
  // at a time, scaled and rotated back.
  const float dks = kLn2;
#pragma unroll
  for (int md = 0; md < MD / 2; ++md) {
    f32x16 x1 = dk[md] * dks, x2 = dk[md + MD / 2] * dks;
    if (rot) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int d = 32 * md + 8 * (r >> 2) + 4 * hi + (r & 3);
        const float cs = a.rope_cos[(int64_t)pos * (D / 2) + d], sn = a.rope_sin[(int64_t)pos * (D / 2) + d];
        const float y1 = x1[r] * cs + x2[r] * sn;
        x2[r] = x2[r] * cs - x1[r] * sn;
        x1[r] = y1;
      }
    }
    put(krow, md, x1);
    put(krow, md + MD / 2, x2);
  }
#pragma unroll
  for (int md = 0; md < MD; ++md) put(vrow, md, dv[md]);
}

// Sum of the nsplit fp32 partials of dk and dv; dk scaled and rotated back.
// One thread per (key, 4 head-dims of the first half and their RoPE partners).
template <typename T, int D>
__global__ void __launch_bounds__(256) bwd_dkv_reduce_kernel(const BwdParams p) {
  typedef typename Vec<T>::v4 v4;
  const goda_prefill_args& a = p.a;
  const int b = blockIdx.z, hk = blockIdx.y;
  const SeqGeom g = seq_geom(b, a.seqlen_q, a.seqlen_k, a.cu_seqlens_q, a.cu_seqlens_k, a.seqused_k);
  const bool varlen = a.cu_seqlens_k != nullptr;
  const int kend = varlen ? g.lk : a.seqlen_k;
  constexpr int G = D / 8;  // groups of 4 head-dims in the first half
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int key = (int)(idx / G);
  const int d0 = (int)(idx % G) * 4;
  if (key >= kend) return;
  const int64_t rows = (int64_t)a.batch * a.seqlen_k;
  const int64_t row = (int64_t)b * a.seqlen_k + key;
  f32x4 k1 = {}, k2 = {}, v1 = {}, v2 = {};
  for (int s = 0; s < p.nsplit; ++s) {
    const float* pk = p.part + (((int64_t)(2 * s) * rows + row) * a.heads_kv + hk) * D;
    const float* pv = p.part + (((int64_t)(2 * s + 1) * rows + row) * a.heads_kv + hk) * D;
    k1 += ld_vec<f32x4>(pk + d0);
    k2 += ld_vec<f32x4>(pk + d0 + D / 2);
    v1 += ld_vec<f32x4>(pv + d0);
    v2 += ld_vec<f32x4>(pv + d0 + D / 2);
  }
  k1 *= kLn2;
  k2 *= kLn2;
  if (a.rope_k && key < g.lk) {
    const int key0 = (int)((int64_t)blockIdx.x * 256 / G);  // of the workgroup
    const int pos = rope_krows(a, g, key0).at(key - key0);
    const f32x4 cs = ld_vec<f32x4>(a.rope_cos + (int64_t)pos * (D / 2) + d0);
    const f32x4 sn = ld_vec<f32x4>(a.rope_sin + (int64_t)pos * (D / 2) + d0);
    const f32x4 y1 = k1 * cs + k2 * sn;
    const f32x4 y2 = k2 * cs - k1 * sn;
    k1 = y1;
    k2 = y2;
  }
  T* krow = reinterpret_cast<T*>(p.g.dk) + (varlen ? 0 : (int64_t)b * p.g.dk_stride_b) +
            (g.k_row0 + key) * p.g.dk_stride_t + (int64_t)hk * p.g.dk_stride_h;
  T* vrow = reinterpret_cast<T*>(p.g.dv) + (varlen ? 0 : (int64_t)b * p.g.dv_stride_b) +
            (g.k_row0 + key) * p.g.dv_stride_t + (int64_t)hk * p.g.dv_stride_h;
  st_vec<v4>(krow + d0, v4{(T)k1[0], (T)k1[1], (T)k1[2], (T)k1[3]});
  st_vec<v4>(krow + d0 + D / 2, v4{(T)k2[0], (T)k2[1], (T)k2[2], (T)k2[3]});
  st_vec<v4>(vrow + d0, v4{(T)v1[0], (T)v1[1], (T)v1[2], (T)v1[3]});
  st_vec<v4>(vrow + d0 + D / 2, v4{(T)v2[0], (T)v2[1], (T)v2[2], (T)v2[3]});
}

// ---------------------------------------------------------------------------
// 4. dq
// ---------------------------------------------------------------------------
template <typename T, int D, bool ALIBI, bool MASK>
__global__ void __launch_bounds__((DqShape<D>::WAVES * 64), (DqShape<D>::OCC)) bwd_dq_mfma_kernel(const BwdParams p) {
  constexpr int kWavesDq = DqShape<D>::WAVES;
  typedef typename Vec<T>::v8 v8;
  typedef typename Vec<T>::v4 v4;
  typedef QImg<T, D> QI;
  typedef KVImg<T, D> KI;
  constexpr int KS = D / 16;
  constexpr int MD = D / 32;
  constexpr int MT = kBKV / 32;   // 32-key blocks of S^T
  constexpr int KS2 = kBKV / 16;  // k-steps of dQ^T over keys
  // Operand reads in flight per product phase with one wave per SIMD (cfg3
  // shape: 2.51 -> 1.99 ms); two waves per SIMD hide each other's latency and
  // keep the scheduler's order (fenced prefetch there: +1-2%).
  constexpr int QL = DqShape<D>::WIDE ? 4 : 0;
  constexpr int LOADS = (KI::CHUNKS + kWavesDq * 64 - 1) / (kWavesDq * 64);
  extern __shared__ __align__(16) unsigned char smem[];

  const goda_prefill_args& a = p.a;
  const int hg = p.heads_per_wg;
  const int nslices = p.group / hg;
  const int qb_rows = (kWavesDq / hg) * 32;
  const int nqt = (a.seqlen_q + qb_rows - 1) / qb_rows;
  int pair, qi;
  chunked_order((int)blockIdx.x, nqt, (int)(gridDim.x / nqt), pair, qi);
  const int qt = nqt - 1 - qi;  // heavy causal tiles first
  const int b = pair / (a.heads_kv * nslices);
  const int rem = pair % (a.heads_kv * nslices);
  const int hk = rem / nslices;
  const int sl = rem % nslices;
  const SeqGeom g = seq_geom(b, a.seqlen_q, a.seqlen_k, a.cu_seqlens_q, a.cu_seqlens_k, a.seqused_k);
  const int qr0 = qt * qb_rows;
  if (qr0 >= g.lq) return;
  const bool varlen = a.cu_seqlens_q != nullptr;

  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63, l32 = lane & 31, hi = lane >> 5;
  const int hq = hk * p.group + sl * hg + (wave % hg);
  const int wrow0 = qr0 + (wave / hg) * 32;  // a 32-row query tile of the images
  const int diag = g.lk - g.lq;
  const bool use_window = a.window_left >= 0 && (a.causal || g.lq == 1);
  const int i = wrow0 + l32;
  const int iabs = diag + i;

  // B operands of this wave's 32 rows: q (rotated) and dO, plus statistics
  // (loaded after the first key tile's copy is issued, so the latencies
  // overlap).
  v8 qf[KS], gf[KS];
  float l2 = kNegInf, dl = 0.f;
  auto load_qg = [&]() {
    if (wrow0 < g.lq) {
      const v8* img = reinterpret_cast<const v8*>(p.qimg + q_tile_index(b, wrow0 / kQRows, hq, p.ntq, a.heads_q) * QI::BYTES);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        qf[ks] = img[QI::QA + (2 * ks + hi) * kQRows + (l32 ^ (QI::SWZ * hi))];
        gf[ks] = img[QI::GA + (2 * ks + hi) * kQRows + (l32 ^ (QI::SWZ * hi))];
      }
      const float* stat = reinterpret_cast<const float*>(img + QI::STAT);
      l2 = stat[l32];
      dl = stat[kQRows + l32];
    } else {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) qf[ks] = gf[ks] = v8{};
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      asm volatile("" : "+v"(qf[ks]));
      asm volatile("" : "+v"(gf[ks]));
    }
  };
  const float slope2 = ALIBI ? a.alibi_slopes[hq] * kLog2e : 0.f;
  // The caller's mask row of this lane's query row (rows past the sequence
  // read the last row's bits and are masked anyway): one word per key tile.
  const uint32_t* mrow = MASK ? mask_row(a, b, hq, min(i, g.lq - 1)) : nullptr;

  // key tiles visible to some row of the workgroup
  const int q_last = min(qr0 + qb_rows, g.lq) - 1;
  int kv_hi = g.lk;
  if (a.causal) kv_hi = min(kv_hi, diag + q_last + 1);
  int kv_lo = 0;
  if (use_window) kv_lo = max(0, diag + qr0 - a.window_left);
  const int j_lo = kv_lo / kBKV;
  const int j_hi = kv_hi > 0 ? (kv_hi + kBKV - 1) / kBKV : 0;
  const int n = max(0, j_hi - j_lo);

  f32x16 dq[MD];
#pragma unroll
  for (int md = 0; md < MD; ++md) dq[md] = f32x16{};

  // Tiles move by direct global->LDS loads (dma_span): wave w copies
  // chunks [w LOADS 64, (w + 1) LOADS 64) of the image to the same offsets
  // of the stage.
  static_assert(KI::CHUNKS % (kWavesDq * 64) == 0, "tile splits over the waves");
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  const unsigned lane_off = (unsigned)((wave_u * LOADS * 64 + lane) * 16);
  auto tile_dma = [&](int it) {
    const unsigned long long base =
        (unsigned long long)(uintptr_t)(p.kvimg + kv_tile_index(b, j_lo + it, hk, p.ntk, a.heads_kv) * KI::BYTES);
    const unsigned lds = (unsigned)(uintptr_t)(smem + (it % 2) * KI::BYTES) + (unsigned)(wave_u * LOADS * 64 * 16);
    dma_span<LOADS>(lds, lane_off, base);
  };
  // Block k of this wave's share of tile `it` (the one-wave kernel spreads a
  // tile's copies over the score products; cfg3-shape backward -3..-9%).
  constexpr bool kSpreadCopies = DqShape<D>::WIDE;
  static_assert(!kSpreadCopies || 2 * LOADS <= 2 * KS, "every copy block issues between score products");
  auto tile_dma_block = [&](int it, int k) {
    const unsigned long long base =
        (unsigned long long)(uintptr_t)(p.kvimg + kv_tile_index(b, j_lo + it, hk, p.ntk, a.heads_kv) * KI::BYTES);
    const unsigned lds = (unsigned)(uintptr_t)(smem + (it % 2) * KI::BYTES) + (unsigned)((wave_u * LOADS + k) * 1024);
    dma_blocks<1>(lds, lane_off, base + k * 1024);
  };
  static_assert(kBKV == 32, "one mask word per key tile");
  auto compute = [&](int it) {
    const int kvb = (j_lo + it) * kBKV;
    const v8* st = reinterpret_cast<const v8*>(smem + (it % 2) * KI::BYTES);
    const uint32_t mword = MASK ? mrow[j_lo + it] >> (4 * hi) : 0u;
    // S^T[keys][rows] and dP^T, starting at -lse2 (+ the ALiBi bias of
    // register r's key offset off = 8 (r/4) + r%4 past kvb + 4 hi) and at
    // -delta: the q operand is prescaled (scale * log2(e)), so they leave the
    // matrix core as the exponents of P and as dP - delta.
    const int rel = kvb + 4 * hi;
    const float base = ALIBI ? slope2 * (float)(rel - iabs) : 0.f;
    f32x16 s[MT], dp[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[mt][r] = (ALIBI ? base + slope2 * (float)(32 * mt + 8 * (r >> 2) + (r & 3)) : 0.f) - l2;
        dp[mt][r] = -dl;
      }
    if constexpr (QL > 0) {
      // One wave per SIMD (head_dim 256): S and dP stay in VGPRs
      // (mfma32_vgpr), where the VALU fills and reads them.
      mfma_vgpr_fill(s[0], dp[0]);
      prefetched_products<2 * KS, QL, v8>(
          [&](int j) { return st[((j & 1) ? KI::VA : KI::KA) + (2 * (j >> 1) + hi) * kBKV + (l32 ^ (KI::SWZ * hi))]; },
          [&](int j, const v8& o) {
            if (j & 1)
              mfma32_vgpr(o, gf[j >> 1], dp[0]);
            else
              mfma32_vgpr(o, qf[j >> 1], s[0]);
          },
          [&](int j) {
            // One wave per SIMD: the next tile's copies go out one block
            // after every other product, beside products in flight (on the
            // last tile: that tile again, into the stage nobody reads).
            if constexpr (kSpreadCopies)
              if ((j & 1) && (j >> 1) < LOADS) tile_dma_block(min(it + 1, n - 1), j >> 1);
          });
      mfma_vgpr_drain(s[0], dp[0]);
    } else {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          s[mt] = mfma32(st[KI::KA + (2 * ks + hi) * kBKV + 32 * mt + (l32 ^ (KI::SWZ * hi))], qf[ks], s[mt]);
          dp[mt] = mfma32(st[KI::VA + (2 * ks + hi) * kBKV + 32 * mt + (l32 ^ (KI::SWZ * hi))], gf[ks], dp[mt]);
        }
      lead_schedule<T, 2 * KS * MT, 4>();
    }
    // masks as ranges of the register's key offset off = key - (kvb + 4 hi)
    int hi_lim = g.lk - 1 - rel;
    if (a.causal) hi_lim = min(hi_lim, iabs - rel);
    const int lo_lim = use_window ? iabs - a.window_left - rel : 0;
    const bool row_ok = i < g.lq;
    // Visible keys as bits (bit off; one key tile is 32 keys); hidden
    // entries are replaced (exp2 of a hidden score may overflow) on the
    // tiles where some lane of the wave has one, a wave-uniform branch.
    static_assert(MT == 1, "one 32-bit visibility word per key tile");
    uint32_t vis = row_ok ? range_bits(lo_lim, hi_lim) : 0u;
    if (MASK) vis &= mword;
    float ds[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) ds[r] = fast_exp2(s[0][r]) * dp[0][r];
    if (__builtin_amdgcn_ballot_w64(vis != ~0u) != 0) {
#pragma unroll
      for (int r = 0; r < 16; ++r) ds[r] = keep_if_bit(ds[r], vis, 8 * (r >> 2) + (r & 3), 0.f);
    }
    v8 dsf[KS2];
    dsf[0] = pack8<v8, T>(ds);
    dsf[1] = pack8<v8, T>(ds + 8);
    // dQ^T += K^T dS^T
    if constexpr (QL > 0) {
      prefetched_products<KS2 * MD, QL, v8>(
          [&](int j) {
            return tr_operand<v8>(reinterpret_cast<const unsigned char*>(st + KI::KA), lane, j / MD, j % MD);
          },
          [&](int j, const v8& o) { dq[j % MD] = mfma32(o, dsf[j / MD], dq[j % MD]); });
    } else {
#pragma unroll
      for (int ks2 = 0; ks2 < KS2; ++ks2)
#pragma unroll
        for (int md = 0; md < MD; ++md)
          dq[md] = mfma32(tr_operand<v8>(reinterpret_cast<const unsigned char*>(st + KI::KA), lane, ks2, md), dsf[ks2], dq[md]);
      lead_schedule<T, KS2 * MD, 4>();
    }
  };

  // Tile it + 1 lands in stage (it + 1) % 2 during interval it: the
  // barrier opening the interval ends every read of tile it - 1 there, and
  // the one opening interval it + 1 waits for the copies (vmcnt(0)).
  if (n > 0) tile_dma(0);
  load_qg();
  for (int it = 0; it < n; ++it) {
    dma_ring_barrier<0>();
    if constexpr (!kSpreadCopies)
      if (it + 1 < n) tile_dma(it + 1);
    compute(it);
  }

  // ---- epilogue: lane l32 owns query row i; register (md, r) is head-dim
  // 32 md + 8 (r/4) + 4 hi + r%4.
  if (i >= g.lq) return;
#pragma unroll
  for (int md = 0; md < MD; ++md) dq[md] *= a.softmax_scale;
  if (a.rope_q) {
    const int pos = rope_qrows(a, g, wrow0).at(l32);
#pragma unroll
    for (int md = 0; md < MD / 2; ++md)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int d = 32 * md + 8 * (r >> 2) + 4 * hi + (r & 3);
        const float cs = a.rope_cos[(int64_t)pos * (D / 2) + d], sn = a.rope_sin[(int64_t)pos * (D / 2) + d];
        const float x1 = dq[md][r], x2 = dq[md + MD / 2][r];
        dq[md][r] = x1 * cs + x2 * sn;
        dq[md + MD / 2][r] = x2 * cs - x1 * sn;
      }
  }
  T* dqrow = reinterpret_cast<T*>(p.g.dq) + (varlen ? 0 : (int64_t)b * p.g.dq_stride_b) +
             (g.q_row0 + i) * p.g.dq_stride_t + (int64_t)hq * p.g.dq_stride_h;
#pragma unroll
  for (int md = 0; md < MD; ++md)
#pragma unroll
    for (int gq = 0; gq < 4; ++gq) {
      const int d0 = 32 * md + 8 * gq + 4 * hi;
      const v4 q4 = {(T)dq[md][4 * gq], (T)dq[md][4 * gq + 1], (T)dq[md][4 * gq + 2], (T)dq[md][4 * gq + 3]};
      st_vec<v4>(dqrow + d0, q4);
    }
}

// ---------------------------------------------------------------------------
// 4b. dq from stored dS tiles
// ---------------------------------------------------------------------------
// With p.ds set the dk/dv kernel stores every dS tile it forms, and dq is one
// product per tile instead of three (S, dP, dQ) plus the exp work:
//   dQ^T [d][rows] += K^T dS^T    A = K^T (transposing reads), B = dS^T (stored)
// Four waves, one per SIMD; a wave owns HW query heads of one 32-row query
// tile, so each K^T operand it reads serves HW products. The key tile (the k
// image only) and the waves' dS tiles move through a STAGES-deep LDS ring by
// direct copies issued STAGES - 1 tiles ahead.
constexpr int kWavesDqS = 4;
// Instances that take dq from stored dS tiles (query heads per wave HW; 0:
// none), and the largest dS store they may use (beyond it dq recomputes S and
// dP).
template <typename T, int D>
constexpr int kDsHeadsPerWave = D == 256 ? 2 : 0;
constexpr int64_t kDsMaxBytes = 8ll << 30;
template <typename T, int D, int HW>
struct DqSShape {
  static constexpr int KBYTES = D * 64;                   // k image of a 32-key tile
  static constexpr int STAGE = KBYTES + kWavesDqS * HW * 2048;
  static constexpr int STAGES = 4 * STAGE <= 160 * 1024 ? 4 : 3;
  static constexpr int KLOADS = KBYTES / 1024 / kWavesDqS;  // 1 KB blocks of k per wave
  static constexpr int LOADS = KLOADS + 2 * HW;             // copies per wave and tile
};

template <typename T, int D, int HW>
__global__ void __launch_bounds__(kWavesDqS * 64, 1) bwd_dq_ds_kernel(const BwdParams p) {
  typedef typename Vec<T>::v8 v8;
  typedef typename Vec<T>::v4 v4;
  typedef KVImg<T, D> KI;
  typedef DqSShape<T, D, HW> S;
  static_assert(sizeof(T) == 2, "16-bit operands");
  static_assert(KI::KA == 0 && S::KBYTES == KI::CH * 16, "the k image opens the key tile image");
  static_assert(S::KLOADS * kWavesDqS * 1024 == S::KBYTES, "the k image splits over the waves");
  static_assert(KI::BYTES >= HW * 2048, "a key tile image can stand in for a wave's dS tiles");
  constexpr int MD = D / 32;
  constexpr int NS = S::STAGES, kAhead = NS - 1;
  constexpr int L = 4;  // operand reads in flight (one wave per SIMD)
  extern __shared__ __align__(16) unsigned char smem[];

  const goda_prefill_args& a = p.a;
  const int hg = p.ds_hpw;   // query heads per workgroup, a multiple of HW
  const int nws = hg / HW;   // waves per query tile
  const int nslices = p.group / hg;
  const int qb_rows = (kWavesDqS / nws) * kQRows;
  const int nqt = (a.seqlen_q + qb_rows - 1) / qb_rows;
  int pair, qi;
  chunked_order((int)blockIdx.x, nqt, (int)(gridDim.x / nqt), pair, qi);
  const int qt = nqt - 1 - qi;  // heavy causal tiles first
  const int b = pair / (a.heads_kv * nslices);
  const int rem = pair % (a.heads_kv * nslices);
  const int hk = rem / nslices;
  const int sl = rem % nslices;
  const SeqGeom g = seq_geom(b, a.seqlen_q, a.seqlen_k, a.cu_seqlens_q, a.cu_seqlens_k, a.seqused_k);
  const int qr0 = qt * qb_rows;
  if (qr0 >= g.lq) return;
  const bool varlen = a.cu_seqlens_q != nullptr;

  const int tid = threadIdx.x;
  const int lane = tid & 63, l32 = lane & 31, hi = lane >> 5;
  const int wave_u = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hq0 = hk * p.group + sl * hg + (wave_u % nws) * HW;
  const int wrow0 = qr0 + (wave_u / nws) * kQRows;
  const int diag = g.lk - g.lq;
  const bool use_window = a.window_left >= 0 && (a.causal || g.lq == 1);

  // Key tiles [lo, hi) some row of r0..r1 sees: the workgroup's walk, and
  // the share of it this wave's tile covers (exactly the tiles the dk/dv
  // kernel stored for it).
  auto tiles = [&](int r0, int r1, int& lo, int& hi_) {
    int kv_hi = g.lk;
    if (a.causal) kv_hi = min(kv_hi, diag + r1 + 1);
    int kv_lo = 0;
    if (use_window) kv_lo = max(0, diag + r0 - a.window_left);
    lo = kv_lo / kBKV;
    hi_ = kv_hi > 0 ? (kv_hi + kBKV - 1) / kBKV : 0;
  };
  int j_lo, j_hi;
  tiles(qr0, min(qr0 + qb_rows, g.lq) - 1, j_lo, j_hi);
  const int n = max(0, j_hi - j_lo);
  int w_lo = 0, w_hi = 0;
  if (wrow0 < g.lq) tiles(wrow0, min(wrow0 + kQRows, g.lq) - 1, w_lo, w_hi);

  // Copies of tile it: this wave's quarter of the k image, and its HW dS
  // tiles (consecutive heads: contiguous); for a key tile outside the wave's
  // share the key tile image stands in (same copy count, never read).
  auto issue = [&](int it) {
    const int kt = j_lo + it;
    const unsigned char* kimg = p.kvimg + kv_tile_index(b, kt, hk, p.ntk, a.heads_kv) * KI::BYTES;
    const unsigned st = (unsigned)(uintptr_t)(smem + (it % NS) * S::STAGE);
    dma_span<S::KLOADS>(st + (unsigned)(wave_u * S::KLOADS * 1024), (unsigned)(lane * 16),
                        (unsigned long long)(uintptr_t)(kimg + wave_u * S::KLOADS * 1024));
    const bool mine = kt >= w_lo && kt < w_hi;
    const unsigned char* dsrc = mine ? p.ds + ds_tile_offset(p, b, wrow0 / kQRows, kt, hq0) : kimg;
    dma_span<2 * HW>(st + (unsigned)(S::KBYTES + wave_u * HW * 2048), (unsigned)(lane * 16),
                     (unsigned long long)(uintptr_t)dsrc);
  };

  f32x16 dq[HW][MD];
#pragma unroll
  for (int h = 0; h < HW; ++h)
#pragma unroll
    for (int md = 0; md < MD; ++md) dq[h][md] = f32x16{};

#pragma unroll
  for (int it = 0; it < kAhead; ++it)
    if (it < n) issue(it);
  for (int it = 0; it < n; ++it) {
    // tile it's copies landed: all but those of the (at most kAhead - 1)
    // tiles issued after it
    const int after = min(kAhead - 1, n - 1 - it);
    if (after >= 2)
      dma_ring_barrier<2 * S::LOADS>();
    else if (after == 1)
      dma_ring_barrier<S::LOADS>();
    else
      dma_ring_barrier<0>();
    // stage (it + kAhead) % NS was last read in interval it - 1
    if (it + kAhead < n) issue(it + kAhead);
    // A key tile outside this wave's share multiplies zeros (a branch around
    // the products makes the compiler keep the accumulators in VGPRs across
    // the loop and copy them into AGPRs for every product).
    const int kt = j_lo + it;
    const bool mine = kt >= w_lo && kt < w_hi;
    const unsigned char* st = smem + (it % NS) * S::STAGE;
    const unsigned char* dst = st + S::KBYTES + wave_u * HW * 2048;
    v8 dsb[HW][2];
#pragma unroll
    for (int h = 0; h < HW; ++h)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        dsb[h][s] = *reinterpret_cast<const v8*>(dst + h * 2048 + ((2 * s + hi) * 32 + l32) * 16);
        if (!mine) dsb[h][s] = v8{};
      }
    // j: k-step j / MD over the tile's keys, head-dim block j % MD
    prefetched_products<2 * MD, L, v8>(
        [&](int j) { return tr_operand<v8>(st, lane, j / MD, j % MD); },
        [&](int j, const v8& o) {
#pragma unroll
          for (int h = 0; h < HW; ++h) dq[h][j % MD] = mfma32(o, dsb[h][j / MD], dq[h][j % MD]);
        });
  }

  // ---- epilogue: lane l32 owns query row i; register (md, r) is head-dim
  // 32 md + 8 (r/4) + 4 hi + r%4.
  const int i = wrow0 + l32;
  if (i >= g.lq) return;
  const int pos = rope_qrows(a, g, wrow0).at(l32);
#pragma unroll
  for (int h = 0; h < HW; ++h) {
#pragma unroll
    for (int md = 0; md < MD; ++md) dq[h][md] *= a.softmax_scale;
    if (a.rope_q) {
#pragma unroll
      for (int md = 0; md < MD / 2; ++md)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int d = 32 * md + 8 * (r >> 2) + 4 * hi + (r & 3);
          const float cs = a.rope_cos[(int64_t)pos * (D / 2) + d], sn = a.rope_sin[(int64_t)pos * (D / 2) + d];
          const float x1 = dq[h][md][r], x2 = dq[h][md + MD / 2][r];
          dq[h][md][r] = x1 * cs + x2 * sn;
          dq[h][md + MD / 2][r] = x2 * cs - x1 * sn;
        }
    }
    T* dqrow = reinterpret_cast<T*>(p.g.dq) + (varlen ? 0 : (int64_t)b * p.g.dq_stride_b) +
               (g.q_row0 + i) * p.g.dq_stride_t + (int64_t)(hq0 + h) * p.g.dq_stride_h;
#pragma unroll
    for (int md = 0; md < MD; ++md)
#pragma unroll
      for (int gq = 0; gq < 4; ++gq) {
        const int d0 = 32 * md + 8 * gq + 4 * hi;
        const v4 q4 = {(T)dq[h][md][4 * gq], (T)dq[h][md][4 * gq + 1], (T)dq[h][md][4 * gq + 2], (T)dq[h][md][4 * gq + 3]};
        st_vec<v4>(dqrow + d0, q4);
      }
  }
}

int gcd_int(int x, int y) {
  while (y) {
    const int t = x % y;
    x = y;
    y = t;
  }
  return x;
}

template <typename T, int D, bool ALIBI, bool MASK>
hipError_t launch_main(const BwdParams& p, hipStream_t s) {
  const goda_prefill_args& a = p.a;
  hipError_t e;
  if ((e = record_timing(p.g.timing_begin, s)) != hipSuccess) return e;
  if (a.seqlen_k > 0) {
    if constexpr (DqShape<D>::WIDE) {
      auto kern = bwd_dkv_wide_kernel<T, D, ALIBI, MASK, false>;
      if constexpr (kDsHeadsPerWave<T, D> > 0)
        if (p.ds) kern = bwd_dkv_wide_kernel<T, D, ALIBI, MASK, true>;
      const size_t lds = 2 * (size_t)QImg<T, D>::BYTES;
      if ((e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)) != hipSuccess)
        return e;
      const dim3 grid((a.seqlen_k + 32 * kWavesWide - 1) / (32 * kWavesWide), a.heads_kv * p.nsplit, a.batch);
      kern<<<grid, kWavesWide * 64, lds, s>>>(p);
      if ((e = hipGetLastError()) != hipSuccess) return e;
      if (p.nsplit > 1) {
        const int64_t threads = (int64_t)a.seqlen_k * (D / 8);
        bwd_dkv_reduce_kernel<T, D><<<dim3((unsigned)((threads + 255) / 256), a.heads_kv, a.batch), 256, 0, s>>>(p);
        if ((e = hipGetLastError()) != hipSuccess) return e;
      }
    } else {
      auto kern = bwd_dkv_mfma_kernel<T, D, ALIBI, MASK>;
      const size_t lds = (size_t)DkvSmem<T, D>::BYTES;
      if ((e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)) != hipSuccess)
        return e;
      const dim3 grid((a.seqlen_k + 127) / 128, a.heads_kv, a.batch);
      kern<<<grid, kWavesKv * 64, lds, s>>>(p);
      if ((e = hipGetLastError()) != hipSuccess) return e;
    }
  }
  constexpr int HW = kDsHeadsPerWave<T, D>;
  if constexpr (HW > 0) {
    if (p.ds && a.seqlen_q > 0) {
      // dq from the dS tiles the dk/dv kernel stored (it ran above: it needs
      // seqlen_k > 0, and with seqlen_k = 0 there are no key tiles to walk)
      auto kern = bwd_dq_ds_kernel<T, D, HW>;
      typedef DqSShape<T, D, HW> S;
      const size_t lds = (size_t)S::STAGES * S::STAGE;
      if ((e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)) != hipSuccess)
        return e;
      const int nws = p.ds_hpw / HW;
      const int qb_rows = (kWavesDqS / nws) * kQRows;
      const int nqt = (a.seqlen_q + qb_rows - 1) / qb_rows;
      const int64_t nblk = (int64_t)nqt * a.batch * a.heads_kv * (p.group / p.ds_hpw);
      if (nblk > 0x7fffffff) return hipErrorInvalidValue;
      kern<<<dim3((unsigned)nblk), kWavesDqS * 64, lds, s>>>(p);
      if ((e = hipGetLastError()) != hipSuccess) return e;
      return record_timing(p.g.timing_end, s);
    }
  }
  if (a.seqlen_q > 0) {
    auto kern = bwd_dq_mfma_kernel<T, D, ALIBI, MASK>;
    const size_t lds = 2 * (size_t)KVImg<T, D>::BYTES;
    if ((e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)) != hipSuccess)
      return e;
    constexpr int kWavesDq = DqShape<D>::WAVES;
    const int qb_rows = (kWavesDq / p.heads_per_wg) * 32;
    const int nqt = (a.seqlen_q + qb_rows - 1) / qb_rows;
    const int64_t nblk = (int64_t)nqt * a.batch * a.heads_kv * (p.group / p.heads_per_wg);
    if (nblk > 0x7fffffff) return hipErrorInvalidValue;
    kern<<<dim3((unsigned)nblk), kWavesDq * 64, lds, s>>>(p);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  return record_timing(p.g.timing_end, s);
}

// Workgroups per key block of the head_dim-256 dk/dv kernel: enough that the
// grid holds ~1024 workgroups (MQA and short batches have few key blocks, and
// causal key blocks differ in work by up to the sequence length), at most 8
// and at most the (query head, query tile) pairs a key block can see.
int dkv_splits(const goda_prefill_args& a) {
  if (a.head_dim < 256 || a.heads_kv <= 0) return 1;
  const int64_t wgs = (int64_t)((a.seqlen_k + 32 * kWavesWide - 1) / (32 * kWavesWide)) * a.heads_kv * a.batch;
  if (wgs <= 0) return 1;
  int64_t ns = (1024 + wgs - 1) / wgs;
  const int64_t pairs = (int64_t)(a.heads_q / a.heads_kv) * ((a.seqlen_q + kQRows - 1) / kQRows);
  ns = std::min<int64_t>(ns, std::max<int64_t>(1, pairs));
  return (int)std::min<int64_t>(ns, 8);
}

int64_t align256(int64_t x) { return (x + 255) / 256 * 256; }

// Workspace: query-tile images, key-tile images, the dk/dv partials, the
// key-major mask words, the dS tiles.
struct BwdLayout {
  int64_t kvimg, part, mask, ds, total;
  int64_t ds_per_b, ds_sink;
  int ds_c, ds_tri;
};
template <typename T, int D>
BwdLayout bwd_layout(const goda_prefill_args& a) {
  BwdLayout l{};
  const int ntq = (a.seqlen_q + kQRows - 1) / kQRows;
  const int ntk = (a.seqlen_k + kBKV - 1) / kBKV;
  l.kvimg = (int64_t)a.batch * ntq * a.heads_q * QImg<T, D>::BYTES;
  l.part = l.kvimg + (int64_t)a.batch * ntk * a.heads_kv * KVImg<T, D>::BYTES;
  l.mask = l.part;
  const int ns = dkv_splits(a);
  if (ns > 1) l.mask += (int64_t)ns * 2 * a.batch * a.seqlen_k * a.heads_kv * D * 4;
  l.ds = l.total = l.mask;
  if (a.mask_bits) {
    l.mask = align256(l.mask);
    l.ds = l.total = l.mask + 4 * bwd_mask_t_words(a);
  }
  constexpr int HW = kDsHeadsPerWave<T, D>;
  const int group = a.heads_kv > 0 ? a.heads_q / a.heads_kv : 0;
  if (HW > 0 && group % HW == 0 && ntq > 0 && ntk > 0) {
    // causal batches of equal lengths keep only the visible key tiles
    const bool varlen = a.cu_seqlens_q != nullptr || a.cu_seqlens_k != nullptr;
    const int diag = a.seqlen_k - a.seqlen_q;
    l.ds_tri = a.causal && !varlen && diag >= 0;
    l.ds_c = l.ds_tri ? (diag + kBKV - 1) / kBKV : 0;
    l.ds_per_b = ds_row_off(ntq, ntk, l.ds_c, l.ds_tri != 0);
    const int64_t bytes = (int64_t)a.batch * l.ds_per_b * a.heads_q * 2048;
    if (bytes <= kDsMaxBytes) {
      l.ds = align256(l.total);
      l.ds_sink = bytes;
      l.total = l.ds + bytes + 2048;
    } else {
      l.ds = -1;
    }
  } else {
    l.ds = -1;
  }
  return l;
}

template <typename T, int D>
int64_t workspace_bytes_d(const goda_prefill_args& a) {
  return bwd_layout<T, D>(a).total;
}

template <typename T, int D>
hipError_t launch_d(BwdParams p, hipStream_t s) {
  const goda_prefill_args& a = p.a;
  const BwdLayout l = bwd_layout<T, D>(a);
  p.ntq = (a.seqlen_q + kQRows - 1) / kQRows;
  p.ntk = (a.seqlen_k + kBKV - 1) / kBKV;
  p.heads_per_wg = gcd_int(p.group, DqShape<D>::WAVES);
  p.qimg = reinterpret_cast<unsigned char*>(p.g.workspace);
  p.kvimg = p.qimg + l.kvimg;
  p.nsplit = dkv_splits(a);
  p.part = reinterpret_cast<float*>(p.qimg + l.part);
  if (l.ds >= 0) {
    p.ds = p.qimg + l.ds;
    p.ds_per_b = l.ds_per_b;
    p.ds_sink = l.ds_sink;
    p.ds_c = l.ds_c;
    p.ds_tri = l.ds_tri;
    p.ds_hpw = gcd_int(p.group, kWavesDqS * kDsHeadsPerWave<T, D>);
  }
  hipError_t e;
  if (a.mask_bits) {
    p.mask_t = reinterpret_cast<uint32_t*>(p.qimg + l.mask);
    if ((e = launch_bwd_mask_t(p, s)) != hipSuccess) return e;
  }
  if (p.ntq > 0) {
    pack_q_bwd_kernel<T, D><<<dim3(p.ntq, a.heads_q, a.batch), 256, 0, s>>>(p);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  if (p.ntk > 0) {
    pack_kv_bwd_kernel<T, D><<<dim3(p.ntk, a.heads_kv, a.batch), 256, 0, s>>>(p);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  if (a.mask_bits)
    return a.alibi_slopes ? launch_main<T, D, true, true>(p, s) : launch_main<T, D, false, true>(p, s);
  return a.alibi_slopes ? launch_main<T, D, true, false>(p, s) : launch_main<T, D, false, false>(p, s);
}

template <typename T>
hipError_t launch_t(const BwdParams& p, hipStream_t s) {
  if (p.a.head_dim == 64) return launch_d<T, 64>(p, s);
  if (p.a.head_dim == 128) return launch_d<T, 128>(p, s);
  if (p.a.head_dim == 256) return launch_d<T, 256>(p, s);
  return hipErrorNotSupported;
}

}  // namespace

int64_t bwd_mask_t_words(const goda_prefill_args& a) {
  if (!a.mask_bits) return 0;
  const int64_t bm = a.mask_stride_b ? a.batch : 1, hm = a.mask_stride_h ? a.heads_q : 1;
  return bm * hm * a.seqlen_k * ((a.seqlen_q + kQRows - 1) / kQRows);
}

hipError_t launch_bwd_mask_t(BwdParams& p, hipStream_t s) {
  const goda_prefill_args& a = p.a;
  const int64_t hm = a.mask_stride_h ? a.heads_q : 1;
  p.mt_stride_h = a.mask_stride_h ? (int64_t)a.seqlen_k * p.ntq : 0;
  p.mt_stride_b = a.mask_stride_b ? hm * a.seqlen_k * p.ntq : 0;
  const int64_t threads = (int64_t)p.ntq * ((a.seqlen_k + 31) / 32);
  if (threads <= 0) return hipSuccess;
  const dim3 grid((unsigned)((threads + 255) / 256), (unsigned)hm, a.mask_stride_b ? a.batch : 1);
  bwd_mask_t_kernel<<<grid, 256, 0, s>>>(p);
  return hipGetLastError();
}

int64_t prefill_bwd_mfma_workspace_bytes(const goda_prefill_args& a) {
  if (a.head_dim == 64) return workspace_bytes_d<bf16, 64>(a);
  if (a.head_dim == 128) return workspace_bytes_d<bf16, 128>(a);
  return workspace_bytes_d<bf16, 256>(a);
}

hipError_t launch_prefill_bwd_mfma(BwdParams p, hipStream_t s) {
  if (p.a.dtype == GODA_DTYPE_BF16) return launch_t<bf16>(p, s);
  if (p.a.dtype == GODA_DTYPE_F16) return launch_t<f16>(p, s);
  return hipErrorNotSupported;
}

}  // namespace goda
