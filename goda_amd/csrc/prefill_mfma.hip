// Causal / non-causal GQA-MQA prefill attention on gfx950 matrix cores
// (bf16 or fp16 operands, fp32 accumulation).
//
// Two launches per call:
//   1. pack_kv_kernel reads every K/V row of a KV head once, rotates K (RoPE,
//      half-split pairing of mint/nn/pos.py:90-98) and writes, per tile of BKV
//      keys, the exact byte image the attention kernel wants in LDS:
//        K' image   [D/8 chunks][BKV keys]    of 16-byte chunks (8 elements)
//        V^T image  [BKV/8 chunks][D dims]    of 16-byte chunks
//      "Chunk-column-major": the 16 lanes of a quarter-wave that read one
//      MFMA operand column touch 256 consecutive bytes, so LDS reads are
//      conflict-free without padding or XOR swizzles, and every operand
//      address is one per-lane base plus a compile-time offset.
//      Inside each 16-key group of the V^T image the keys are stored in the
//      order the P^T register fragment holds them (kPermKey), so one 16-byte
//      read yields a whole MFMA operand.
//   2. prefill_fa_kernel: one workgroup (8 waves, two per SIMD) per
//      (query tile, query-head slice, sequence). All waves
//      belong to query heads of ONE KV head, so every K/V tile streamed into
//      LDS serves the whole query-head group ("read once per group"). Tiles
//      move through a ring of 4 LDS stages: during the interval that reads
//      tiles j and j+1, each wave moves its share of tile j+3 into a free
//      stage (kStages below), for 16-bit tiles by direct global->LDS loads
//      (global_load_lds_dwordx4) issued from inline asm and waited for at the
//      ring barrier (the compiler's own form of those loads makes it wait for
//      them before every LDS operand read), for fp32 tiles through registers.
//
// Per wave and KV tile (32x32x16 MFMA, 32*NT query rows of one head):
//   S^T[kv][q] = K'[kv][d] . Q^T[d][q] - m[q] + bias[kv][q]
//                                          A = K' (LDS), B = Q^T (registers)
//   O^T[d][q] += V^T[d][kv] . P^T[kv][q]   A = V^T (LDS), B = P^T (registers)
// Q^T holds q * scale * log2(e) and the accumulators start at the row's
// reference max m (negated) plus the ALiBi bias, so the scores leave the
// MFMA as the exponents of P: the softmax spends no VALU instruction on
// scaling, biasing or shifting them (every VALU instruction of the softmax
// lengthens the interval: the two waves of a SIMD share its VALU, and the
// row sums' packed dot products wait out the other wave's MFMAs).
// Every query row lives in one lane pair (l, l^32), so the row max needs one
// permlane32 swap and any rescale is lane-local.
// Rescaling is lazy: a row's reference max only moves (and its O and l are
// rescaled) when the tile max exceeds it by more than kRescaleThresh (log2
// units), so O is untouched by the VALU on almost every tile. The result is
// exact either way: numerator and denominator share the reference max.
//
// MFMA 32x32 accumulator layout (gfx9 family): lane l, register r holds
// row 8*(r/4) + 4*(l/32) + r%4, column l%32. The K dimension of the A and B
// operands uses the same (lane half, element) assignment, so the P^T operand
// is the S^T accumulator re-packed in place.

#include <algorithm>
#include <mutex>

#include "common.h"
#include "launch.h"
#include "mfma_common.h"

namespace goda {
namespace {

// Rescale margin in log2 units: P entries stay <= 2^margin. fp16 operands
// hold P up to 2^14 (largest finite 65504). bf16 and fp32 share fp32's
// exponent range, and the products and row sums accumulate in fp32: 2^60
// leaves a row of 2^20 keys with values up to 1e4 some 2^30 below fp32's
// largest value. ALiBi moves the row max along the keys, so a wider margin
// saves rescales: cfg3 kernel (bf16) 915.8 us at 8, 907.5 at 12, 904.9 at 14
// in one same-box A/B; 954.2 at 14, 936.8 at 24, 932.1 at 30 in another;
// 942.6 at 30, 928.2 at 60 in a third; cfg2 unchanged.
template <typename T>
constexpr float kRescaleThresh = std::is_same<T, f16>::value ? 14.0f : 60.0f;


template <typename T, int D, int BKV, int WAVES>
struct TileGeom {
  static constexpr int CHB = (int)sizeof(typename Vec<T>::v8);  // bytes per 8-element chunk
  static constexpr int K_CHUNKS = D / 8 * BKV;  // 16-byte chunks of the K' image
  static constexpr int V_CHUNKS = BKV / 8 * D;
  static constexpr int BYTES = (K_CHUNKS + V_CHUNKS) * CHB;
  static constexpr int LOADS_PER_LANE = (K_CHUNKS + V_CHUNKS) / (64 * WAVES);  // 16-byte loads
  static_assert((K_CHUNKS + V_CHUNKS) % (64 * WAVES) == 0, "tile must split evenly over the waves");
};
// LDS ring of kStages tile stages: interval j reads tiles j (V) and j+1 (K)
// and writes tile j + kAhead; a workgroup barrier opens every kBarrierEvery-th
// interval. Safe when kAhead >= kBarrierEvery + 1 (every tile read was
// written before the last barrier) and kStages >= kAhead + kBarrierEvery (no
// stage is overwritten before every wave is past its last read).
// (4 stages, tiles 3 intervals ahead, a barrier every interval: the extra
// stage of prefetch is worth 1.5-2% at D = 256; halving the barriers with 5
// stages changed nothing measurable.)
constexpr int kStages = 4, kAhead = 3, kBarrierEvery = 1;
static_assert(kAhead >= kBarrierEvery + 1 && kStages >= kAhead + kBarrierEvery, "ring shape");
// Packed batches: the query tiles of each (sequence, head slice) pair are dealt
// round-robin over a group of this many XCDs (see the workgroup order below).
// Kernel time over five packed batches (cfg5's and three other draws of 16
// lengths in [128, 4096], one of 16 in [512, 8192]): 8 XCDs 3379 us, groups
// of 4 3391, of 2 3752, whole pairs per XCD 4024.
constexpr int kVarlenXcdGroup = 8;
// Packed batches of at most 64 sequences: the shortest kPackedTailNum /
// kPackedTailDen of the sequences are dealt level by level at the end of each
// XCD's walk (see grid_item). cfg5's packed prefill kernel, same-box A/B:
// a quarter 517.6 -> 504.5 us, a half 507.2, three quarters 508.3, all 523.2
// (the more sequences interleave, the more of their K/V tiles miss L2; a
// schedule simulation without that cost gave 539 -> 521 / 505 / 500 / 500).
constexpr int kPackedTailNum = 1, kPackedTailDen = 4;
// Packed batches whose longest sequence has at most this many query tiles per
// XCD: tile qt of the pair at place i of the walk goes to XCD (qt - i) mod 8.
// With qt mod 8 the first XCDs took nearly all tiles of short sequences (of a
// batch with one tile each, XCD 0 all). Packed prefill, us, before / now, 4
// to 48 sequences of 1/16 .. all of the longest, causal:
//   longest, tiles      1          4          8         16         24        32
//   16/16 D=64    275 / 191  220 / 169  147 / 129  225 / 206  247 / 248  502 / 458
//   32/8 D=128    143 / 100  164 / 121  195 / 172  277 / 258  226 / 231  376 / 359
//   8/1 D=256      34 /  21   42 /  28   47 /  41   77 /  70   85 /  89  120 / 106
// (24 and 32 tiles turned as well: the tail's order, below, is then lost.)
constexpr int kRotateTiles = 2;
// Move each tile in two halves through half the staging registers: register
// relief for D = 256 (whose two-waves-per-SIMD form is at the limit), and at
// D = 128 half of the LDS stores move from the end of the interval, where
// the ring barrier waits for them, to its middle (cfg2 +2-4%).
template <int D>
constexpr bool kSplitStaging = D >= 128;

// Head dims whose dense batches take the persistent grid (prefill_fa_kernel;
// head_dim 256 has no registers to spare for it, nor have the instances with
// a caller's mask).
template <int D>
constexpr bool kPersistent = D <= 128;

// With a caller's mask: key tiles that no row of the workgroup sees are not
// walked. The pre-pass marks, per 32 query rows, the tiles that one of them sees
// (mark_tiles); a workgroup lists those of its rows behind the LDS ring, for up
// to kListTiles tiles (more: all are walked).
constexpr int kListTiles = 4096;
constexpr int kListBytes = kListTiles * 2;

// Split keys (KSPLIT instances): an item's key tiles are cut into pieces that
// workgroups of their own walk, for dense batches whose items are too few to
// fill the GPU (see key_pieces). A piece of a cut item leaves its
// sums in the workspace, and merge_pieces_kernel adds them: rows' O^T as
// 16-byte quarters of 8 head-dims, [D/4][256 rows] per piece (a wave stores 1 KB
// runs), then m and l of the 256 rows.
constexpr int kPieceRows = 256;  // 8 waves of 32 rows
template <int D>
constexpr int64_t kPieceBytes = (int64_t)kPieceRows * (D + 2) * 4;
constexpr int kCus = 256;
constexpr int kMostPieceBatch = 64;

// Key tiles per piece for this launch: p.piece_tiles, or (lengths on the
// device, of at most 64 sequences: key_pieces) an equal share of all items'
// tiles, at least what keeps the longest sequence to p.ksplit pieces.
__device__ __forceinline__ int piece_tiles(const PrefillParams& p, int bkv) {
  if (p.piece_tiles > 0) return p.piece_tiles;
  const goda_prefill_args& a = p.a;
  const int lane = threadIdx.x & 63;
  int sum = lane < a.batch ? (max(0, min(a.seqused_k[lane], a.seqlen_k)) + bkv - 1) / bkv : 0;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) sum += __shfl_xor(sum, o, 64);
  const long long tiles = (long long)sum * p.qtiles * a.heads_kv * (p.group / p.heads_per_wg);
  const int share = (int)min((long long)p.ntiles_k, (tiles + kCus - 1) / kCus);
  return max(max(share, p.min_piece), (p.ntiles_k + p.ksplit - 1) / p.ksplit);
}
// Pieces of an item of n tiles, of equal length; a remainder of at most a
// quarter piece makes them longer instead of one more.
__device__ __forceinline__ int piece_count(int n, int per, int most) {
  return max(1, min(most, (n + per - 1 - per / 4) / per));
}

// Index of workspace tile j of sequence b, KV head hk.
__device__ __forceinline__ int64_t ws_tile(int b, int j, int hk, int ntiles, int hkv) {
  return ((int64_t)b * ntiles + j) * hkv + hk;
}

// Bits of the caller's boolean mask for one key tile of one query row: 64
// keys in one 8-byte word, 32 in a 4-byte one.
template <int BKV>
struct MaskWord;
template <>
struct MaskWord<64> {
  typedef uint64_t t;
  static constexpr t kAll = ~0ull;
};
template <>
struct MaskWord<32> {
  typedef uint32_t t;
  static constexpr t kAll = ~0u;
};

// Marks of the caller's mask, [sequence][query head][32 query rows][64 key
// tiles], one bit a tile; dimensions that the mask broadcasts have size 1.
struct Marks {
  int batch, heads, blocks, words;
};
__host__ __device__ __forceinline__ Marks marks_of(const goda_prefill_args& a, int ntiles) {
  return Marks{a.mask_stride_b ? a.batch : 1, a.mask_stride_h ? a.heads_q : 1, a.mask_stride_q ? (a.seqlen_q + 31) / 32 : 1,
               (ntiles + 63) / 64};
}
// One wave: the marks of block `u` of 32 rows. A lane holds a tile, so that a
// row's words are one run of memory, and eight rows are in flight.
template <int BKV>
__device__ __forceinline__ void mark_tiles(const PrefillParams& p, int64_t u) {
  typedef typename MaskWord<BKV>::t mword_t;
  const goda_prefill_args& a = p.a;
  const Marks k = marks_of(a, p.ntiles_k);
  if (u >= (int64_t)k.batch * k.heads * k.blocks) return;
  const int lane = threadIdx.x & 63;
  const int block = (int)(u % k.blocks);
  const int h = (int)(u / k.blocks % k.heads), b = (int)(u / k.blocks / k.heads);
  const uint32_t* rows = mask_row(a, b, h, 32 * block);
  const int last = a.mask_stride_q ? min(32, a.seqlen_q - 32 * block) - 1 : 0;
  for (int w = 0; w < k.words; ++w) {
    const int t = min(64 * w + lane, p.ntiles_k - 1);
    mword_t any = 0;
    for (int r0 = 0; r0 <= last; r0 += 8) {
#pragma unroll
      for (int r = 0; r < 8; ++r)
        any |= reinterpret_cast<const mword_t*>(rows + min(r0 + r, last) * a.mask_stride_q)[t];
    }
    const uint64_t m = __builtin_amdgcn_ballot_w64(any != 0 && 64 * w + lane < p.ntiles_k);
    if (lane == 0) p.marks[u * k.words + w] = m;
  }
}

// ---------------------------------------------------------------------------
// 1. pack K (rotated) and V^T into tile images; with a caller's mask, blocks
// past the tiles mark what its rows see
// ---------------------------------------------------------------------------
template <typename T, int D, int BKV, bool MASK>
__global__ void __launch_bounds__(256) pack_kv_kernel(const PrefillParams p) {
  typedef typename Vec<T>::v8 v8;
  typedef TileGeom<T, D, BKV, 1> TG;
  const goda_prefill_args& a = p.a;
  const int j = blockIdx.x;
  const int hk = blockIdx.y;
  const int b = blockIdx.z;
  if constexpr (MASK) {
    if (j >= p.ntiles_k) {
      const int64_t group = ((int64_t)b * a.heads_kv + hk) * (gridDim.x - p.ntiles_k) + j - p.ntiles_k;
      mark_tiles<BKV>(p, 4 * group + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
      return;
    }
  }
  const SeqGeom g = seq_geom(b, a.seqlen_q, a.seqlen_k, a.cu_seqlens_q, a.cu_seqlens_k,
                             a.seqused_k);
  const int kv0 = j * BKV;
  if (kv0 >= g.lk) return;

  unsigned char* tile = reinterpret_cast<unsigned char*>(a.workspace) +
                        ws_tile(b, j, hk, p.ntiles_k, a.heads_kv) * TG::BYTES;
  v8* kimg = reinterpret_cast<v8*>(tile);
  v8* vimg = reinterpret_cast<v8*>(tile + TG::K_CHUNKS * TG::CHB);

  const T* kbase = reinterpret_cast<const T*>(a.k) +
                   (a.cu_seqlens_k ? 0 : (int64_t)b * a.k_stride_b) + (int64_t)hk * a.k_stride_h;
  const T* vbase = reinterpret_cast<const T*>(a.v) +
                   (a.cu_seqlens_k ? 0 : (int64_t)b * a.v_stride_b) + (int64_t)hk * a.v_stride_h;

  // One row-major staging buffer, used for K then for V; +8 elements per row
  // keep the column reads of the transposes off a single bank.
  __shared__ __align__(16) T rows[BKV][D + 8];
  __shared__ float inv_rms[BKV];
  const int tid = threadIdx.x;
  constexpr int HALF8 = D / 16;  // 8-element chunks per half row
  RopePos rope{};
  if (a.rope_k) rope = rope_krows(a, g, kv0);

  if (a.k_norm_weight) {
    // Fused QK-RMSNorm: raw rows staged first, then each row's scale, then
    // normalisation and rotation in fp32 in place (one rounding).
    for (int idx = tid; idx < BKV * (D / 8); idx += 256) {
      const int r = idx / (D / 8);
      const int c = (idx % (D / 8)) * 8;
      const int row = kv0 + r;
      v8 x = {};
      if (row < g.lk) x = ld_stream<v8>(kbase + (g.k_row0 + row) * a.k_stride_t + c);
      st_vec<v8>(&rows[r][c], x);
    }
    __syncthreads();
    {
      constexpr int TPN = 256 / BKV;  // threads per row
      const int r = tid / TPN, part = tid % TPN;
      float ss = 0.f;
      for (int d = part; d < D; d += TPN) {
        const float x = (float)rows[r][d];
        ss = fmaf(x, x, ss);
      }
#pragma unroll
      for (int o = 1; o < TPN; o <<= 1) ss += shfl_xor_f(ss, o);
      if (part == 0) inv_rms[r] = rms_scale(ss, D, a.norm_eps);
    }
    __syncthreads();
    for (int idx = tid; idx < BKV * HALF8; idx += 256) {
      const int r = idx / HALF8;
      const int c = (idx % HALF8) * 8;
      const int row = kv0 + r;
      const float inv = inv_rms[r];
      v8 k1 = ld_vec<v8>(&rows[r][c]);
      v8 k2 = ld_vec<v8>(&rows[r][c + D / 2]);
      float x1[8], x2[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        x1[e] = (float)k1[e] * inv * (1.f + a.k_norm_weight[c + e]);
        x2[e] = (float)k2[e] * inv * (1.f + a.k_norm_weight[c + D / 2 + e]);
      }
      if (a.rope_k && row < g.lk) {
        const int pos = rope.at(r);
        const float* cs = a.rope_cos + (int64_t)pos * (D / 2) + c;
        const float* sn = a.rope_sin + (int64_t)pos * (D / 2) + c;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float y1 = x1[e] * cs[e] - x2[e] * sn[e];
          const float y2 = x1[e] * sn[e] + x2[e] * cs[e];
          x1[e] = y1;
          x2[e] = y2;
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        k1[e] = (T)x1[e];
        k2[e] = (T)x2[e];
      }
      st_vec<v8>(&rows[r][c], k1);
      st_vec<v8>(&rows[r][c + D / 2], k2);
    }
  } else {
  // K: coalesced row loads, rotation of the (i, i + D/2) pairs, staged.
  for (int idx = tid; idx < BKV * HALF8; idx += 256) {
    const int r = idx / HALF8;
    const int c = (idx % HALF8) * 8;
    const int row = kv0 + r;
    v8 k1 = {}, k2 = {};
    if (row < g.lk) {
      const T* kr = kbase + (g.k_row0 + row) * a.k_stride_t;
      k1 = ld_stream<v8>(kr + c);
      k2 = ld_stream<v8>(kr + c + D / 2);
      if (a.rope_k) {
        const int pos = rope.at(r);
        const float* cs = a.rope_cos + (int64_t)pos * (D / 2) + c;
        const float* sn = a.rope_sin + (int64_t)pos * (D / 2) + c;
        const f32x4 c0 = ld_vec<f32x4>(cs), c1 = ld_vec<f32x4>(cs + 4);
        const f32x4 s0 = ld_vec<f32x4>(sn), s1 = ld_vec<f32x4>(sn + 4);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float x1 = (float)k1[e], x2 = (float)k2[e];
          const float cc = e < 4 ? c0[e & 3] : c1[e & 3];
          const float ss = e < 4 ? s0[e & 3] : s1[e & 3];
          k1[e] = (T)(x1 * cc - x2 * ss);
          k2[e] = (T)(x1 * ss + x2 * cc);
        }
      }
    }
    st_vec<v8>(&rows[r][c], k1);
    st_vec<v8>(&rows[r][c + D / 2], k2);
  }
  }
  __syncthreads();
  // K' image: chunk (c, r) at c*BKV + r; consecutive threads write
  // consecutive chunks.
  for (int idx = tid; idx < TG::K_CHUNKS; idx += 256) {
    const int c = idx / BKV, r = idx % BKV;
    kimg[idx] = ld_vec<v8>(&rows[r][8 * c]);
  }
  __syncthreads();
  // V rows; rows past the sequence end are zero, so P = 0 there meets a
  // finite value.
  for (int idx = tid; idx < BKV * (D / 8); idx += 256) {
    const int r = idx / (D / 8);
    const int c = (idx % (D / 8)) * 8;
    const int row = kv0 + r;
    v8 v = {};
    if (row < g.lk) v = ld_stream<v8>(vbase + (g.k_row0 + row) * a.v_stride_t + c);
    st_vec<v8>(&rows[r][c], v);
  }
  __syncthreads();
  // V^T image: chunk (kc, d) at kc*D + d holds keys kPermKey(8*(kc%2) + e),
  // e = 0..7, of the 16-key group kc/2.
  for (int idx = tid; idx < TG::V_CHUNKS; idx += 256) {
    const int kc = idx / D, d = idx % D;
    const int k0 = 16 * (kc / 2);
    v8 out;
#pragma unroll
    for (int e = 0; e < 8; ++e) out[e] = rows[k0 + kPermKey(8 * (kc % 2) + e)][d];
    vimg[idx] = out;
  }
}

// ---------------------------------------------------------------------------
// 2. attention
// ---------------------------------------------------------------------------
__device__ __forceinline__ float max3f(float a, float b, float c) { return fmaxf(fmaxf(a, b), c); }

// After permlane32_swap(x, x), r[0] holds x of lane l%32 and r[1] x of lane
// 32 + l%32: the two halves of a query row.
__device__ __forceinline__ float half_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// acc + p[2i] + p[2i+1] on the rounded probabilities (the values the PV
// product uses).
__device__ __forceinline__ float dot2_ones(bf16x8 p, int i, float acc) {
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  const b2 v = {p[2 * i], p[2 * i + 1]};
  const b2 one = {(__bf16)1.0f, (__bf16)1.0f};
  return __builtin_amdgcn_fdot2_f32_bf16(v, one, acc, false);
}
__device__ __forceinline__ float dot2_ones(f32x8 p, int i, float acc) { return acc + p[2 * i] + p[2 * i + 1]; }
__device__ __forceinline__ float dot2_ones(f16x8 p, int i, float acc) {
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  const h2 v = {p[2 * i], p[2 * i + 1]};
  const h2 one = {(_Float16)1.0f, (_Float16)1.0f};
  return __builtin_amdgcn_fdot2(v, one, acc, false);
}

// Non-persistent grid: the work item of workgroup `lin` of `nblk`.
__device__ __forceinline__ void grid_item(const PrefillParams& p, const int lin, const int nblk, const int qb_rows,
                                          int& pair, int& qt) {
  const goda_prefill_args& a = p.a;
  const int nqt = p.qtiles;
  // XCD-aware order: consecutive dispatch slots rotate over the 8 XCDs
  // (XCD = blockIdx % 8). Dense batches: each XCD gets a contiguous range of
  // (sequence, head-slice) pairs, so the workgroups sharing K/V tiles share
  // that XCD's L2; heavy causal query tiles go first. Packed batches of
  // unequal lengths would leave the XCDs very unequally loaded that way
  // (random draws of 16 lengths in [128, 4096]: busiest XCD 1.5-2x the mean),
  // so there XCD x takes the query tiles qt = x (mod kXg) of the pairs of its
  // group, pair after pair, heaviest tile first: every XCD stays within ~3%
  // of the mean, and the XCDs work on the same pair at the same time, so each
  // XCD's L2 still serves one pair's K/V stream to all its workgroups.
  // XCDs sharing one pair's query tiles (a power of two: shifts): fewer where a
  // pair has fewer (packed_tiles).
  static_assert(kVarlenXcdGroup == 8, "log2 below");
  const int log_xg = nqt >= kVarlenXcdGroup ? 3 : nqt >= 4 ? 2 : nqt >= 2 ? 1 : 0;
  const int kXg = 1 << log_xg;
  const int npairs = nblk / nqt;
  if (a.cu_seqlens_q && nblk % 8 == 0 && (nqt & (kXg - 1)) == 0 && (npairs & ((8 >> log_xg) - 1)) == 0) {
    const int x = lin % 8, s = lin / 8;
    const int per = nqt >> log_xg;                               // query tiles of one pair on one XCD
    pair = (s / per << (3 - log_xg)) + (x >> log_xg);            // place in the walk
    // Short sequences: turned by the pair's place in the walk (kRotateTiles).
    const bool rotate = per <= kRotateTiles;
    qt = ((per - 1 - s % per) << log_xg) + ((x + (rotate ? pair : 0)) & (kXg - 1));
    if (a.batch <= 64) {
      // Longest sequences first, so the heaviest tiles are not the last ones
      // dispatched: position `pair` in the walk is served by the sequence of
      // that length rank (ties by index; one wave-wide pass over the lengths).
      const int per_seq = npairs / a.batch;  // pairs of one sequence
      const int ln = threadIdx.x & 63;
      const int len = ln < a.batch ? a.cu_seqlens_q[ln + 1] - a.cu_seqlens_q[ln] : -1;
      int rank = 0;
      for (int j = 0; j < a.batch; ++j) {
        const int lj = __shfl(len, j, 64);
        rank += (lj > len || (lj == len && j < ln)) ? 1 : 0;
      }
      // The shortest kPackedTailNum / kPackedTailDen of the sequences (ranks
      // >= r0) form the tail of each XCD's walk. Pair by pair, their heaviest
      // tiles would start late and end the kernel, so the tail deals its
      // tiles level by level instead: every tail sequence's tile at the
      // highest level first (longest sequence first within a level), then
      // the next level down.
      // Level i of XCD x is query tile (per - 1 - i) * 8 + x; sequence r has
      // n_r = ceil((nq_r - x) / 8) tiles there, its levels per - n_r .. per - 1.
      const int r0 = rotate ? a.batch : a.batch - (a.batch * kPackedTailNum) / kPackedTailDen;
      const int s0 = r0 * per_seq * per;  // the tail's first slot on this XCD
      if (s < s0 || r0 >= a.batch) {
        const int r = pair / per_seq;
        const uint64_t hit = __builtin_amdgcn_ballot_w64(ln < a.batch && rank == r);
        if (hit == 0) {  // (only with inconsistent sequence lengths) an empty item
          pair = 0;
          qt = nqt;
          return;
        }
        pair = __builtin_ctzll(hit) * per_seq + pair % per_seq;
      } else {
        const int k = s - s0;
        const bool tail = ln < a.batch && rank >= r0;
        const int nq = (len + qb_rows - 1) / qb_rows;
        const int n_l = tail && nq > x ? (nq - x + 7) / 8 : 0;
        // tail items at levels 0 .. i
        auto count = [&](int i) {
          int c = max(0, i - (per - n_l) + 1);
#pragma unroll
          for (int o = 32; o >= 1; o >>= 1) c += __shfl_xor(c, o, 64);
          return c * per_seq;
        };
        if (count(per - 1) <= k) {
          pair = 0;  // past the tail's tiles: an empty item
          qt = nqt;
          return;
        }
        int lo = 0, hi = per - 1;  // smallest level i with count(i) > k
        while (lo < hi) {
          const int mid = (lo + hi) / 2;
          if (count(mid) > k)
            hi = mid;
          else
            lo = mid + 1;
        }
        const int j = k - (lo > 0 ? count(lo - 1) : 0);
        const int m = j / per_seq;
        // the m-th (by rank) tail sequence with a tile at level lo
        const bool act = tail && n_l >= per - lo;
        int before = 0;
        for (int t = 0; t < a.batch; ++t) {
          const int rt = __shfl(rank, t, 64);
          const bool at = __shfl(act ? 1 : 0, t, 64) != 0;
          before += (at && rt < rank) ? 1 : 0;
        }
        const uint64_t hit = __builtin_amdgcn_ballot_w64(act && before == m);
        if (hit == 0) {  // (only with inconsistent sequence lengths) an empty item
          pair = 0;
          qt = nqt;
          return;
        }
        pair = __builtin_ctzll(hit) * per_seq + j % per_seq;
        qt = ((per - 1 - lo) << log_xg) + (x & (kXg - 1));
      }
    }
  } else {
    const int vid = (nblk % 8 == 0) ? (lin % 8) * (nblk / 8) + lin / 8 : lin;
    pair = vid / nqt;
    qt = nqt - 1 - (vid % nqt);
  }
}

// One work item of the attention kernel: query tile qt of (sequence, head
// slice) pair `pair`.
template <typename T, int D, int BKV, int NT, int WAVES, bool ALIBI, bool MASK, bool KSPLIT = false>
__device__ __forceinline__ void fa_item(const PrefillParams& p, unsigned char* smem, const int pair, const int qt,
                                        const int piece = 0) {
  typedef typename Vec<T>::v8 v8;
  typedef typename Vec<T>::v4 v4;
  typedef TileGeom<T, D, BKV, WAVES> TG;
  constexpr int MT = BKV / 32;   // 32-key row tiles of S^T
  constexpr int KS = D / 16;     // k-steps of QK^T
  constexpr int MD = D / 32;     // 32-wide head-dim tiles of O^T
  constexpr int KS2 = BKV / 16;  // k-steps of PV
  static_assert(MT >= 1, "tile shape");
  static_assert(WAVES == 8, "two waves per SIMD, in two groups half an interval apart");

  const goda_prefill_args& a = p.a;
  // Fields the key loop reads, copied once: read through `a` and `p` inside
  // the loop they were loaded again every step (as far as the compiler knows
  // the inline-asm barriers and copies write memory), each scalar load then
  // waited for with the counter the LDS operand reads share.
  const int causal = a.causal;
  const int window_left = a.window_left;
  const int ntiles_k = p.ntiles_k;
  const int heads_kv = a.heads_kv;
  const int hg = p.heads_per_wg;
  const int nslices = p.group / hg;
  const int qb_rows = (WAVES / hg) * 32 * NT;  // query rows per workgroup

  const int b = pair / (heads_kv * nslices);
  const int rem = pair % (heads_kv * nslices);
  const int hk = rem / nslices;
  const int sl = rem % nslices;

  const SeqGeom g = seq_geom(b, a.seqlen_q, a.seqlen_k, a.cu_seqlens_q, a.cu_seqlens_k,
                             a.seqused_k);
  const int qr0 = qt * qb_rows;
  if (qr0 >= g.lq) return;

  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int l32 = lane & 31;
  const int hi = lane >> 5;  // lane half
  const int hq = hk * p.group + sl * hg + (wave % hg);
  const int wrow0 = qr0 + (__builtin_amdgcn_readfirstlane(wave) / hg) * 32 * NT;  // first query row of this wave (scalar)
  const int diag = g.lk - g.lq;
  const bool use_window = window_left >= 0 && (causal || g.lq == 1);

  // ---- Q^T operand fragments (rotated) ---------------------------------------
  v8 qf[NT][KS];
  // (invoked in the prologue, after the first tiles' copies are issued; part 1:
  // the loads alone, 2: what comes after them)
  auto load_q = [&](auto part) {
    constexpr int PART = decltype(part)::value;
    const T* qbase = reinterpret_cast<const T*>(a.q) +
                     (a.cu_seqlens_q ? 0 : (int64_t)b * a.q_stride_b) + (int64_t)hq * a.q_stride_h;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int qi = wrow0 + 32 * nt + l32;
      if (qi < g.lq) {
        const T* qr = qbase + (g.q_row0 + qi) * a.q_stride_t;
        if constexpr (PART != 2)
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) qf[nt][ks] = ld_vec<v8>(qr + 16 * ks + 8 * hi);
        if constexpr (PART != 1) {
          // fp32 round trip: fused QK-RMSNorm, then RoPE, then the softmax
          // scale in log2 units (scores come out of the MFMA ready for exp2),
          // one rounding.
          float xf[KS][8];
#pragma unroll
          for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int e = 0; e < 8; ++e) xf[ks][e] = (float)qf[nt][ks][e];
          if (a.q_norm_weight) {
            float ss = 0.f;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
#pragma unroll
              for (int e = 0; e < 8; ++e) ss = fmaf(xf[ks][e], xf[ks][e], ss);
            const float inv = rms_scale(half_sum(ss), D, a.norm_eps);  // lanes l, l^32 hold the row
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
              const float* w = a.q_norm_weight + 16 * ks + 8 * hi;
#pragma unroll
              for (int e = 0; e < 8; ++e) xf[ks][e] *= inv * (1.f + w[e]);
            }
          }
          if (a.rope_q) {
            const int pos = rope_qrows(a, g, wrow0 + 32 * nt).at(l32);
#pragma unroll
            for (int ks = 0; ks < KS / 2; ++ks) {
              const int f0 = 16 * ks + 8 * hi;
              const float* cs = a.rope_cos + (int64_t)pos * (D / 2) + f0;
              const float* sn = a.rope_sin + (int64_t)pos * (D / 2) + f0;
              const f32x4 c0 = ld_vec<f32x4>(cs), c1 = ld_vec<f32x4>(cs + 4);
              const f32x4 s0 = ld_vec<f32x4>(sn), s1 = ld_vec<f32x4>(sn + 4);
#pragma unroll
              for (int e = 0; e < 8; ++e) {
                const float cc = e < 4 ? c0[e & 3] : c1[e & 3];
                const float ss = e < 4 ? s0[e & 3] : s1[e & 3];
                const float x1 = xf[ks][e], x2 = xf[ks + KS / 2][e];
                xf[ks][e] = x1 * cc - x2 * ss;
                xf[ks + KS / 2][e] = x1 * ss + x2 * cc;
              }
            }
          }
#pragma unroll
          for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int e = 0; e < 8; ++e) qf[nt][ks][e] = (T)(xf[ks][e] * p.scale_log2);
        }
      } else if constexpr (PART != 2) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) qf[nt][ks] = v8{};
      }
    }
    // Pin the fragments in registers: without this the compiler treats the
    // (read-only) q loads as rematerializable and re-reads q from global
    // memory inside the key loop.
    if constexpr (PART != 1)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(qf[nt][ks]));
  };

  // ---- key tile range ---------------------------------------------------------
  const int q_last = min(qr0 + qb_rows, g.lq) - 1;
  int kv_hi = g.lk;
  if (causal) kv_hi = min(kv_hi, diag + q_last + 1);
  int kv_lo = 0;
  if (use_window) kv_lo = max(0, diag + qr0 - window_left);
  int j_lo = kv_lo / BKV;
  int j_hi = kv_hi > 0 ? (kv_hi + BKV - 1) / BKV : 0;
  int npieces = 1;
  if constexpr (KSPLIT) {
    const int all = max(0, j_hi - j_lo);
    npieces = __builtin_amdgcn_readfirstlane(piece_count(all, piece_tiles(p, BKV), p.ksplit));
    if (piece >= npieces) return;
    const int len = (all + npieces - 1) / npieces;
    j_lo += piece * len;
    j_hi = min(j_hi, j_lo + len);
  }
  // Key tile of step j. With ALiBi the steps walk the tiles from the last
  // down: the bias slope*(key - row) grows along the keys, so the first tile
  // holds (nearly) every row's max and the lazy rescale seldom fires again;
  // in key order the max moved by the slope per key and rescaled often.
  // Stages and loop bounds stay in step order.
  // With a caller's mask the steps are those of the tiles that some row sees,
  // counted from 0, and a list in LDS has their tiles (`listed`: some tile is
  // hidden). Lane i of `walk` holds the tile of step walk0 + i, so that a tile is
  // read by one v_readlane, without a branch or a wait; head_dim 256, which has
  // no register for it, reads the list. `ahead`: the tiles of the steps j .. j +
  // kAhead, read one step before the first use.
  constexpr bool WALK = D <= 128;
  uint16_t* list = reinterpret_cast<uint16_t*>(smem + kStages * TG::BYTES);
  bool listed = false;
  const int first_tile = j_lo;
  if constexpr (MASK) {
    j_hi = max(j_hi - j_lo, 0);
    j_lo = 0;
  }
  const int j_rev = j_lo + j_hi - 1;
  int walk = 0, walk0 = 0, ahead[kAhead + 1];
  // Lane i's tile of the 64 steps from j (the last ones' where there are fewer).
  auto fill_walk = [&](int j) {
    if constexpr (WALK) {
      walk0 = j;
      const int i = min(j + lane, j_hi - 1);
      walk = first_tile + (listed ? (int)list[i] : ALIBI ? j_rev - i : i);
    }
  };
  auto tile_of = [&](int j) {
    if constexpr (MASK && WALK) return __builtin_amdgcn_readlane(walk, j - walk0);
    if constexpr (MASK) {
      const int i = min(j, j_hi - 1);
      return first_tile + (listed ? __builtin_amdgcn_readfirstlane((int)list[i]) : ALIBI ? j_rev - i : i);
    }
    return ALIBI ? j_rev - j : j;
  };
  // The tile of step j in the key loop, j being `K` steps past the current one.
  typedef std::integral_constant<int, 0> Now;
  typedef std::integral_constant<int, 1> Next;
  typedef std::integral_constant<int, kAhead> Copied;
  auto tile_at = [&](auto k, int j) {
    if constexpr (MASK) return ahead[decltype(k)::value];
    return tile_of(j);
  };

  f32x16 oacc[MD][NT];
#pragma unroll
  for (int md = 0; md < MD; ++md)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) oacc[md][nt] = f32x16{};
  float m_run[NT];
  float l_run[NT][4];  // row sum in four independent chains (one per dot-product slot), added at the end
  // Rescale test of a tile against its own reference: the reference moves
  // when the tile's max (relative to the reference) exceeds gthr, which is
  // kRescaleThresh once the row has a finite reference and -inf before.
  float gthr[NT];
  // Without ALiBi every accumulator of a lane starts at -m of its query row:
  // minit holds that block and is the C operand of each S tile's first
  // product, so no VALU instruction refills the accumulators per tile
  // (cfg2 kernel -1.2%; head_dim 256 has no 16 registers to spare for it).
  constexpr bool MINIT = !ALIBI && D <= 128;
  f32x16 minit[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    m_run[nt] = kNegInf;
    l_run[nt][0] = l_run[nt][1] = l_run[nt][2] = l_run[nt][3] = 0.f;
    gthr[nt] = kNegInf;
    minit[nt] = f32x16{};
  }
  if constexpr (MINIT) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) asm volatile("" : "+v"(minit[nt]));
  }
  const float slope2 = ALIBI ? a.alibi_slopes[hq] * kLog2e : 0.f;
  const float alibi_s1 = slope2, alibi_s2 = 2.f * slope2, alibi_s3 = 3.f * slope2, alibi_s8 = 8.f * slope2;

  // Caller's mask: this lane's query rows (rows past the sequence read the
  // last row's bits, and are never stored). A tile's word is loaded with the
  // tile's score products and applied in its softmax phase.
  typedef typename MaskWord<BKV>::t mword_t;
  const mword_t* mrow[NT];
  mword_t mw[NT];
  if constexpr (MASK) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      mrow[nt] = reinterpret_cast<const mword_t*>(mask_row(a, b, hq, min(wrow0 + 32 * nt + l32, g.lq - 1)));
      mw[nt] = MaskWord<BKV>::kAll;
    }
  }

  // ---- tile ring ----------------------------------------------------------------
  // Lane chunk c of this wave's share sits at the same offset in the
  // workspace tile and in the LDS stage.
  constexpr int LOADS = TG::LOADS_PER_LANE;
  const unsigned char* ws = reinterpret_cast<const unsigned char*>(a.workspace);
  const int my_chunk0 = wave * LOADS * 64 + lane;
  // (Stored and later read through the same operand type v8.) With SPLIT the
  // tile moves in two halves through half the staging registers: the first
  // half is loaded at the start of the interval and stored mid-interval, when
  // the second half is loaded; that one is stored at the end.
  constexpr bool SPLIT = kSplitStaging<D> && WAVES == 8 && LOADS % 2 == 0;
  constexpr int NSTG = SPLIT ? LOADS / 2 : LOADS;
  v8 stg[NSTG];
  auto tile_load_part = [&](int tile, int part) {
    const v8* src = reinterpret_cast<const v8*>(ws + ws_tile(b, tile, hk, ntiles_k, heads_kv) * TG::BYTES) +
                    my_chunk0 + part * NSTG * 64;
#pragma unroll
    for (int i = 0; i < NSTG; ++i) stg[i] = src[i * 64];
  };
  auto tile_store_part = [&](int j, int part) {
    v8* dst = reinterpret_cast<v8*>(smem + ((j - j_lo) & (kStages - 1)) * TG::BYTES) + my_chunk0 + part * NSTG * 64;
#pragma unroll
    for (int i = 0; i < NSTG; ++i) dst[i * 64] = stg[i];
  };
  auto tile_load = [&](int j, int tile) {
    tile_load_part(tile, 0);
    if constexpr (SPLIT) {
      tile_store_part(j, 0);
      tile_load_part(tile, 1);
    }
  };
  auto tile_store = [&](int j) { tile_store_part(j, SPLIT ? 1 : 0); };
  // 16-bit tiles move by direct global->LDS loads instead (dma_blocks): wave
  // w's share of a tile is LOADS blocks of 64 consecutive 16-byte chunks, the
  // same offsets in the workspace tile and in the LDS stage. The barrier
  // opening interval j must see tile j + 1 (its K part is read in interval
  // j), copied in interval j - 2. When interval j - 1 copied tile j + 2 the
  // barrier waits vmcnt(LOADS): every batch but that newest one has landed.
  // In the last kAhead - 1 intervals no batch is issued, so the newest
  // outstanding batch is tile j + 1 itself and the barrier waits vmcnt(0).
  // Tile t sits in stage (t - j_lo) mod kStages (counted from the
  // workgroup's first tile, so the loop unrolled by kStages sees constant
  // stage addresses); tile j + kAhead lands in a stage no wave reads between
  // its issue (interval j, after the barrier) and the barrier opening
  // interval j + kAhead - 1, where it is first read.
  constexpr bool DMA = sizeof(T) == 2;
  static_assert(!DMA || LOADS == 2 || LOADS == 4, "DMA share of 2 or 4 blocks");
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  const unsigned lane_off = (unsigned)((wave_u * LOADS * 64 + lane) * 16);
  auto tile_dma = [&](int j, int tile) {
    const unsigned long long base =
        (unsigned long long)(uintptr_t)(ws + ws_tile(b, tile, hk, ntiles_k, heads_kv) * TG::BYTES);
    const unsigned lds0 =
        (unsigned)(uintptr_t)(smem + ((j - j_lo) & (kStages - 1)) * TG::BYTES) + (unsigned)(wave_u * LOADS * 64 * 16);
    dma_blocks<LOADS>(lds0, lane_off, base);
  };
  auto dma_barrier = [&](int j) {
    if (j + kAhead - 1 < j_hi)
      dma_ring_barrier<LOADS>();
    else
      dma_ring_barrier<0>();
  };

  // This lane's K' operand for (ks, mt) is chunk (2ks + hi)*BKV + 32mt + l32;
  // its V^T operand for (ks2, md) is chunk (2ks2 + hi)*D + 32md + l32.
  // S^T(j) in log2 units relative to the row's current reference max: the
  // accumulators start at -m (plus the ALiBi bias slope*(kv - i) of each
  // register), so a score leaves the MFMA as the exponent of its P.
  // js is the tile whose stage the products read: j itself, except on the
  // last step of a workgroup that does not peel it (head_dim 256), where j is
  // clamped for the mask words and the bias and the products read stage
  // j + 1 (whatever it holds; they are never used).
  auto qk = [&](auto k, int j, f32x16 (&s)[MT][NT], int js) {
    if constexpr (MASK) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) mw[nt] = mrow[nt][tile_at(k, j)];
    }
    const v8* kp = reinterpret_cast<const v8*>(smem + ((js - j_lo) & (kStages - 1)) * TG::BYTES) + hi * BKV + l32;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const float m0 = (m_run[nt] == kNegInf) ? 0.f : -m_run[nt];
      if (ALIBI) {
        const int iabs = diag + wrow0 + 32 * nt + l32;
        float bg = m0 + slope2 * (float)(tile_at(k, j) * BKV + 4 * hi - iabs);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            if ((r & 3) == 0 && (mt | r) != 0) bg += alibi_s8;
            s[mt][nt][r] = (r & 3) == 0 ? bg : (r & 3) == 1 ? bg + alibi_s1 : (r & 3) == 2 ? bg + alibi_s2 : bg + alibi_s3;
          }
      } else if constexpr (!MINIT) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int r = 0; r < 16; ++r) s[mt][nt][r] = m0;
      }
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const v8 av = kp[ks * 2 * BKV + mt * 32];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          s[mt][nt] = mfma32(av, qf[nt][ks], (ks == 0 && MINIT) ? minit[nt] : s[mt][nt]);
      }
  };

  // ---- softmax half of a step: scores s of tile j -> probabilities pf --------------
  // The scores arrive as exponents relative to the reference max the row had
  // when S(j) was issued (the same m_run as now: nothing updates it between
  // an S tile's products and its softmax).
  auto vpart = [&](auto k, int j, f32x16 (&s)[MT][NT], v8 (&pf)[NT][KS2]) {
    const int kvb = tile_at(k, j) * BKV;
    const bool need_mask = (kvb + BKV > g.lk) || (causal && kvb + BKV - 1 > diag + wrow0) ||
                           (use_window && kvb < diag + wrow0 + 32 * NT - 1 - window_left);
    if (need_mask) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const int iabs = diag + wrow0 + 32 * nt + l32;
        // Visibility as a range of the register's key offset
        // off = kv - (kvb + 4 hi), a compile-time constant per register:
        // lo_lim <= off <= hi_lim (no per-register key index is formed).
        const int rel = kvb + 4 * hi;
        int hi_lim = g.lk - 1 - rel;
        if (causal) hi_lim = min(hi_lim, iabs - rel);
        const int lo_lim = use_window ? iabs - window_left - rel : 0;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int off = 32 * mt + 8 * (r >> 2) + (r & 3);
            s[mt][nt][r] = (off >= lo_lim && off <= hi_lim) ? s[mt][nt][r] : kNegInf;
          }
      }
    }
    if constexpr (MASK) {
      // Register (mt, r) holds key kvb + 4 hi + 32 mt + 8 (r/4) + r%4.
      bool partial = false;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) partial = partial || (mw[nt] != MaskWord<BKV>::kAll);
      if (__builtin_amdgcn_ballot_w64(partial) != 0) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          const mword_t w = mw[nt] >> (4 * hi);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) {
            const uint32_t w32 = (uint32_t)(w >> (32 * mt));
#pragma unroll
            for (int r = 0; r < 16; ++r) s[mt][nt][r] = keep_if_bit(s[mt][nt][r], w32, 8 * (r >> 2) + (r & 3), kNegInf);
          }
        }
      }
    }
    // Row max (relative to the reference, log2 units) and lazy rescale. The
    // test runs on each lane's half of the row: a row's max exceeds the
    // threshold iff one of its halves does, and the ballot spans both, so
    // the two halves are only combined on the (rare) rescale path.
    float mhalf[NT];
    bool grow = false;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      float mx = kNegInf;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < 16; r += 2) mx = max3f(mx, s[mt][nt][r], s[mt][nt][r + 1]);
      mhalf[nt] = mx;
      grow = grow || (mx > gthr[nt]);
    }
    if (__builtin_amdgcn_ballot_w64(grow) != 0) {
      // the max moved: rescale O and l, and bring the scores to the new
      // reference (rare: the reference only moves by more than the threshold)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const float mq = (m_run[nt] == kNegInf) ? 0.f : m_run[nt];  // the reference the scores carry
        const float mn = fmaxf(m_run[nt], half_max(mhalf[nt]) + mq);
        const float alpha = (m_run[nt] == kNegInf) ? 0.f : fast_exp2(m_run[nt] - mn);
        const float shift = (mn == kNegInf) ? 0.f : mn - mq;
        m_run[nt] = mn;
        gthr[nt] = (mn == kNegInf) ? kNegInf : kRescaleThresh<T>;
        if constexpr (MINIT) {
          const float mi = (mn == kNegInf) ? 0.f : -mn;
#pragma unroll
          for (int r = 0; r < 16; ++r) minit[nt][r] = mi;
          asm volatile("" : "+v"(minit[nt]));
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) l_run[nt][i] *= alpha;
#pragma unroll
        for (int md = 0; md < MD; ++md) oacc[md][nt] *= alpha;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int r = 0; r < 16; ++r) s[mt][nt][r] -= shift;
      }
    }
    // probabilities (rounded to the operand type) and their row sums
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      // Four independent row-sum chains (one per dot-product slot) instead of
      // one chain of 2*MT*4 dependent dot products: cfg2 +1.1-1.5%; kept
      // apart across tiles and added once in the epilogue (cfg2 -0.8%).
      float (&ls)[4] = l_run[nt];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          v8 pv;
#pragma unroll
          for (int e = 0; e < 8; ++e) pv[e] = (T)fast_exp2(s[mt][nt][8 * h + e]);
#pragma unroll
          for (int i = 0; i < 4; ++i) ls[i] = dot2_ones(pv, i, ls[i]);
          pf[nt][2 * mt + h] = pv;
        }
      }
    }
  };

  // ---- O^T += V^T P^T for tile j ----------------------------------------------------
  auto pv_mfma = [&](int j, const v8 (&pf)[NT][KS2]) {
    const v8* vp = reinterpret_cast<const v8*>(smem + ((j - j_lo) & (kStages - 1)) * TG::BYTES + TG::K_CHUNKS * TG::CHB) +
                   hi * D + l32;
#pragma unroll
    for (int ks2 = 0; ks2 < KS2; ++ks2) {
#pragma unroll
      for (int md = 0; md < MD; ++md) {
        const v8 av = vp[ks2 * 2 * D + md * 32];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) oacc[md][nt] = mfma32(av, pf[nt][ks2], oacc[md][nt]);
      }
    }
  };

  // MFMA half of a step: O += P(j)V(j), then S(j+1) = K(j+1)Q^T.
  // The schedule keeps the LDS operand reads kLead MFMAs ahead of their use,
  // so each wave's MFMA phase runs back to back instead of waiting out an
  // LDS round trip every two MFMAs.
  // The workgroup's last step has no next tile. At head_dim <= 128 it is
  // peeled (last = true) and issues P(j)V(j) only: its score products were
  // 0.8% of cfg2's MFMAs (cfg2 kernel -0.7%). At head_dim 256 the peeled copy
  // cost cfg3 5% (its instances use 252-256 registers), so there the last
  // step runs the whole phase on a clamped tile and discards the scores.
  auto mphase = [&](auto last, int j, const v8 (&pf)[NT][KS2], f32x16 (&s)[MT][NT]) {
    constexpr bool LAST = decltype(last)::value;
    pv_mfma(j, pf);
    if constexpr (!LAST) qk(Next{}, j + 1 < j_hi ? j + 1 : j, s, j + 1);
    // counted in instructions: an fp32 step is 8 MFMAs and its 32-byte
    // operand two 16-byte LDS reads
    constexpr int kMfma = (KS2 * MD * NT + (LAST ? 0 : KS * MT * NT)) * kMfmaPerStep<T>;
    constexpr int kReads = (KS2 * MD + (LAST ? 0 : KS * MT)) * TG::CHB / 16;
    // (same-box A/B: at D = 128, 4 beats 2, 6 and 8 by 0.5-0.7%; at D = 256,
    // 3 beats 4 by 6.4% on cfg3 and ties on cfg5)
    constexpr int kLead = D >= 256 ? 3 : 4;
    static_assert(kReads > kLead, "phase too short");
    __builtin_amdgcn_sched_group_barrier(0x100, kLead, 0);
#pragma unroll
    for (int i = 0; i < kReads - kLead; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, kMfma / kReads, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, kLead * (kMfma / kReads), 0);
  };

  // Start of the ring interval that reads tiles j (V) and j+1 (K) and writes
  // tile j + kAhead. Register-staged tiles: the global loads are issued now,
  // the LDS stores go out mid-interval and at the end. Direct copies: issued
  // mid-interval (ring_mid), after each wave's first phase. Issued right
  // after the barrier, the 32 copies of a workgroup's 8 waves queue at the
  // CU's address unit together and hold every wave of a SIMD at once
  // (s_memtime probe: 120-300 clocks of a ~3600-clock interval); after the
  // first phase, the two groups issue at different times and the partner
  // wave keeps computing (cfg2 kernel -3.4% in a same-box A/B; issuing them
  // all from group 0, or between a wave's PV and QK products, was slower).
  // With a caller's mask they stay at the barrier: the compiler's wait for a
  // mask word (loaded with the score products, used in the softmax) cannot
  // see the inline-asm copies and would wait for a copy issued just before.
  constexpr bool kDmaMid = DMA && !MASK;
  auto ring_begin = [&](int j) {
    if constexpr (DMA) {
      dma_barrier(j);
      if constexpr (!kDmaMid)
        if (j + kAhead < j_hi) tile_dma(j + kAhead, tile_at(Copied{}, j + kAhead));
      return;
    }
    if ((j - j_lo) % kBarrierEvery == kBarrierEvery - 1) ring_barrier();  // the prologue's barrier opens interval j_lo
    if (j + kAhead < j_hi) tile_load_part(tile_at(Copied{}, j + kAhead), 0);
  };
  auto ring_mid = [&](int j) {
    if constexpr (kDmaMid) {
      if (j + kAhead < j_hi) tile_dma(j + kAhead, tile_at(Copied{}, j + kAhead));
    } else if constexpr (SPLIT && !DMA) {
      if (j + kAhead < j_hi) {
        tile_store_part(j + kAhead, 0);
        tile_load_part(tile_at(Copied{}, j + kAhead), 1);
      }
    }
  };
  auto ring_end = [&](int j) {
    if constexpr (!DMA)
      if (j + kAhead < j_hi) tile_store(j + kAhead);
  };

  // ---- prologue: tiles j_lo .. j_lo + kAhead - 1 resident, scores of tile j_lo --------
  // With a caller's mask, the tiles to walk: lane w takes word w of the marks of
  // the workgroup's rows, and every wave writes the whole list, the same words
  // from each. Meanwhile the tiles that are the first if none is hidden are
  // copied, and the q rows loaded. bf16, us, every tile walked / this: B=4,
  // T=2048, 16/4 heads, D=128: half the tiles hidden 133 / 83, a prefix mask
  // 137 / 130, nothing hidden 139 / 141; B=1, T=8192, 32/8 heads: six documents
  // 470 / 139, nothing hidden 929 / 940; small ones up to 1 us more (T=300: 14.3 /
  // 15.4). With the marks taken in this kernel and the list read from LDS three
  // times a step, nothing hidden was 156, 1074 and 16.1.
  if constexpr (MASK) {
    const int ntl = j_hi;
    if (ntl > 0) {
      fill_walk(0);
      if constexpr (DMA)
        for (int t = 0; t < kAhead && t < ntl; ++t) tile_dma(t, tile_of(t));
      const int w0 = first_tile / 64, nw = (first_tile + ntl - 1) / 64 - w0 + 1;
      const bool marked = p.marks && nw <= kListTiles / 64;
      uint64_t m = 0;
      if (marked && lane < nw) {
        const Marks k = marks_of(a, ntiles_k);
        const int64_t bh = (int64_t)(a.mask_stride_b ? b : 0) * k.heads;
#pragma unroll
        for (int i = 0; i < WAVES; ++i) {
          const int h = a.mask_stride_h ? hk * p.group + sl * hg + i % hg : 0;
          const int block = a.mask_stride_q ? min(qr0 / 32 + i / hg, k.blocks - 1) : 0;
          m |= p.marks[((bh + h) * k.blocks + block) * k.words + w0 + lane];
        }
        // the tiles of the walk alone
        const int lo = first_tile - 64 * (w0 + lane), n = first_tile + ntl - 64 * (w0 + lane);
        if (lo > 0) m &= ~0ull << lo;
        if (n < 64) m &= ~0ull >> (64 - n);
      }
      load_q(std::integral_constant<int, 1>{});
      if (marked) {
        int upto = __popcll(m);
        if (nw > 1) {
#pragma unroll
          for (int o = 1; o < 64; o <<= 1) {
            const int t = __shfl_up(upto, o, 64);
            if (lane >= o) upto += t;
          }
        }
        const int total = __builtin_amdgcn_readlane(upto, nw - 1);
        if (total < ntl) {
          for (int w = 0; w < nw; ++w) {
            const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)m, w), up = __builtin_amdgcn_readlane((uint32_t)(m >> 32), w);
            const int before = __builtin_amdgcn_readlane(upto, w) - __popc(lo) - __popc(up);
            const int at = before + (int)__builtin_amdgcn_mbcnt_hi(up, __builtin_amdgcn_mbcnt_lo(lo, 0));
            if (((lane < 32 ? lo : up) >> l32) & 1u)
              list[ALIBI ? total - 1 - at : at] = (uint16_t)(64 * (w0 + w) + lane - first_tile);
          }
          j_hi = total;
          listed = true;
          if (total > 0) fill_walk(0);
          // The first tiles are others than those copied: again, behind this
          // wave's earlier copies to the same places. No tile at all: every
          // wave's copies are done with before the stages serve the outputs.
          bool same = total > 0;
          for (int t = 0; t < kAhead && t < total; ++t) same = same && tile_of(t) == first_tile + (ALIBI ? j_rev - t : t);
          if (DMA && !same) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            for (int t = 0; t < kAhead && t < total; ++t) tile_dma(t, tile_of(t));
          }
          if (total == 0) __syncthreads();
        }
      }
      if (j_hi > 0)
        for (int t = 0; t <= kAhead; ++t) ahead[t] = tile_of(t);
    }
  }
  const int ntile = j_hi - j_lo;
  f32x16 s_a[MT][NT];
  v8 pf[NT][KS2];
  if (ntile > 0) {
    if constexpr (DMA) {
      if constexpr (!MASK)
        for (int t = 0; t < kAhead && t < ntile; ++t) tile_dma(j_lo + t, tile_of(j_lo + t));
      load_q(std::integral_constant<int, MASK ? 2 : 0>{});
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    } else {
      load_q(std::integral_constant<int, MASK ? 2 : 0>{});
      for (int t = 0; t < kAhead && t < ntile; ++t) {
        tile_load(j_lo + t, tile_of(j_lo + t));
        tile_store(j_lo + t);
      }
    }
    ring_barrier();
    qk(Now{}, j_lo, s_a, j_lo);
  }

  {
    // Two waves share each SIMD (waves w and w+4). They run the same
    // sequence of tiles half an interval apart, so one wave's MFMA work
    // (P(j)V(j) and S(j+1)) overlaps the other's softmax:
    //   group 0: | softmax(j)  MFMA(j)       | softmax(j+1) MFMA(j+1) | ...
    //   group 1: | MFMA(j)     softmax(j+1)  | MFMA(j+1)    ...
    // Both groups touch tiles j and j+1 in interval j, so the ring is the
    // same for both.
    if (wave >= 4 && ntile > 0) vpart(Now{}, j_lo, s_a, pf);
    auto step = [&](auto last, int j) {
      ring_begin(j);
      if (wave < 4) {
        vpart(Now{}, j, s_a, pf);
        ring_mid(j);
        mphase(last, j, pf, s_a);
      } else {
        mphase(last, j, pf, s_a);
        ring_mid(j);
        if constexpr (!decltype(last)::value)
          if (j + 1 < j_hi) vpart(Next{}, j + 1, s_a, pf);
      }
      ring_end(j);
      if constexpr (MASK) {
#pragma unroll
        for (int t = 0; t < kAhead; ++t) ahead[t] = ahead[t + 1];
        ahead[kAhead] = tile_of(j + 1 + kAhead);
      }
    };
    // Unrolled by the ring depth, so every stage address is a constant; the
    // last step is peeled at head_dim <= 128.
    constexpr bool kPeel = D <= 128;
    const std::false_type more{};
    const int nmid = kPeel ? ntile - 1 : ntile;
    for (int t = 0; t < nmid; t += kStages) {
      // (the steps from t look at most kStages + kAhead ahead of it)
      if constexpr (MASK && WALK)
        if (t - walk0 >= 32) fill_walk(t);
      step(more, j_lo + t);
      if (t + 1 < nmid) step(more, j_lo + t + 1);
      if (t + 2 < nmid) step(more, j_lo + t + 2);
      if (t + 3 < nmid) step(more, j_lo + t + 3);
    }
    if constexpr (kPeel)
      if (ntile > 0) step(std::true_type{}, j_hi - 1);
  }

  // ---- epilogue ------------------------------------------------------------
  T* obase = reinterpret_cast<T*>(a.o) + (a.cu_seqlens_q ? 0 : (int64_t)b * a.o_stride_b) +
             (int64_t)hq * a.o_stride_h;
  // 16-bit rows go out through LDS. A lane holds 4-element pieces of its
  // query row, so direct stores hand L2 16-byte pieces of 32 rows per
  // instruction: ~4000 partial-line writes per workgroup and item at D = 128,
  // 4500-8300 clocks to issue on cfg2 (s_memtime probe) while the next item
  // waits at its first barrier. Through LDS each store instruction writes 4
  // (D = 128, 256) or 8 (D = 64) whole 256-byte (128-byte) row pieces; rows of
  // D = 256 go in two 128-column halves through the same space. The staging
  // stages are those of tiles j_hi - 3 and j_hi - 2 (or of no tile): every
  // wave passed its last read of them before the barrier that opened
  // interval j_hi - 1, no copy into them is outstanding, and the last
  // interval reads only V^T(j_hi - 1) (and, unpeeled, stage j_hi's K').
  // Chunk c of row r sits at chunk c ^ (r mod CH) of the row, so neither the
  // writes (one row per lane) nor the reads (a row per CH lanes) meet on a
  // few banks.
  if constexpr (KSPLIT) {
    if (npieces > 1) {
      static_assert(NT == 1 && WAVES * 32 == kPieceRows, "a piece is 256 rows");
      const int64_t slot = ((int64_t)pair * p.qtiles + qt) * p.ksplit + piece;
      float* po = p.pieces + slot * (kPieceBytes<D> / 4);
      const int row = wave_u * 32 + l32;
#pragma unroll
      for (int md = 0; md < MD; ++md)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr)
          st_vec<f32x4>(po + ((8 * md + 2 * rr + hi) * kPieceRows + row) * 4,
                        f32x4{oacc[md][0][4 * rr], oacc[md][0][4 * rr + 1], oacc[md][0][4 * rr + 2], oacc[md][0][4 * rr + 3]});
      const float lsum = half_sum((l_run[0][0] + l_run[0][1]) + (l_run[0][2] + l_run[0][3]));
      if (hi == 0) {
        po[kPieceRows * D + row] = m_run[0];
        po[kPieceRows * (D + 1) + row] = lsum;
      }
      return;
    }
  }
  constexpr bool kStageO = DMA && NT == 1;
  if constexpr (kStageO) {
    constexpr int DH = D < 128 ? D : 128;  // columns staged at a time
    constexpr int RB = DH * (int)sizeof(T);  // bytes of a staged row piece
    constexpr int CH = DH / 8;               // 16-byte chunks per piece
    constexpr int RPI = 64 / CH;             // row pieces per store instruction
    static_assert(32 * RB * 4 <= TG::BYTES, "a wave's 32 row pieces in a quarter stage");
    static_assert(kStages == 4 && kAhead == 3 && kBarrierEvery == 1,
                  "the staging stages are those no interval past j_hi - 2 reads or fills");
    const int64_t o_stride_t = a.o_stride_t;  // (read once: the stores below may alias `a` for the compiler)
    const int st = ((j_hi + 1 + (wave_u >> 2) - j_lo) & (kStages - 1));
    unsigned char* rows = smem + st * TG::BYTES + (wave_u & 3) * (32 * RB);
    const float ltot = half_sum((l_run[0][0] + l_run[0][1]) + (l_run[0][2] + l_run[0][3]));
    const float inv = ltot > 0.f ? 1.f / ltot : 0.f;
#pragma unroll
    for (int h = 0; h < D / DH; ++h) {
#pragma unroll
      for (int md = h * (DH / 32); md < (h + 1) * (DH / 32); ++md)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
          const int c = 4 * (md - h * (DH / 32)) + rr;
          const v4 ov = {(T)(oacc[md][0][4 * rr + 0] * inv), (T)(oacc[md][0][4 * rr + 1] * inv),
                         (T)(oacc[md][0][4 * rr + 2] * inv), (T)(oacc[md][0][4 * rr + 3] * inv)};
          st_vec<v4>(reinterpret_cast<T*>(rows + l32 * RB + ((c ^ (l32 & (CH - 1))) * 16) + hi * 8), ov);
        }
      // the wave's own rows: its LDS accesses complete in order
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int k = 0; k < 32 / RPI; ++k) {
        const int r = k * RPI + lane / CH;
        const int c = lane % CH;
        const v8 val = *reinterpret_cast<const v8*>(rows + r * RB + ((c ^ (r & (CH - 1))) * 16));
        const int qo = wrow0 + r;
        if (qo < g.lq) st_vec<v8>(obase + (g.q_row0 + qo) * o_stride_t + h * DH + 8 * c, val);
      }
      // (the next half's writes follow these reads in the wave's LDS order)
      asm volatile("" ::: "memory");
    }
    const int qi = wrow0 + l32;
    if (a.lse && hi == 0 && qi < g.lq) {
      const float lse = ltot > 0.f ? (m_run[0] + log2f(ltot)) * kLn2 : kNegInf;
      if (a.cu_seqlens_q)
        a.lse[(int64_t)hq * a.lse_stride_h + g.q_row0 + qi] = lse;
      else
        a.lse[(int64_t)b * a.lse_stride_b + (int64_t)hq * a.lse_stride_h + qi] = lse;
    }
    return;
  }
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const float ltot = half_sum((l_run[nt][0] + l_run[nt][1]) + (l_run[nt][2] + l_run[nt][3]));
    const float inv = ltot > 0.f ? 1.f / ltot : 0.f;
    const int qi = wrow0 + 32 * nt + l32;
    if (qi < g.lq) {
      T* orow = obase + (g.q_row0 + qi) * a.o_stride_t;
#pragma unroll
      for (int md = 0; md < MD; ++md)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
          const int d0 = 32 * md + 8 * rr + 4 * hi;
          const v4 ov = {(T)(oacc[md][nt][4 * rr + 0] * inv), (T)(oacc[md][nt][4 * rr + 1] * inv),
                         (T)(oacc[md][nt][4 * rr + 2] * inv), (T)(oacc[md][nt][4 * rr + 3] * inv)};
          st_vec<v4>(orow + d0, ov);
        }
      if (a.lse && hi == 0) {
        const float lse = ltot > 0.f ? (m_run[nt] + log2f(ltot)) * kLn2 : kNegInf;
        if (a.cu_seqlens_q)
          a.lse[(int64_t)hq * a.lse_stride_h + g.q_row0 + qi] = lse;
        else
          a.lse[(int64_t)b * a.lse_stride_b + (int64_t)hq * a.lse_stride_h + qi] = lse;
      }
    }
  }
}

// Non-persistent grid (p.persist_slots = 0): each workgroup is one item,
// ordered by grid_item. Persistent grid (dense batches with enough work, see
// the launcher): p.persist_slots resident workgroups per XCD walk a fixed
// list. The (sequence, head slice) pairs are split over the 8 XCDs in
// contiguous ranges (XCD = blockIdx % 8, as the hardware deals workgroups);
// within a pair the query tiles form couples (c, nqt - 1 - c), whose key
// tiles add up to the same count under a causal mask, and the couples are
// dealt round-robin over the XCD's workgroups (rotated by pair, so remainders
// spread). Every workgroup thus carries the same work, the XCD's workgroups
// move through its pairs together (one pair's K/V in its L2 at a time), and a
// workgroup's launch is paid once instead of per item (measured per item on
// cfg2 with one workgroup each: 3.8 us between workgroups on a CU and 0.7 us
// from launch to the first copy, beside ~1.5 us per key tile).
template <typename T, int D, int BKV, int NT, int WAVES, bool ALIBI, bool MASK, bool PERSIST>
__global__ void __launch_bounds__(WAVES * 64, 1) prefill_fa_kernel(const PrefillParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  if constexpr (!PERSIST) {
    int pair, qt;
    grid_item(p, blockIdx.x, gridDim.x, (WAVES / p.heads_per_wg) * 32 * NT, pair, qt);
    // wave-uniform by construction (the packed tail order comes out of
    // cross-lane reductions the compiler cannot see are uniform)
    pair = __builtin_amdgcn_readfirstlane(pair);
    qt = __builtin_amdgcn_readfirstlane(qt);
    fa_item<T, D, BKV, NT, WAVES, ALIBI, MASK>(p, smem, pair, qt);
  } else {
    // The arguments are read through a pointer the compiler cannot prove
    // constant across items, so it loads them again per item instead of
    // holding every one in registers across the loop (SGPR spills).
    auto args = [&]() -> const PrefillParams& {
      const __attribute__((address_space(4))) PrefillParams* pp =
          (const __attribute__((address_space(4))) PrefillParams*)__builtin_amdgcn_kernarg_segment_ptr();
      asm volatile("" : "+s"(pp));
      return *(const PrefillParams*)pp;
    };
    const int S = p.persist_slots;
    const int nqt = p.qtiles;
    const int ppx = p.persist_pairs;  // pairs per XCD
    const int ncouple = (nqt + 1) / 2;
    const int x = blockIdx.x & 7, w = blockIdx.x >> 3;
    // walk: pair i of this XCD, couple c, which tile of the couple
    int i = 0, c = w, half = 0;
    auto advance = [&](int& pair, int& qt) {
      while (c >= ncouple) {
        // next pair; this workgroup's first couple there
        if (++i >= ppx) {
          pair = -1;
          return;
        }
        c = ((w - i * ncouple) % S + S) % S;
        half = 0;
      }
      pair = x * ppx + i;
      qt = half == 0 ? nqt - 1 - c : c;
      if (half == 0 && c != nqt - 1 - c) {
        half = 1;
      } else {
        half = 0;
        c += S;
      }
    };
    int pair, qt;
    for (advance(pair, qt); pair >= 0; advance(pair, qt)) {
      fa_item<T, D, BKV, NT, WAVES, ALIBI, MASK>(args(), smem, pair, qt);
      // every wave is past its last LDS read of this item (no wait for the
      // item's output stores)
      ring_barrier();
    }
  }
}

// The pieces' grid: every item's first piece, then every item's second, ...
// (grid_item's order within each), so that the full pieces come first.
template <typename T, int D, int BKV, bool ALIBI>
__global__ void __launch_bounds__(512, 1) prefill_fa_pieces_kernel(const PrefillParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int nblk = gridDim.x / p.ksplit;
  const int piece = blockIdx.x / nblk;
  int pair, qt;
  grid_item(p, blockIdx.x % nblk, nblk, (8 / p.heads_per_wg) * 32, pair, qt);
  fa_item<T, D, BKV, 1, 8, ALIBI, false, true>(p, smem, pair, qt, piece);
}

// Adds the pieces of cut items. A workgroup takes 32 rows of an item, a thread
// one row's D/32 quarters: 8 rows x 8 quarters a wave, so that it reads
// 128-byte runs and writes 64-byte ones.
template <typename T, int D, int BKV>
__global__ void __launch_bounds__(256) merge_pieces_kernel(const PrefillParams p) {
  typedef typename Vec<T>::v4 v4;
  const goda_prefill_args& a = p.a;
  const int qt = blockIdx.x / 8, wave32 = blockIdx.x % 8, pair = blockIdx.y;
  const int hg = p.heads_per_wg, nslices = p.group / hg;
  const int qb_rows = (8 / hg) * 32;
  const int b = pair / (a.heads_kv * nslices), rem = pair % (a.heads_kv * nslices);
  const int hq = rem / nslices * p.group + rem % nslices * hg + wave32 % hg;
  const SeqGeom g = seq_geom(b, a.seqlen_q, a.seqlen_k, nullptr, nullptr, a.seqused_k);
  // the item's pieces, as fa_item counts them
  const int qr0 = qt * qb_rows;
  if (qr0 >= g.lq) return;
  const int diag = g.lk - g.lq;
  const bool use_window = a.window_left >= 0 && (a.causal || g.lq == 1);
  int kv_hi = g.lk;
  if (a.causal) kv_hi = min(kv_hi, diag + min(qr0 + qb_rows, g.lq));
  const int kv_lo = use_window ? max(0, diag + qr0 - a.window_left) : 0;
  const int all = max(0, (kv_hi > 0 ? (kv_hi + BKV - 1) / BKV : 0) - kv_lo / BKV);
  const int n = piece_count(all, piece_tiles(p, BKV), p.ksplit);
  if (n == 1) return;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int rr = 8 * wave + (lane & 7);  // row of the 32
  const int row = wave32 * 32 + rr;
  const int qi = qr0 + wave32 / hg * 32 + rr;
  const float* po = p.pieces + ((int64_t)pair * p.qtiles + qt) * p.ksplit * (kPieceBytes<D> / 4);
  constexpr int64_t kStep = kPieceBytes<D> / 4;
  float M = kNegInf;
  for (int s = 0; s < n; ++s) M = fmaxf(M, po[s * kStep + kPieceRows * D + row]);
  const float Mu = (M == kNegInf) ? 0.f : M;
  float l = 0.f;
  f32x4 o[D / 32];
#pragma unroll
  for (int c = 0; c < D / 32; ++c) o[c] = f32x4{};
  for (int s = 0; s < n; ++s) {
    const float* ps = po + s * kStep;
    const float w = fast_exp2(ps[kPieceRows * D + row] - Mu);
    l = fmaf(w, ps[kPieceRows * (D + 1) + row], l);
#pragma unroll
    for (int c = 0; c < D / 32; ++c) o[c] += w * ld_vec<f32x4>(ps + ((8 * c + (lane >> 3)) * kPieceRows + row) * 4);
  }
  if (qi >= g.lq) return;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  T* orow = reinterpret_cast<T*>(a.o) + (int64_t)b * a.o_stride_b + (int64_t)qi * a.o_stride_t + (int64_t)hq * a.o_stride_h;
#pragma unroll
  for (int c = 0; c < D / 32; ++c)
    st_vec<v4>(orow + 4 * (8 * c + (lane >> 3)), v4{(T)(o[c][0] * inv), (T)(o[c][1] * inv), (T)(o[c][2] * inv), (T)(o[c][3] * inv)});
  if (a.lse && lane < 8)
    a.lse[(int64_t)b * a.lse_stride_b + (int64_t)hq * a.lse_stride_h + qi] = l > 0.f ? (M + log2f(l)) * kLn2 : kNegInf;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// Tile shape per head dim: keys per tile, 32-row query tiles per wave, waves
// per workgroup (8 = two per SIMD, in two groups half an interval apart).
// D = 256 fits two waves per SIMD with 32-key tiles (measured 1.5x a form
// with one wave per SIMD on cfg3/cfg5).
// fp32 operands (D <= 128) double the tile bytes: D = 128 takes 32-key tiles
// so three LDS stages still fit.
template <typename T, int D>
struct Config;
template <typename T>
struct Config<T, 64> {
  static constexpr int BKV = 64, NT = 1, WAVES = 8;
};
template <typename T>
struct Config<T, 128> {
  static constexpr int BKV = sizeof(T) == 4 ? 32 : 64, NT = 1, WAVES = 8;
};
template <typename T>
struct Config<T, 256> {
  static_assert(sizeof(T) == 2, "fp32 at head_dim 256 takes prefill_f32.hip");
  static constexpr int BKV = 32, NT = 1, WAVES = 8;
};

int kv_tile_for(int d, int dtype) {
  if (dtype == GODA_DTYPE_F32) return d >= 128 ? Config<float, 128>::BKV : Config<float, 64>::BKV;
  return d >= 256 ? Config<bf16, 256>::BKV : d >= 128 ? Config<bf16, 128>::BKV : Config<bf16, 64>::BKV;
}

// Bytes of the K/V tile images in the workspace.
int64_t image_bytes(const goda_prefill_args& a) {
  const int bkv = kv_tile_for(a.head_dim, a.dtype);
  const int64_t ntiles = (a.seqlen_k + bkv - 1) / bkv;
  const int64_t elem = a.dtype == GODA_DTYPE_F32 ? 4 : 2;
  return 2 * (int64_t)a.batch * ntiles * a.heads_kv * bkv * a.head_dim * elem;
}

// Marks of the caller's mask behind the images.
int64_t marks_bytes(const goda_prefill_args& a) {
  if (!a.mask_bits) return 0;
  const int bkv = kv_tile_for(a.head_dim, a.dtype);
  const Marks k = marks_of(a, (a.seqlen_k + bkv - 1) / bkv);
  return (int64_t)k.batch * k.heads * k.blocks * k.words * 8;
}

// Workgroups of `kern` resident on the whole device at once (cached per
// device and kernel).
hipError_t resident_slots(const void* kern, int threads, size_t lds, int* out) {
  struct Entry {
    const void* kern;
    int dev, slots;
  };
  static Entry cache[64];
  static std::mutex mu;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lock(mu);
  for (const Entry& c : cache)
    if (c.kern == kern && c.dev == dev) {
      *out = c.slots;
      return hipSuccess;
    }
  int ncu = 0, per = 0;
  if ((e = hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev)) != hipSuccess) return e;
  if ((e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kern, threads, lds)) != hipSuccess) return e;
  *out = ncu * per;
  for (Entry& c : cache)
    if (!c.kern) {
      c = Entry{kern, dev, *out};
      break;
    }
  return hipSuccess;
}

int gcd_int(int x, int y) {
  while (y) {
    int t = x % y;
    x = y;
    y = t;
  }
  return x;
}

// Whether the keys of a launch's items are cut, and how (PrefillParams fields).
struct KeyPieces {
  int ksplit = 1, tiles = 0, min_piece = 0;
  int64_t items = 0;
};
// Cut where few items leave most CUs idle and the
// longest is well past an equal share of the work: a piece costs a prologue
// (about 5 tiles' time), and the cut items' sums a second launch and their way
// through memory (130 KB a piece at head_dim 128). Whole call, us, uncut / cut,
// bf16, causal (chunks: keys of 1/8 .. all of the cache):
//   items  32  B=1, 256 rows on 8448 keys, 32/8 D=128     171 /  67
//   items  16  B=2, 16 rows on 8000 keys, 32/8 D=128      137 /  54
//   items  64  B=8, 64 rows on 8448 keys, 32/8 D=128      172 / 124
//   items  96  B=1 T=4096 6/2 D=128                        92 /  66
//   items 128  B=2 T=4096 4/4 D=128                        95 /  79
//   items 128  B=1 T=4096 8/2 D=256                       169 / 156
//   items 128  B=1 T=2048 16/1 D=256                       96 / 105
//   items 128  B=4, 256 rows on 1024 keys, 32/8 D=128      41 /  44
//   items 256  B=8, 256 rows on 8448 keys, 32/8 D=128     244 / 257
//   items 256  B=2 T=2048 16/16 D=64                       48 /  62
KeyPieces key_pieces(const goda_prefill_args& a) {
  KeyPieces k;
  if (a.dtype == GODA_DTYPE_F32 || a.mask_bits || a.cu_seqlens_q || a.seqlen_q <= 0 || a.seqlen_k <= 0 || a.heads_kv <= 0) return k;
  const int bkv = kv_tile_for(a.head_dim, a.dtype);
  const int group = a.heads_q / a.heads_kv;
  const int hg = gcd_int(group, 8);
  const int rows = 8 / hg * 32;
  const int nqt = (a.seqlen_q + rows - 1) / rows;
  const int64_t per_qt = (int64_t)a.batch * a.heads_kv * (group / hg);
  k.items = prefill_mfma_workgroups(a);
  // Lengths on the device, seen by the host as the capacity alone: where they are
  // all short nothing is cut, and the second launch and the reading of the
  // lengths cost 3 to 4 us a call (capacity 8192: 8 x 16 rows on 256 keys 26 / 30,
  // on 1024 44 / 48, on 2048 68 / 60), so fewer items.
  const bool long_keys = a.seqlen_k >= 4096;
  static_assert(kMostPieceBatch == 64, "piece_tiles reads the lengths of 64 sequences, and an item is of one");
  if (a.seqused_k ? k.items > (long_keys ? kMostPieceBatch : 48) || a.seqlen_k < 2048
                  : k.items > (a.head_dim == 64 ? 64 : long_keys ? 128 : 96))
    return k;
  const int diag = a.seqlen_k - a.seqlen_q;
  const bool window = a.window_left >= 0 && (a.causal || a.seqlen_q == 1);
  int64_t total = 0;
  int longest = 0;
  for (int qt = 0; qt < nqt; ++qt) {
    const int64_t q_last = std::min<int64_t>((int64_t)(qt + 1) * rows, a.seqlen_q);
    const int64_t hi = a.causal ? std::min<int64_t>(a.seqlen_k, diag + q_last) : a.seqlen_k;
    const int64_t lo = window ? std::max<int64_t>(0, diag + (int64_t)qt * rows - a.window_left) : 0;
    const int n = (int)std::max<int64_t>(0, (hi + bkv - 1) / bkv - lo / bkv);
    total += n * per_qt;
    longest = std::max(longest, n);
  }
  k.min_piece = 8;
  const int share = (int)std::max<int64_t>(k.min_piece, (total + kCus - 1) / kCus);
  if (longest < (a.seqused_k ? 16 : share + 12)) return k;
  constexpr int most = 8;  // (bounds the workspace)
  if (a.seqused_k) {
    k.ksplit = std::min(most, (longest + k.min_piece - 1) / k.min_piece);
  } else {
    k.tiles = std::max(share, (longest + most - 1) / most);
    k.ksplit = (longest + k.tiles - 1) / k.tiles;
  }
  return k;
}
int64_t piece_bytes(int d) {
  return d == 64 ? kPieceBytes<64> : d == 128 ? kPieceBytes<128> : kPieceBytes<256>;
}

// Query tiles per pair of a packed grid: whole rounds over the 8 XCDs (extra
// tiles exit at once), or 1, 2 or 4 where the longest sequence has no more and
// the pairs divide over the XCDs' groups: the extra tiles would be up to seven
// in eight workgroups, some 4 us each. Packed prefill, 8 tiles / this: longest
// sequence of 1 tile, 16/16 D=64 191 / 57 us, 32/8 D=128 100 / 30; of 4 tiles
// 170 / 144 and 121 / 99 (longer ones: within 1.5%).
int packed_tiles(int nqt, int64_t pairs) {
  for (int g = 1; g < 8; g *= 2)
    if (nqt <= g && pairs % (8 / g) == 0) return g;
  return (nqt + 7) / 8 * 8;
}

template <typename T, int D, bool ALIBI, bool MASK>
hipError_t launch_attn(PrefillParams p, hipStream_t s) {
  typedef Config<T, D> C;
  const goda_prefill_args& a = p.a;
  const int hg = gcd_int(p.group, C::WAVES);
  p.heads_per_wg = hg;
  const int qb_rows = (C::WAVES / hg) * 32 * C::NT;
  int nqt = (a.seqlen_q + qb_rows - 1) / qb_rows;
  if (a.cu_seqlens_q) nqt = packed_tiles(nqt, (int64_t)a.batch * a.heads_kv * (p.group / hg));
  p.qtiles = nqt;
  const int64_t nblk = (int64_t)nqt * a.batch * a.heads_kv * (p.group / hg);
  if (nblk <= 0) return hipSuccess;
  if (nblk > 0x7fffffff) return hipErrorInvalidValue;
  const size_t lds = (size_t)kStages * TileGeom<T, D, C::BKV, C::WAVES>::BYTES + (MASK ? kListBytes : 0);
  auto kern = prefill_fa_kernel<T, D, C::BKV, C::NT, C::WAVES, ALIBI, MASK, false>;
  hipError_t e;
  if constexpr (!MASK && sizeof(T) == 2) {
    const KeyPieces k = key_pieces(a);
    // (a workspace that holds the tile images alone is enough for uncut items)
    if (k.ksplit > 1 && a.workspace_bytes >= prefill_mfma_workspace_bytes(a)) {
      p.ksplit = k.ksplit;
      p.piece_tiles = k.tiles;
      p.min_piece = k.min_piece;
      p.pieces = reinterpret_cast<float*>(reinterpret_cast<unsigned char*>(a.workspace) + image_bytes(a));
      auto pk = prefill_fa_pieces_kernel<T, D, C::BKV, ALIBI>;
      if ((e = hipFuncSetAttribute((const void*)pk, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)) != hipSuccess) return e;
      if ((e = record_timing(a.timing_begin, s)) != hipSuccess) return e;
      pk<<<dim3((unsigned)(nblk * k.ksplit)), 512, lds, s>>>(p);
      if ((e = hipGetLastError()) != hipSuccess) return e;
      merge_pieces_kernel<T, D, C::BKV><<<dim3(8 * nqt, (unsigned)(nblk / nqt)), 256, 0, s>>>(p);
      if ((e = hipGetLastError()) != hipSuccess) return e;
      return record_timing(a.timing_end, s);
    }
  }
  // Persistent grid (see prefill_fa_kernel): head_dim <= 128, dense batches
  // whose pairs split evenly over the 8 XCDs, more items than resident
  // workgroups.
  int64_t grid = nblk;
  p.persist_slots = p.persist_pairs = 0;
  const int64_t npairs = nblk / nqt;
  if constexpr (kPersistent<D> && !MASK) {
    if (!a.cu_seqlens_q && !a.cu_seqlens_k && npairs % 8 == 0) {
      auto pk = prefill_fa_kernel<T, D, C::BKV, C::NT, C::WAVES, ALIBI, MASK, true>;
      if ((e = hipFuncSetAttribute((const void*)pk, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)) !=
          hipSuccess)
        return e;
      int slots = 0;
      if ((e = resident_slots((const void*)pk, C::WAVES * 64, lds, &slots)) != hipSuccess) return e;
      slots -= slots % 8;
      if (slots >= 8 && nblk > slots) {
        grid = slots;
        p.persist_slots = slots / 8;
        p.persist_pairs = (int)(npairs / 8);
        kern = pk;
      }
    }
  }
  if ((e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)) !=
      hipSuccess)
    return e;
  if ((e = record_timing(a.timing_begin, s)) != hipSuccess) return e;
  kern<<<dim3((unsigned)grid), dim3(C::WAVES * 64), lds, s>>>(p);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  return record_timing(a.timing_end, s);
}

template <typename T, int D>
hipError_t launch_d(PrefillParams p, hipStream_t s) {
  constexpr int BKV = Config<T, D>::BKV;
  const goda_prefill_args& a = p.a;
  p.kv_tile = BKV;
  p.ntiles_k = (a.seqlen_k + BKV - 1) / BKV;
  if (p.ntiles_k > 0) {
    dim3 grid(p.ntiles_k, a.heads_kv, a.batch);
    if (a.mask_bits && a.workspace_bytes >= image_bytes(a) + marks_bytes(a)) {
      p.marks = reinterpret_cast<uint64_t*>(reinterpret_cast<unsigned char*>(a.workspace) + image_bytes(a));
      const int64_t waves = marks_bytes(a) / 8 / ((p.ntiles_k + 63) / 64), rows = (int64_t)a.heads_kv * a.batch;
      grid.x += (unsigned)((waves + 4 * rows - 1) / (4 * rows));
      pack_kv_kernel<T, D, BKV, true><<<grid, 256, 0, s>>>(p);
    } else {
      pack_kv_kernel<T, D, BKV, false><<<grid, 256, 0, s>>>(p);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (a.mask_bits) return a.alibi_slopes ? launch_attn<T, D, true, true>(p, s) : launch_attn<T, D, false, true>(p, s);
  return a.alibi_slopes ? launch_attn<T, D, true, false>(p, s) : launch_attn<T, D, false, false>(p, s);
}

template <typename T>
hipError_t launch_t(const PrefillParams& p, hipStream_t s) {
  switch (p.a.head_dim) {
    case 64:
      return launch_d<T, 64>(p, s);
    case 128:
      return launch_d<T, 128>(p, s);
    case 256:
      if constexpr (sizeof(T) == 2) return launch_d<T, 256>(p, s);
      return hipErrorNotSupported;
    default:
      return hipErrorNotSupported;
  }
}

}  // namespace

bool prefill_mfma_supported(const goda_prefill_args& a) {
  if (a.dtype == GODA_DTYPE_F32) return a.head_dim == 64 || a.head_dim == 128;
  if (a.dtype != GODA_DTYPE_BF16 && a.dtype != GODA_DTYPE_F16) return false;
  return a.head_dim == 64 || a.head_dim == 128 || a.head_dim == 256;
}

int64_t prefill_mfma_workgroups(const goda_prefill_args& a) {
  const int group = a.heads_q / a.heads_kv, hg = gcd_int(group, 8);
  const int rows = 8 / hg * 32;
  return (int64_t)((a.seqlen_q + rows - 1) / rows) * a.batch * a.heads_kv * (group / hg);
}

int64_t prefill_mfma_least_bytes(const goda_prefill_args& a) { return image_bytes(a); }

int64_t prefill_mfma_workspace_bytes(const goda_prefill_args& a) {
  const KeyPieces k = key_pieces(a);
  return image_bytes(a) + marks_bytes(a) + (k.ksplit > 1 ? k.items * k.ksplit * piece_bytes(a.head_dim) : 0);
}

hipError_t launch_prefill_mfma(const PrefillParams& p, hipStream_t s) {
  if (p.a.dtype == GODA_DTYPE_BF16) return launch_t<bf16>(p, s);
  if (p.a.dtype == GODA_DTYPE_F16) return launch_t<f16>(p, s);
  if (p.a.dtype == GODA_DTYPE_F32) return launch_t<float>(p, s);
  return hipErrorNotSupported;
}

}  // namespace goda
