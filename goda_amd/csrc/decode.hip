// One-token decode attention over a contiguous KV cache (bf16 / fp16 / fp32) with
// per-sequence lengths, plus the KV append.
//
// Work decomposition (balanced split-K). The visible keys of every unit
// (sequence b, KV head, slice of that head's query heads) are laid end to end,
// sequence-major, in one flattened key space of `total` keys. The space is cut
// into ranges of `per` keys that a persistent grid of workgroups (as many as
// the GPU holds at once) takes in turn. With the default per = total / grid
// every workgroup reads the same number of cache bytes whatever the mix of
// lengths, and nothing is launched for keys that do not exist. A range covers
// pieces (segments) of one or more units:
//   - a segment that is a whole unit writes o and lse directly;
//   - a partial segment writes (o normalised, lse) to one of the range's two
//     workspace slots (slot 0: its first segment, slot 1: its last), and
//     merge_kernel combines a unit's partials:
//       lse = log sum_s exp(lse_s), o = sum_s exp(lse_s - lse) o_s.
// Inside a segment the workgroup's 4 waves take 16-key chunks in turn, each
// with its own online-softmax state, and merge through LDS at the end:
//   scores  S^T[16 keys][16 heads] = K[16 keys][D] . Q^T[D][heads]
//           on 16x16x32 MFMA; K rows are loaded straight from the cache into
//           the A operand (16 bytes per lane), Q^T lives in VGPRs. All query
//           heads of the KV head's group are served by the same K/V bytes.
//   values  O[head][d] += p[head][key] * V[key][d] on the vector ALUs, p
//           broadcast through LDS (16-bit types: packed dot products over
//           key pairs, p rounded to T); the lane mapping is described at VRows.

#include <algorithm>
#include <map>
#include <mutex>
#include <utility>

#include "common.h"
#include "launch.h"

// Split-K partials of goda_attn_decode_noalloc: a fixed device-resident array
// instead of a caller workspace, for callers that cannot allocate. Each GPU
// holds its own copy for the life of the process; every call on that GPU
// shares it, so calls that overlap on one GPU race. Nothing in it has to
// start at zero: the decode kernel writes every partial slot that the merge
// kernel of the same call reads.
static __device__ __align__(256) unsigned char scratch[goda::kDecodeScratchBytes];

namespace goda {

hipError_t decode_scratch(void** ptr) {
  // Host code must never pass `scratch` itself to a kernel (it is a host-side
  // stand-in, not a device address): its address on each device is looked up
  // once, with that device current, and kept per device.
  constexpr int kMaxDevices = 64;
  static std::mutex mu;
  static void* addr[kMaxDevices] = {};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(mu);
  if (!addr[dev]) {
    void* p = nullptr;
    if ((e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch))) != hipSuccess) return e;
    if (!p) return hipErrorInvalidSymbol;
    addr[dev] = p;
  }
  *ptr = addr[dev];
  return hipSuccess;
}

namespace {

constexpr int kWaves = 4;
constexpr int kChunk = 16;              // keys per wave step
constexpr float kRescaleThresh = 8.0f;  // log2 units
// 16-key chunks in flight per wave (depth of the register ring).
template <int D>
constexpr int kNbuf = 2;
constexpr int kMinRange = 64;           // keys; ranges are multiples of this
constexpr int kMaxGrid = 2048;          // persistent grid bound (sizes the workspace)

// Max over the four lanes l16, l16+16, l16+32, l16+48 (the key groups of one
// head): permlane16/32 swaps exchange the halves without an LDS round trip.
__device__ __forceinline__ float group_max(float x) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// Sum over the same four lanes.
__device__ __forceinline__ float group_sum(float x) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <typename T>
struct V8;
template <>
struct V8<bf16> {
  typedef bf16x8 t;
};
template <>
struct V8<f16> {
  typedef f16x8 t;
};
template <>
struct V8<float> {
  typedef f32x8 t;
};
template <typename T>
struct V4;
template <>
struct V4<bf16> {
  typedef bf16x4 t;
};
template <>
struct V4<f16> {
  typedef f16x4 t;
};
template <>
struct V4<float> {
  typedef f32x4 t;
};

// P.V lane mapping. Default: lane (kg, l16) owns head-dim chunks l16 (+16 i)
// over the chunk's keys 4 kg .. 4 kg + 3, so the four key groups hold
// partial sums of every output (reduced across lanes at the end). Slice
// (head_dim 64 or 256, or 16 query heads per workgroup): lane l owns head-dim
// elements D/64 * l .. + D/64 - 1 over all 16 keys: a quarter of the
// accumulators (D = 256, 8 heads: 32 registers instead of 128), no
// cross-lane reduction, and two waves per SIMD instead of one (cfg5 decode
// 94 -> 84 us; D = 128 with 16 heads 278 -> 212 us). With 4 or 8 heads at
// D = 128 the default mapping already fits 3 or 2 waves per SIMD and its
// 16-byte loads are 0-3% faster.
template <int D, int HMAX>
constexpr bool kPvSlice = D != 128 || HMAX >= 16;  // head_dim 64 and 256, or 16 heads
template <typename T, int D, bool SLICE>
struct VRows;
template <typename T, int D>
struct VRows<T, D, false> {
  typename V8<T>::t x[4][D / 128];  // keys 4 kg + kk, chunks l16 + 16 i
};
template <typename T, int D>
struct VRows<T, D, true> {
  static constexpr int DPL = D / 64;
  typedef T vec __attribute__((ext_vector_type(DPL)));
  vec x[kChunk];  // keys kk, elements DPL l .. DPL l + DPL - 1
};

// Wave-uniform copies (scalar registers) of values every lane holds equally.
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ long long uniform(long long x) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)x);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)((unsigned long long)x >> 32));
  return (long long)(((unsigned long long)hi << 32) | lo);
}

// Visible keys of sequence b: [kbeg, kbeg + n) with kbeg + n = its length.
__device__ __forceinline__ int visible(const goda_decode_args& a, int b, int* kbeg) {
  int L = a.cache_seqlens[b];
  L = max(0, min(L, a.max_seqlen));
  const int k0 = (a.window_left >= 0) ? max(0, L - 1 - a.window_left) : 0;
  *kbeg = k0;
  return L - k0;
}

// x / y for wave-uniform x >= 0, y > 0: in 32 bits where both fit (a 64-bit
// division is some 150 instructions).
__device__ __forceinline__ int64_t udiv(int64_t x, int64_t y) {
  if (((x | y) >> 32) == 0) return (int64_t)((uint32_t)x / (uint32_t)y);
  return x / y;
}

// Keys per range: the caller's split, else total / grid rounded up.
__device__ __forceinline__ int64_t range_keys(int64_t total, int grid, int split) {
  if (split > 0) return split;
  const int64_t q = udiv(total + grid - 1, grid);
  static_assert((kMinRange & (kMinRange - 1)) == 0, "ranges rounded up by a mask");
  return max((int64_t)kMinRange, (q + kMinRange - 1) & ~(int64_t)(kMinRange - 1));
}

// The visible key counts of up to 64 sequences in one register of the wave
// (lane = sequence) with their running sums: read and summed once for the
// total, the position of a range and the keys before a sequence. `ok` where
// 32 bits hold the sums; other batches go through the loops below.
struct Lens {
  bool ok;
  int n, k0, incl;
  __device__ __forceinline__ explicit Lens(const goda_decode_args& a) : ok(a.batch <= 64 && a.max_seqlen < (1 << 25)), n(0), k0(0), incl(0) {
    if (!ok) return;
    const int lane = threadIdx.x & 63;
    if (lane < a.batch) n = visible(a, lane, &k0);
    incl = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(incl, o, 64);
      if (lane >= o) incl += t;
    }
  }
  __device__ __forceinline__ int at(int v, int l) const { return __builtin_amdgcn_readlane(v, l); }
};

// Wave-wide sums of the visible key counts: over all sequences, and over the
// sequences before `b` (every lane returns both).
__device__ __forceinline__ void visible_sums(const goda_decode_args& a, const Lens& s64, int b, long long* all,
                                             long long* before) {
  if (s64.ok) {
    *all = s64.at(s64.incl, 63);
    *before = s64.at(s64.incl, b) - s64.at(s64.n, b);
    return;
  }
  const int lane = threadIdx.x & 63;
  long long s = 0, sb = 0;
  for (int i = lane; i < a.batch; i += 64) {
    int k0;
    const int n = visible(a, i, &k0);
    s += n;
    if (i < b) sb += n;
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    s += __shfl_xor(s, o, 64);
    sb += __shfl_xor(sb, o, 64);
  }
  *all = uniform(s);
  *before = uniform(sb);
}

// Position in the flattened key space: sequence b whose block of U * n keys
// starts at `base` and holds the position.
struct Cursor {
  int b, kbeg, n;
  int64_t base;
};

// The sequence holding flattened position R (R < total), by a wave-wide
// inclusive scan of U * n over 64 sequences at a time.
__device__ Cursor locate(const goda_decode_args& a, const Lens& s64, int U, int64_t R) {
  const int lane = threadIdx.x & 63;
  if (s64.ok) {
    const uint64_t hit = __builtin_amdgcn_ballot_w64((int64_t)U * s64.incl > R);
    const int l = __builtin_ctzll(hit);  // (R < total: some lane's sum exceeds it)
    const int n = s64.at(s64.n, l);
    return Cursor{l, s64.at(s64.k0, l), n, (int64_t)U * (s64.at(s64.incl, l) - n)};
  }
  long long base = 0;
  Cursor c{0, 0, 0, 0};
  for (int b0 = 0; b0 < a.batch; b0 += 64) {
    const int b = b0 + lane;
    int k0 = 0;
    const long long n = b < a.batch ? (long long)U * visible(a, b, &k0) : 0;
    long long incl = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const long long t = __shfl_up(incl, o, 64);
      if (lane >= o) incl += t;
    }
    const uint64_t hit = __builtin_amdgcn_ballot_w64(base + incl > R);
    if (hit != 0) {
      const int l = __builtin_ctzll(hit);
      c.b = b0 + l;
      c.base = base + uniform(__shfl(incl - n, l, 64));
      c.n = uniform(__shfl((int)(n / U), l, 64));
      c.kbeg = uniform(__shfl(k0, l, 64));
      return c;
    }
    base += uniform(__shfl(incl, 63, 64));
  }
  return c;  // not reached for R < total
}

// Moves the cursor to the next sequence with visible keys; false if none.
__device__ __forceinline__ bool advance(const goda_decode_args& a, int U, Cursor& c) {
  c.base += (int64_t)U * c.n;
  while (c.b + 1 < a.batch) {
    ++c.b;
    c.n = visible(a, c.b, &c.kbeg);
    if (c.n > 0) return true;
  }
  return false;
}

struct Segment {
  int b, hk, hs;   // sequence, KV head, slice of its query heads
  int sbeg, send;  // absolute key positions [sbeg, send)
  int qpos;        // absolute position of the query token
  bool whole;      // the segment is the whole unit: write o directly
  int64_t slot;    // workspace slot of a partial segment
};

// The launch parameters, re-read from the kernel argument segment (scalar
// loads) wherever this is called, instead of being held in scalar registers
// across the segment loop, which spills them. The kernel's only argument sits
// at offset 0 of that segment.
__device__ __forceinline__ const DecodeParams& reload_params() {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef __attribute__((address_space(4))) const DecodeParams* ParamsPtr;
  ParamsPtr pp = (ParamsPtr)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(pp));
  return *pp;
#else
  static const DecodeParams unused{};  // host pass: never executed
  return unused;
#endif
}

template <int D, int HMAX>
struct DecodeSmem {
  float p[kWaves][kChunk][16];
  uint32_t pp[kWaves][kChunk / 2][16];  // 16-bit types: (p[key 2i], p[key 2i+1]) as T per head
  float alpha[kWaves][16];
  float m[kWaves][HMAX];
  float l[kWaves][HMAX];
  float o[kWaves][HMAX][D];
};

// 16-bit P.V on packed dot products: acc + p0 v0 + p1 v1 for the probabilities
// of two keys (rounded to T, as the row sums count them) and the two keys'
// values of one head-dim element.
__device__ __forceinline__ uint32_t pack_pair(bf16 x, bf16 y) {
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, b2{x, y});
}
__device__ __forceinline__ uint32_t pack_pair(f16 x, f16 y) {
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, h2{x, y});
}
__device__ __forceinline__ float dot2_acc(uint32_t p2, uint32_t v2, float acc, bf16) {
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(b2, p2), __builtin_bit_cast(b2, v2), acc, false);
}
__device__ __forceinline__ float dot2_acc(uint32_t p2, uint32_t v2, float acc, f16) {
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  return __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, p2), __builtin_bit_cast(h2, v2), acc, false);
}

// Attention of the segment's query heads over its keys; ends with a
// workgroup barrier so the LDS can be reused by the next segment.
template <typename T, int D, int HMAX>
__device__ __forceinline__ void run_segment(DecodeSmem<D, HMAX>& sm, const Segment& sg) {
  const DecodeParams& p = reload_params();
  typedef typename V8<T>::t v8;
  constexpr int KS = D / 32;    // k-steps of the 16x16x32 score MFMA
  constexpr int CPL = D / 128;  // 8-element head-dim chunks per lane in PV
  constexpr bool SLICE = kPvSlice<D, HMAX>;
  constexpr bool DOT2 = sizeof(T) == 2;  // packed dot products for P.V
  static_assert(CPL >= 1 || SLICE, "the default mapping needs head_dim >= 128");
  constexpr int NACC = SLICE ? D / 64 : CPL * 8;  // accumulators per head and lane
  typedef VRows<T, D, SLICE> VR;
  const goda_decode_args& a = p.a;

  const int b = sg.b;
  const int hq0 = sg.hk * p.group + sg.hs * HMAX;
  const int nh = min(HMAX, p.group - sg.hs * HMAX);
  const int sbeg = sg.sbeg, send = sg.send;
  // The lane index is made opaque per segment: otherwise the compiler hoists
  // every lane-dependent address product out of the segment loop and keeps
  // them all live through the chunk loop.
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int l16 = lane & 15;
  const int kg = lane >> 4;  // 4 lane groups of 16
  const bool head_ok = l16 < nh;
  const int qpos = sg.qpos;

  // Q^T operand: lane -> head l16, head-dim 32*ks + 8*kg + e.
  v8 qf[KS];
  {
    const T* qr = reinterpret_cast<const T*>(a.q) + (int64_t)b * a.q_stride_b +
                  (int64_t)(hq0 + min(l16, nh - 1)) * a.q_stride_h;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = head_ok ? ld_vec<v8>(qr + 32 * ks + 8 * kg) : v8{};
    if (a.q_norm_weight || a.rope_q) {
      // fp32 round trip: fused QK-RMSNorm, then RoPE, one rounding.
      float xf[KS][8];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int e = 0; e < 8; ++e) xf[ks][e] = (float)qf[ks][e];
      if (a.q_norm_weight) {
        float ss = 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int e = 0; e < 8; ++e) ss = fmaf(xf[ks][e], xf[ks][e], ss);
        const float inv = rms_scale(group_sum(ss), D, a.norm_eps);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const float* w = a.q_norm_weight + 32 * ks + 8 * kg;
#pragma unroll
          for (int e = 0; e < 8; ++e) xf[ks][e] *= inv * (1.f + w[e]);
        }
      }
      if (a.rope_q && head_ok) {
        const int pos = (a.rope_pos_abs ? 0 : qpos) + a.rope_q_offset;
#pragma unroll
        for (int ks = 0; ks < KS / 2; ++ks) {
          const int f0 = 32 * ks + 8 * kg;
          const float* cs = a.rope_cos + (int64_t)pos * (D / 2) + f0;
          const float* sn = a.rope_sin + (int64_t)pos * (D / 2) + f0;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float x1 = xf[ks][e], x2 = xf[ks + KS / 2][e];
            xf[ks][e] = x1 * cs[e] - x2 * sn[e];
            xf[ks + KS / 2][e] = x1 * sn[e] + x2 * cs[e];
          }
        }
      }
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int e = 0; e < 8; ++e) qf[ks][e] = (T)xf[ks][e];
    }
  }
  const float c = p.scale_log2;
  const bool alibi = a.alibi_slopes != nullptr;
  const float slope2 = (alibi && head_ok) ? a.alibi_slopes[hq0 + l16] * kLog2e : 0.f;

  const T* kbase = reinterpret_cast<const T*>(a.k_cache) + (int64_t)b * a.k_stride_b +
                   (int64_t)sg.hk * a.k_stride_h;
  const T* vbase = reinterpret_cast<const T*>(a.v_cache) + (int64_t)b * a.v_stride_b +
                   (int64_t)sg.hk * a.v_stride_h;

  float acc[HMAX][NACC];
#pragma unroll
  for (int h = 0; h < HMAX; ++h)
#pragma unroll
    for (int i = 0; i < NACC; ++i) acc[h][i] = 0.f;
  float m_run = kNegInf, l_run = 0.f;  // for head l16 over this lane's keys

  // Each wave takes chunks wave, wave+4, ... of 16 keys.
  const int nchunks = (send - sbeg + kChunk - 1) / kChunk;
  auto load = [&](int ch, v8 (&kf)[KS], VR& vf) {
    const int k0 = sbeg + ch * kChunk;
    // K operand rows (clamped inside the segment; masked in the softmax).
    const T* kp = kbase + (int64_t)min(k0 + l16, send - 1) * a.k_stride_t;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) kf[ks] = ld_stream<v8>(kp + 32 * ks + 8 * kg);
    if constexpr (SLICE) {
      // V rows for the PV step: every key of the chunk, this lane's elements.
#pragma unroll
      for (int kk = 0; kk < kChunk; ++kk) {
        const T* vp = vbase + (int64_t)min(k0 + kk, send - 1) * a.v_stride_t;
        vf.x[kk] = ld_stream<typename VR::vec>(vp + NACC * lane);
      }
    } else {
      // V rows for the PV step: keys k0 + 4*kg + kk, head-dim chunk l16 (+16 i).
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        const T* vp = vbase + (int64_t)min(k0 + 4 * kg + kk, send - 1) * a.v_stride_t;
#pragma unroll
        for (int i = 0; i < CPL; ++i) vf.x[kk][i] = ld_stream<v8>(vp + 8 * (l16 + 16 * i));
      }
    }
  };
  auto process = [&](int ch, const v8 (&kf)[KS], const VR& vf) {
    const int k0 = sbeg + ch * kChunk;
    f32x4 sc = f32x4{};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) sc = mfma16(kf[ks], qf[ks], sc);
    // sc[r]: head l16, key k0 + 4*kg + r.
    float t[4];
    float mx = kNegInf;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int key = k0 + 4 * kg + r;
      float x = sc[r] * c;
      if (alibi) x = fmaf(slope2, (float)(key - qpos), x);
      t[r] = (key < send) ? x : kNegInf;
      mx = fmaxf(mx, t[r]);
    }
    mx = group_max(mx);
    // Lazy rescale: the reference max of a head only moves when the chunk
    // max exceeds it by more than kRescaleThresh (log2 units).
    if (__builtin_amdgcn_ballot_w64(mx > m_run + kRescaleThresh) != 0) {
      const float m_new = fmaxf(m_run, mx);
      const float alpha = (m_run == kNegInf) ? 0.f : fast_exp2(m_run - m_new);
      m_run = m_new;
      l_run *= alpha;
      if (kg == 0) sm.alpha[wave][l16] = alpha;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int h4 = 0; h4 < HMAX / 4; ++h4) {
        const f32x4 al = ld_vec<f32x4>(&sm.alpha[wave][4 * h4]);
#pragma unroll
        for (int hh = 0; hh < 4; ++hh)
#pragma unroll
          for (int i = 0; i < NACC; ++i) acc[4 * h4 + hh][i] *= al[hh];
      }
    }
    const float m_use = (m_run == kNegInf) ? 0.f : m_run;
    if constexpr (DOT2) {
      // the probabilities as T, in key pairs; the row sum counts the rounded
      // values the products use
      T pt[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        pt[r] = (T)fast_exp2(t[r] - m_use);
        l_run += (float)pt[r];
      }
      sm.pp[wave][2 * kg][l16] = pack_pair(pt[0], pt[1]);
      sm.pp[wave][2 * kg + 1][l16] = pack_pair(pt[2], pt[3]);
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float pr = fast_exp2(t[r] - m_use);
        l_run += pr;
        sm.p[wave][4 * kg + r][l16] = pr;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if constexpr (DOT2 && SLICE) {
      // Key pairs: one packed dot product per (pair, head, element) instead
      // of two FMAs and the values' conversions (p pairs read as a broadcast).
#pragma unroll
      for (int kp = 0; kp < kChunk / 2; ++kp) {
        uint32_t vv[NACC];
#pragma unroll
        for (int e = 0; e < NACC; ++e) vv[e] = pack_pair(vf.x[2 * kp][e], vf.x[2 * kp + 1][e]);
#pragma unroll
        for (int h4 = 0; h4 < HMAX / 4; ++h4) {
          const u32x4 pv = ld_vec<u32x4>(&sm.pp[wave][kp][4 * h4]);
#pragma unroll
          for (int hh = 0; hh < 4; ++hh)
#pragma unroll
            for (int e = 0; e < NACC; ++e) acc[4 * h4 + hh][e] = dot2_acc(pv[hh], vv[e], acc[4 * h4 + hh][e], T{});
        }
      }
    } else if constexpr (SLICE) {
      // Every key of the chunk for this lane's elements and every head
      // (p is read as a broadcast: all lanes load the same LDS words).
#pragma unroll
      for (int kk = 0; kk < kChunk; ++kk) {
        float vv[NACC];
#pragma unroll
        for (int e = 0; e < NACC; ++e) vv[e] = (float)vf.x[kk][e];
#pragma unroll
        for (int h4 = 0; h4 < HMAX / 4; ++h4) {
          const f32x4 pv = ld_vec<f32x4>(&sm.p[wave][kk][4 * h4]);
#pragma unroll
          for (int hh = 0; hh < 4; ++hh)
#pragma unroll
            for (int e = 0; e < NACC; ++e) acc[4 * h4 + hh][e] = fmaf(pv[hh], vv[e], acc[4 * h4 + hh][e]);
        }
      }
    } else if constexpr (DOT2) {
      // This lane's 4 keys as two pairs, for every head of the slice.
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        uint32_t vv[CPL][8];
#pragma unroll
        for (int i = 0; i < CPL; ++i)
#pragma unroll
          for (int e = 0; e < 8; ++e) vv[i][e] = pack_pair(vf.x[2 * j][i][e], vf.x[2 * j + 1][i][e]);
#pragma unroll
        for (int h4 = 0; h4 < HMAX / 4; ++h4) {
          const u32x4 pv = ld_vec<u32x4>(&sm.pp[wave][2 * kg + j][4 * h4]);
#pragma unroll
          for (int hh = 0; hh < 4; ++hh)
#pragma unroll
            for (int i = 0; i < CPL; ++i)
#pragma unroll
              for (int e = 0; e < 8; ++e)
                acc[4 * h4 + hh][8 * i + e] = dot2_acc(pv[hh], vv[i][e], acc[4 * h4 + hh][8 * i + e], T{});
        }
      }
    } else {
      // Accumulate this lane's 4 keys for every head of the slice.
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        float vv[CPL][8];
#pragma unroll
        for (int i = 0; i < CPL; ++i)
#pragma unroll
          for (int e = 0; e < 8; ++e) vv[i][e] = (float)vf.x[kk][i][e];
#pragma unroll
        for (int h4 = 0; h4 < HMAX / 4; ++h4) {
          const f32x4 pv = ld_vec<f32x4>(&sm.p[wave][4 * kg + kk][4 * h4]);
#pragma unroll
          for (int hh = 0; hh < 4; ++hh)
#pragma unroll
            for (int i = 0; i < CPL; ++i)
#pragma unroll
              for (int e = 0; e < 8; ++e)
                acc[4 * h4 + hh][8 * i + e] = fmaf(pv[hh], vv[i][e], acc[4 * h4 + hh][8 * i + e]);
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };

  // Ring of NBUF register sets: chunk ch + (NBUF-1)*kWaves is in flight while
  // chunk ch is processed (the unrolled loop keeps every buffer index static).
  constexpr int NBUF = kNbuf<D>;
  v8 kb[NBUF][KS];
  VR vb[NBUF];
#pragma unroll
  for (int i = 0; i < NBUF - 1; ++i)
    if (wave + i * kWaves < nchunks) load(wave + i * kWaves, kb[i], vb[i]);
  for (int base = wave; base < nchunks; base += NBUF * kWaves) {
#pragma unroll
    for (int u = 0; u < NBUF; ++u) {
      const int ch = base + u * kWaves;
      if (ch < nchunks) {
        const int nxt = ch + (NBUF - 1) * kWaves;
        if (nxt < nchunks) load(nxt, kb[(u + NBUF - 1) % NBUF], vb[(u + NBUF - 1) % NBUF]);
        process(ch, kb[u], vb[u]);
      }
    }
  }

  // ---- reduce within the wave -------------------------------------------------
  l_run += shfl_xor_f(l_run, 16);
  l_run += shfl_xor_f(l_run, 32);
  if (kg == 0 && l16 < HMAX) {
    sm.m[wave][l16] = m_run;
    sm.l[wave][l16] = l_run;
  }
  if constexpr (SLICE) {
#pragma unroll
    for (int h = 0; h < HMAX; ++h)
#pragma unroll
      for (int e = 0; e < NACC; ++e) sm.o[wave][h][NACC * lane + e] = acc[h][e];
  } else {
#pragma unroll
    for (int h = 0; h < HMAX; ++h)
#pragma unroll
      for (int i = 0; i < NACC; ++i) {
        float v = acc[h][i];
        v += shfl_xor_f(v, 16);
        v += shfl_xor_f(v, 32);
        acc[h][i] = v;
      }
    if (kg == 0) {
#pragma unroll
      for (int h = 0; h < HMAX; ++h)
#pragma unroll
        for (int i = 0; i < CPL; ++i)
#pragma unroll
          for (int e = 0; e < 8; ++e) sm.o[wave][h][8 * (l16 + 16 * i) + e] = acc[h][8 * i + e];
    }
  }
  __syncthreads();

  // ---- merge the waves, write the output or the partial ----------------------
  T* obase = reinterpret_cast<T*>(a.o) + (int64_t)b * a.o_stride_b;
  float* part_o = reinterpret_cast<float*>(a.workspace);
  float* part_lse = part_o + p.nslots * HMAX * D;
  for (int idx = tid; idx < nh * D; idx += kWaves * 64) {
    const int h = idx / D, d = idx % D;
    float M = kNegInf;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) M = fmaxf(M, sm.m[w][h]);
    const float Mu = (M == kNegInf) ? 0.f : M;
    float lsum = 0.f, o = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const float f = fast_exp2(sm.m[w][h] - Mu);
      lsum = fmaf(f, sm.l[w][h], lsum);
      o = fmaf(f, sm.o[w][h][d], o);
    }
    const float inv = lsum > 0.f ? 1.f / lsum : 0.f;
    const float lse = lsum > 0.f ? (M + log2f(lsum)) * kLn2 : kNegInf;
    const int hq = hq0 + h;
    if (sg.whole) {
      obase[(int64_t)hq * a.o_stride_h + d] = (T)(o * inv);
      if (a.lse && d == 0) a.lse[(int64_t)b * a.lse_stride_b + hq] = lse;
    } else {
      part_o[(sg.slot * HMAX + h) * D + d] = o * inv;
      if (d == 0) part_lse[sg.slot * HMAX + h] = lse;
    }
  }
  __syncthreads();
}

// Waves per SIMD the register allocation must allow (1: no constraint). fp32
// operands and V rows take twice the registers of 16-bit ones.
template <typename T, int D, int HMAX>
constexpr int kDecodeOcc = sizeof(T) == 4 ? ((D == 128 && HMAX == 4) ? 2 : 1)
                                          : (D == 128 && HMAX == 4) ? 3 : kPvSlice<D, HMAX> ? 2 : 1;

// The kernel's only argument sits at offset 0 of the kernel argument segment
// (reload_params reads it from there).
template <typename T, int D, int HMAX>
__global__ void __launch_bounds__(kWaves * 64) __attribute__((amdgpu_waves_per_eu(kDecodeOcc<T, D, HMAX>)))
decode_splitk_kernel(const DecodeParams p) {
  __shared__ DecodeSmem<D, HMAX> sm;
  const goda_decode_args& a = p.a;
  const int nhs = (p.group + HMAX - 1) / HMAX;
  const int U = a.heads_kv * nhs;
  const Lens lens(a);
  long long all, unused;
  visible_sums(a, lens, 0, &all, &unused);
  const int64_t total = (int64_t)U * all;
  const int64_t per = range_keys(total, gridDim.x, p.split);
  const int64_t nranges = udiv(total + per - 1, per);

  for (int64_t r = blockIdx.x; r < nranges; r += gridDim.x) {
    const int64_t R0 = r * per;
    const int64_t R1 = min(total, R0 + per);
    Cursor cur = locate(a, lens, U, R0);
    int64_t pos = R0;
    bool first = true;
    while (pos < R1) {
      if (pos >= cur.base + (int64_t)U * cur.n && !advance(a, U, cur)) return;
      const int64_t in_b = pos - cur.base;
      const int j = uniform((int)udiv(in_b, cur.n));
      const int off = uniform((int)(in_b - (int64_t)j * cur.n));
      const int len = (int)min((int64_t)(cur.n - off), R1 - pos);
      Segment sg;
      sg.b = cur.b;
      sg.hk = j / nhs;
      sg.hs = j % nhs;
      sg.sbeg = cur.kbeg + off;
      sg.send = sg.sbeg + len;
      sg.qpos = cur.kbeg + cur.n - 1;
      sg.whole = (off == 0 && len == cur.n);
      sg.slot = 2 * r + (first ? 0 : 1);
      run_segment<T, D, HMAX>(sm, sg);
      pos += len;
      first = false;
    }
  }
}

// Combines the partials of a unit that spans several ranges, and writes
// o = 0, lse = -inf for a sequence with no visible key; units held whole by
// one range were written by the main kernel. Grid (head-dim blocks, unit,
// sequence): each thread owns one (head, d) output element.
constexpr int kMergeThreads = 256;
constexpr int kMergeBatch = 8;

template <typename T, int D, int HMAX>
__global__ void __launch_bounds__(kMergeThreads) merge_kernel(const DecodeParams p) {
  const goda_decode_args& a = p.a;
  const int nhs = (p.group + HMAX - 1) / HMAX;
  const int U = a.heads_kv * nhs;
  const int j = blockIdx.y;
  const int b = blockIdx.z;
  const int hk = j / nhs, hs = j % nhs;
  const int hq0 = hk * p.group + hs * HMAX;
  const int nh = min(HMAX, p.group - hs * HMAX);
  const int idx = blockIdx.x * kMergeThreads + threadIdx.x;
  const int h = idx / D, d = idx % D;
  const Lens lens(a);
  long long all, before;
  visible_sums(a, lens, b, &all, &before);
  if (h >= nh) return;
  int kbeg;
  const int n = visible(a, b, &kbeg);
  T* orow = reinterpret_cast<T*>(a.o) + (int64_t)b * a.o_stride_b + (int64_t)(hq0 + h) * a.o_stride_h;
  float* lse_out = a.lse ? a.lse + (int64_t)b * a.lse_stride_b + hq0 + h : nullptr;
  if (n == 0) {
    orow[d] = (T)0.f;
    if (lse_out && d == 0) *lse_out = kNegInf;
    return;
  }
  const int64_t total = (int64_t)U * all;
  const int64_t per = range_keys(total, p.grid, p.split);
  const int64_t S = (int64_t)U * before + (int64_t)j * n;
  const int64_t r0 = udiv(S, per), r1 = udiv(S + n - 1, per);
  if (r0 == r1) return;  // written whole by the range that holds it
  const float* part_o = reinterpret_cast<const float*>(a.workspace);
  const float* part_lse = part_o + p.nslots * HMAX * D;
  // The unit is the last segment of range r0 (slot 1) unless it starts that
  // range (slot 0), and the first segment (slot 0) of every later range.
  const int64_t slot0 = 2 * r0 + (S == r0 * per ? 0 : 1);
  // One pass, kMergeBatch partials' loads in flight: each batch moves the
  // reference max and brings the sums so far to it. (A pass over the lse values
  // and then one over both, four at a time, took 8.6 us for units of some 16
  // partials: a chain of round trips to memory.)
  float M = kNegInf, wsum = 0.f, o = 0.f;
  for (int64_t rb = r0; rb <= r1; rb += kMergeBatch) {
    float ls[kMergeBatch], ov[kMergeBatch];
#pragma unroll
    for (int i = 0; i < kMergeBatch; ++i) {
      const int64_t r = min(rb + i, r1);
      const int64_t sl = r == r0 ? slot0 : 2 * r;
      ls[i] = part_lse[sl * HMAX + h];
      ov[i] = part_o[(sl * HMAX + h) * D + d];
    }
    float m = M;
#pragma unroll
    for (int i = 0; i < kMergeBatch; ++i) {
      if (rb + i > r1) {
        ls[i] = kNegInf;
        ov[i] = 0.f;
      }
      m = fmaxf(m, ls[i]);
    }
    const float mu = (m == kNegInf) ? 0.f : m;
    const float f = __expf(M - mu);
    wsum *= f;
    o *= f;
#pragma unroll
    for (int i = 0; i < kMergeBatch; ++i) {
      const float w = __expf(ls[i] - mu);
      wsum += w;
      o = fmaf(w, ov[i], o);
    }
    M = m;
  }
  orow[d] = (T)(wsum > 0.f ? o / wsum : 0.f);
  if (lse_out && d == 0) *lse_out = wsum > 0.f ? M + logf(wsum) : kNegInf;
}

// Workgroups of `kernel` the device holds at once (cached per device).
hipError_t persistent_grid(const void* kernel, int* grid) {
  static std::mutex mu;
  static std::map<std::pair<const void*, int>, int> cache;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lock(mu);
  auto it = cache.find({kernel, dev});
  if (it != cache.end()) {
    *grid = it->second;
    return hipSuccess;
  }
  int cus = 0, occ = 0;
  if ((e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)) != hipSuccess) return e;
  if ((e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kernel, kWaves * 64, 0)) != hipSuccess) return e;
  const int g = max(1, min(kMaxGrid, cus * max(1, occ)));
  cache[{kernel, dev}] = g;
  *grid = g;
  return hipSuccess;
}

template <typename T, int D, int HMAX>
hipError_t launch_hd(DecodeParams p, hipStream_t s) {
  const goda_decode_args& a = p.a;
  hipError_t e =
      persistent_grid(reinterpret_cast<const void*>(&decode_splitk_kernel<T, D, HMAX>), &p.grid);
  if (e != hipSuccess) return e;
  if ((e = record_timing(a.timing_begin, s)) != hipSuccess) return e;
  decode_splitk_kernel<T, D, HMAX><<<p.grid, kWaves * 64, 0, s>>>(p);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if ((e = record_timing(a.timing_end, s)) != hipSuccess) return e;
  const int nhs = (p.group + HMAX - 1) / HMAX;
  const dim3 mgrid((HMAX * D + kMergeThreads - 1) / kMergeThreads, a.heads_kv * nhs, a.batch);
  merge_kernel<T, D, HMAX><<<mgrid, kMergeThreads, 0, s>>>(p);
  return hipGetLastError();
}

// Query heads per workgroup for a GQA group size (the launch_d dispatch).
int decode_hmax(const goda_decode_args& a) {
  const int group = a.heads_q / a.heads_kv;
  if (group <= 4) return 4;
  if (group <= 8 || a.head_dim > 128) return 8;
  return 16;
}

template <typename T, int D>
hipError_t launch_d(const DecodeParams& p, hipStream_t s) {
  if (p.group <= 4) return launch_hd<T, D, 4>(p, s);
  if constexpr (D > 128) {
    return launch_hd<T, D, 8>(p, s);
  } else {
    if (p.group <= 8) return launch_hd<T, D, 8>(p, s);
    return launch_hd<T, D, 16>(p, s);
  }
}

template <typename T>
hipError_t launch_t(const DecodeParams& p, hipStream_t s) {
  if (p.a.head_dim == 64) return launch_d<T, 64>(p, s);
  if (p.a.head_dim == 128) return launch_d<T, 128>(p, s);
  if (p.a.head_dim == 256) return launch_d<T, 256>(p, s);
  return hipErrorNotSupported;
}

// ---------------------------------------------------------------------------
// KV append: rows [pos_b, pos_b + T_new) of sequence b receive the new k
// (optionally RMS-normalised, then rotated at its absolute position) and v,
// with pos_b = cache_seqlens[b] read on the device. One workgroup per (new
// row, sequence), one wave per KV head at a time: lane l holds head-dim
// elements l + 64 m, so a row's norm is one wave reduction and each RoPE pair
// (i, i + D/2) sits in one lane (D >= 128) or in lanes l, l ^ 32 (D = 64).
// The lengths are advanced by a second launch on the same stream, so every
// workgroup of the first one has read the old positions before they change;
// kv_append_few_kernel does both where one workgroup holds a sequence's rows.
// ---------------------------------------------------------------------------
template <typename T, int D>
__device__ __forceinline__ void append_row(const goda_kv_append_args& a, int b, int t, int h, int pos, int lane) {
  constexpr int M = D / 64;  // elements per lane
  const T* kn = reinterpret_cast<const T*>(a.k_new) + (int64_t)b * a.kn_stride_b + (int64_t)t * a.kn_stride_t + (int64_t)h * a.kn_stride_h;
  const T* vn = reinterpret_cast<const T*>(a.v_new) + (int64_t)b * a.vn_stride_b + (int64_t)t * a.vn_stride_t + (int64_t)h * a.vn_stride_h;
  T* kc = reinterpret_cast<T*>(a.k_cache) + (int64_t)b * a.k_stride_b + (int64_t)pos * a.k_stride_t + (int64_t)h * a.k_stride_h;
  T* vc = reinterpret_cast<T*>(a.v_cache) + (int64_t)b * a.v_stride_b + (int64_t)pos * a.v_stride_t + (int64_t)h * a.v_stride_h;
  const int rp = (a.rope_pos_abs ? t : pos) + a.rope_k_offset;
  float x[M];
  T v[M];
#pragma unroll
  for (int m = 0; m < M; ++m) {
    x[m] = Elem<T>::to_f32(kn[lane + 64 * m]);
    v[m] = vn[lane + 64 * m];
  }
  if (a.k_norm_weight) {
    float ss = 0.f;
#pragma unroll
    for (int m = 0; m < M; ++m) ss = fmaf(x[m], x[m], ss);
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) ss += shfl_xor_f(ss, o);
    const float inv = rms_scale(ss, D, a.norm_eps);
#pragma unroll
    for (int m = 0; m < M; ++m) x[m] *= inv * (1.f + a.k_norm_weight[lane + 64 * m]);
  }
  if (a.rope_k) {
    if constexpr (M == 1) {
      // pair (l, l + 32): lanes l < 32 hold x1, lanes l >= 32 hold x2
      const float other = shfl_xor_f(x[0], 32);
      const int f = lane & 31;
      const float c = a.rope_cos[(int64_t)rp * (D / 2) + f], sn = a.rope_sin[(int64_t)rp * (D / 2) + f];
      x[0] = lane < 32 ? x[0] * c - other * sn : other * sn + x[0] * c;
    } else {
#pragma unroll
      for (int m = 0; m < M / 2; ++m) {
        const int f = lane + 64 * m;
        const float c = a.rope_cos[(int64_t)rp * (D / 2) + f], sn = a.rope_sin[(int64_t)rp * (D / 2) + f];
        const float x1 = x[m], x2 = x[m + M / 2];
        x[m] = x1 * c - x2 * sn;
        x[m + M / 2] = x1 * sn + x2 * c;
      }
    }
  }
#pragma unroll
  for (int m = 0; m < M; ++m) {
    kc[lane + 64 * m] = Elem<T>::from_f32(x[m]);
    vc[lane + 64 * m] = v[m];
  }
}

template <typename T, int D>
__global__ void __launch_bounds__(256) kv_append_kernel(const goda_kv_append_args a) {
  const int t = blockIdx.x;
  const int b = blockIdx.y;
  const int pos = a.cache_seqlens[b] + t;
  if (pos < 0 || pos >= a.max_seqlen) return;
  for (int h = threadIdx.x >> 6; h < a.heads_kv; h += 4) append_row<T, D>(a, b, t, h, pos, threadIdx.x & 63);
}

// Length `len` plus `add`, clamped to [0, lmax] (a sequence that would pass the
// end keeps the rows that fit); the overflow is reported through `status`.
__device__ __forceinline__ void bump(int32_t* len, int add, int lmax, int32_t* status) {
  const int64_t to = (int64_t)*len + add;
  *len = (int32_t)(to > lmax ? lmax : to < 0 ? 0 : to);
  if ((to > lmax || to < 0) && status) *status = 1;
}

// A few rows (a generation step's token): one workgroup writes all rows of a
// sequence, a wave per (row, head), and then advances its length, in one launch.
constexpr int kFewRows = 64;  // (row, head) pairs of a sequence: four rounds of the 16 waves
template <typename T, int D>
__global__ void __launch_bounds__(1024) kv_append_few_kernel(const goda_kv_append_args a) {
  const int b = blockIdx.x;
  const int pos = a.cache_seqlens[b];
  for (int i = threadIdx.x >> 6; i < a.seqlen_new * a.heads_kv; i += blockDim.x >> 6) {
    const int t = i / a.heads_kv;
    if (pos + t >= 0 && pos + t < a.max_seqlen) append_row<T, D>(a, b, t, i % a.heads_kv, pos + t, threadIdx.x & 63);
  }
  __syncthreads();  // every wave has read the old length
  if (threadIdx.x == 0) bump(a.cache_seqlens + b, a.seqlen_new, a.max_seqlen, a.status);
}

__global__ void kv_bump_kernel(int32_t* seqlens, int n, int add, int lmax, int32_t* status) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b < n) bump(seqlens + b, add, lmax, status);
}

template <typename T>
hipError_t launch_append_few(const goda_kv_append_args& a, hipStream_t s) {
  const int waves = std::min(16, a.seqlen_new * a.heads_kv);
  switch (a.head_dim) {
    case 64:
      kv_append_few_kernel<T, 64><<<a.batch, 64 * waves, 0, s>>>(a);
      break;
    case 128:
      kv_append_few_kernel<T, 128><<<a.batch, 64 * waves, 0, s>>>(a);
      break;
    case 256:
      kv_append_few_kernel<T, 256><<<a.batch, 64 * waves, 0, s>>>(a);
      break;
    default:
      return hipErrorNotSupported;
  }
  return hipGetLastError();
}

template <typename T>
hipError_t launch_append_t(const goda_kv_append_args& a, hipStream_t s) {
  if (a.seqlen_new > 0 && (int64_t)a.seqlen_new * a.heads_kv <= kFewRows) return launch_append_few<T>(a, s);
  if (a.seqlen_new > 0) {
    const dim3 grid(a.seqlen_new, a.batch);
    switch (a.head_dim) {
      case 64:
        kv_append_kernel<T, 64><<<grid, 256, 0, s>>>(a);
        break;
      case 128:
        kv_append_kernel<T, 128><<<grid, 256, 0, s>>>(a);
        break;
      case 256:
        kv_append_kernel<T, 256><<<grid, 256, 0, s>>>(a);
        break;
      default:
        return hipErrorNotSupported;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  kv_bump_kernel<<<(a.batch + 255) / 256, 256, 0, s>>>(a.cache_seqlens, a.batch, a.seqlen_new, a.max_seqlen,
                                                        a.status);
  return hipGetLastError();
}

}  // namespace

int64_t decode_slots(const goda_decode_args& a) {
  // Ranges are at most ceil(total / split), or with the balanced default at
  // most min(grid, ceil(total / kMinRange)); total <= units * batch * max_seqlen.
  const int group = a.heads_q / a.heads_kv;
  const int hmax = decode_hmax(a);
  const int64_t units = (int64_t)a.heads_kv * ((group + hmax - 1) / hmax);
  const int64_t tmax = units * a.batch * (int64_t)a.max_seqlen;
  const int64_t per = a.split_size > 0 ? a.split_size : kMinRange;
  int64_t ranges = (tmax + per - 1) / per;
  if (a.split_size <= 0) ranges = std::min<int64_t>(ranges, kMaxGrid);
  return 2 * ranges;
}

int64_t decode_workspace_bytes(const goda_decode_args& a) {
  if (a.batch <= 0 || a.max_seqlen <= 0) return 0;
  return decode_slots(a) * decode_hmax(a) * (a.head_dim + 1) * (int64_t)sizeof(float);
}

hipError_t launch_decode(const DecodeParams& p, hipStream_t s) {
  if (p.a.dtype == GODA_DTYPE_BF16) return launch_t<bf16>(p, s);
  if (p.a.dtype == GODA_DTYPE_F16) return launch_t<f16>(p, s);
  if (p.a.dtype == GODA_DTYPE_F32) return launch_t<float>(p, s);
  return hipErrorNotSupported;
}

hipError_t launch_kv_append(const goda_kv_append_args& a, hipStream_t s) {
  switch (a.dtype) {
    case GODA_DTYPE_F32:
      return launch_append_t<float>(a, s);
    case GODA_DTYPE_F16:
      return launch_append_t<f16>(a, s);
    case GODA_DTYPE_BF16:
      return launch_append_t<bf16>(a, s);
    default:
      return hipErrorNotSupported;
  }
}

}  // namespace goda
