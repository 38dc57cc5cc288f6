// Helpers shared by the matrix-core attention kernels (prefill forward and
// backward).
#pragma once

#include "common.h"

namespace goda {

template <typename T>
struct Vec;
template <>
struct Vec<bf16> {
  typedef bf16x8 v8;
  typedef bf16x4 v4;
};
template <>
struct Vec<f16> {
  typedef f16x8 v8;
  typedef f16x4 v4;
};
template <>
struct Vec<float> {
  typedef f32x8 v8;
  typedef f32x4 v4;
};
// Matrix instructions issued per mfma32() call (a 32x32 tile, 16 steps of K).
template <typename T>
constexpr int kMfmaPerStep = sizeof(T) == 4 ? 8 : 1;

// 32x32 MFMA accumulator layout (gfx9 family): lane l, register r holds row
// 8*(r/4) + 4*(l/32) + r%4, column l%32; the K dimension of the A and B
// operands is split the same way (lane half h holds k = 8h..8h+7 of each
// 16-step). So the 8 accumulator registers 8g..8g+7 of one column, packed,
// form a B (or A) operand whose k index p maps to accumulator row
// 16g + kPermKey(p): a transposed operand image built in that order (an
// "image" with its 16-row groups permuted by kPermKey) multiplies the packed
// registers directly, with no register shuffles.
__host__ __device__ constexpr int kPermKey(int p) { return 8 * ((p % 8) / 4) + 4 * (p / 8) + p % 4; }

// Direct global->LDS copy by one wave of N (1, 2 or 4) consecutive 1 KB
// blocks: lane i's 16 bytes of block k go from base + lane_off + 1024 k to
// LDS byte address lds + 16 i + 1024 k (global_load_lds_dwordx4 writes lane
// i's data at m0 + 16 i, and its immediate offset moves the global source and
// the LDS destination alike; both checked in bounds on the GPU). Lanes
// outside EXEC copy nothing. Issued from inline asm, so the compiler neither
// counts these loads nor makes LDS reads wait for them: the caller waits
// (vmcnt) before the barrier that publishes the data. Sets m0, which no code
// of these kernels otherwise uses.
template <int N>
__device__ __forceinline__ void dma_blocks(unsigned lds, unsigned lane_off, unsigned long long base) {
  static_assert(N == 1 || N == 2 || N == 4, "1, 2 or 4 blocks");
  // Both are wave-uniform; readfirstlane keeps them in scalar registers where
  // the compiler would otherwise hand the "s" operands a VGPR copy (it costs
  // nothing for a value already in SGPRs).
  // (The builtin is 32-bit and returns int: each half goes back through
  // unsigned, so the low half is not sign-extended into the high one.)
  lds = (unsigned)__builtin_amdgcn_readfirstlane(lds);
  const unsigned base_hi = (unsigned)__builtin_amdgcn_readfirstlane((unsigned)(base >> 32));
  const unsigned base_lo = (unsigned)__builtin_amdgcn_readfirstlane((unsigned)base);
  base = ((unsigned long long)base_hi << 32) | base_lo;
  if constexpr (N == 1)
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds), "v"(lane_off), "s"(base) : "memory");
  else if constexpr (N == 2)
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2\n\tglobal_load_lds_dwordx4 %1, %2 offset:1024"
                 :
                 : "s"(lds), "v"(lane_off), "s"(base)
                 : "memory");
  else
    asm volatile(
        "s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2\n\tglobal_load_lds_dwordx4 %1, %2 offset:1024\n\t"
        "global_load_lds_dwordx4 %1, %2 offset:2048\n\tglobal_load_lds_dwordx4 %1, %2 offset:3072"
        :
        : "s"(lds), "v"(lane_off), "s"(base)
        : "memory");
}

// N blocks (N = 1, 2, or a multiple of 4) as dma_blocks calls of at most 4
// (the immediate offset reaches 4095 bytes).
template <int N>
__device__ __forceinline__ void dma_span(unsigned lds, unsigned lane_off, unsigned long long base) {
  if constexpr (N <= 4) {
    dma_blocks<N>(lds, lane_off, base);
  } else {
    static_assert(N % 4 == 0, "spans beyond 4 blocks come in 4s");
    dma_blocks<4>(lds, lane_off, base);
    dma_span<N - 4>(lds + 4096, lane_off, base + 4096);
  }
}

// The tile rings' barrier when their tiles arrive by dma_blocks: this wave's
// copies have landed (vmcnt(N): all but its N most recent loads), then the
// workgroup barrier makes every wave's copies visible.
template <int N>
__device__ __forceinline__ void dma_ring_barrier() {
  static_assert(N >= 0 && N < 64, "vmcnt holds 0..63");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(N) : "memory");
}

// A 32x32x16 product whose accumulator stays in VGPRs. Kernels that need
// AGPRs (more than 256 registers a wave) get the AGPR form for every
// builtin product, so score tiles that the VALU fills and reads would be
// copied into AGPRs before their products and back after them (64 moves per
// step in the head_dim-256 backward). As inline asm the compiler neither
// classifies it as a matrix product nor inserts its hazard wait states:
// mfma_vgpr_fill() separates the VALU writes of the accumulators from the
// first product, mfma_vgpr_drain() the last product from the VALU reads
// (both tie the accumulators as operands, so nothing that reads them can be
// scheduled across). Every operand is a VGPR the caller's code waits for.
__device__ __forceinline__ void mfma32_vgpr(const bf16x8& a, const bf16x8& b, f32x16& c) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
}
__device__ __forceinline__ void mfma32_vgpr(const f16x8& a, const f16x8& b, f32x16& c) {
  asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
}
// VALU write -> matrix-core read of the same VGPR: at most a few wait states.
__device__ __forceinline__ void mfma_vgpr_fill(f32x16& x, f32x16& y) {
  asm volatile("s_nop 4" : "+v"(x), "+v"(y));
}
// Matrix-core write -> VALU read: up to (passes + 3) wait states; 24 cover
// the 16-pass products.
__device__ __forceinline__ void mfma_vgpr_drain(f32x16& x, f32x16& y) {
  asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" : "+v"(x), "+v"(y));
}

// Dispatch order of a grid of `units` x `nblk` workgroups whose work falls
// with the block index (block 0: the earliest keys, or the last query tile,
// which the most causal rows / keys reach). Unit after unit, the last unit's
// heaviest block would start when little work is left (simulated makespan
// 1.19-1.23x the ideal at the cfg2 shape); here units go in chunks of
// kOrderChunk, heaviest block of every unit of the chunk first (1.0x).
// Measured: cfg2-shape backward 13.5 -> 10.7 ms, cfg3 shape 9.2 -> 6.4 ms
// (chunks of 8, 16 and 32 alike then; 4: 10.7 and 7.3 ms).
// Chunks of 8: consecutive workgroups go round-robin to the 8 XCDs, so every
// block of one unit runs on the same XCD and each XCD runs one unit at a
// time. With the dk/dv walk that reads the same query tiles in every key
// block of a unit, one unit per XCD halves the distinct tiles streaming
// through each L2 (16: two units per XCD): cfg2-shape dk/dv 5.10 -> 4.89 ms,
// dq 2.99 -> 2.89 ms.
constexpr int kOrderChunk = 8;
__device__ __forceinline__ void chunked_order(int lin, int nblk, int units, int& unit, int& blk) {
  const int base = lin / (kOrderChunk * nblk) * kOrderChunk;
  const int cc = min(kOrderChunk, units - base);
  const int r = lin - base * nblk;
  blk = r / cc;
  unit = base + r % cc;
}

// Workgroup barrier for the tile rings. __syncthreads() would also wait for
// every outstanding global access (vmcnt(0)), i.e. for the registers of the
// tile being prefetched; a ring only needs this wave's LDS accesses retired.
// The "memory" clobber keeps the compiler from moving LDS accesses across it.
__device__ __forceinline__ void ring_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

}  // namespace goda
