// Operand images and products shared by the fp32 matrix-core kernels
// (prefill_f32.hip, backward_f32.hip).
//
// v_mfma_f32_32x32x2_f32 multiplies true fp32 operands; a 32x32 tile takes 64
// clocks per two steps of K, one 4-byte operand element a lane each. A chunk
// is four such products: 16 bytes a lane, 256 clocks. Lane half h of a chunk
// holds k = 4h .. 4h + 3 of each 8 steps of K, the same on both operands.
// An image is the D/8 chunks of a 32-row tile in the order a kernel reads
// them, 1 KB each, lane l (half h = l / 32) at 16 l:
//   row image         chunk s holds elements 8s + 4h + e of row l % 32: the A
//                     or B operand of a product over head_dim
//   transposed image  chunk g * D/32 + md holds rows 8g + 4h + e of head-dim
//                     32 md + l % 32: the A operand of a product over the
//                     tile's rows; accumulator register 4g + e of lane half h
//                     is row 8g + 4h + e, so a 32x32 accumulator is the B
//                     operand in place
#pragma once

#include "common.h"
#include "mfma_common.h"

namespace goda {

constexpr int kF32Rows = 32;  // rows (queries or keys) of a tile

// Bytes of one image of a tile.
template <int D>
constexpr int kF32Img = D * kF32Rows * 4;

// c += the four products of one chunk.
__device__ __forceinline__ f32x16 mfma_chunk(f32x4 a, f32x4 b, f32x16 c) {
#pragma unroll
  for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], b[e], c, 0, 0, 0);
  return c;
}
// Accumulator registers 4g .. 4g + 3 as a B operand chunk.
__device__ __forceinline__ f32x4 acc_chunk(const f32x16& x, int g) {
  return f32x4{x[4 * g], x[4 * g + 1], x[4 * g + 2], x[4 * g + 3]};
}

// Chunk c of an image: a wave-uniform base and this lane's byte offset 16 l.
__device__ __forceinline__ f32x4 img_chunk(const unsigned char* img, int c, unsigned lane16) {
  return *reinterpret_cast<const f32x4*>(img + c * 1024 + lane16);
}

// Writes the images of one staged 32-row tile from LDS, 256 threads: chunk c
// goes to chunk position c * STEP of img.
template <int D, int STEP = 1>
__device__ __forceinline__ void write_row_image(const float (*rows)[D + 4], unsigned char* img, int tid, float scale = 1.f) {
#pragma unroll 4
  for (int i = tid; i < D / 8 * 64; i += 256) {
    const int c = i / 64, l = i % 64;  // row l % 32, elements 8 c + 4 (l / 32) ..
    *reinterpret_cast<f32x4*>(img + c * STEP * 1024 + l * 16) = ld_vec<f32x4>(&rows[l % 32][8 * c + 4 * (l / 32)]) * scale;
  }
}
template <int D, int STEP = 1>
__device__ __forceinline__ void write_tr_image(const float (*rows)[D + 4], unsigned char* img, int tid) {
#pragma unroll 4
  for (int i = tid; i < D / 8 * 64; i += 256) {
    const int c = i / 64, l = i % 64;
    const int k = 8 * (c / (D / 32)) + 4 * (l / 32), d = 32 * (c % (D / 32)) + l % 32;
    *reinterpret_cast<f32x4*>(img + c * STEP * 1024 + l * 16) = f32x4{rows[k][d], rows[k + 1][d], rows[k + 2][d], rows[k + 3][d]};
  }
}

// Elements c .. c + 3 and their rotation partners c + D/2 .. of a row held by
// D/8 consecutive lanes (all of which call this): goda's RMSNorm (weight w, or
// none), then the half-split rotation at `pos` (when `rot`).
template <int D>
__device__ __forceinline__ void norm_rope_f32(f32x4& x1, f32x4& x2, int c, const float* w, float eps, bool rot, int pos,
                                              const float* rope_cos, const float* rope_sin) {
  if (w) {
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) ss = fmaf(x1[e], x1[e], fmaf(x2[e], x2[e], ss));
    const float inv = rms_scale(lane_group_sum<D / 8>(ss), D, eps);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x1[e] *= inv * (1.f + w[c + e]);
      x2[e] *= inv * (1.f + w[c + D / 2 + e]);
    }
  }
  if (rot) {
    const f32x4 cs = ld_vec<f32x4>(rope_cos + (int64_t)pos * (D / 2) + c);
    const f32x4 sn = ld_vec<f32x4>(rope_sin + (int64_t)pos * (D / 2) + c);
    const f32x4 y1 = x1 * cs - x2 * sn;
    x2 = x1 * sn + x2 * cs;
    x1 = y1;
  }
}

}  // namespace goda
