// Bit-packs a boolean mask along the key axis (goda_prefill_args.mask_bits):
// a thread forms one 32-key word. Bound by the one read of the mask (a byte a
// key): four 8-byte loads a thread where the keys are contiguous and aligned.
// The chain of elementwise launches and a reduction that it replaces took
// 126 us for [4, 1, 2048, 2048] and waited for a host copy on every call.

#include "common.h"
#include "launch.h"

namespace goda {
namespace {

__global__ void __launch_bounds__(256) pack_mask_kernel(const goda_pack_mask_args a) {
  const int words = 2 * ((a.keys + 63) / 64);
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t row = idx / words;
  if (row >= (int64_t)a.batch * a.heads * a.rows) return;
  const int w = (int)(idx % words);
  const int q = (int)(row % a.rows);
  const int64_t bh = row / a.rows;
  const int h = (int)(bh % a.heads), b = (int)(bh / a.heads);
  const unsigned char* src = reinterpret_cast<const unsigned char*>(a.mask) + b * a.stride_b + h * a.stride_h + q * a.stride_q;
  const int k0 = 32 * w;
  uint32_t out = 0;
  if (a.stride_k == 1 && k0 + 32 <= a.mask_keys && (reinterpret_cast<uintptr_t>(src + k0) & 7) == 0) {
    uint64_t x[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = reinterpret_cast<const uint64_t*>(src + k0)[i];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // 1 in every nonzero byte, then byte k's 1 to bit 56 + k
      const uint64_t low = 0x7f7f7f7f7f7f7f7full;
      const uint64_t one = ((((x[i] & low) + low) | x[i]) >> 7) & 0x0101010101010101ull;
      out |= (uint32_t)((one * 0x0102040810204080ull) >> 56) << (8 * i);
    }
  } else {
    for (int i = 0; i < 32; ++i)
      if (k0 + i < a.mask_keys && src[(int64_t)(k0 + i) * a.stride_k]) out |= 1u << i;
  }
  reinterpret_cast<uint32_t*>(a.bits)[idx] = out;
}

}  // namespace

hipError_t launch_pack_mask(const goda_pack_mask_args& a, hipStream_t s) {
  const int64_t n = (int64_t)a.batch * a.heads * a.rows * 2 * ((a.keys + 63) / 64);
  if (n <= 0) return hipSuccess;
  if ((n + 255) / 256 > 0x7fffffff) return hipErrorInvalidValue;
  pack_mask_kernel<<<dim3((unsigned)((n + 255) / 256)), 256, 0, s>>>(a);
  return hipGetLastError();
}

}  // namespace goda
