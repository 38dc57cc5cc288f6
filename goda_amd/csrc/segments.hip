// Document segments of packed rows (goda's doc_ids, mint/nn/flashattn.py:98-137):
// the cumulative starts of the maximal runs of equal ids inside each row, the
// longest run, and whether an id occupies more than one run of its row. Two
// launches and one small read-back take the place of a chain of some 25
// elementwise, sort, scan and reduction launches with two read-backs (a
// training pass over B=4, T=2048, 6 documents a row spent about 140 us of GPU
// time and two synchronizations there). Latency-bound: a workgroup per row.

#include "common.h"
#include "launch.h"

namespace goda {
namespace {

constexpr int kThreads = 256;
// Rows whose ids are not strictly monotonic over their runs are checked pair by
// pair, up to this many runs.
constexpr int kMaxPairs = 1024;

__device__ __forceinline__ int block_sum(int x, int* sh) {
  for (int o = 32; o >= 1; o >>= 1) x += __shfl_xor(x, o, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = x;
  __syncthreads();
  return sh[0] + sh[1] + sh[2] + sh[3];
}
__device__ __forceinline__ int block_max(int x, int* sh) {
  for (int o = 32; o >= 1; o >>= 1) x = max(x, __shfl_xor(x, o, 64));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = x;
  __syncthreads();
  return max(max(sh[0], sh[1]), max(sh[2], sh[3]));
}

// Per row: the columns at which runs start (starts[row][0 .. count)), and
// stat[row] = {count, longest run, recurring (0 no, 1 yes, 2 not determined)}.
template <typename I>
__global__ void __launch_bounds__(kThreads) row_runs_kernel(const I* ids, int64_t stride, int cols, int32_t* starts,
                                                            int32_t* stat) {
  const int row = blockIdx.x, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const I* r = ids + row * stride;
  int32_t* out = starts + (int64_t)row * cols;
  __shared__ int sh[4];
  __shared__ I run_id[kMaxPairs];
  int count = 0;
  for (int c0 = 0; c0 < cols; c0 += kThreads) {
    const int c = c0 + tid;
    const bool start = c < cols && (c == 0 || r[c] != r[c - 1]);
    const uint64_t m = __builtin_amdgcn_ballot_w64(start);
    __syncthreads();
    if (lane == 0) sh[wave] = __popcll(m);
    __syncthreads();
    int at = count;
    for (int w = 0; w < wave; ++w) at += sh[w];
    at += __popcll(m & ((1ull << lane) - 1));
    if (start) {
      out[at] = c;
      if (at < kMaxPairs) run_id[at] = r[c];
    }
    count += sh[0] + sh[1] + sh[2] + sh[3];
  }
  __threadfence_block();
  __syncthreads();
  int longest = 0;
  bool up = true, down = true;
  for (int k = tid; k < count; k += kThreads) {
    const int next = k + 1 < count ? out[k + 1] : cols;
    longest = max(longest, next - out[k]);
    if (k + 1 < count) {
      const I x = r[out[k]], y = r[next];
      up = up && x < y;
      down = down && x > y;
    }
  }
  longest = block_max(longest, sh);
  const bool monotonic = block_sum(up ? 0 : 1, sh) == 0 || block_sum(down ? 0 : 1, sh) == 0;
  int rec = 0;
  if (!monotonic) {
    if (count > kMaxPairs) {
      rec = 2;
    } else {
      int hit = 0;
      for (int k = tid; k < count; k += kThreads)
        for (int j = 0; j < k; ++j) hit |= run_id[j] == run_id[k] ? 1 : 0;
      rec = block_max(hit, sh);
    }
  }
  if (tid == 0) {
    stat[3 * row] = count;
    stat[3 * row + 1] = longest;
    stat[3 * row + 2] = rec;
  }
}

// cu[0 .. total]: every row's starts behind those of the rows before it, and
// the end; out = {total, longest run, recurring}.
__global__ void __launch_bounds__(kThreads) compact_kernel(const int32_t* starts, const int32_t* stat, int rows, int cols,
                                                           int32_t* cu, int32_t* out) {
  const int row = blockIdx.x, tid = threadIdx.x;
  __shared__ int sh[4];
  int before = 0;
  for (int i = tid; i < row; i += kThreads) before += stat[3 * i];
  before = block_sum(before, sh);
  const int count = stat[3 * row];
  for (int k = tid; k < count; k += kThreads) cu[before + k] = row * cols + starts[(int64_t)row * cols + k];
  if (row == rows - 1) {
    int longest = 0, rec = 0;
    for (int i = tid; i < rows; i += kThreads) {
      longest = max(longest, stat[3 * i + 1]);
      rec = max(rec, stat[3 * i + 2]);
    }
    longest = block_max(longest, sh);
    rec = block_max(rec, sh);
    if (tid == 0) {
      cu[before + count] = rows * cols;
      out[0] = before + count;
      out[1] = longest;
      out[2] = rec;
    }
  }
}

}  // namespace

// Scratch: starts [rows][cols], then 3 words a row.
hipError_t launch_doc_segments(const void* ids, int elem_bytes, int64_t stride, int rows, int cols, int32_t* scratch,
                               int32_t* cu, int32_t* out, hipStream_t s) {
  int32_t* stat = scratch + (int64_t)rows * cols;
  if (elem_bytes == 8)
    row_runs_kernel<int64_t><<<rows, kThreads, 0, s>>>(reinterpret_cast<const int64_t*>(ids), stride, cols, scratch, stat);
  else
    row_runs_kernel<int32_t><<<rows, kThreads, 0, s>>>(reinterpret_cast<const int32_t*>(ids), stride, cols, scratch, stat);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  compact_kernel<<<rows, kThreads, 0, s>>>(scratch, stat, rows, cols, cu, out);
  return hipGetLastError();
}

}  // namespace goda
