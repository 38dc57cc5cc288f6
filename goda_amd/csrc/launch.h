// Host-side launcher declarations shared between the C-ABI layer (api.hip)
// and the kernel translation units. Internal to libgoda_attn.so.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "goda_attn.h"

namespace goda {

// Launch-ready prefill parameters: the caller's arguments plus values derived
// once on the host.
struct PrefillParams {
  goda_prefill_args a;
  int group;          // heads_q / heads_kv
  float scale_log2;   // softmax_scale * log2(e)
  int kv_tile;        // keys per workspace tile (MFMA path)
  int ntiles_k;       // ceil(seqlen_k / kv_tile)
  int heads_per_wg;   // query heads sharing one workgroup (MFMA path)
  int qtiles;         // query tiles per (sequence, head slice) in the grid (MFMA path)
  int persist_slots;  // persistent grid: resident workgroups per XCD (0: one workgroup per item)
  int persist_pairs;  // persistent grid: (sequence, head slice) pairs per XCD
  int key_split;      // fp32: waves of a workgroup sharing an item's key tiles
  int ksplit;         // 16-bit, split keys: most pieces of an item, slots an item has
  int piece_tiles;    // key tiles per piece; 0: from the lengths, on the device
  int min_piece;
  float* pieces;      // the pieces' sums, behind the tile images
  uint64_t* marks;    // key tiles that 32 query rows see of the caller's mask, behind the images; or NULL
};

struct DecodeParams {
  goda_decode_args a;
  int group;
  float scale_log2;
  int split;          // keys per work range; 0: balanced over the grid
  int grid;           // persistent workgroups (set by the launcher)
  int64_t nslots;     // partial slots in the workspace
};

// Launch-ready backward parameters.
struct BwdParams {
  goda_prefill_args a;   // the forward's arguments (o, lse: its outputs)
  goda_prefill_grads g;
  int group;
  float scale_log2;
  // Operand images in the workspace (set by the launcher).
  int ntq, ntk;          // 32-row query tiles / key tiles per sequence
  int heads_per_wg;      // query heads per dq workgroup
  int key_split;         // fp32 dq: waves of a workgroup sharing an item's key tiles
  unsigned char* qimg;   // [batch][ntq][heads_q] query-tile images
  unsigned char* kvimg;  // [batch][ntk][heads_kv] key-tile images
  // head_dim 256 or fp32: the dk/dv walk over (query head, query tile) pairs is split
  // over nsplit workgroups per key block; with nsplit > 1 they write fp32
  // partials [nsplit][dk, dv][batch * seqlen_k][heads_kv][head_dim] here.
  int nsplit;
  float* part;
  // Caller's mask, key-major for the dk/dv kernels (whose lanes hold keys):
  // word [b][h][key][query tile] holds bit r for query row 32*tile + r.
  // Broadcast dimensions of the mask keep a zero stride.
  uint32_t* mask_t;
  int64_t mt_stride_b, mt_stride_h;
  // dq from stored dS tiles (set when the launcher takes that path, else
  // null): the dk/dv kernel stores each dS tile it forms (32 query rows x 32
  // keys, 2 KB) at tile index (b * ds_per_b + row offset of its query tile +
  // key tile) * heads_q + query head. Causal batches of equal lengths keep only
  // the key tiles a query tile can see (ds_tri: query tile q holds
  // min(ntk, q + ds_c + 1) of them), others all ntk.
  unsigned char* ds;
  int64_t ds_per_b;
  int64_t ds_sink;       // byte offset past the tiles: 2 KB that only take writes
  // fp32: the (sequence, KV head) pairs of this launch, whose dS tiles the
  // buffer holds, and a pair's tiles per query head. ds_band > 0: query tile q
  // holds ds_band key tiles from the first that its window reaches.
  int pair0, npairs;
  int ds_band;
  int64_t ds_per_pair;
  int ds_c, ds_tri;
  int ds_hpw;            // query heads per workgroup of the dq-from-dS kernel
};

// Stored dS tiles: key tiles held before query tile qt of a sequence. With
// `tri`, query tile q holds min(ntk, q + c + 1) key tiles (a causal sequence
// whose keys run c tiles past its queries), else ntk.
__host__ __device__ __forceinline__ int64_t ds_row_off(int qt, int ntk, int c, bool tri) {
  if (!tri) return (int64_t)qt * ntk;
  const int m = ntk - c > 0 ? ntk - c : 0;  // tiles below m are not yet full
  const int q1 = qt < m ? qt : m;
  return (int64_t)q1 * (q1 - 1) / 2 + (int64_t)q1 * (c + 1) + (int64_t)(qt - q1) * ntk;
}
// Backward: workspace bytes (the most that a launch uses, the least that it
// runs with) and the launch.
int64_t prefill_bwd_workspace_bytes(const goda_prefill_args& a);
int64_t prefill_bwd_least_bytes(const goda_prefill_args& a);
hipError_t launch_prefill_bwd(const BwdParams& p, hipStream_t s);
// Fused QK-RMSNorm backward (norm_bwd.hip): fp32 dw partials' bytes, and dx /
// dw from the attention backward's dq / dk (gradients of the normalized rows).
int64_t norm_bwd_part_bytes(const goda_prefill_args& a);
// dL/dw of the fused norms as zeros (an empty backward: no rows, no keys).
hipError_t zero_norm_dw(const goda_prefill_args& a, const goda_prefill_grads& g, hipStream_t s);
hipError_t launch_norm_bwd(const goda_prefill_args& a, const goda_prefill_grads& g, float* part, hipStream_t s);
// Key-major mask words of the backward: (batches, heads) of the mask (1 where it
// broadcasts) x keys x 32-row query tiles; the launch that writes them to
// p.mask_t and sets their strides.
int64_t bwd_mask_t_words(const goda_prefill_args& a);
hipError_t launch_bwd_mask_t(BwdParams& p, hipStream_t s);
// fp32 backward with operands streamed from L2: bytes of the largest layout
// that `room` bytes hold, or of the smallest.
int64_t prefill_bwd_f32_workspace_bytes(const goda_prefill_args& a, int64_t room);
hipError_t launch_prefill_bwd_f32(const BwdParams& p, int64_t room, hipStream_t s);
int64_t prefill_bwd_mfma_workspace_bytes(const goda_prefill_args& a);
hipError_t launch_prefill_bwd_mfma(BwdParams p, hipStream_t s);

// Generic (VALU) prefill: any dtype, head_dim in {64,128,256}.
hipError_t launch_prefill_generic(const PrefillParams& p, hipStream_t s);

// MFMA prefill for bf16/fp16, head_dim in {64,128,256}. Returns
// hipErrorNotSupported when no tuned instance covers the arguments.
bool prefill_mfma_supported(const goda_prefill_args& a);
int64_t prefill_mfma_workspace_bytes(const goda_prefill_args& a);
// What it runs with at the least: the K/V tile images, without the room for the
// sums of items whose keys are cut (then none are) and for a mask's marks (then
// all tiles are walked).
int64_t prefill_mfma_least_bytes(const goda_prefill_args& a);
hipError_t launch_prefill_mfma(const PrefillParams& p, hipStream_t s);
// Workgroups of a dense launch (8 waves of 32 query rows each).
int64_t prefill_mfma_workgroups(const goda_prefill_args& a);

// fp32 prefill on the matrix cores with operands streamed from L2: head_dim
// 256 (more than two key tiles), and 64 / 128 where the work is small.
bool prefill_f32_streams(const goda_prefill_args& a);
int64_t prefill_f32_workspace_bytes(const goda_prefill_args& a);
hipError_t launch_prefill_f32(const PrefillParams& p, hipStream_t s);
// Waves of a workgroup that share the key tiles of an fp32 item (32 query rows
// of one head; `items` of them). Few items: four waves each, so that they fill
// the GPU. More: the longest items of a long walk still end the kernel, so they
// are shared (four ways, two at head_dim 256 with its one wave per SIMD); a
// short walk only pays the sums. Forward us at 1 / 2 / 4 waves, causal:
//   B=2 T=512 6/2 D=128      192 items   75 /  46 /  32
//   B=2 T=1000 8/2 D=256     512 items  280 / 161 / 119
//   B=16 T=512 4/4 D=128    1024 items   89 /  92 /  95 (window 128: 48 / 50 / 64)
//   B=1 T=2048 16/1 D=256   1024 items  542 / 324 / 348
//   B=1 T=2048 32/8 D=128   2048 items  430 / 308 / 320
//   B=4 T=2048 16/16 D=64   4096 items  443 / 413 / 375
//   B=8 T=4096 16/1 D=256  16384 items 8660 / 8941 / 9371
inline int f32_key_split(const goda_prefill_args& a, int64_t items) {
  int tiles = (a.seqlen_k + 31) / 32;
  if (a.window_left >= 0 && a.causal && a.window_left / 32 + 2 < tiles) tiles = a.window_left / 32 + 2;
  const int split = items <= 512 ? 4 : items > 4096 || tiles < 32 ? 1 : a.head_dim == 256 ? 2 : 4;
  return tiles >= split ? split : tiles >= 2 ? 2 : 1;
}

// Split-K decode (bf16 / fp16 / fp32).
int64_t decode_slots(const goda_decode_args& a);
int64_t decode_workspace_bytes(const goda_decode_args& a);
hipError_t launch_decode(const DecodeParams& p, hipStream_t s);

// Size of the device-resident scratch array of goda_attn_decode_noalloc: the
// split-K partials of any decode with the balanced default split
// (split_size = 0) fit, the largest being head_dim 128 with 16 query heads
// per workgroup: 2 * 2048 slots * 16 heads * (128 + 1) floats = 33.8 MB.
constexpr int64_t kDecodeScratchBytes = GODA_DECODE_NOALLOC_SCRATCH_BYTES;
// Device address of that array on the current device (looked up once per
// device with hipGetSymbolAddress).
hipError_t decode_scratch(void** ptr);

// Bit-packed boolean mask (mask.hip).
hipError_t launch_pack_mask(const goda_pack_mask_args& a, hipStream_t s);

// Document segments of packed rows (segments.hip).
hipError_t launch_doc_segments(const void* ids, int elem_bytes, int64_t stride, int rows, int cols, int32_t* scratch,
                               int32_t* cu, int32_t* out, hipStream_t s);

hipError_t launch_kv_append(const goda_kv_append_args& a, hipStream_t s);

// Records the caller's optional timing event (a hipEvent_t or NULL) on s.
inline hipError_t record_timing(void* ev, hipStream_t s) {
  if (!ev) return hipSuccess;
  return hipEventRecord(reinterpret_cast<hipEvent_t>(ev), s);
}

}  // namespace goda
