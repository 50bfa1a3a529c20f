// Internal declarations shared by the kernel launchers and the C ABI layer.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kvx.h"

namespace kvx {

// Blocks handled by one save/restore launch. The list travels in the kernel
// argument segment (ids + entry addresses: 12 bytes per block), so a launch
// needs no device-side index buffer and stays capturable in a HIP graph.
constexpr int kMaxBatch = 128;

struct BlockBatch {
  int32_t n;
  int32_t ids[kMaxBatch];
  uint64_t entries[kMaxBatch];
};

// n / d for 0 <= n < 2^31 and 1 <= d < 2^31 by one multiplication: with
// 2^l >= d and mul = floor(2^(31 + l) / d) + 1, mul * d exceeds 2^(31 + l) by at
// most d <= 2^l, so n times that excess stays below 2^(31 + l) and the quotient
// is exact. mul < 2^33 / 2 fits 32 bits. The kernels find a tile's entry and
// plane by it, ahead of a workgroup's first load. With two integer divisions
// instead, measured on MI355X on one card (us): FP8 saves of 128 / 48 / 16 / 1
// Qwen3-8B blocks 1108 / 466 / 141.1 / 12.2, 1092 / 436 / 137.2 / 11.7 so;
// their restores 1139.5 and 1139.1 for 128 blocks, 12.6 and 12.4 for one; BF16
// copies of 32 Qwen3-0.6B blocks 562 and 560, but of 4 Qwen3-8B ones 92.2 and
// 92.8.
struct FastDiv {
  uint32_t mul;
  uint32_t shift;
  FastDiv() = default;
  explicit FastDiv(uint32_t d) {
    uint32_t l = 0;
    while ((1u << l) < d) ++l;
    shift = 31 + l;
    mul = (uint32_t)((uint64_t{1} << shift) / d + 1);
  }
  __device__ __forceinline__ int operator()(int n) const { return (int)(((uint64_t)(uint32_t)n * mul) >> shift); }
};

// Launch-time geometry derived from kvx_block_layout. For FP8 entries, the
// payload of (entry e, plane p, row r) is at
//   entries[e] + p * payload_plane_stride + r * head_dim
// and its scale at
//   entries[e] + scale_offset + e * scale_entry_step + p * scale_plane_stride + r * scale_bytes.
// Block entries are dense per block (payload_plane_stride = plane_rows *
// head_dim, scale_plane_stride = plane_rows * scale_bytes, no entry step);
// token entries (KV handoff) are one block's rows of a [planes][rows][hd]
// payload and a [planes][rows] scale array. The batch's last entry has
// last_rows valid rows per plane (a sequence's partial final block), the
// others plane_rows.
struct PlaneGeom {
  int64_t plane_stride;  // elements
  int64_t block_stride;  // elements
  int64_t scale_offset;  // bytes from an entry's payload to its scales
  int64_t payload_plane_stride;  // bytes (FP8)
  int64_t scale_plane_stride;    // bytes (FP8)
  int64_t scale_entry_step;      // bytes (FP8)
  int32_t planes;
  int32_t plane_rows;
  int32_t last_rows;
  int32_t head_dim;
  int32_t scales16;      // every plane's scales start on 16 bytes (given 16-byte entries)
  int32_t chunks;        // tiles per plane of an entry (fewer in the last of a batch of token entries)
  int32_t outer_tiles;   // tiles per entry, or for token entries per plane over the entries of the batch
  FastDiv outer_of;      // tile -> entry, or for token entries plane (/ outer_tiles)
  FastDiv inner_of;      // tile of that -> plane, or for token entries entry (/ chunks)
};

// FP8 token entries of one launch (see PlaneGeom).
struct TokenSpan {
  int64_t payload_plane_stride;
  int64_t scale_plane_stride;
  int64_t scale_entry_step;
  int32_t last_rows;
};

// Records a message for kvx_last_error() and returns `code`.
int set_error(int code, const char* fmt, ...);
// Converts a HIP status into the ABI convention, recording a message.
int hip_status(hipError_t err, const char* what);

int check_layout(const kvx_block_layout* layout, int32_t format);

// What a pool and its entries' addresses allow. The pool's base and strides
// are multiples of 16 bytes for the last two, and the entries of 16
// (kVectorAccess: the tiled kernels) or of 8 (kPieceAccess: FP8 payloads
// written and read 8 codes at a time). kAnyAccess runs the element-granular
// kernels. Scales may start at any element in all of them.
enum Access { kAnyAccess, kPieceAccess, kVectorAccess };

// Kernel launchers: arguments are validated by the caller.
// `max_grid` > 0 caps a vector kernel's workgroups (they then stride over
// the tiles): for saves written to and restores read from host memory, which
// hold their workgroups while the bytes cross the host link.
hipError_t launch_save(const void* pool, const kvx_block_layout& layout, int32_t format,
                       const BlockBatch& batch, int64_t scale_offset, Access access, int32_t max_grid,
                       hipStream_t stream);
hipError_t launch_restore(void* pool, const kvx_block_layout& layout, int32_t format,
                          const BlockBatch& batch, int64_t scale_offset, Access access, int32_t max_grid,
                          hipStream_t stream);
// True when a restore launched with max_grid > 0 runs the striding kernel,
// whose reads of host entries are system-scope loads (the element-granular
// kernels read with plain loads and must not read host memory).
bool striding_restore_supported(const kvx_block_layout& layout, int32_t format, Access access);
// Token gather/scatter between a sequence's blocks and a dense
// [planes][rows][head_dim] buffer: entries are the dense buffer at
// block_index * plane_bytes, dense_plane_stride apart per plane, and the
// batch's last block copies last_bytes per plane.
hipError_t launch_token_copy(bool gather, void* pool, const kvx_block_layout& layout, const BlockBatch& batch,
                             Access access, int64_t dense_plane_stride, int64_t last_bytes, hipStream_t stream);
// The same with FP8 quantisation (gather) or dequantisation (scatter):
// entries are the payload rows of each block, scales per `span`.
hipError_t launch_token_fp8(bool gather, void* pool, const kvx_block_layout& layout, const BlockBatch& batch,
                            int64_t scale_offset, const TokenSpan& span, Access access, hipStream_t stream);
// The widest access this pool/entry combination allows.
Access access_of(const void* pool, const kvx_block_layout& layout, const uint64_t* entries, int32_t n);
hipError_t launch_store_kvcache(const void* key, int64_t key_stride, const void* value,
                                int64_t value_stride, void* k_cache, void* v_cache,
                                const int32_t* slot_mapping, int64_t num_tokens, int64_t row_elems,
                                int32_t elem_bytes, int64_t cache_slots, hipStream_t stream);
// Copies n bytes of pinned host memory at `src` (a device-accessible address)
// to device memory at `dst` with a kernel on `stream`; n < 2^31.
hipError_t launch_upload(void* dst, const void* src, int64_t n, hipStream_t stream);
hipError_t launch_sleep(hipStream_t stream, int64_t microseconds);
hipError_t launch_selftest(uint64_t* counters, hipStream_t stream);

}  // namespace kvx
