// Arguments and host entry points shared by the paged attention kernels (attention.hip: the key-
// streaming kernel of short entries, attn_tile.hip: the row-tiled kernel of long ones).
#pragma once

#include "lse_common.h"

namespace lse {

// Orders of the key-streaming kernel's grid (attn_order, attention.hip).
enum { kAttnByEntry, kAttnByTile, kAttnFirstTiles, kAttnCompact,
       kAttnCompactSplit };

struct PagedAttnArgs {
  const uint16_t* q;  // bf16, element (h, t, d) at h * sq_h + t * sq_t + d
  int64_t sq_h, sq_t;
  const uint16_t* k_pool;  // bf16 (blocks, block_size, H_KV, D): (b, w, h, d) at b sb + w sw + h sh + d
  const uint16_t* v_pool;
  int64_t sb, sw, sh;
  const int32_t* block_table;  // (entries, max_blocks), row stride sbt
  int64_t sbt;
  const int32_t* context_len;
  const int32_t* query_offset;
  const int32_t* q_start;
  const int32_t* q_len;
  uint16_t* o;  // bf16, same indexing as q with strides so_h, so_t
  int64_t so_h, so_t;
  int entries, H, HKV, G, block_size, max_q_len;
  int bs_shift;      // log2(block_size) when it is a power of two, else -1
  int tq;            // query tokens per tile: floor(16 / G)
  int qtiles;        // ceil(max_q_len / tq)
  int parts;         // 1: a workgroup folds every chunk of its item; > 1: one chunk per workgroup
  int sorted;        // entries are taken in descending order of context length...
  int first_round;   // ...and, where > 0, those from this rank on in ascending order
  float scale_log2;  // softmax scale x log2(e): scores are kept in the base-2 domain
  float* ws_o;       // parts > 1: chunk states' O [parts][entries][H][max_q_len][D], fp32
  float* ws_ml;      // parts > 1: chunk states' max and sum [parts][entries][H][max_q_len][2]
  int tiled;         // the row-tiled kernel runs too and takes the long entries (attn_is_long)
};

// Whether the row-tiled kernel takes an entry of `rows` = q_len x G query rows per K/V head; the
// key-streaming kernel takes it otherwise. The choice depends on the entry alone, so a row's bits do
// not depend on the rest of the call. Measured on MI355X (32 heads over 8; us, key-streaming against
// row-tiled): 8 entries of 64 tokens behind 1000 positions 60.0 / 27.2, one of them 23.1 / 24.2; of
// 32 tokens 49 / 26 and 22.5 / 24.3, fresh prompts of 32 tokens 6.7 / 11.5 (two launches), so 256 rows
// is where it starts. A workgroup walks its rows' whole context, so a lone short chunk far into a
// long one leaves the chip idle: one entry behind 8000 positions 55 / 98 at 64 tokens, 97 / 99 at 128,
// 181 / 102 at 256.
constexpr int kAttnTileRows = 256, kAttnTileRowsFar = 512, kAttnTileNear = 2048;
__host__ __device__ inline bool attn_is_long(int64_t rows, int ctx) {
  return rows >= kAttnTileRowsFar || (rows >= kAttnTileRows && ctx <= kAttnTileNear);
}

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

// 16-lane transposing LDS read: in each 16-lane group, lane i receives element i & 3 of the 8-byte
// reads of lanes (i >> 2) + 4 j, j = 0..3.
__device__ __forceinline__ bf16x4 lds_read_tr16(const unsigned char* p) {
  typedef __attribute__((address_space(3))) bf16x4* LdsV4;
  return __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
      (LdsV4)((__attribute__((address_space(3))) unsigned char*)p));
}

__device__ __forceinline__ float exp2_fast(float v) { return __builtin_amdgcn_exp2f(v); }

// Launches the row-tiled kernel over every entry that attn_is_long.
int launch_attn_tile(const PagedAttnArgs& a, int cus, hipStream_t stream);

}  // namespace lse
