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
  int qtiles;        // query tiles of the longest entry of this kernel
  int parts;         // 1: a workgroup folds every chunk of its item; > 1: one chunk per workgroup
  int sorted;        // entries are taken in descending order of context length...
  int first_round;   // ...and, where > 0, those from this rank on in ascending order
  float scale_log2;  // softmax scale x log2(e): scores are kept in the base-2 domain
  float* ws_o;       // parts > 1: chunk states' O [parts][entries][H][max_q_len][D], fp32
  float* ws_ml;      // parts > 1: chunk states' max and sum [parts][entries][H][max_q_len][2]
  int tiled;         // the row-tiled kernel runs too and takes the long entries (attn_is_long)
};

// Whether the row-tiled kernel takes an entry of q_len tokens; the key-streaming kernel takes it
// otherwise. The choice depends on the entry and the heads alone, so a row's bits do not depend on the
// rest of the call, and it is fitted so that an entry alone in its call is not slower for it (among
// others it gains more). The key-streaming kernel's time grows with the (query row, key) pairs; the
// row-tiled one's, with fewer items than CUs, with the context its workgroups walk, 13 us per 1000
// positions, on top of some 12 us for both launches. Measured on MI355X, us, key-streaming / row-tiled:
//  * fresh prompts, 32 heads over 8: one of 64 tokens 6 / 12, 128: 7 / 12, 256: 12 / 14, 320: 19 / 16, 512:
//    27 / 18; four of 128: 16 / 13, of 256: 36 / 16; one of 512, 8 heads over 2: 12 / 17; of 2048: 71 / 37;
//  * one entry behind 500 positions, 32 over 8: 128 tokens 14 / 19, 256: 22 / 20;
//  * behind 2000: 64 tokens 31 / 33, 128: 44 / 39; 8 heads over 2, 128: 22 / 39, 512: 49 / 45; 4 over 1,
//    512: 30 / 43, 1024: 49 / 50;
//  * behind 8000: 32 over 8, 128 tokens 101 / 114, 200: 163 / 116; 4 over 1, 512: 73 / 119, 2048: 207 / 136.
// An item is 128 rows of a K/V head, so fewer than 256 would leave much of them idle. With fewer than 8
// K/V heads (a shard's), the same work is more tokens, whose workgroups walk more of their own keys: there
// the gain alone is small (8 over 2, 512 tokens behind 2000 positions, above), and beside decode rows,
// which run after the row-tiled kernel and beside the other, it turns into a loss (50 / 72).
constexpr int kAttnTileRows = 256;            // query rows per K/V head
constexpr int kAttnTileHeads = 4096;          // q_len x H, from which with kAttnTilePairs...
constexpr int kAttnTileHeadsFar = 5120;       // ...(contexts longer than kAttnTileNear)
constexpr int kAttnTileHeadsFew = 8192;       // ...(fewer than 8 K/V heads)
constexpr int kAttnTileNear = 4096;
constexpr int64_t kAttnTilePairs = 4000000;   // (query row, key) pairs over all heads
constexpr int kAttnTileAlways = 10240;        // q_len x H, from which in any case
__host__ __device__ inline bool attn_is_long(int64_t q_len, int G, int HKV, int ctx) {
  const int64_t rows = q_len * G, heads = rows * HKV;
  const int from = HKV < 8 ? kAttnTileHeadsFew
                           : ctx > kAttnTileNear ? kAttnTileHeadsFar : kAttnTileHeads;
  return rows >= kAttnTileRows &&
         (heads >= kAttnTileAlways ||
          (heads >= from && heads * (2 * (int64_t)ctx - q_len) >= 2 * kAttnTilePairs));
}
// Whether a call may hold a long entry, from what the host knows: no more than max_q_len tokens, contexts
// within the block table's max_ctx positions.
inline bool attn_may_be_long(int64_t max_q_len, int G, int HKV, int64_t max_ctx) {
  const int64_t rows = max_q_len * G, heads = rows * HKV;
  const int64_t q = max_q_len < max_ctx ? max_q_len : max_ctx;
  return rows >= kAttnTileRows &&
         (heads >= kAttnTileAlways ||
          (heads >= (HKV < 8 ? kAttnTileHeadsFew : kAttnTileHeads) &&
           q * G * HKV * (2 * max_ctx - q) >= 2 * kAttnTilePairs));
}
// The most tokens of an entry that is not long whatever its context.
inline int64_t attn_short_tokens(int G, int HKV) {
  const int64_t by_heads = (kAttnTileAlways - 1) / (G * HKV), by_rows = (kAttnTileRows - 1) / G;
  return by_heads > by_rows ? by_heads : by_rows;
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
