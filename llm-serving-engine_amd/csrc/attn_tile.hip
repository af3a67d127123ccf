// Paged attention of long entries (prompts and prompt chunks): the row-tiled kernel beside
// attention.hip's key-streaming one, with the same semantics and arguments. It takes every
// entry that attn_is_long.
//
// What bounds the key-streaming kernel there is that a K/V byte it reads serves only 16 MFMA rows:
// at 2048-token prompts it reads, stages and transposes each key once per 4 tokens. Here a workgroup
// owns 128 rows (tokens x the G query heads of one K/V head, token-major, so any G packs without idle
// rows), and each of its waves 32 of them on v_mfma_f32_32x32x16_bf16:
//  * S^T = K Q^T: K rows from LDS are the A operand, Q stays in registers as the B operand, so lane
//    l holds the scores of row l % 32 only: keys 8 b + 4 (l / 32) + r of a 32-key block.
//  * O^T += V^T P^T: those scores, rounded to bf16, are already the B operand for the contraction
//    order {8 b + 4 h + r}; V^T comes out of row-major V rows in LDS by ds_read_b64_tr_b16. O^T's
//    columns are the rows l % 32 again, so the softmax factors are per-lane scalars: no shuffle but
//    one 32-lane swap for the row maximum.
//
// Two streams. The 8 waves are two groups of 4, each over all 128 rows and every second 64-key
// tile with its own softmax state; the two states are merged at the end. Each SIMD holds one wave
// of either group, and the groups run half a step apart: between two barriers one group issues its
// MFMAs (P V of the last tile and K Q^T of this one) while the other does its softmax, so the matrix
// cores and the VALU (about 1000 clocks each per tile and wave) run at the same time.
//
// K and V tiles go straight from the pool to LDS (global_load_lds, 16 bytes per lane), two slots
// each per stream, issued three phases before their use. LDS rows are 256 bytes, 16-byte chunk c of
// row r stored at c ^ (r & 15) (K) or c ^ 4 (r & 3) (V): K fragment reads of 16 rows at one chunk
// and the transposing reads of 4 rows x 64 bytes then cover every bank once. The swizzle is applied
// to the global addresses, since the LDS side of these loads is linear in the lane.
//
// Work list. Items are (entry, K/V head, row tile). The grid is one workgroup per CU; every
// workgroup computes the same order of items from q_len (row tiles in descending order, so the
// longest causal ranges come first, K/V heads fastest, so with 8 heads an XCD's L2 holds one head)
// and takes every grid-th one, alternating direction so that the sums of lengths even out. No item
// is launched for entries that are not long, however many there are.
//
// Order of summation: tiles 2 j + s of stream s in order, then the two streams. It depends on the
// row's own entry only.
//
// Measured on MI355X, against the key-streaming kernel: three fresh prompts of 1285-1321 tokens, 32
// heads over 8, 268 -> 74 us (570 TFLOP/s of the causal half; a dense bf16 product of 8192^3 reaches
// 1434); a 735-token chunk behind 1291 positions, 24 heads over 8, 107 -> 38. A phase takes 1300-1600 clocks of which
// 1024 are MFMA issue; an item's first loads and its merge another 10000 or so, about a third of
// the time at these prompt lengths. Without gain, against 66-68 us: the next item's first loads
// issued before the merge (69 us); the tiles of consecutive items in one pipeline (73-105 us: the
// softmax phase grows by the item cursors and the waits for Q); the loads in pairs between the
// exponentials (68.5 us).
#include <algorithm>
#include <type_traits>

#include "attention.h"

namespace lse {

constexpr int kTileRowsQ = 128;    // query rows of a workgroup
constexpr int kTileKeys = 64;      // keys of a tile
constexpr int kTileWaves = 8;      // two streams of four waves
constexpr int kTileBytesKV = kTileKeys * 256;
constexpr int kTileMaxEntries = 1024;  // entries of one launch (their tile counts lie in LDS)
constexpr int kTileMaxLevels = 1024;
constexpr int kTileListMax = 512;  // items of a workgroup whose list lies in LDS at a time
// A row's reference m (probabilities are exp2(s - m)) is its running maximum plus what makes it a whole
// number above the tile's own maximum, so that the tile's largest probability is a power of two and
// is rounded to bf16 without error; tiles whose maximum lies more than kAlign below it keep m. Relative
// error against fp64 before the output is rounded (a model of the arithmetic, 1300 keys; scores of
// standard deviation 1 and, where few keys matter, 3): 0.00125 and 0.00028; with the running
// maximum itself 0.00142 and 0.00049 (the key-streaming kernel, which has one in each of 8 parts: 0.00131
// and 0.00034); with one that lags by up to 8, which saves most rescales of O and 3 us of 70,
// 0.00161 and 0.00142.
constexpr float kAlign = 9.0f;
// The exponent s - m is one fused multiply-add of the unscaled score, while m holds a rounded product:
// the largest score's exponent is off by that rounding, at most 2^-10 up to this magnitude of m (no
// bf16 probability changes). Past it the product is rounded first, as m's was.
constexpr float kFarScore = 16384.0f;

struct AttnTileArgs {
  int e0, entries;  // this launch's entries e0 .. e0 + entries - 1
  int sh;           // row tiles per level of the work list: 1 << sh
  int levels;
  int fast;  // a wave's 16 rows of a tile lie in one block, and offsets inside it fit 32 bits
};

__device__ __forceinline__ f32x16 mfma32x32x16(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// Four 16-byte global loads straight to LDS: lane l's bytes of load i land at lds + 1024 i + 16 l.
// Not tracked by the compiler: ordered by explicit vmcnt waits and barriers. M0 (the LDS address) is
// restored. A vector-memory read of an SGPR that a VALU instruction wrote (v_readlane of a spilled base,
// v_readfirstlane) needs five wait states between the two, and the compiler does not look into the block:
// its three instructions before the first load make five.
__device__ __forceinline__ void dma4_saddr(uint32_t lds, const void* base, const uint32_t (&off)[4]) {
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %1\n\t"
      "s_nop 2\n\t"
      "global_load_lds_dwordx4 %2, %6\n\t"
      "s_add_u32 m0, m0, 0x400\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %3, %6\n\t"
      "s_add_u32 m0, m0, 0x400\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %4, %6\n\t"
      "s_add_u32 m0, m0, 0x400\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %5, %6\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(saved)
      : "s"(lds), "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "s"(base)
      : "memory", "scc");
}
__device__ __forceinline__ void dma4_vaddr(uint32_t lds, const char* const (&p)[4]) {
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %1\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %2, off\n\t"
      "s_add_u32 m0, m0, 0x400\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %3, off\n\t"
      "s_add_u32 m0, m0, 0x400\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %4, off\n\t"
      "s_add_u32 m0, m0, 0x400\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %5, off\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(saved)
      : "s"(lds), "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3])
      : "memory", "scc");
}

// A 64-bit value that is the same in every lane, as a scalar.
__device__ __forceinline__ int64_t uniform64(int64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return (int64_t)((uint64_t)hi << 32 | lo);
}

// Every LDS read of this wave is done, then the workgroup's barrier.
__device__ __forceinline__ void phase_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// A lane's value and that of lane l ^ 32, in either order: the instruction exchanges the upper half of
// its first operand with the lower half of its second. Written in assembly because the compiler
// takes the builtin's two results to be equal when both come from one value, and uses one twice.
struct Halves {
  float a, b;
};
__device__ __forceinline__ Halves both_halves(float v) {
  Halves h{v, v};
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(h.a), "+v"(h.b));
  return h;
}

template <bool POW2>
__global__ void __launch_bounds__(64 * kTileWaves)
attn_tile_kernel(PagedAttnArgs a, AttnTileArgs t) {
  constexpr float NEG_INF = -__builtin_huge_valf();
  // K slots [stream][2], then V slots; reused for the streams' O at the end of an item.
  __shared__ __attribute__((aligned(16))) unsigned char kv[8 * kTileBytesKV];
  __shared__ int ntile[kTileMaxEntries], pre[kTileMaxLevels + 1];
  __shared__ float mbuf[2][kTileRowsQ], lbuf[2][kTileRowsQ];
  __shared__ int list_e[kTileListMax], list_kvh[kTileListMax], list_qt[kTileListMax];
  static_assert(kTileListMax == 64 * kTileWaves, "one item per thread");

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int stream = wave >> 2, w = wave & 3;
  const int n32 = lane & 31, half = lane >> 5;
  const int G = a.G;

  // The work list: level l holds row tiles [l << sh, (l + 1) << sh) of every entry, and pre[l] is
  // the number of row tiles in the levels above it.
  for (int i = threadIdx.x; i < t.entries; i += 64 * kTileWaves) {
    const int qlen = a.q_len[t.e0 + i];
    ntile[i] = attn_is_long(qlen, G, a.HKV, a.context_len[t.e0 + i])
                   ? (qlen * G + kTileRowsQ - 1) / kTileRowsQ
                   : 0;
  }
  __syncthreads();
  for (int l = threadIdx.x; l <= t.levels; l += 64 * kTileWaves) {
    int above = 0;  // pre[l] for l < levels; pre[levels] = all row tiles
    const int from = l < t.levels ? (l + 1) << t.sh : 0;
    for (int i = 0; i < t.entries; ++i) above += max(0, ntile[i] - from);
    pre[l] = above;
  }
  __syncthreads();
  const int64_t total = (int64_t)pre[t.levels] * a.HKV;

  // Lane constants of the tile loads: instruction i of a wave fills rows 16 w + 4 i + lane / 16,
  // chunk lane % 16 of LDS, from the logical chunk that the row's swizzle puts there.
  const int lrow = lane >> 4, lchunk = lane & 15;
  const uint32_t lds0 = lds_addr(kv);
  const uint32_t kslot = lds0 + stream * 2 * kTileBytesKV + w * 4096;
  const uint32_t vslot = kslot + 4 * kTileBytesKV;
  const int rowb = t.fast ? (int)(a.sw * 2) : 0;  // bytes from a key to the next
  uint32_t ksrc[4], vsrc[4];  // byte offsets from the wave's first row
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t row = (uint32_t)((4 * i + lrow) * rowb);
    ksrc[i] = row + 16 * (lchunk ^ (4 * i + lrow));
    vsrc[i] = row + 16 * (lchunk ^ (4 * lrow));
  }

  // LDS addresses of the fragment reads, relative to a slot.
  const unsigned char* kread = kv + stream * 2 * kTileBytesKV + n32 * 256;
  const int kswz = half ^ (n32 & 15);  // chunk of K fragment kk: (2 kk) ^ kswz
  const int g16 = lane >> 4, s16 = lane & 15;
  const unsigned char* vread = kv + (4 + stream * 2) * kTileBytesKV +
                               (4 * half + (s16 >> 2)) * 256 + 8 * (s16 & 1);
  const int vchunk = 2 * (g16 & 1) + ((s16 & 3) >> 1), vswz = 4 * (s16 >> 2);

  const int groups = gridDim.x >> 3;
  for (int round = 0;; ++round) {
    // This workgroup's next kTileListMax items, one per thread: (entry, K/V head, row tile).
    if (round % kTileListMax == 0) {
      const int64_t rd = round + (int)threadIdx.x;
      int slot_id = blockIdx.x;
      if ((rd & 1) && (gridDim.x & 7) == 0)
        slot_id = (groups - 1 - (slot_id >> 3)) * 8 + (slot_id & 7);
      const int64_t item = rd * gridDim.x + slot_id;
      int e = -1, kvh = 0, qt = 0;
      if (item < total) {
        const int p = (int)item / a.HKV;
        kvh = (int)item - p * a.HKV;
        int lo = 0, hi = t.levels - 1;  // the level of row tile p: the smallest l with pre[l] <= p
        while (lo < hi) {
          const int mid = (lo + hi) >> 1;
          if (pre[mid] <= p) hi = mid; else lo = mid + 1;
        }
        int left = p - pre[lo], cnt = 0;  // then its entry and tile inside the level
        for (e = 0; e < t.entries; ++e) {
          cnt = min(max(ntile[e] - (lo << t.sh), 0), 1 << t.sh);
          if (left < cnt) break;
          left -= cnt;
        }
        qt = (lo << t.sh) + cnt - 1 - left;
      }
      __syncthreads();
      list_e[threadIdx.x] = e, list_kvh[threadIdx.x] = kvh, list_qt[threadIdx.x] = qt;
      __syncthreads();
    }
    const int at = round % kTileListMax;
    const int e_in = __builtin_amdgcn_readfirstlane(list_e[at]);
    if (e_in < 0) break;
    const int e = t.e0 + e_in;
    const int kvh = __builtin_amdgcn_readfirstlane(list_kvh[at]);
    const int qt = __builtin_amdgcn_readfirstlane(list_qt[at]);

    const int qlen = a.q_len[e], ctx = a.context_len[e], qo = a.query_offset[e], qs = a.q_start[e];
    const int rows = qlen * G, row0 = qt * kTileRowsQ;
    const int last_tok = min(qlen - 1, (row0 + kTileRowsQ - 1) / G);
    const int end_n = min(qo + last_tok + 1, ctx);
    const int steps = end_n > 0 ? (end_n + 2 * kTileKeys - 1) / (2 * kTileKeys) : 0;

    // This lane's row and, below, the last position it sees (relative ones are compared with
    // constants in the masked tiles).
    const int r = row0 + 32 * w + n32;
    const int tok = r / G, gq = r - tok * G;
    const bool row_ok = r < rows;
    const int lim = row_ok ? min(qo + tok, end_n - 1) : -1;
    // Keys up to here are seen by every row of the wave: tiles inside need no mask.
    const int all_see = min(qo + (row0 + 32 * w) / G, end_n - 1);

    typedef const __attribute__((address_space(4))) int32_t* ConstI32;
    const int32_t* bt = a.block_table + (int64_t)e * a.sbt;
    const int bs = a.block_size;
    const char* kbase = reinterpret_cast<const char*>(a.k_pool + (int64_t)kvh * a.sh);
    const char* vbase = reinterpret_cast<const char*>(a.v_pool + (int64_t)kvh * a.sh);
    auto blk_of = [&](int n) { return POW2 ? n >> a.bs_shift : n / bs; };
    // The block of this wave's first key of the stream's tile j, and that key's byte offset in a
    // pool. Keys past the item's last one are clamped to it, here and below, so every read stays
    // inside the entry's own slots.
    auto first_key = [&](int j) { return kTileKeys * (2 * j + stream) + 16 * w; };
    auto tile_blk = [&](int j) {
      const int n = min(first_key(j), end_n - 1);
      return __builtin_amdgcn_readfirstlane(
          ((ConstI32)(uintptr_t)bt)[__builtin_amdgcn_readfirstlane(blk_of(n))]);
    };
    auto tile_off = [&](int j, int blk) {
      const int n = min(first_key(j), end_n - 1);
      const int within = POW2 ? n & (bs - 1) : n % bs;
      return 2 * ((int64_t)blk * a.sb + (int64_t)within * a.sw);
    };
    // Loads the wave's 16 rows of tile j from `pool` into slot j & 1; `off` is tile_off's.
    auto load_tile = [&](int j, const char* pool, int64_t off, uint32_t slot,
                         const uint32_t (&src)[4], int swz4) {
      slot += (j & 1) * kTileBytesKV;
      const int n0 = first_key(j);
      if (t.fast) {
        const void* base = reinterpret_cast<const void*>(uniform64((int64_t)(pool + off)));
        if (n0 + 16 <= end_n) {
          dma4_saddr(slot, base, src);
        } else {  // rows past the last key's: that row again
          const int most = max(end_n - 1 - n0, 0);
          uint32_t to[4];
#pragma unroll
          for (int i = 0; i < 4; ++i)
            to[i] = src[i] - (uint32_t)(max(4 * i + lrow - most, 0) * rowb);
          dma4_saddr(slot, base, to);
        }
      } else {
        // Opaque, so that nothing of this path is kept in registers across the loop.
        int ln = lane;
        asm volatile("" : "+v"(ln));
        int n[4], bi[4], blk[4];
        const char* p[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          n[i] = min(n0 + 4 * i + (ln >> 4), end_n - 1);
          bi[i] = blk_of(n[i]);
          blk[i] = bt[bi[i]];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t chunk = (ln & 15) ^ (swz4 ? 4 * (ln >> 4) : 4 * i + (ln >> 4));
          p[i] = pool + 2 * ((int64_t)blk[i] * a.sb + (int64_t)(n[i] - bi[i] * bs) * a.sw) +
                 16 * chunk;
        }
        dma4_vaddr(slot, p);
      }
    };

    const float sc = a.scale_log2 == 0.0f ? 1.0f : __builtin_fabsf(a.scale_log2);
    bf16x8 qf[8];
    float m_run = NEG_INF, m_max = NEG_INF, l_run = 0.0f;
    f32x16 oacc[4], st[2];
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int i = 0; i < 16; ++i) oacc[d][i] = 0.0f;
    bf16x8 pa[4];

    // Probabilities 16 k .. 16 k + 15 of the tile, rounded to bf16.
    auto to_pa = [&](int k) {
      f32x8 v;
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = st[k >> 1][8 * (k & 1) + i];
      pa[k] = __builtin_convertvector(v, bf16x8);
    };
    // A matrix phase: P V of tile j (PV) and K Q^T of tile jq into st (QK), 16 MFMAs each. Their
    // fragments are read kAhead MFMAs before use, in exactly this order: left to itself the compiler
    // reads each one right before its MFMA and waits out LDS's latency 32 times. The row sums and the
    // rest of the roundings of tile j's probabilities go between its P V MFMAs, where the VALU is
    // free, which brings the two phases to about the same length.
    auto matrix = [&](auto PV, auto QK, int j, int jq) {
      constexpr int kAhead = 4, U0 = PV.value ? 0 : 16, U1 = QK.value ? 32 : 16;
      const unsigned char* vr = vread + (j & 1) * kTileBytesKV;
      const unsigned char* kr = kread + (jq & 1) * kTileBytesKV;
      bf16x8 fr[kAhead];
      f32x16 zero;
#pragma unroll
      for (int i = 0; i < 16; ++i) zero[i] = 0.0f;
      auto read = [&](int u) -> bf16x8 {
        if (u < 16) {
          const unsigned char* src = vr + 16 * ((4 * (u & 3) + vchunk) ^ vswz) + (u >> 2) * 16 * 256;
          return __builtin_shufflevector(lds_read_tr16(src), lds_read_tr16(src + 8 * 256), 0, 1, 2,
                                         3, 4, 5, 6, 7);
        }
        const int kk = (u - 16) >> 1, b = u & 1;
        return as_bf16x8(
            *reinterpret_cast<const uint4*>(kr + 16 * ((2 * kk) ^ kswz) + b * 32 * 256));
      };
      float sum[4] = {0, 0, 0, 0};
#pragma unroll
      for (int u = U0; u < U0 + kAhead; ++u) fr[u % kAhead] = read(u);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = U0; u < U1; ++u) {
        if (u < 16)
          oacc[u & 3] = mfma32x32x16(fr[u % kAhead], pa[u >> 2], oacc[u & 3]);
        else
          st[u & 1] = mfma32x32x16(fr[u % kAhead], qf[(u - 16) >> 1], u < 18 ? zero : st[u & 1]);
        if (u + kAhead < U1) fr[u % kAhead] = read(u + kAhead);
        if (u < 16) {
          if ((u & 3) == 0 && u < 12) to_pa((u >> 2) + 1);
          sum[u & 1] += st[u >> 3][2 * (u & 7)];
          sum[2 + (u & 1)] += st[u >> 3][2 * (u & 7) + 1];
        }
        if (u == 15) l_run += (sum[0] + sum[1]) + (sum[2] + sum[3]);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    const std::true_type on{};
    const std::false_type off{};
    // Rows that see less than the stream's first tile: few probabilities, all about as large, so that their
    // rounding to bf16 averages out least, and the largest rows of a prompt's output (its size falls with
    // the square root of the keys). For the waves that hold some, P V of what the rounding leaves is added
    // too: 16 MFMAs, in the first items of an entry only. Relative error against fp64 of fresh
    // prompts of 417 / 1300 tokens, scores of standard deviation 1, output rounding included: 0.00176 /
    // 0.00182; without it 0.00194 / 0.00196, with it in every masked tile 0.00175 / 0.00181 (and 4 %
    // slower, against 1.5 %); the key-streaming kernel 0.00191 / 0.00195.
    const bool few_keys = kTileKeys * (stream + 1) - 1 > all_see;
    auto matrix_rest = [&] {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        f32x8 v;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float p = st[k >> 1][8 * (k & 1) + i];
          v[i] = p - (float)(__bf16)p;
        }
        const bf16x8 rest = __builtin_convertvector(v, bf16x8);
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const unsigned char* src = vread + 16 * ((4 * d + vchunk) ^ vswz) + k * 16 * 256;
          const bf16x8 fr = __builtin_shufflevector(lds_read_tr16(src), lds_read_tr16(src + 8 * 256),
                                                    0, 1, 2, 3, 4, 5, 6, 7);
          oacc[d] = mfma32x32x16(fr, rest, oacc[d]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    // The softmax of st, tile j's scores: probabilities to pa, the running state and O rescaled.
    auto softmax = [&](int j) {
#pragma clang fp contract(off)  // the maximum is a rounded product wherever it is used
      const int n0 = kTileKeys * (2 * j + stream);
      if (n0 + kTileKeys - 1 > all_see) {
        const int rel = lim - n0 - 4 * half;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            st[b][i] = 32 * b + 8 * (i >> 2) + (i & 3) <= rel ? st[b][i] : NEG_INF;
      }
      float mx = st[0][0];
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, st[b][i]);
      const Halves hm = both_halves(mx);
      const float m_tile = fmaxf(hm.a, hm.b) * sc;
      m_max = fmaxf(m_max, m_tile);
      const float below = m_max - m_tile;  // not <= kAlign where no key is seen yet (NaN)
      const float m_new = below <= kAlign ? m_tile + __builtin_ceilf(below) : m_run;
      const float mref = m_new == NEG_INF ? 0.0f : m_new;  // a row with no key yet keeps p = 0
      const float alpha = m_new == m_run ? 1.0f : exp2_fast(m_run - mref);
      float mul = sc, sub = mref;
      if (__ballot(__builtin_fabsf(mref) > kFarScore)) {
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int i = 0; i < 16; ++i) st[b][i] = st[b][i] * sc - mref;
        mul = 1.0f, sub = 0.0f;
      }
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) st[b][i] = exp2_fast(__builtin_fmaf(st[b][i], mul, -sub));
      l_run *= alpha;
      m_run = m_new;
      to_pa(0);
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) oacc[d][i] *= alpha;
    };

    if (steps > 0) {
      // The first loads of an item, none waiting for another: K, Q, then the rest in flight.
      int64_t off1 = tile_off(0, tile_blk(0));
      const int64_t off_v0 = off1;
      load_tile(0, kbase, off1, kslot, ksrc, 0);
      uint4 qv[8];
      const uint16_t* qp = a.q + (int64_t)(kvh * G + (row_ok ? gq : 0)) * a.sq_h +
                           (int64_t)(qs + (row_ok ? tok : 0)) * a.sq_t + 8 * half;
#pragma unroll
      for (int kk = 0; kk < 8; ++kk) qv[kk] = *reinterpret_cast<const uint4*>(qp + 16 * kk);
      if (steps > 1) {
        off1 = tile_off(1, tile_blk(1));
        load_tile(1, kbase, off1, kslot, ksrc, 0);
      }
      load_tile(0, vbase, off_v0, vslot, vsrc, 1);
      // A negative or zero softmax scale moves into Q (exactly), so that the row maximum can be
      // taken before the scaling.
      const uint32_t flip = a.scale_log2 < 0.0f ? 0x80008000u : 0u;
      const bool keep = row_ok && a.scale_log2 != 0.0f;
#pragma unroll
      for (int kk = 0; kk < 8; ++kk) {
        const uint4 v = make_uint4(qv[kk].x ^ flip, qv[kk].y ^ flip, qv[kk].z ^ flip,
                                   qv[kk].w ^ flip);
        qf[kk] = as_bf16x8(keep ? v : make_uint4(0, 0, 0, 0));
      }
      int blk2 = tile_blk(2);
      if (stream == 1) phase_barrier();
      if (steps > 1)
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(8));
      else
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(4));
      phase_barrier();
      matrix(off, on, 0, 0);
      phase_barrier();
      for (int j = 0; j + 1 < steps; ++j) {
        // Softmax phase, with the loads of K two tiles on and V one tile on.
        if (j + 2 < steps) {
          const int64_t off2 = tile_off(j + 2, blk2);
          load_tile(j + 2, kbase, off2, kslot, ksrc, 0);
          load_tile(j + 1, vbase, off1, vslot, vsrc, 1);
          off1 = off2;
          blk2 = tile_blk(j + 3);
        } else {
          load_tile(j + 1, vbase, off1, vslot, vsrc, 1);
        }
        softmax(j);
        if (j + 2 < steps)
          __builtin_amdgcn_s_waitcnt(vmcnt_imm(8));
        else
          __builtin_amdgcn_s_waitcnt(vmcnt_imm(4));
        phase_barrier();
        if (j == 0 && few_keys) matrix_rest();
        matrix(on, on, j, j + 1);
        phase_barrier();
      }
      softmax(steps - 1);
      __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
      phase_barrier();
      if (steps == 1 && few_keys) matrix_rest();
      matrix(on, off, steps - 1, 0);
      phase_barrier();
      if (stream == 0) phase_barrier();
    }

    // The streams' states to LDS (O as [stream][row][32 chunks of 4 columns], chunk c of row r at
    // c ^ (r & 31)), then each thread merges and writes 8-column pieces of one row.
    const int lr = 32 * w + n32;
    {
      const Halves hl = both_halves(l_run);
      l_run = hl.a + hl.b;
      if (half == 0) {
        mbuf[stream][lr] = m_run;
        lbuf[stream][lr] = l_run;
      }
      unsigned char* ob = kv + stream * (kTileRowsQ * 512) + lr * 512;
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int b = 0; b < 4; ++b)
          *reinterpret_cast<float4*>(ob + 16 * ((8 * d + 2 * b + half) ^ n32)) =
              make_float4(oacc[d][4 * b], oacc[d][4 * b + 1], oacc[d][4 * b + 2],
                          oacc[d][4 * b + 3]);
    }
    __syncthreads();
    {
      const int orow = threadIdx.x >> 2, part = threadIdx.x & 3;
      const int ro = row0 + orow;
      const float m0 = mbuf[0][orow], m1 = mbuf[1][orow];
      const float mm = fmaxf(m0, m1);
      const float ref = mm == NEG_INF ? 0.0f : mm;
      const float f0 = exp2_fast(m0 - ref), f1 = exp2_fast(m1 - ref);
      const float L = __builtin_fmaf(lbuf[1][orow], f1, lbuf[0][orow] * f0);
      const float inv = L > 0.0f ? 1.0f / L : 0.0f;
      if (ro < rows) {
        const int to = ro / G;
        uint16_t* out = a.o + (int64_t)(kvh * G + ro - to * G) * a.so_h + (int64_t)(qs + to) * a.so_t;
        const unsigned char* o0 = kv + orow * 512;
        const unsigned char* o1 = o0 + kTileRowsQ * 512;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int c = 2 * (4 * i + part);
          float v[8];
#pragma unroll
          for (int hh = 0; hh < 2; ++hh) {
            const int pc = 16 * ((c + hh) ^ (orow & 31));
            const float4 x = *reinterpret_cast<const float4*>(o0 + pc);
            const float4 y = *reinterpret_cast<const float4*>(o1 + pc);
            v[4 * hh] = __builtin_fmaf(y.x, f1, x.x * f0) * inv;
            v[4 * hh + 1] = __builtin_fmaf(y.y, f1, x.y * f0) * inv;
            v[4 * hh + 2] = __builtin_fmaf(y.z, f1, x.z * f0) * inv;
            v[4 * hh + 3] = __builtin_fmaf(y.w, f1, x.w * f0) * inv;
          }
          *reinterpret_cast<uint4*>(out + 4 * c) =
              make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]),
                         pack_bf16x2(v[6], v[7]));
        }
      }
    }
    __syncthreads();
  }
}

// One workgroup per CU, or per item where those are fewer, in whole rounds over the 8 XCDs: rounded up
// (workgroups without an item leave at once), since rounding down gave some workgroups two items
// one after the other while most CUs had none (200 tokens behind 2000 positions, 8 heads over 2: 14
// items, 41 us in 16 workgroups, 73 in 8).
static int64_t attn_tile_grid(int64_t items, int cus) {
  const int64_t grid = std::min<int64_t>(cus, ceil_div(items, 8) * 8);
  return grid >= 8 ? grid & ~(int64_t)7 : grid;
}

int launch_attn_tile(const PagedAttnArgs& a0, int cus, hipStream_t stream) {
  PagedAttnArgs a = a0;
  const int64_t tiles = ceil_div((int64_t)a.max_q_len * a.G, kTileRowsQ);
  AttnTileArgs t{};
  t.fast = a.block_size % 16 == 0 && a.sw < (int64_t)1 << 25;
  while (ceil_div(tiles, (int64_t)1 << t.sh) > kTileMaxLevels) ++t.sh;
  t.levels = (int)ceil_div(tiles, (int64_t)1 << t.sh);
  const void* fn = a.bs_shift >= 0 ? reinterpret_cast<const void*>(&attn_tile_kernel<true>)
                                   : reinterpret_cast<const void*>(&attn_tile_kernel<false>);
  for (t.e0 = 0; t.e0 < a.entries; t.e0 += kTileMaxEntries) {
    t.entries = std::min(kTileMaxEntries, a.entries - t.e0);
    const int64_t grid = attn_tile_grid(t.entries * tiles * a.HKV, cus);
    void* args[] = {&a, &t};
    const hipError_t err = hipLaunchKernel(fn, dim3((unsigned)grid), dim3(64 * kTileWaves), args, 0,
                                           stream);
    if (err != hipSuccess) return (int)err;
  }
  return launch_status();
}

}  // namespace lse
