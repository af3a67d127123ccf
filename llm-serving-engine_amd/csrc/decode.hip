// The elementwise work between a decoder layer's GEMMs and its attention, each as one launch:
//  * rope_kv_kernel: rotates q and k (apply_rotary_pos_emb) and writes q, k and v where the
//    attention reads them (q token-major, K/V rows in the contiguous cache and the paged pool);
//  * add_rmsnorm_kernel: the residual addition and the RMSNorm that follows it.
// At decode sizes (64 tokens of 6144 and of 4096 bf16 values, under 2 MB) both are bound by their
// launch. In the eager operations of the reference's path a layer runs about 40 such launches of
// 2 to 8 us around 5 GEMMs and one attention; four layers and the lm_head at 64 sequences behind 1024
// positions took 1384 us a step replayed from a graph, about 600 of it there; with these two, 813 us.
// Every rounding to bf16 of those eager operations is kept, so the rotation is bit-identical to
// them; the norm's sum of squares runs in another order.
#include "lse_common.h"

namespace lse {

struct RopeArgs {
  const uint16_t *q, *k, *v;  // (tokens, heads x D) rows, strides sq, sk, sv
  int64_t sq, sk, sv;
  const uint16_t *cos, *sin;  // (tokens, D) rows, stride sc
  int64_t sc;
  uint16_t* q_out;            // (tokens, H, D)
  uint16_t *k_cache, *v_cache;  // element (seq, head, position, d), strides below; may be null
  int64_t cs, ch, cp;
  uint16_t *k_pool, *v_pool;  // element (block, slot, head, d); may be null
  int64_t pb, pw, ph;
  const int32_t* table;  // (sequences, blocks), row stride st
  int64_t st;
  int H, HKV, D, ntok, start, block_size, units;
};

// Rotates eight pairs (x[d], x[d + D/2]) as two bf16 products rounded, then their sum rounded.
__device__ __forceinline__ void rope8(const uint4& a, const uint4& b, const uint4& ca,
                                      const uint4& cb, const uint4& sa, const uint4& sb, uint4& oa,
                                      uint4& ob) {
  const uint32_t A[4] = {a.x, a.y, a.z, a.w}, B[4] = {b.x, b.y, b.z, b.w};
  const uint32_t CA[4] = {ca.x, ca.y, ca.z, ca.w}, CB[4] = {cb.x, cb.y, cb.z, cb.w};
  const uint32_t SA[4] = {sa.x, sa.y, sa.z, sa.w}, SB[4] = {sb.x, sb.y, sb.z, sb.w};
  uint32_t X[4], Y[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t x = 0, y = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      auto val = [&](uint32_t w) { return bf16_to_f32((uint16_t)(w >> (16 * h))); };
      auto rnd = [](float f) { return bf16_to_f32(f32_to_bf16(f)); };
      const float lo = val(A[i]), hi = val(B[i]);
      const float p = rnd(lo * val(CA[i])), q = rnd(-hi * val(SA[i]));
      const float r = rnd(hi * val(CB[i])), s = rnd(lo * val(SB[i]));
      x |= (uint32_t)f32_to_bf16(p + q) << (16 * h);
      y |= (uint32_t)f32_to_bf16(r + s) << (16 * h);
    }
    X[i] = x, Y[i] = y;
  }
  oa = make_uint4(X[0], X[1], X[2], X[3]);
  ob = make_uint4(Y[0], Y[1], Y[2], Y[3]);
}

// One thread per eight pairs of one head of one token: heads 0 .. H-1 are q's, then k's, then v's.
__global__ void __launch_bounds__(256) rope_kv_kernel(RopeArgs a) {
  const int per_head = a.D / 16;
  const int u = blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= a.units) return;
  const int t = blockIdx.y;
  const int head = u / per_head, d = 8 * (u - head * per_head), half = a.D / 2;
  const int seq = t / a.ntok, pos = a.start + t - seq * a.ntok;
  const int what = head < a.H ? 0 : head < a.H + a.HKV ? 1 : 2;
  const int h = head - (what == 0 ? 0 : what == 1 ? a.H : a.H + a.HKV);
  const uint16_t* src = (what == 0   ? a.q + t * a.sq
                         : what == 1 ? a.k + t * a.sk
                                     : a.v + t * a.sv) +
                        (int64_t)h * a.D + d;
  uint4 x = *reinterpret_cast<const uint4*>(src);
  uint4 y = *reinterpret_cast<const uint4*>(src + half);
  if (what < 2) {
    const uint16_t* c = a.cos + t * a.sc + d;
    const uint16_t* s = a.sin + t * a.sc + d;
    const uint4 x0 = x, y0 = y;
    rope8(x0, y0, *reinterpret_cast<const uint4*>(c), *reinterpret_cast<const uint4*>(c + half),
          *reinterpret_cast<const uint4*>(s), *reinterpret_cast<const uint4*>(s + half), x, y);
  }
  auto put = [&](uint16_t* dst) {
    *reinterpret_cast<uint4*>(dst) = x;
    *reinterpret_cast<uint4*>(dst + half) = y;
  };
  if (what == 0) {
    put(a.q_out + ((int64_t)t * a.H + h) * a.D + d);
    return;
  }
  uint16_t* cache = what == 1 ? a.k_cache : a.v_cache;
  if (cache) put(cache + seq * a.cs + h * a.ch + pos * a.cp + d);
  uint16_t* pool = what == 1 ? a.k_pool : a.v_pool;
  if (pool) {
    const int bi = pos / a.block_size;
    const int64_t block = a.table[seq * a.st + bi];
    put(pool + block * a.pb + (int64_t)(pos - bi * a.block_size) * a.pw + h * a.ph + d);
  }
}

constexpr int kNormThreads = 512;

// One workgroup per row, thread t holding elements 8 t + 4096 i (i < NV): s = bf16(x + res) (or x),
// y = bf16(w * bf16(s * r)), r = 1 / sqrt(mean(s^2) + eps), the roundings of LlamaRMSNorm
// (modeling_llama.py:62-67). The sum of squares: each thread's in order, then a fixed tree. `sum` may be x
// or res: a thread reads all of its elements before it writes any.
template <int NV>
__global__ void __launch_bounds__(kNormThreads)
add_rmsnorm_kernel(const uint16_t* x, int64_t ldx, const uint16_t* res, int64_t ldr,
                   const uint16_t* __restrict__ w, float eps, uint16_t* sum,
                   uint16_t* __restrict__ y, int K) {
  __shared__ float red[kNormThreads / 64];
  const int64_t m = blockIdx.x;
  uint32_t u[NV][4], g[NV][4];
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int k = 8 * (threadIdx.x + kNormThreads * i);
    const uint4 zero = make_uint4(0, 0, 0, 0);
    const uint4 a = k < K ? *reinterpret_cast<const uint4*>(x + m * ldx + k) : zero;
    const uint4 b = res && k < K ? *reinterpret_cast<const uint4*>(res + m * ldr + k) : zero;
    const uint4 c = k < K ? *reinterpret_cast<const uint4*>(w + k) : zero;
    u[i][0] = a.x, u[i][1] = a.y, u[i][2] = a.z, u[i][3] = a.w;
    g[i][0] = c.x, g[i][1] = c.y, g[i][2] = c.z, g[i][3] = c.w;
    const uint32_t r[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float lo = __builtin_bit_cast(float, u[i][j] << 16);
      float hi = __builtin_bit_cast(float, u[i][j] & 0xffff0000u);
      if (res) {
        u[i][j] = pack_bf16x2(lo + __builtin_bit_cast(float, r[j] << 16),
                              hi + __builtin_bit_cast(float, r[j] & 0xffff0000u));
        lo = __builtin_bit_cast(float, u[i][j] << 16);
        hi = __builtin_bit_cast(float, u[i][j] & 0xffff0000u);
      }
      ss = __builtin_fmaf(lo, lo, ss);
      ss = __builtin_fmaf(hi, hi, ss);
    }
  }
  if (sum) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int k = 8 * (threadIdx.x + kNormThreads * i);
      if (k < K)
        *reinterpret_cast<uint4*>(sum + m * K + k) = make_uint4(u[i][0], u[i][1], u[i][2], u[i][3]);
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  float total = red[0];
#pragma unroll
  for (int i = 1; i < kNormThreads / 64; ++i) total += red[i];
  const float r = 1.0f / __builtin_sqrtf(total / (float)K + eps);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int k = 8 * (threadIdx.x + kNormThreads * i);
    uint32_t o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      auto norm = [&](uint32_t xb, uint32_t wb) {
        const float h = bf16_to_f32(f32_to_bf16(__builtin_bit_cast(float, xb) * r));
        return __builtin_bit_cast(float, wb) * h;
      };
      o[j] = pack_bf16x2(norm(u[i][j] << 16, g[i][j] << 16),
                         norm(u[i][j] & 0xffff0000u, g[i][j] & 0xffff0000u));
    }
    if (k < K) *reinterpret_cast<uint4*>(y + m * K + k) = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

int launch_rope_kv(const RopeArgs& a, int64_t tokens, hipStream_t stream) {
  hipLaunchKernelGGL(rope_kv_kernel, dim3((unsigned)ceil_div(a.units, 256), (unsigned)tokens),
                     dim3(256), 0, stream, a);
  return launch_status();
}

int launch_add_rmsnorm(const uint16_t* x, int64_t ldx, const uint16_t* res, int64_t ldr,
                       const uint16_t* w, float eps, uint16_t* sum, uint16_t* y, int64_t M,
                       int64_t K, hipStream_t stream) {
  const dim3 grid((unsigned)M), block(kNormThreads);
  if (K <= 8 * kNormThreads)
    hipLaunchKernelGGL(add_rmsnorm_kernel<1>, grid, block, 0, stream, x, ldx, res, ldr, w, eps, sum,
                       y, (int)K);
  else if (K <= 16 * kNormThreads)
    hipLaunchKernelGGL(add_rmsnorm_kernel<2>, grid, block, 0, stream, x, ldx, res, ldr, w, eps, sum,
                       y, (int)K);
  else
    hipLaunchKernelGGL(add_rmsnorm_kernel<4>, grid, block, 0, stream, x, ldx, res, ldr, w, eps, sum,
                       y, (int)K);
  return launch_status();
}

}  // namespace lse

namespace {
bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }
}  // namespace

extern "C" {

int lse_add_rmsnorm(const void* x, int64_t ldx, const void* res, int64_t ldr, const void* weight,
                    float eps, void* sum, void* y, int64_t M, int64_t K, void* stream) {
  if (M < 0 || K < 0 || M > 2147483647) return LSE_E_SHAPE;
  if (K % 8) return LSE_E_ALIGN;
  if (K > LSE_NORM_MAX_K) return LSE_E_RANGE;
  if (M == 0 || K == 0) return LSE_OK;
  if (!x || !weight || !y) return LSE_E_NULL;
  if (ldx < K || (res && ldr < K)) return LSE_E_SHAPE;
  if (ldx % 8 || (res && ldr % 8) || !aligned16(x) || !aligned16(res) || !aligned16(weight) ||
      !aligned16(sum) || !aligned16(y))
    return LSE_E_ALIGN;
  if (!(eps >= 0.0f)) return LSE_E_SHAPE;
  return lse::launch_add_rmsnorm((const uint16_t*)x, ldx, (const uint16_t*)res, ldr,
                                 (const uint16_t*)weight, eps, (uint16_t*)sum, (uint16_t*)y, M, K,
                                 (hipStream_t)stream);
}

int lse_rope_kv(const void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v,
                int64_t v_stride, const void* cos, const void* sin, int64_t cs_stride, void* q_out,
                void* k_cache, void* v_cache, int64_t cache_stride_seq, int64_t cache_stride_head,
                int64_t cache_stride_pos, void* k_pool, void* v_pool, int64_t pool_stride_block,
                int64_t pool_stride_slot, int64_t pool_stride_head, const int32_t* block_table,
                int64_t block_table_stride, int64_t block_size, int64_t H, int64_t H_KV, int64_t D,
                int64_t sequences, int64_t tokens_per_sequence, int64_t start, void* stream) {
  if (H < 1 || H_KV < 1 || H > 65536 || H_KV > 65536 || D < 16 || D > 1024 || D % 16 ||
      sequences < 0 || tokens_per_sequence < 0 || start < 0 || block_size < 1 ||
      block_size > 2147483647)
    return LSE_E_SHAPE;
  const int64_t tokens = sequences * tokens_per_sequence;
  if (tokens == 0) return LSE_OK;
  if (tokens > 65535 || start + tokens_per_sequence > 2147483647) return LSE_E_RANGE;
  if (!q || !k || !v || !cos || !sin || !q_out || !k_cache != !v_cache || !k_pool != !v_pool ||
      (k_pool && !block_table))
    return LSE_E_NULL;
  if (q_stride < H * D || k_stride < H_KV * D || v_stride < H_KV * D || cs_stride < D ||
      cache_stride_seq < 0 || cache_stride_head < 0 || cache_stride_pos < 0 ||
      pool_stride_block < 0 || pool_stride_slot < 0 || pool_stride_head < 0 ||
      block_table_stride < 0)
    return LSE_E_SHAPE;
  const int64_t strides[] = {q_stride,         k_stride,          v_stride,
                             cs_stride,        cache_stride_seq,  cache_stride_head,
                             cache_stride_pos, pool_stride_block, pool_stride_slot,
                             pool_stride_head};
  for (int64_t s : strides)
    if (s % 8) return LSE_E_ALIGN;
  const void* ptrs[] = {q, k, v, cos, sin, q_out, k_cache, v_cache, k_pool, v_pool};
  for (const void* p : ptrs)
    if (!aligned16(p)) return LSE_E_ALIGN;
  lse::RopeArgs a{};
  a.q = (const uint16_t*)q, a.k = (const uint16_t*)k, a.v = (const uint16_t*)v;
  a.sq = q_stride, a.sk = k_stride, a.sv = v_stride;
  a.cos = (const uint16_t*)cos, a.sin = (const uint16_t*)sin, a.sc = cs_stride;
  a.q_out = (uint16_t*)q_out;
  a.k_cache = (uint16_t*)k_cache, a.v_cache = (uint16_t*)v_cache;
  a.cs = cache_stride_seq, a.ch = cache_stride_head, a.cp = cache_stride_pos;
  a.k_pool = (uint16_t*)k_pool, a.v_pool = (uint16_t*)v_pool;
  a.pb = pool_stride_block, a.pw = pool_stride_slot, a.ph = pool_stride_head;
  a.table = block_table, a.st = block_table_stride;
  a.H = (int)H, a.HKV = (int)H_KV, a.D = (int)D, a.ntok = (int)tokens_per_sequence;
  a.start = (int)start, a.block_size = (int)block_size;
  a.units = (int)((H + 2 * H_KV) * (D / 16));
  return lse::launch_rope_kv(a, tokens, (hipStream_t)stream);
}

}  // extern "C"
