// Attention over a prompt (qtip_prefill_attention): rotary embedding and cache update, then causal attention of many
// queries against the key / value cache.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/qtip_hip.h"
#include "qtip_setup.h"
#include "qtip_wht.h"

namespace {

typedef _Float16 half4v __attribute__((ext_vector_type(4)));
typedef _Float16 half8v __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));

// x * cos + rotate_half(x) * sin on eight elements of either half, every product and sum rounded to fp16
__device__ __forceinline__ void rope8(half8v& lo, half8v& hi, half8v c_lo, half8v s_lo, half8v c_hi, half8v s_hi) {
#pragma clang fp contract(off)
  const half8v a = lo * c_lo, b = -hi * s_lo, c = hi * c_hi, d = lo * s_hi;
  lo = a + b;
  hi = c + d;
}

// ---- rotary tables: one launch for the seven library passes of a prompt (30 us of 1000 tokens, 5 here)
constexpr int kBlock = 256;

__global__ __launch_bounds__(kBlock) void rotary_tables_kernel(_Float16* __restrict__ cos_t, _Float16* __restrict__ sin_t,
                                                               const int64_t* __restrict__ pos,
                                                               const float* __restrict__ inv_freq, int n, int half) {
  const long idx = (long)blockIdx.x * kBlock + threadIdx.x;
  if (idx >= (long)n * half) return;
  const int i = (int)(idx / half), d = (int)(idx % half);
  const float angle = (float)pos[i] * inv_freq[d];
  const _Float16 c = (_Float16)cosf(angle), s = (_Float16)sinf(angle);
  const size_t o = (size_t)i * 2 * half + d;
  cos_t[o] = cos_t[o + half] = c;
  sin_t[o] = sin_t[o + half] = s;
}

// ---- keys (with the rotary embedding) and values of the new tokens into their cache slots ------------------
// A thread takes eight elements of either half of a head's key, and of its value.
__global__ __launch_bounds__(kBlock) void cache_rows_kernel(
    _Float16* __restrict__ k_cache, _Float16* __restrict__ v_cache, const _Float16* __restrict__ k,
    const _Float16* __restrict__ v, int k_stride, int v_stride, const _Float16* __restrict__ cos_t,
    const _Float16* __restrict__ sin_t, const int64_t* __restrict__ pos, int n, int kv_heads, int hd, int slots) {
  const int cph = hd >> 4;  // chunk pairs per head
  const long idx = (long)blockIdx.x * kBlock + threadIdx.x;
  if (idx >= (long)n * kv_heads * cph) return;
  const int c = (int)(idx % cph);
  const long rest = idx / cph;
  const int h = (int)(rest % kv_heads), i = (int)(rest / kv_heads);
  const int64_t p = pos[i];
  if (p < 0 || p >= slots) return;
  const int lo = 8 * c, hi = lo + (hd >> 1);
  auto ld = [](const _Float16* q) { return *reinterpret_cast<const half8v*>(q); };
  const _Float16* kr = k + (size_t)i * k_stride + h * hd;
  const _Float16* vr = v + (size_t)i * v_stride + h * hd;
  const _Float16* cr = cos_t + (size_t)i * hd;
  const _Float16* sr = sin_t + (size_t)i * hd;
  half8v a = ld(kr + lo), b = ld(kr + hi);
  rope8(a, b, ld(cr + lo), ld(sr + lo), ld(cr + hi), ld(sr + hi));
  const size_t o = ((size_t)h * slots + (size_t)p) * hd;
  *reinterpret_cast<half8v*>(k_cache + o + lo) = a;
  *reinterpret_cast<half8v*>(k_cache + o + hi) = b;
  *reinterpret_cast<half8v*>(v_cache + o + lo) = ld(vr + lo);
  *reinterpret_cast<half8v*>(v_cache + o + hi) = ld(vr + hi);
}

// ---- attention -------------------------------------------------------------------------------------------
// A workgroup takes 64 queries of one head, a wave 16 of them; the 64-key tiles up to the last position a query of
// the group attends to pass through LDS, the next one waiting in registers.  Both products run on
// v_mfma_f32_16x16x32_f16 with the queries along N, so that everything about a query - scores, maximum, sum,
// output - sits in the lanes l % 16 of one column:
//   scores   A = 16 keys x 32 dims, B = the queries (registers): lane (g, q) gets keys 16 t + 4 g + r of query q
//   output   A = 16 dims x 32 keys of V^T, B = the probabilities as they stand: K slot 8 g + j of tile pair kk is
//            key 32 kk + 4 g + j (j < 4) or 32 kk + 16 + 4 g + j - 4, and V^T is laid out in that order
// V goes to LDS transposed (four keys of one dim in 8 bytes); dim 8 c + e sits in row 16 e + c, which keeps the
// writes of a phase on distinct banks and makes tile e hold the dims 8 c + e, so a lane ends with eight
// consecutive dims per register.  Scores, softmax and sums in fp32; a probability enters the second product as two fp16
// numbers, its rounded value and the rest, 22 bits of it or 2^-25 of the largest: rounded to one, outputs
// were up to 1.013 times as far from float64 as the library's attention (2.38e-4 and 2.35e-4 at 150 tokens of 32
// heads of 128), with two they are the correctly rounded ones (1.96e-4).  The rests have accumulators of their own: an
// infinite value times a rest of zero is a NaN where times the probability it is infinite, and is left out.
// Bound by a wave's chain through a tile (products, maximum, exponentials, products), and 16-query waves give two workgroups
// per CU at 1000 tokens of 32 heads: so it matters which two.  With a head's workgroups side by side an XCD had those of two lengths
// only, 2.4 times as many keys as another, and a CU two of the same length.  us with the launch for the caches, 1000 tokens, 32 heads
// of 128: 50.7, with no mask where every key is seen 49.8, in the order below too 40.6; the library's attention under a dense mask
// took 193 beside about 150 of small passes (rotation, cache writes, copies of heads).
constexpr int kQ = 64, kKeys = 64;

// the larger of v and lane ^ 16 (b = 4) or lane ^ 32 (5)
__device__ __forceinline__ float lane_max(float v, int b) {
  const auto s = qtip_wht::lane_pair(v, b);
  return fmaxf(s.x, s.y);
}

template <int HD>
__global__ __launch_bounds__(kBlock, 2) void prefill_attn_kernel(
    _Float16* __restrict__ out, const _Float16* __restrict__ q, int q_stride, const _Float16* __restrict__ cos_t,
    const _Float16* __restrict__ sin_t, const _Float16* __restrict__ k_cache, const _Float16* __restrict__ v_cache,
    const int64_t* __restrict__ pos, int n, int heads, int group, int slots, float scale_log2, int turn) {
  constexpr int KSTR = HD * 2 + 16, VSTR = kKeys * 2 + 16;  // bytes per key, per dim
  constexpr int NS = HD / 32, NE = HD / 16;                 // K steps of the scores, dim tiles
  constexpr int CPK = HD / 8;                               // 16-byte chunks per key
  constexpr int NKL = kKeys * CPK / kBlock;                 // chunks of K per thread
  __shared__ __align__(16) uint8_t lds_k[kKeys * KSTR];
  __shared__ __align__(16) uint8_t lds_v[HD * VSTR];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ql = lane & 15, g = lane >> 4;
  // rank 0 has the most keys; heads side by side, so that an XCD (every eighth workgroup) has the same mix of ranks as the others
  // and, of eight heads or a multiple, heads of its own
  // (grid = (heads, tiles of queries): only the workgroups behind the turn divide, 0.1 us in front of the first load)
  int h = blockIdx.x, qt = (int)gridDim.y - 1 - (int)blockIdx.y;
  const int id = (int)blockIdx.y * heads + h;
  if (id >= turn) {  // rank = workgroups - 1 - (id - turn)
    h = (heads - 1) - (id - turn) % heads;
    qt = (id - turn) / heads;
  }
  const size_t head = (size_t)(h / group) * slots * HD;
  const _Float16* kc = k_cache + head;
  const _Float16* vc = v_cache + head;
  auto position = [&](int i) {
    const int64_t p = pos[i < n ? i : n - 1];
    return p < 0 ? -1 : p < slots ? (int)p : slots - 1;  // (no such slot: nothing outside the cache is read)
  };
  int last = position(kQ * qt + lane);
#pragma unroll
  for (int m = 32; m; m >>= 1) {
    const int o = __shfl_xor(last, m);
    last = o > last ? o : last;
  }
  const int kmax = __builtin_amdgcn_readfirstlane(last) + 1;  // keys the workgroup looks at
  const int i = kQ * qt + 16 * wave + ql;
  const int ir = i < n ? i : n - 1;
  const int limit = position(ir);

  // ---- the wave's queries, rotated: dims 32 s + 8 g .. + 7 of query ql
  half8v qv[NS];
  {
    const _Float16* qr = q + (size_t)ir * q_stride + h * HD + 8 * g;
    const _Float16* cr = cos_t + (size_t)ir * HD + 8 * g;
    const _Float16* sr = sin_t + (size_t)ir * HD + 8 * g;
    auto ld = [](const _Float16* p) { return *reinterpret_cast<const half8v*>(p); };
#pragma unroll
    for (int s = 0; s < NS; ++s) qv[s] = ld(qr + 32 * s);
#pragma unroll
    for (int s = 0; s < NS / 2; ++s) {
      constexpr int H = HD / 2;
      rope8(qv[s], qv[s + NS / 2], ld(cr + 32 * s), ld(sr + 32 * s), ld(cr + 32 * s + H), ld(sr + 32 * s + H));
    }
  }

  // ---- tiles: keys kk0 .. kk0 + 63; past the last one a query looks at, zeros
  const u32x4v zero = {0u, 0u, 0u, 0u};
  u32x4v kr[NKL], vr[4];
  const int vq = tid / CPK, vch = tid % CPK;  // key quad and chunk of V this thread turns round
  const bool v_on = vq < kKeys / 4;
  auto load_tile = [&](int kk0) {
#pragma unroll
    for (int j = 0; j < NKL; ++j) {
      const int key = kk0 + (j * kBlock + tid) / CPK;
      kr[j] = key < kmax ? *reinterpret_cast<const u32x4v*>(kc + (size_t)key * HD + 8 * (tid % CPK)) : zero;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int key = kk0 + 4 * vq + j;
      vr[j] = v_on && key < kmax ? *reinterpret_cast<const u32x4v*>(vc + (size_t)key * HD + 8 * vch) : zero;
    }
  };
  auto store_tile = [&]() {
#pragma unroll
    for (int j = 0; j < NKL; ++j)
      *reinterpret_cast<u32x4v*>(lds_k + ((j * kBlock + tid) / CPK) * KSTR + 16 * (tid % CPK)) = kr[j];
    if (v_on) {
      // quads in the order the second product reads them: pairs (quad, quad + 4) of eight
      uint8_t* dst = lds_v + vch * VSTR + (vq >> 3) * 64 + (2 * (vq & 3) + ((vq >> 2) & 1)) * 8;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        uint2 w;
        const uint32_t sel = (e & 1) ? 0x07060302u : 0x05040100u;
        w.x = __builtin_amdgcn_perm(vr[1][e >> 1], vr[0][e >> 1], sel);
        w.y = __builtin_amdgcn_perm(vr[3][e >> 1], vr[2][e >> 1], sel);
        *reinterpret_cast<uint2*>(dst + e * CPK * VSTR) = w;
      }
    }
  };

  float4v o[NE], rest_o[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e) o[e] = rest_o[e] = float4v{0.f, 0.f, 0.f, 0.f};
  float mx = -__builtin_inff(), sum = 0.f;  // the query's maximum; this lane's share of its sum
  load_tile(0);
  for (int kk0 = 0; kk0 < kmax; kk0 += kKeys) {
    __syncthreads();  // the previous tile has been read
    store_tile();
    if (kk0 + kKeys < kmax) load_tile(kk0 + kKeys);
    __syncthreads();
    float4v s[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      s[t] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < NS; ++ks) {
        const half8v a = *reinterpret_cast<const half8v*>(lds_k + (16 * t + ql) * KSTR + 64 * ks + 16 * g);
        s[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, qv[ks], s[t], 0, 0, 0);
      }
    }
    float tile_max = mx;
#pragma unroll
    for (int t = 0; t < 4; ++t) s[t] *= scale_log2;
    if (__any(kk0 + kKeys - 1 > limit)) {  // (a tile that every query of the wave sees all of needs no mask)
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (kk0 + 16 * t + 4 * g + r > limit) s[t][r] = -__builtin_inff();
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) tile_max = fmaxf(tile_max, s[t][r]);
    tile_max = lane_max(tile_max, 4);
    tile_max = lane_max(tile_max, 5);
    const float base = fmaxf(tile_max, -3.0e38f);  // (nothing but scores of -inf so far)
    // (Also where the maximum stays, by 1: behind a branch that asks the wave for a maximum that changed the fade and the sum's first
    // addition are two roundings, and 1000 tokens of 32 heads of 128 take 41.8 us, without it 40.6; 16 heads 33.8 and 32.8.)
    const float fade = __builtin_amdgcn_exp2f(mx - base);
    mx = tile_max;
    sum *= fade;
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      o[e] *= fade;
      rest_o[e] *= fade;
    }
    half8v p[2], rest[2];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float x = __builtin_amdgcn_exp2f(s[t][r] - base);
        sum += x;
        const _Float16 h = (_Float16)x;
        p[t >> 1][4 * (t & 1) + r] = h;
        rest[t >> 1][4 * (t & 1) + r] = (_Float16)(x - (float)h);
      }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int e0 = 0; e0 < NE; e0 += 4) {  // (four reads in flight)
        half8v a[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) a[e] = *reinterpret_cast<const half8v*>(lds_v + (16 * (e0 + e) + ql) * VSTR + 64 * kk + 16 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e0 + e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[e], p[kk], o[e0 + e], 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) rest_o[e0 + e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[e], rest[kk], rest_o[e0 + e], 0, 0, 0);
      }
  }
  sum = qtip_wht::lane_add(sum, 4);
  sum = qtip_wht::lane_add(sum, 5);
  const float inv = 1.f / sum;
#pragma unroll
  for (int e = 0; e < NE; ++e)
#pragma unroll
    for (int r = 0; r < 4; ++r) o[e][r] += __builtin_isfinite(rest_o[e][r]) ? rest_o[e][r] : 0.f;
  if (i >= n) return;
  // row 16 e + x of V^T is dim 8 c + e' with e' * CPK + c = 16 e + x
  _Float16* dst = out + ((size_t)i * heads + h) * HD;
  if constexpr (CPK == 16) {  // tile e: dims 8 c + e, c = 4 g + r
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      half8v y;
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = (_Float16)(o[e][r] * inv);
      *reinterpret_cast<half8v*>(dst + 8 * (4 * g + r)) = y;
    }
  } else {  // 8 chunks: tile e holds dims 8 c + 2 e (rows 0..7) and 8 c + 2 e + 1 (rows 8..15), c = (4 g + r) % 8
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int e = 0; e < NE; ++e) dst[8 * ((4 * g + r) & 7) + 2 * e + (g >> 1)] = (_Float16)(o[e][r] * inv);
  }
}

}  // namespace

extern "C" int qtip_rotary_tables(void* cos_f16, void* sin_f16, const void* positions_i64, const float* inv_freq, long n,
                                  int half, void* stream) {
  if (!cos_f16 || !sin_f16 || !positions_i64 || !inv_freq) return QTIP_E_NULL;
  if (n < 1 || half < 1 || half > 1 << 20) return QTIP_E_SHAPE;
  const long step = (1 << 30) / half;  // (a launch holds fewer than 2^32 threads)
  for (long i = 0; i < n; i += step) {
    const long m = n - i < step ? n - i : step;
    rotary_tables_kernel<<<(unsigned)((m * half + kBlock - 1) / kBlock), kBlock, 0, (hipStream_t)stream>>>(
        (_Float16*)cos_f16 + i * 2 * half, (_Float16*)sin_f16 + i * 2 * half, (const int64_t*)positions_i64 + i, inv_freq,
        (int)m, half);
    if (const hipError_t e = hipGetLastError()) return (int)e;
  }
  return 0;
}

extern "C" int qtip_prefill_attention(void* out_f16, const void* q_f16, const void* k_f16, const void* v_f16,
                                      int q_stride, int k_stride, int v_stride, const void* cos_f16,
                                      const void* sin_f16, void* k_cache_f16, void* v_cache_f16, const int64_t* pos,
                                      int n, int heads, int kv_heads, int head_dim, int slots, void* stream) {
  if (!out_f16 || !q_f16 || !k_f16 || !v_f16 || !cos_f16 || !sin_f16 || !k_cache_f16 || !v_cache_f16 || !pos)
    return QTIP_E_NULL;
  if (n < 1 || n > 65535 || heads < 1 || heads > 65535 || kv_heads < 1 || heads % kv_heads || slots < 1 ||
      (head_dim != 64 && head_dim != 128))
    return QTIP_E_SHAPE;
  if (q_stride < heads * head_dim || k_stride < kv_heads * head_dim || v_stride < kv_heads * head_dim) return QTIP_E_SHAPE;
  if (!aligned16(out_f16) || !aligned16(q_f16) || !aligned16(k_f16) || !aligned16(v_f16) || !aligned16(cos_f16) ||
      !aligned16(sin_f16) || !aligned16(k_cache_f16) || !aligned16(v_cache_f16) || ((q_stride | k_stride | v_stride) & 7) ||
      (reinterpret_cast<uintptr_t>(pos) & 7u))
    return QTIP_E_ALIGN;
  hipStream_t st = (hipStream_t)stream;
  auto* kc = (_Float16*)k_cache_f16;
  auto* vc = (_Float16*)v_cache_f16;
  auto* c = (const _Float16*)cos_f16;
  auto* s = (const _Float16*)sin_f16;
  const long items = (long)n * kv_heads * (head_dim >> 4);
  cache_rows_kernel<<<(unsigned)((items + kBlock - 1) / kBlock), kBlock, 0, st>>>(
      kc, vc, (const _Float16*)k_f16, (const _Float16*)v_f16, k_stride, v_stride, c, s, pos, n, kv_heads, head_dim, slots);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return (int)e;
  const int tiles = (n + kQ - 1) / kQ;
  const long wgs = (long)tiles * heads;
  const dim3 grid((unsigned)heads, (unsigned)tiles);
  // Two workgroups a CU at most: the second ones come shortest first, beside the longest (32 heads, 1000 tokens: 16 tiles of keys
  // and 1 to 9 and 8).  More of them take the place of those that end, longest first.
  const int cus = qtip_device_cus(), turn = cus > 0 && wgs <= 2L * cus ? cus : (int)wgs;
  const int group = heads / kv_heads;
  const float log2e = 1.44269504088896340736f;
  if (head_dim == 128)
    prefill_attn_kernel<128><<<grid, kBlock, 0, st>>>((_Float16*)out_f16, (const _Float16*)q_f16, q_stride, c, s, kc, vc, pos,
                                                      n, heads, group, slots, log2e * 0.08838834764831845f, turn);
  else
    prefill_attn_kernel<64><<<grid, kBlock, 0, st>>>((_Float16*)out_f16, (const _Float16*)q_f16, q_stride, c, s, kc, vc, pos,
                                                     n, heads, group, slots, log2e * 0.125f, turn);
  return (int)hipGetLastError();
}
