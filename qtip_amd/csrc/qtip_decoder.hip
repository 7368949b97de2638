// Single-token decode attention for the end-to-end decode loop: rotary
// embedding of q and k, KV-cache write and attention over the cache in one
// launch (the reference runs these as a dozen framework kernels:
// model/llama.py:264-295 RoPE, model/cache_utils.py:1173-1193 cache update,
// model/llama.py:866-880 scaled-dot-product attention).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/qtip_hip.h"
#include "qtip_shares.h"
#include "qtip_wht.h"

namespace {

constexpr int kAttnThreads = 1024;
constexpr int kMaxHeadDim = 256;

// Cross-lane exchanges go through qtip_wht::lane_xor (DPP, ds_swizzle, v_permlane32_swap: a few
// cycles each); a generic shuffle is a ds_bpermute with an LDS round trip per step, which these
// latency-bound kernels feel.
__device__ __forceinline__ int lane_xor_i(int v, int b) {
  return __builtin_bit_cast(int, qtip_wht::lane_xor(__builtin_bit_cast(float, v), b));
}
// The qkv projection's output transform, for the XF form of the kernel: the new token's
// [q | k | v] vector (n = order * 2^logp2 elements) is
//   post * scale * (H_order (x) H_{2^logp2}) (sum of the in_parts partial sums),
// and a workgroup needs three D-long slices of it.  A slice (table row iK, block b of the
// power-of-two part) is the D-point Walsh-Hadamard transform of
//   u[c] = sum_{jK, b'} (-1)^(bits[jK][iK] + popcount(b & b')) v[(jK * 2^logp2) + b' * D + c],
// n additions per slice instead of a launch of its own for the whole vector.
// XF = 1: q, k and v are slices of one transformed vector [q | k | v] (fused projection; entry 0
// of the arrays below describes it).  XF = 2: three vectors with a transform each (separate
// projections): q of heads * D elements, k and v of kv_heads * D.
struct AttnXf {
  const float* parts[3];
  const float* post[3];
  const uint32_t* had_bits[3];
  size_t part_stride;
  float scale[3];
  int order[3], logp2[3], n[3];
  int in_parts;
};

typedef float float4a __attribute__((ext_vector_type(4)));
typedef uint32_t uint4a __attribute__((ext_vector_type(4)));
typedef _Float16 half8a __attribute__((ext_vector_type(8)));

// value of lane 7 - i of the eight lanes (sums of four equal lanes: the other four)
__device__ __forceinline__ float dpp_half_mirror(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xF, 0xF, false));
}

// x * c + y * s, both products and the sum rounded to fp16 as in the prompt's kernels and the module's own arithmetic.  (Left
// to itself the compiler makes one product and the sum a single operation of one rounding, in some instances of a kernel and
// not in others.)
__device__ __forceinline__ _Float16 rotated(_Float16 x, _Float16 c, _Float16 y, _Float16 s) {
#pragma clang fp contract(off)
  const _Float16 a = x * c, b = y * s;
  return a + b;
}

// One workgroup per query head and key range.  qkv: [H*D | Hkv*D | Hkv*D] fp16 of the new
// token; k_cache / v_cache: [Hkv][max_len][D] fp16; pos_ptr: position of the
// new token (device memory, so that a recorded graph follows the position).
// nsplit > 1 (long contexts): workgroup blockIdx.z takes the keys
// [z * keys_per_split, (z + 1) * keys_per_split) and leaves its share - the D unnormalised output
// sums, its score maximum and its sum of exponentials - in split_ws[head][z][D + 2] for
// attn_combine_kernel; every workgroup repeats the prologue (transform, rotary embedding), the
// one of range 0 writes the cache.
// keys_per_split = 0: the ranges of qtip_shares.h, whose shares the next matvec reads; no workgroup past those in use does
// anything.
template <int D, int XF>
__global__ __launch_bounds__(kAttnThreads) void decode_attn_kernel(
    _Float16* __restrict__ out, const _Float16* __restrict__ qkv, _Float16* __restrict__ k_cache,
    _Float16* __restrict__ v_cache, const long* __restrict__ pos_ptr,
    const float* __restrict__ inv_freq, int H, int Hkv, int max_len, const AttnXf X, int nsplit,
    int keys_per_split, float* __restrict__ split_ws) {
  extern __shared__ __align__(16) uint8_t smem[];
  float* new_s = reinterpret_cast<float*>(smem);  // [3][kMaxHeadDim] rotated query, rotated new key, new value (fp16 values)
  float* swap_s = new_s + 3 * kMaxHeadDim;        // [3][kMaxHeadDim] last level of the prologue's transform
  float* red = swap_s + 3 * kMaxHeadDim;          // [2][16] maxima and sums of the waves
  float* acc = red + 32;                          // [16][D] outputs of the waves; the prologue's [3][16][D] before that
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // grid = (query heads per kv head, kv heads): no integer division on the way to the loads
  const int rep = gridDim.x, kvh = blockIdx.y, h = kvh * rep + blockIdx.x;
  const int pos = (int)pos_ptr[0];
  constexpr int LOGD = D == 64 ? 6 : (D == 128 ? 7 : 8);
  constexpr int half = D >> 1;
  _Float16* kc = k_cache + (size_t)kvh * max_len * D;
  _Float16* vc = v_cache + (size_t)kvh * max_len * D;
  // threads tid < 3 * D hold element c of the new token's query (s3 = 0), key (1) and value (2)
  const int s3 = tid >> LOGD, place = qtip_wht::wht_place(lane), c = ((tid & ~63) | place) & (D - 1);
  const float freq = tid < 2 * D ? inv_freq[c & (half - 1)] : 0.f;
  float postv = 1.f, postp = 1.f;
  _Float16 own = (_Float16)0.f, pair = (_Float16)0.f;  // element c and the one that it is rotated with
  if constexpr (!XF) {
    if (tid < 3 * D) {
      const _Float16* e = qkv + (size_t)(s3 == 0 ? h : (s3 == 1 ? H + kvh : H + Hkv + kvh)) * D;
      own = e[c];
      pair = e[c ^ half];
    }
  }

  // rotary angle of the thread's element: the fp32 product the reference forms; its reduction to a fraction of a
  // turn is done in fp64 (exact to 2^-29 of a turn at position 4096), the hardware cos / sin take
  // turns.  (cosf / sinf with their large-argument paths cost ~0.5 us on this kernel's critical path.)
  _Float16 rc = (_Float16)1.f, rs = (_Float16)0.f;
  auto rotary = [&] {
    const float ang = (float)pos * freq;
    const double turns = (double)ang * 0.15915494309189535;
    const float fr = (float)(turns - __builtin_floor(turns));
    rc = (_Float16)__builtin_amdgcn_cosf(fr);
    rs = (_Float16)__builtin_amdgcn_sinf(fr);
  };

  // ---- the cached keys [k0, kend) of this workgroup, in units of U: wave w takes keys t0 + w * KPW .. + KPW - 1 of
  // a unit, a key of D values on D / 8 lanes.  One pass with a running maximum, a wave by itself, NU units of keys and
  // values in flight, the first ones from before the transform's last levels and the rotary embedding on.  The part of the
  // launch that grows with the keys is what one CU draws from memory, 50 to 60 bytes a ns: more in flight is no
  // faster (a token of 8 layers, 500 keys: two units 548 us, four 549, eight 560), and loads of nothing take the
  // memory unit 0.15 us a unit.  us a token of 8 layers of 4096 (32 heads of 128), 60 / 200 / 500 / 900 keys, scores and
  // values in two passes over all keys with six barriers / here: 531 537 562 599 / 523 529 549 587; separate
  // projections 528 537 562 / 520 527 547.
  constexpr int LPK = D / 8, KPW = 64 / LPK, U = 16 * KPW, NU = 2;
  const int nkeys = pos + 1 < max_len ? pos + 1 : max_len;
  const bool open = keys_per_split == 0;
  const int used = open ? qtip_shares::active(nkeys, nsplit, H) : nsplit;
  if ((int)blockIdx.z >= used) return;
  const int kps = open ? qtip_shares::keys_of(nkeys, used) : keys_per_split;
  const int k0 = (int)blockIdx.z * kps;  // this workgroup's keys: [k0, k1)
  const int k1 = k0 + kps < nkeys ? k0 + kps : nkeys;
  const int kend = k1 < pos ? k1 : pos;             // (the new key comes from LDS)
  const __amdgpu_buffer_rsrc_t rs_k = __builtin_amdgcn_make_buffer_rsrc(kc, 0, max_len * D * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t rs_v = __builtin_amdgcn_make_buffer_rsrc(vc, 0, max_len * D * 2, 0x00020000);
  const int tl = wave * KPW + lane / LPK, dl = lane & (LPK - 1);
  // the keys and values of a unit are requested together; a lane offset past the end of the cache returns zeros
  auto request = [&](uint4a& k, uint4a& v, int t0) {
    const int off = t0 + tl < kend ? ((t0 + tl) * D + dl * 8) * 2 : 0x7FFFFF00;
    k = __builtin_amdgcn_raw_buffer_load_b128(rs_k, off, 0, 0);
    v = __builtin_amdgcn_raw_buffer_load_b128(rs_v, off, 0, 0);
  };

  if constexpr (XF) {
    static_assert(D == 64 || D == 128, "the transform prologue holds 3 x 16 x D partial sums in LDS");
    constexpr int G = D / 4, R = kAttnThreads / G;  // float4 column groups, chunk rows per pass
    constexpr bool SEP = XF == 2;
    const int g = tid & (G - 1), r = tid >> (LOGD - 2);
    // slices: q of head h, k and v of its kv head - of the one vector, or each of its own
    const int off[3] = {h * D, SEP ? kvh * D : (H + kvh) * D, SEP ? kvh * D : (H + Hkv + kvh) * D};
    int iK[3], bb[3], lgb[3];
#pragma unroll
    for (int s3 = 0; s3 < 3; ++s3) {
      const int lp = X.logp2[SEP ? s3 : 0];
      lgb[s3] = lp - LOGD;
      iK[s3] = off[s3] >> lp;
      bb[s3] = (off[s3] >> LOGD) & ((1 << lgb[s3]) - 1);
    }
    // the epilogue's operands, requested with everything else
    const int sx = SEP ? (s3 < 3 ? s3 : 0) : 0;  // descriptor of this thread's slice
    const float* post = sx == 0 ? X.post[0] : (sx == 1 ? X.post[1] : X.post[2]);
    if (tid < 3 * D && post) {
      const float* e = post + (s3 == 0 ? off[0] : (s3 == 1 ? off[1] : off[2]));
      postv = e[c];
      postp = e[c ^ half];
    }
    float a[3][4];  // (plain arrays: element-wise bit operations on vector-typed values went wrong in the compiler)
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) a[i][e] = 0.f;
    // (chunk rows past the last are out of the descriptor's range and come back as zeros)
    // NV vectors, QP chunk rows and WP partial sums of each in flight (more would spill)
    constexpr int NV = SEP ? 3 : 1, QP = SEP ? 1 : 4, WP = 2;
    auto load = [&](float4a (&raw)[NV][QP][WP], int j0, int w0) {
#pragma unroll
      for (int u = 0; u < WP; ++u)
#pragma unroll
        for (int i = 0; i < NV; ++i) {
          if (w0 + u < X.in_parts) {
            const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<float*>(X.parts[i] + (size_t)(w0 + u) * X.part_stride), 0, X.n[i] * 4, 0x00020000);
#pragma unroll
            for (int q = 0; q < QP; ++q)
              raw[i][q][u] = __builtin_bit_cast(
                  float4a, __builtin_amdgcn_raw_buffer_load_b128(rs, (((j0 + r + q * R) << LOGD) + 4 * g) * 4, 0, 0));
          } else {
#pragma unroll
            for (int q = 0; q < QP; ++q) raw[i][q][u] = float4a{0.f, 0.f, 0.f, 0.f};
          }
        }
    };
    // the table words of the rows.  (With order 1 the index is 0 and the word is masked out: any readable address does.)
    auto words = [&](uint32_t (&hw)[QP][3], int j0) {
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const int x = SEP ? i : 0;
        const uint32_t* hb = X.order[x] > 1 ? X.had_bits[x] : reinterpret_cast<const uint32_t*>(X.parts[x]);
        const int nrows = X.n[x] >> LOGD;
#pragma unroll
        for (int q = 0; q < QP; ++q) {
          const int j = j0 + r + q * R;
          const unsigned bit = (unsigned)((j < nrows ? j : 0) >> lgb[x]) * X.order[x] + iK[i];
          hw[q][i] = hb[bit >> 5] >> (bit & 31);
        }
      }
    };
    auto add = [&](float (&v)[NV][QP][4], const float4a (&raw)[NV][QP][WP]) {
#pragma unroll
      for (int u = 0; u < WP; ++u)
#pragma unroll
        for (int i = 0; i < NV; ++i)
#pragma unroll
          for (int q = 0; q < QP; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[i][q][e] += raw[i][q][u][e];
    };
    auto pass = [&](float4a (&raw)[NV][QP][WP], const uint32_t (&hw)[QP][3], int j0) {
      float v[NV][QP][4] = {};
      add(v, raw);
      for (int w0 = WP; w0 < X.in_parts; w0 += WP) {
        load(raw, j0, w0);
        add(v, raw);
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const int x = SEP ? i : 0;
        const uint32_t omask = X.order[x] > 1 ? 1u : 0u;
        const int bmask = (1 << lgb[x]) - 1;
#pragma unroll
        for (int q = 0; q < QP; ++q) {
          const uint32_t sg =
              (((hw[q][i] & omask) ^ (uint32_t)__builtin_popcount(bb[i] & (j0 + r + q * R) & bmask)) & 1u) << 31;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            a[i][e] += __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v[x][q][e]) ^ sg);
        }
      }
    };
    int maxrows = X.n[0] >> LOGD;
    if constexpr (SEP) {
      maxrows = X.n[1] >> LOGD > maxrows ? X.n[1] >> LOGD : maxrows;
      maxrows = X.n[2] >> LOGD > maxrows ? X.n[2] >> LOGD : maxrows;
    }
    {
      float4a raw[NV][QP][WP];
      uint32_t hw[QP][3];
      words(hw, 0);
      load(raw, 0, 0);
      rotary();
      pass(raw, hw, 0);
      for (int j0 = QP * R; j0 < maxrows; j0 += QP * R) {
        words(hw, j0);
        load(raw, j0, 0);
        pass(raw, hw, j0);
      }
    }
    // rows that share a wave, then one partial slice per wave
#pragma unroll
    for (int b = 5; (1 << b) >= G; --b)
#pragma unroll
      for (int s3 = 0; s3 < 3; ++s3)
#pragma unroll
        for (int e = 0; e < 4; ++e) a[s3][e] += qtip_wht::lane_xor(a[s3][e], b);
    if (lane < G) {
#pragma unroll
      for (int s3 = 0; s3 < 3; ++s3)
        *reinterpret_cast<float4a*>(acc + (s3 * 16 + wave) * D + 4 * g) =
            float4a{a[s3][0], a[s3][1], a[s3][2], a[s3][3]};
    }
  } else {
    rotary();
  }

  // (the registers of the partial sums are free)
  uint4a kb[NU], vb[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) request(kb[u], vb[u], k0 + u * U);
  if constexpr (XF) {
    constexpr bool SEP = XF == 2;
    const int sx = SEP ? (s3 < 3 ? s3 : 0) : 0;
    const float scalev = sx == 0 ? X.scale[0] : (sx == 1 ? X.scale[1] : X.scale[2]);
    __syncthreads();
    // the other half of a slice, behind the last level of the transform, is what an element is rotated with
    float y = 0.f, z = 0.f;
    if (tid < 3 * D) {
#pragma unroll
      for (int w = 0; w < 16; ++w) y += acc[(s3 * 16 + w) * D + c];
      y = qtip_wht::wht_places(y, 6, place);
      if constexpr (D > 64) swap_s[s3 * kMaxHeadDim + c] = y;
      else z = qtip_wht::lane_xor(y, 5);
    }
    if constexpr (D > 64) {
      __syncthreads();
      if (tid < 3 * D) {
        const float other = swap_s[s3 * kMaxHeadDim + (c ^ 64)];
        z = (c & 64) ? other + y : y - other;
        y = (c & 64) ? other - y : y + other;
      }
    }
    own = (_Float16)(y * scalev * postv);
    pair = (_Float16)(z * scalev * postp);
  }

  // ---- rotary embedding in fp16 arithmetic: x*cos + rotate_half(x)*sin
  if (tid < 3 * D) {
    const _Float16 rot = c < half ? (_Float16)(-(float)pair) : pair;
    _Float16 e = rotated(own, rc, rot, rs);
    if (s3 == 2) e = own;
    new_s[s3 * kMaxHeadDim + c] = (float)e;
    if (s3 && blockIdx.x == 0 && blockIdx.z == 0 && pos < max_len) (s3 == 1 ? kc : vc)[(size_t)pos * D + c] = e;
  }
  __syncthreads();

  // ---- softmax(q k) v of the lane group's keys with a running maximum: mx, the sum of exponentials l and the
  // unnormalised outputs o (dims 8 * dl ..); the first group of wave 0 starts with the new key
  const float sm_scale = rsqrtf((float)D);
  float q[8], o[8], mx = -INFINITY, l = 0.f;
  auto row_sum = [&](float s) {  // over the lanes of a key
    s += qtip_wht::lane_xor(s, 0);
    s += qtip_wht::lane_xor(s, 1);
    s += dpp_half_mirror(s);
    if constexpr (LPK >= 16) s += qtip_wht::lane_xor(s, 3);
    if constexpr (LPK >= 32) s += qtip_wht::lane_xor(s, 4);
    return s;
  };
  {
    const bool fresh = tl == 0 && pos >= k0 && pos < k1;
    float s = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      q[e] = new_s[dl * 8 + e];
      s += q[e] * new_s[kMaxHeadDim + dl * 8 + e];
    }
    s = row_sum(s) * sm_scale;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = 0.f;
    if (fresh) {
      mx = s;
      l = __expf(s - (s == -INFINITY ? 0.f : s));  // 1; 0 for -inf, NaN for NaN and inf
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = l * new_s[2 * kMaxHeadDim + dl * 8 + e];
    }
  }
  for (int t0 = k0;;) {
    float s[NU], m = mx;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const half8a kv = __builtin_bit_cast(half8a, kb[u]);
      float d = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) d += q[e] * (float)kv[e];
      d = row_sum(d) * sm_scale;
      s[u] = t0 + u * U + tl < kend ? d : -INFINITY;
      m = fmaxf(m, s[u]);
    }
    const float ms = m == -INFINITY ? 0.f : m;  // (nothing but scores of -inf so far: all of weight 0)
    const float keep = __expf(mx - ms);
    mx = m;
    l *= keep;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] *= keep;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const half8a vv = __builtin_bit_cast(half8a, vb[u]);
      const float pt = __expf(s[u] - ms);
      l += pt;
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] += pt * (float)vv[e];
    }
    t0 += NU * U;
    if (t0 >= kend) break;
#pragma unroll
    for (int u = 0; u < NU; ++u) request(kb[u], vb[u], t0 + u * U);
  }

  // ---- the lane groups of a wave, then the waves
  {
    float m = mx;
#pragma unroll
    for (int b = 5; (1 << b) >= LPK; --b) m = fmaxf(m, qtip_wht::lane_xor(m, b));
    const float f = m == -INFINITY ? 0.f : __expf(mx - m);
    l *= f;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] *= f;
#pragma unroll
    for (int b = 5; (1 << b) >= LPK; --b) {
      l += qtip_wht::lane_xor(l, b);
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] += qtip_wht::lane_xor(o[e], b);
    }
    if (lane < LPK) {
      *reinterpret_cast<float4a*>(acc + wave * D + dl * 8) = float4a{o[0], o[1], o[2], o[3]};
      *reinterpret_cast<float4a*>(acc + wave * D + dl * 8 + 4) = float4a{o[4], o[5], o[6], o[7]};
    }
    if (lane == 0) {
      red[wave] = m;
      red[16 + wave] = l;
    }
  }
  __syncthreads();
  if (tid >= D) return;
  mx = -INFINITY;
#pragma unroll
  for (int w = 0; w < 16; ++w) mx = fmaxf(mx, red[w]);
  float sum = 0.f, tot = 0.f;
#pragma unroll
  for (int w = 0; w < 16; ++w) {
    const float f = red[w] == -INFINITY ? 0.f : __expf(red[w] - mx);
    tot += f * red[16 + w];
    sum += f * acc[w * D + tid];
  }
  if (nsplit == 1 && !open) {
    out[(size_t)h * D + tid] = (_Float16)(sum * (1.f / tot));
  } else {
    float* w = split_ws + ((size_t)h * nsplit + blockIdx.z) * (open ? qtip_shares::floats(D) : D + 2);
    w[tid] = sum;       // 0 for a range past the last key
    if (tid == 0) {
      w[D] = mx;        // -inf for an empty range
      w[D + 1] = tot;
    }
  }
}

// out[head] = sum_z exp(m_z - M) o_z / sum_z exp(m_z - M) l_z over the key ranges of a head
// (M = max_z m_z): the softmax of the whole context from the shares of its ranges.
__global__ __launch_bounds__(kMaxHeadDim) void attn_combine_kernel(_Float16* __restrict__ out,
                                                                  const float* __restrict__ split_ws,
                                                                  int nsplit, int D) {
  const int h = blockIdx.x, d = threadIdx.x;
  const float* w = split_ws + (size_t)h * nsplit * (D + 2);
  float M = -INFINITY;
  for (int z = 0; z < nsplit; ++z) M = fmaxf(M, w[z * (D + 2) + D]);
  float num = 0.f, den = 0.f;
  for (int z = 0; z < nsplit; ++z) {
    const float mz = w[z * (D + 2) + D];
    const float e = mz == -INFINITY ? 0.f : __expf(mz - M);
    num += e * w[z * (D + 2) + d];
    den += e * w[z * (D + 2) + D + 1];
  }
  out[(size_t)h * D + d] = (_Float16)(num / den);
}

}  // namespace

static int launch_attention(void* out_f16, const void* qkv_f16, const AttnXf* xf, int xf_mode, void* k_cache_f16,
                            void* v_cache_f16, const void* pos_i64, const float* inv_freq, int heads,
                            int kv_heads, int head_dim, int max_len, int key_splits, float* split_ws,
                            void* stream, bool open = false) {
  if ((!out_f16 && !open) || !k_cache_f16 || !v_cache_f16 || !pos_i64 || !inv_freq) return QTIP_E_NULL;
  if (key_splits < 1 || key_splits > 16) return QTIP_E_SHAPE;
  if ((key_splits > 1 || open) && !split_ws) return QTIP_E_NULL;
  if ((key_splits > 1 || open) && (reinterpret_cast<uintptr_t>(split_ws) & 15)) return QTIP_E_ALIGN;
  if (heads < 1 || kv_heads < 1 || heads % kv_heads || head_dim < 64 || head_dim > kMaxHeadDim ||
      (head_dim & (head_dim - 1)) || max_len < 1 || max_len > 4096)  // (positions the rotary reduction is stated for)
    return QTIP_E_SHAPE;
  const size_t lds = (size_t)(6 * kMaxHeadDim + 32 + (xf ? 3 : 1) * 16 * head_dim) * sizeof(float);
  const dim3 grid((unsigned)(heads / kv_heads), (unsigned)kv_heads, (unsigned)key_splits);
  const int kps = open ? 0 : (max_len + key_splits - 1) / key_splits;  // keys per range
#define QTIP_ATTN(DD, XX, ARG)                                                                      \
  decode_attn_kernel<DD, XX><<<grid, kAttnThreads, lds, (hipStream_t)stream>>>(                      \
      (_Float16*)out_f16, (const _Float16*)qkv_f16, (_Float16*)k_cache_f16, (_Float16*)v_cache_f16,  \
      (const long*)pos_i64, inv_freq, heads, kv_heads, max_len, ARG, key_splits, kps, split_ws)
  if (xf) {
    if (head_dim != 64 && head_dim != 128) return QTIP_E_SHAPE;
    if (xf_mode == 1) {
      if (head_dim == 64) QTIP_ATTN(64, 1, *xf); else QTIP_ATTN(128, 1, *xf);
    } else {
      if (head_dim == 64) QTIP_ATTN(64, 2, *xf); else QTIP_ATTN(128, 2, *xf);
    }
  } else {
    switch (head_dim) {
      case 64: QTIP_ATTN(64, 0, AttnXf{}); break;
      case 128: QTIP_ATTN(128, 0, AttnXf{}); break;
      default: QTIP_ATTN(256, 0, AttnXf{}); break;
    }
  }
#undef QTIP_ATTN
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || key_splits == 1 || open) return (int)e;
  attn_combine_kernel<<<heads, head_dim, 0, (hipStream_t)stream>>>((_Float16*)out_f16, split_ws, key_splits,
                                                                   head_dim);
  return (int)hipGetLastError();
}

// one transformed vector of n elements: table order and log2 of the power-of-two part
static int fill_xf_slot(AttnXf& x, int slot, const float* parts, const float* post, const uint32_t* had_bits,
                        float scale, int order, long n, int head_dim) {
  if (!parts || (order > 1 && !had_bits)) return QTIP_E_NULL;
  if (order < 1 || order > 256 || n % order) return QTIP_E_SHAPE;
  const long p2 = n / order;
  if ((p2 & (p2 - 1)) || p2 < head_dim || n > (1 << 20)) return QTIP_E_SHAPE;
  if (reinterpret_cast<uintptr_t>(parts) & 15) return QTIP_E_ALIGN;
  x.parts[slot] = parts;
  x.post[slot] = post;
  x.had_bits[slot] = had_bits;
  x.scale[slot] = scale;
  x.order[slot] = order;
  x.logp2[slot] = 0;
  while ((1L << x.logp2[slot]) < p2) ++x.logp2[slot];
  x.n[slot] = (int)n;
  return QTIP_OK;
}

extern "C" int qtip_decode_attention(void* out_f16, const void* qkv_f16, void* k_cache_f16,
                                     void* v_cache_f16, const void* pos_i64, const float* inv_freq,
                                     int heads, int kv_heads, int head_dim, int max_len, int key_splits,
                                     float* split_workspace, void* stream) {
  if (!qkv_f16) return QTIP_E_NULL;
  return launch_attention(out_f16, qkv_f16, nullptr, 0, k_cache_f16, v_cache_f16, pos_i64, inv_freq, heads,
                          kv_heads, head_dim, max_len, key_splits, split_workspace, stream);
}

extern "C" int qtip_decode_attention_rht(void* out_f16, const float* parts, int in_parts, size_t part_stride,
                                         const float* post_f32, float scale, const uint32_t* had_bits,
                                         int order, void* k_cache_f16, void* v_cache_f16,
                                         const void* pos_i64, const float* inv_freq, int heads,
                                         int kv_heads, int head_dim, int max_len, int key_splits,
                                         float* split_workspace, void* stream) {
  if (in_parts < 1 || in_parts > 16 || heads < 1 || kv_heads < 1 || head_dim < 64 || head_dim > 128 ||
      (part_stride & 3))
    return QTIP_E_SHAPE;
  AttnXf x = {};
  const int rc = fill_xf_slot(x, 0, parts, post_f32, had_bits, scale, order,
                              (long)(heads + 2 * kv_heads) * head_dim, head_dim);
  if (rc) return rc;
  x.part_stride = part_stride;
  x.in_parts = in_parts;
  return launch_attention(out_f16, nullptr, &x, 1, k_cache_f16, v_cache_f16, pos_i64, inv_freq, heads, kv_heads,
                          head_dim, max_len, key_splits, split_workspace, stream);
}

extern "C" int qtip_decode_attention_rht3(void* out_f16, const float* const* parts, int in_parts,
                                          size_t part_stride, const float* const* post_f32, const float* scale,
                                          const uint32_t* const* had_bits, const int* order, void* k_cache_f16,
                                          void* v_cache_f16, const void* pos_i64, const float* inv_freq,
                                          int heads, int kv_heads, int head_dim, int max_len, int key_splits,
                                          float* split_workspace, void* stream) {
  if (!parts || !post_f32 || !scale || !had_bits || !order) return QTIP_E_NULL;
  if (in_parts < 1 || in_parts > 16 || heads < 1 || kv_heads < 1 || head_dim < 64 || head_dim > 128 ||
      (part_stride & 3))
    return QTIP_E_SHAPE;
  AttnXf x = {};
  for (int s = 0; s < 3; ++s) {
    const long n = (long)(s == 0 ? heads : kv_heads) * head_dim;
    const int rc = fill_xf_slot(x, s, parts[s], post_f32[s], had_bits[s], scale[s], order[s], n, head_dim);
    if (rc) return rc;
  }
  x.part_stride = part_stride;
  x.in_parts = in_parts;
  return launch_attention(out_f16, nullptr, &x, 2, k_cache_f16, v_cache_f16, pos_i64, inv_freq, heads, kv_heads,
                          head_dim, max_len, key_splits, split_workspace, stream);
}

extern "C" int qtip_decode_attention_shares(float* shares, int ranges, int vectors, const float* const* parts, int in_parts,
                                            size_t part_stride, const float* const* post_f32, const float* scale,
                                            const uint32_t* const* had_bits, const int* order, void* k_cache_f16,
                                            void* v_cache_f16, const void* pos_i64, const float* inv_freq, int heads, int kv_heads,
                                            int head_dim, int max_len, void* stream) {
  if (!parts || !post_f32 || !scale || !had_bits || !order) return QTIP_E_NULL;
  if ((vectors != 1 && vectors != 3) || ranges < 1 || ranges > qtip_shares::kMaxRanges || in_parts < 1 || in_parts > 16 ||
      heads < 1 || kv_heads < 1 || head_dim < 64 || head_dim > 128 || (part_stride & 3))
    return QTIP_E_SHAPE;
  AttnXf x = {};
  for (int s = 0; s < vectors; ++s) {
    const long n = (long)(vectors == 1 ? heads + 2 * kv_heads : (s == 0 ? heads : kv_heads)) * head_dim;
    const int rc = fill_xf_slot(x, s, parts[s], post_f32[s], had_bits[s], scale[s], order[s], n, head_dim);
    if (rc) return rc;
  }
  x.part_stride = part_stride;
  x.in_parts = in_parts;
  return launch_attention(nullptr, nullptr, &x, vectors == 1 ? 1 : 2, k_cache_f16, v_cache_f16, pos_i64, inv_freq, heads, kv_heads,
                          head_dim, max_len, ranges, shares, stream, true);
}

// ---- token head of the decode loop: final RMSNorm and the greedy pick ------------------------

namespace {

constexpr int kHeadThreads = 1024;

// out = w * fp16(x * rsqrt(mean(x^2) + eps)) for a row of n (model/llama.py:129-135), one workgroup.
// Bound by one cold read: V elements a load, 8 where the vectors start on 16 bytes and n is a multiple of 8 (one
// element at a time, sixteen loads of either vector: 4096 6.1 us in a token, 8192 9.7; now 5.0 and 5.2).  Workgroups are as
// wide as the row: 1000 rows of 4096 take 6 us, the eight library passes of the module's formula 64.
template <int V>
__global__ __launch_bounds__(kHeadThreads) void rmsnorm_kernel(_Float16* __restrict__ out,
                                                               const _Float16* __restrict__ x,
                                                               const _Float16* __restrict__ w, float eps,
                                                               int n) {
  __shared__ float wsum[16];
  typedef _Float16 vec __attribute__((ext_vector_type(V)));
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, waves = blockDim.x >> 6;
  x += (size_t)blockIdx.x * n;
  out += (size_t)blockIdx.x * n;
  constexpr int MAXE = 16 / V;  // n <= 16384
  vec v[MAXE], g[MAXE];
#pragma unroll
  for (int e = 0; e < MAXE; ++e) {
    const int i = (tid + e * (int)blockDim.x) * V;
    v[e] = vec{};
    if (i < n) {
      v[e] = *reinterpret_cast<const vec*>(x + i);
      g[e] = *reinterpret_cast<const vec*>(w + i);
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < MAXE; ++e)
#pragma unroll
    for (int q = 0; q < V; ++q) ss += (float)v[e][q] * (float)v[e][q];
  ss = qtip_wht::wave_sum(ss);
  if (lane == 0) wsum[wave] = ss;
  __syncthreads();
  float tot = 0.f;
#pragma unroll
  for (int q = 0; q < 16; ++q) tot += q < waves ? wsum[q] : 0.f;
  const float rs = __builtin_amdgcn_rsqf(tot / (float)n + eps);
#pragma unroll
  for (int e = 0; e < MAXE; ++e) {
    const int i = (tid + e * (int)blockDim.x) * V;
    if (i < n) {
      vec y;
#pragma unroll
      for (int q = 0; q < V; ++q) y[q] = (_Float16)((float)g[e][q] * (float)(_Float16)((float)v[e][q] * rs));
      *reinterpret_cast<vec*>(out + i) = y;
    }
  }
}

// argmax of fp16 logits (first index among equal maxima, NaNs never win), stored as the next
// input token and into the history slot of this position; the position advances by one.  All in
// device memory, so a recorded graph decodes token after token without host work in between
// (eval/interactive_gen.py:43-69 does this with argmax, copies and an increment per token).
__global__ __launch_bounds__(kHeadThreads) void greedy_pick_kernel(const _Float16* __restrict__ logits, int vocab,
                                                                   long* __restrict__ tok, long* __restrict__ pos,
                                                                   long* __restrict__ hist, long hist_len,
                                                                   long hist_base) {
  __shared__ float bv[16];
  __shared__ int bi[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  float best = -INFINITY;
  int idx = 0x7fffffff;
  const int nch = vocab >> 3;  // 16-byte chunks
  for (int c = tid; c < nch; c += kHeadThreads) {
    const uint4 raw = reinterpret_cast<const uint4*>(logits)[c];
    const _Float16* h = reinterpret_cast<const _Float16*>(&raw);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float f = (float)h[e];
      if (f > best) {  // chunks come in increasing order per thread: the first maximum stays
        best = f;
        idx = c * 8 + e;
      }
    }
  }
  for (int i = (nch << 3) + tid; i < vocab; i += kHeadThreads) {
    const float f = (float)logits[i];
    if (f > best) {
      best = f;
      idx = i;
    }
  }
#pragma unroll
  for (int b = 0; b < 6; ++b) {
    const float ob = qtip_wht::lane_xor(best, b);
    const int oi = lane_xor_i(idx, b);
    if (ob > best || (ob == best && oi < idx)) {
      best = ob;
      idx = oi;
    }
  }
  if (lane == 0) {
    bv[wave] = best;
    bi[wave] = idx;
  }
  __syncthreads();
  if (tid == 0) {
    for (int q = 1; q < 16; ++q)
      if (bv[q] > best || (bv[q] == best && bi[q] < idx)) {
        best = bv[q];
        idx = bi[q];
      }
    if (idx == 0x7fffffff) idx = 0;  // nothing compared greater than -inf
    const long p = pos[0];
    const long slot = p - hist_base;
    if (hist && slot >= 0 && slot < hist_len) hist[slot] = idx;
    tok[0] = idx;
    pos[0] = p + 1;
  }
}

}  // namespace

extern "C" int qtip_rmsnorm_rows(void* out_f16, const void* x_f16, const void* weight_f16, float eps, long rows, int n,
                                 void* stream) {
  if (!out_f16 || !x_f16 || !weight_f16) return QTIP_E_NULL;
  if (n < 1 || n > 16 * kHeadThreads || rows < 1) return QTIP_E_SHAPE;
  const bool wide = !(n & 7) && !((reinterpret_cast<uintptr_t>(out_f16) | reinterpret_cast<uintptr_t>(x_f16) |
                                   reinterpret_cast<uintptr_t>(weight_f16)) & 15);
  auto* kernel = wide ? rmsnorm_kernel<8> : rmsnorm_kernel<1>;
  const int loads = wide ? n >> 3 : n;
  const int threads = loads < kHeadThreads ? (loads + 63) & ~63 : kHeadThreads;
  for (long r = 0; r < rows; r += 1 << 20) {  // (a launch holds fewer than 2^32 threads)
    kernel<<<(unsigned)(rows - r < 1 << 20 ? rows - r : 1 << 20), threads, 0, (hipStream_t)stream>>>(
        (_Float16*)out_f16 + r * n, (const _Float16*)x_f16 + r * n, (const _Float16*)weight_f16, eps, n);
    if (const hipError_t e = hipGetLastError()) return (int)e;
  }
  return 0;
}

extern "C" int qtip_rmsnorm(void* out_f16, const void* x_f16, const void* weight_f16, float eps, int n, void* stream) {
  return qtip_rmsnorm_rows(out_f16, x_f16, weight_f16, eps, 1, n, stream);
}

extern "C" int qtip_greedy_pick(const void* logits_f16, int vocab, void* tok_i64, void* pos_i64,
                                void* history_i64, long history_len, long history_base, void* stream) {
  if (!logits_f16 || !tok_i64 || !pos_i64) return QTIP_E_NULL;
  if (vocab < 1 || history_len < 0 || (reinterpret_cast<uintptr_t>(logits_f16) & 15)) return QTIP_E_SHAPE;
  greedy_pick_kernel<<<1, kHeadThreads, 0, (hipStream_t)stream>>>((const _Float16*)logits_f16, vocab, (long*)tok_i64,
                                                                 (long*)pos_i64, (long*)history_i64, history_len,
                                                                 history_base);
  return (int)hipGetLastError();
}

// ---- sampled token pick ----------------------------------------------------------------------

namespace {

__device__ __forceinline__ uint32_t mix32(uint32_t x) {
  x ^= x >> 16;
  x *= 0x7feb352dU;
  x ^= x >> 15;
  x *= 0x846ca68bU;
  x ^= x >> 16;
  return x;
}

// (value, index) pairs ordered by value descending, index ascending; `before(a, b)`: a comes first
__device__ __forceinline__ bool before(float av, int ai, float bv, int bi) {
  return av > bv || (av == bv && ai < bi);
}

// Sampling of eval/interactive_gen.py:15-40 in one launch: logits / temperature, everything below
// the top_k-th largest logit removed (ties with it stay, as torch.where(logits < kth, -inf, logits)
// keeps them), softmax, and a draw by the exponential race argmax(p_i / q_i), q_i ~ Exp(1) - which
// is argmax(logit_i / T - log q_i).  The q_i come from a counter-based generator keyed by (seed,
// draw counter, i); the counter lives in device memory and advances with every launch, so a
// recorded graph draws fresh numbers at every replay.  Bookkeeping as in greedy_pick_kernel.
__global__ __launch_bounds__(kHeadThreads) void sample_pick_kernel(const _Float16* __restrict__ logits, int vocab,
                                                                   float inv_temperature, int top_k, uint32_t seed,
                                                                   long* __restrict__ counter, long* __restrict__ tok,
                                                                   long* __restrict__ pos, long* __restrict__ hist,
                                                                   long hist_len, long hist_base) {
  __shared__ float bv[16];
  __shared__ int bi[16];
  __shared__ float sel_v;
  __shared__ int sel_i;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // block-wide first element in (value desc, index asc) order among those after (pv, pi)
  auto next_after = [&](float pv, int pi, auto&& score) {
    float best = -INFINITY;
    int idx = 0x7fffffff;
    for (int i = tid; i < vocab; i += kHeadThreads) {
      const float raw = (float)logits[i];
      if (before(pv, pi, raw, i)) {  // strictly after the previous pick
        const float f = score(raw, i);
        if (before(f, i, best, idx)) {
          best = f;
          idx = i;
        }
      }
    }
#pragma unroll
    for (int b = 0; b < 6; ++b) {
      const float ob = qtip_wht::lane_xor(best, b);
      const int oi = lane_xor_i(idx, b);
      if (before(ob, oi, best, idx)) {
        best = ob;
        idx = oi;
      }
    }
    __syncthreads();  // the previous round's result has been read by everyone
    if (lane == 0) {
      bv[wave] = best;
      bi[wave] = idx;
    }
    __syncthreads();
    if (tid == 0) {
      for (int q = 1; q < 16; ++q)
        if (before(bv[q], bi[q], best, idx)) {
          best = bv[q];
          idx = bi[q];
        }
      sel_v = best;
      sel_i = idx;
    }
    __syncthreads();
  };
  // ---- the top_k-th largest logit (with multiplicity): top_k rounds of "next in order"
  float kth = -INFINITY;
  if (top_k > 0 && top_k < vocab) {
    float pv = INFINITY;
    int pi = -1;
    for (int r = 0; r < top_k; ++r) {
      next_after(pv, pi, [](float raw, int) { return raw; });
      pv = sel_v;
      pi = sel_i;
    }
    kth = pv;
  }
  // ---- the race: argmax over the kept entries of logit / T - log(q), q = -log(u)
  const uint32_t draw = (uint32_t)counter[0];
  const uint32_t key = mix32(seed ^ mix32(draw + 0x9e3779b9U));
  next_after(INFINITY, -1, [&](float raw, int i) {
    if (raw < kth) return -INFINITY;
    const uint32_t h = mix32(key ^ mix32((uint32_t)i * 0x85ebca6bU + 1u));
    const float u = ((float)(h >> 8) + 0.5f) * (1.0f / 16777216.0f);  // (0, 1)
    return raw * inv_temperature - __logf(-__logf(u));
  });
  if (tid == 0) {
    int idx = sel_i;
    if (idx == 0x7fffffff) idx = 0;
    const long p = pos[0];
    const long slot = p - hist_base;
    if (hist && slot >= 0 && slot < hist_len) hist[slot] = idx;
    tok[0] = idx;
    pos[0] = p + 1;
    counter[0] = (long)draw + 1;
  }
}

}  // namespace

extern "C" int qtip_sample_pick(const void* logits_f16, int vocab, float temperature, int top_k,
                                unsigned seed, void* counter_i64, void* tok_i64, void* pos_i64,
                                void* history_i64, long history_len, long history_base, void* stream) {
  if (!logits_f16 || !counter_i64 || !tok_i64 || !pos_i64) return QTIP_E_NULL;
  if (vocab < 1 || history_len < 0 || top_k < 0 || top_k > 64) return QTIP_E_SHAPE;
  const float t = temperature > 1e-5f ? temperature : 1e-5f;  // max(temperature, 1e-5) as the reference
  sample_pick_kernel<<<1, kHeadThreads, 0, (hipStream_t)stream>>>((const _Float16*)logits_f16, vocab, 1.0f / t, top_k,
                                                                 seed, (long*)counter_i64, (long*)tok_i64,
                                                                 (long*)pos_i64, (long*)history_i64, history_len,
                                                                 history_base);
  return (int)hipGetLastError();
}
