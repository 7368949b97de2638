// The (table (x) H_A) factor of a randomised Hadamard transform as a +-1 operand of the matrix cores, shared by the
// transforms of many rows and the transform in front of a matvec.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "qtip_wht.h"

namespace qtip_mix {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 half8m __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4m __attribute__((ext_vector_type(4)));
typedef float float4m __attribute__((ext_vector_type(4)));

// eight +-1 values (`one` = twice the 16-bit pattern of 1) from the bits of a byte (1 = -1)
__device__ __forceinline__ u32x4m expand_signs(uint32_t b, uint32_t one) {
  const uint32_t u = b | (b << 15);
  u32x4m r;
#pragma unroll
  for (int q = 0; q < 4; ++q) r[q] = ((u << (15 - 2 * q)) & 0x80008000u) | one;
  return r;
}

// Signs of output row row0 + a (a = lane % 16, row0 a multiple of 16) against rows 32 * kt + 8 * g + e of v (g = lane / 16):
// byte kt of (sb0, sb1), bit e.  hb: the table's bits in LDS (words of zeros for order 1); on = order << logA.
// (the lookups of all k tiles are issued together: a wait per lookup costs more than the transform)
template <int KTC>
__device__ __forceinline__ void mix_signs(uint32_t& sb0, uint32_t& sb1, const uint32_t* hb, int order, int logA, int row0, int on,
                                          int lane) {
  const int a = lane & 15, g = lane >> 4, Am = (1 << logA) - 1, nw = (order * order + 31) >> 5;
  uint32_t sb[2] = {0u, 0u};
  // H_A: within eight rows a pattern of iA's low bits (the rows differ in theirs), and for A > 8 a
  // sign per eight rows
  const int i = row0 + a, iA = i & Am;
  const uint32_t pat = ((iA & 1) ? 0xAAu : 0u) ^ ((iA & 2) ? 0xCCu : 0u) ^ ((iA & 4) ? 0xF0u : 0u);
  uint32_t f[KTC];
  if (logA >= 3) {  // one table column
    const int iK = (i < on ? i : 0) >> logA;
#pragma unroll
    for (int kt = 0; kt < KTC; ++kt) {
      const int q = ((32 * kt + 8 * g) >> logA) * order + iK;
      f[kt] = hb[q >> 5 < nw ? q >> 5 : 0] >> (q & 31);
    }
#pragma unroll
    for (int kt = 0; kt < KTC; ++kt) {
      const uint32_t b = f[kt] ^ (uint32_t)__builtin_popcount(iA & (32 * kt + 8 * g) & Am);
      sb[kt >> 2] |= ((0u - (b & 1u)) & 0xFFu) << (8 * (kt & 3));
    }
  } else {
    // lane e = a % 8 takes the bits of the eight output rows of its half of the wave against v row
    // 32 * kt + 8 * g + e, adjacent in the table's words, and the eight lanes transpose their bytes
    const int iK = (row0 + (a & 8)) >> logA;
    uint32_t hi[KTC], sh[KTC];
#pragma unroll
    for (int kt = 0; kt < KTC; ++kt) {
      const int q = ((32 * kt + 8 * g + (a & 7)) >> logA) * order + iK, w = q >> 5;
      f[kt] = hb[w < nw ? w : 0];  // (rows past the table meet zeros of v, or are not stored)
      hi[kt] = hb[w + 1 < nw ? w + 1 : 0];
      sh[kt] = q & 31;
    }
#pragma unroll
    for (int kt = 0; kt < KTC; ++kt) f[kt] = __builtin_amdgcn_alignbit(hi[kt], f[kt], sh[kt]) & 0xFFu;
    if (logA == 1) {  // four bits, each for two rows
#pragma unroll
      for (int kt = 0; kt < KTC; ++kt) {
        uint32_t x = f[kt];
        x = (x & 3u) | ((x & 0xCu) << 2);
        x = (x & 0x11u) | ((x & 0x22u) << 1);
        f[kt] = x * 3u;
      }
    } else if (logA == 2) {  // two bits, each for four rows
#pragma unroll
      for (int kt = 0; kt < KTC; ++kt) f[kt] = (f[kt] & 1u) * 0x0Fu | (f[kt] & 2u) * 0x78u;
    }
#pragma unroll
    for (int kt = 0; kt < KTC; ++kt) sb[kt >> 2] |= f[kt] << (8 * (kt & 3));
#pragma unroll
    for (int h = 0; h < (KTC > 4 ? 2 : 1); ++h) {
      auto step = [&](int b, uint32_t m) {  // the off-diagonal quarters change places
        const int s = 1 << b;
        const uint32_t o = __builtin_bit_cast(uint32_t, qtip_wht::lane_xor(__builtin_bit_cast(float, sb[h]), b));
        sb[h] = (a & s) ? (sb[h] & ~m) | ((o >> s) & m) : (sb[h] & m) | ((o & m) << s);
      };
      step(2, 0x0F0F0F0Fu);
      step(1, 0x33333333u);
      step(0, 0x55555555u);
    }
  }
  sb0 = sb[0] ^ pat * 0x01010101u;
  sb1 = sb[1] ^ pat * 0x01010101u;
}

// ---- One vector of k = order * A * pp elements in front of a matvec: x_t = fp16(scale * ((table (x) H_A) (x) H_pp)(su * x)),
// by a workgroup of 16 waves, pp = 16 * NT.  As in the transforms of many rows v = su * x is the matrix v[j][c] of on = order * A
// rows, exact on one fp16 plane under a sign vector of +-1 and on three bf16 planes otherwise; sums are fp32.
// Takes the place of a launch of its own, at the price of a chain of one cold read, the plane, the products and the butterflies of a
// tile's wave (0.7 us each) in every workgroup: past the first barrier after 4.1 us where the plain matvec is after 1.4.  us from cold
// memory, two launches / one, 2 bits and 4: 11008 -> 4096 10.1 / 8.7 and 12.1 / 10.2, 14336 -> 4096 10.7 / 9.9 and 13.4 / 11.7,
// 13824 -> 5120 13.0 / 12.2 and 15.5 / 13.8, 5504 -> 2048 7.9 / 6.8 and 8.9 / 7.4, 5120 -> 5120 9.0 / 8.1 and 10.2 / 8.8.  A token of
// 8 layers of 4096 473 -> 463.  (Two waves to a tile, each with half of the k tiles: what they hand each other costs what it saves.)
struct MixArgs {
  const uint32_t* sign_rows;  // [on][8] words: bit j of row i is set where entry (i, j) of table (x) H_A is -1
  int on;
};
constexpr int kMixInMaxRows = 256;  // of v: 16 to a wave

// LDS: the plane (column position major: 64 bytes per k tile and 16 to spread the columns over the banks) and flags
struct MixInLds {
  int stride, flags, bytes;
};
__host__ __device__ constexpr MixInLds mix_in_lds(int on, int nt) {
  MixInLds l{};
  l.stride = 64 * ((on + 31) >> 5) + 16;
  l.flags = 16 * nt * l.stride;
  l.bytes = l.flags + 64;
  return l;
}

template <int NT>
struct MixInRegs {
  u32x4m x[4], su[4];  // eight columns of four rows
  u32x4m rows[2];      // the signs of the lane's output row
};

// the thread's requests, every one of them without a condition, so that a wait for one is not a wait for all
template <int NT>
__device__ __forceinline__ void mix_in_load(MixInRegs<NT>& r, const MixArgs& M, const _Float16* x, const _Float16* su,
                                            int row0, int tid) {
  constexpr int PP = 16 * NT;
  const int lane = tid & 63, wave = tid >> 6, a = lane & 15, g = lane >> 4;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int j = 16 * wave + 4 * g + i;
    const uint32_t e = j < M.on && 8 * a < PP ? (uint32_t)(j * PP + 8 * a) : 0u;
    r.x[i] = *reinterpret_cast<const u32x4m*>(x + e);
    r.su[i] = *reinterpret_cast<const u32x4m*>(su + e);
  }
  const int i = (row0 & ~15) + 16 * wave + a;
  const uint32_t* row = M.sign_rows + (i < M.on ? i : 0) * 8;
  r.rows[0] = *reinterpret_cast<const u32x4m*>(row);
  r.rows[1] = *reinterpret_cast<const u32x4m*>(row + 4);
}

// Rows [row0, row1) of the result to xs (row0 first), which may lie in the mix_in_lds bytes at smem: those are free when the
// workgroup is past a barrier again.
// A wave's lane (g, a) holds columns 8a .. 8a + 7 of rows 16 * wave + 4g .. + 3 and writes them to LDS transposed; then wave w
// owns output rows 16 (row0 / 16 + w) .. + 15, column tile t its columns NT * n + t (n = place of the lane): four or two
// consecutive columns of four rows end in a lane.
template <int NT>
__device__ __forceinline__ void mix_in_compute(const MixInRegs<NT>& r, const MixArgs& M, float scale, uint8_t* smem,
                                               _Float16* xs, const _Float16* x, const _Float16* su, int row0,
                                               int row1, int tid, unsigned long long* sv = nullptr) {
  using namespace qtip_wht;
  constexpr int PP = 16 * NT, LOGNT = NT == 4 ? 2 : 1;
  const int lane = tid & 63, a = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int on = M.on, KT = (on + 31) >> 5;
  const MixInLds L = mix_in_lds(on, NT);
  uint32_t* flags = reinterpret_cast<uint32_t*>(smem + L.flags);
  (void)sv;
  QTIP_STAMP_SV(6)
  // ---- the plane
  const int j0 = 16 * wave + 4 * g;
  const bool loader = 16 * wave < 32 * KT && 8 * a < PP;  // (rows past the matrix, up to a whole k tile, are zeros)
  auto put = [&](int e, uint32_t lo, uint32_t hi) {       // rows j0, j0 + 1 and j0 + 2, j0 + 3 of column 8a + e
    const int pos = 16 * (e & (NT - 1)) + a * (8 / NT) + (e >> LOGNT);
    *reinterpret_cast<uint2*>(smem + pos * L.stride + j0 * 2) = uint2{lo, hi};
  };
  uint32_t off = 0;
  if (loader) {
    u32x4m h[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool live = j0 + i < on;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        off |= live ? (r.su[i][q] & 0x7FFF7FFFu) ^ 0x3C003C00u : 0u;
        h[i][q] = live ? r.x[i][q] ^ (r.su[i][q] & 0x80008000u) : 0u;
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t sel = (e & 1) ? 0x07060302u : 0x05040100u;
      put(e, __builtin_amdgcn_perm(h[1][e >> 1], h[0][e >> 1], sel), __builtin_amdgcn_perm(h[3][e >> 1], h[2][e >> 1], sel));
    }
  }
  const bool mine = __any(off != 0);
  if (lane == 0) flags[wave] = mine;
  __syncthreads();
  QTIP_STAMP_SV(7)
  const bool fast = !__any(flags[a] != 0);  // the sign vector is one of +-1

  // ---- products
  float4m acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = float4m{0.f, 0.f, 0.f, 0.f};
  const int place = wht_place(lane) & 15;
  const uint8_t* rd = smem + place * L.stride + g * 16;
  const int base = (row0 & ~15) + 16 * wave;
  const bool busy = base < row1;
  auto products = [&](uint32_t one, auto mfma) {
    if (!busy) return;
    u32x4m b[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) b[t] = *reinterpret_cast<const u32x4m*>(rd + 16 * t * L.stride);
#pragma unroll
    for (int kt = 0; kt < kMixInMaxRows / 32; ++kt)
      if (kt < KT) {
        const u32x4m fa = expand_signs((r.rows[kt >> 2][kt & 3] >> (8 * g)) & 0xFFu, one);
        const int next = kt + 1 < KT ? kt + 1 : kt;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          acc[t] = mfma(fa, b[t], acc[t]);
          b[t] = *reinterpret_cast<const u32x4m*>(rd + 16 * t * L.stride + next * 64);
        }
      }
  };
  if (fast) {
    products(0x3C003C00u, [](u32x4m fa, u32x4m b, float4m c) {
      return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8m, fa), __builtin_bit_cast(half8m, b), c, 0, 0, 0);
    });
  } else {
    // the exact products su * x in three planes of eight bits each (read again: kept, they would cost the other way 32 registers)
    MixInRegs<NT> again;
    mix_in_load<NT>(again, M, x, su, row0, tid);
    float v[4][8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const half8m xv = __builtin_bit_cast(half8m, again.x[i]), sv = __builtin_bit_cast(half8m, again.su[i]);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[i][e] = j0 + i < on ? (float)xv[e] * (float)sv[e] : 0.f;
    }
    for (int p = 0; p < 3; ++p) {
      __syncthreads();  // the plane has been read
      if (loader) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          uint32_t b[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            b[i] = __builtin_bit_cast(uint32_t, v[i][e]);
            // (nothing is left of an infinity: the difference would turn it into a NaN)
            const float rest = v[i][e] - __builtin_bit_cast(float, b[i] & 0xFFFF0000u);
            v[i][e] = __builtin_isinf(v[i][e]) ? 0.f : rest;
          }
          put(e, __builtin_amdgcn_perm(b[1], b[0], 0x07060302u), __builtin_amdgcn_perm(b[3], b[2], 0x07060302u));
        }
      }
      __syncthreads();
      products(0x3F803F80u, [](u32x4m fa, u32x4m b, float4m c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, fa), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
      });
    }
  }
  QTIP_STAMP_SV(8)
  __syncthreads();  // the plane has been read
  QTIP_STAMP_SV(9)
  if (!busy) return;
  // ---- H_pp: the low bits of a column are t, the others the lane's place
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float y[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) y[t] = acc[t][q];
    wht_regs<NT>(y);
    wht_places<NT>(y, 4, place);
    const int i = base + 4 * g + q;
    _Float16 o[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) o[t] = (_Float16)(y[t] * scale);
    if (i >= row0 && i < row1) st_f16<NT>(xs + (i - row0) * PP + NT * place, o);
  }
}

}  // namespace qtip_mix
