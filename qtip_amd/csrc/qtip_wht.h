// Walsh-Hadamard building blocks shared by the transform kernels and the matvec prologue:
// cross-lane exchanges of a wave64, butterflies over lane bits and over a thread's registers,
// and the vector loads / stores of EPT consecutive elements.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace qtip_wht {

typedef float float4w __attribute__((ext_vector_type(4)));

// value of lane ^ (1 << b) for b = 0..5
__device__ __forceinline__ float lane_xor(float v, int b) {
  const int u = __builtin_bit_cast(int, v);
  int r;
  switch (b) {
    case 0: r = __builtin_amdgcn_update_dpp(0, u, 0xB1, 0xF, 0xF, false); break;  // quad_perm 1,0,3,2
    case 1: r = __builtin_amdgcn_update_dpp(0, u, 0x4E, 0xF, 0xF, false); break;  // quad_perm 2,3,0,1
    // xor 4 and xor 16 go through the LDS crossbar: one instruction outside the vector pipe (two
    // bank-masked row rotations do xor 4 as well, but cost two vector instructions that cannot
    // ride on the addition; the transforms are bound by vector issue)
    case 2: r = __builtin_amdgcn_ds_swizzle(u, 0x101F); break;                    // xor 4
    case 3: r = __builtin_amdgcn_update_dpp(0, u, 0x128, 0xF, 0xF, false); break;  // xor 8 = row_ror:8
    case 4: r = __builtin_amdgcn_ds_swizzle(u, 0x401F); break;                    // xor 16
    default: {
      auto sw = __builtin_amdgcn_permlane32_swap((uint32_t)u, (uint32_t)u, false, false);
      r = (int)((threadIdx.x & 32) ? sw[0] : sw[1]);
    }
  }
  return __builtin_bit_cast(float, r);
}

// Transforms whose elements may sit in any lane keep element `place` of a wave in lane place ^ (3 if bit 2 of it is set).
// A step over bit 2 of the place then exchanges lanes l and l ^ 7, a mirror of eight lanes that rides on the addition
// as a DPP operand, and the one over bit 4 is a row swap: no step goes through the LDS crossbar, whose round trip (a wave
// of a boundary waited for sixteen of them in a row) was most of a transform's time.
__device__ __forceinline__ int wht_place(int lane) {
  return lane ^ ((lane & 4) ? 3 : 0);
}
// the value of element `lane` of a wave -> that of element wht_place(lane), in every lane
__device__ __forceinline__ float wht_to_place(float v, int lane) {
  const float m = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x1B, 0xF, 0xF, false));
  return (lane & 4) ? m : v;  // (quads with bit 2 set run backwards)
}
__device__ __forceinline__ float half_mirror(float v) {  // value of lane ^ 7
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xF, 0xF, false));
}
// One butterfly over bit b of the place: lanes with the bit clear get v + partner, the others partner - v.
// Written as partner + (v with its sign flipped where the bit is set): an xor and an addition (the
// exchange rides on the addition as a DPP operand) instead of an addition, a subtraction and a
// select; the sums are the same floating-point operations on the same operands.  The swaps exchange odd rows (or the
// upper half) of their first operand with even rows (the lower half) of their second: with (v, flipped v) the first result holds
// the lower partner's values in either and the second the upper one's, negated where they stayed at home - their sum is the butterfly.
__device__ __forceinline__ float wht_place_stage(float v, int b, int place) {
  const uint32_t flip = ((uint32_t)place << (31 - b)) & 0x80000000u;
  const uint32_t u = __builtin_bit_cast(uint32_t, v), f = u ^ flip;
  if (b >= 4) {
    auto sw = b == 4 ? __builtin_amdgcn_permlane16_swap(u, f, false, false) : __builtin_amdgcn_permlane32_swap(u, f, false, false);
    return __builtin_bit_cast(float, (uint32_t)sw[0]) + __builtin_bit_cast(float, (uint32_t)sw[1]);
  }
  return (b == 2 ? half_mirror(v) : lane_xor(v, b)) + __builtin_bit_cast(float, f);
}
// butterflies over place bits lo .. nbits-1 of EPT values
template <int EPT>
__device__ __forceinline__ void wht_places(float (&v)[EPT], int nbits, int place, int lo = 0) {
#pragma unroll
  for (int b = 0; b < 6; ++b)
    if (b >= lo && b < nbits) {
#pragma unroll
      for (int i = 0; i < EPT; ++i) v[i] = wht_place_stage(v[i], b, place);
    }
}

__device__ __forceinline__ float wht_places(float v, int nbits, int place, int lo = 0) {
#pragma unroll
  for (int b = 0; b < 6; ++b)
    if (b >= lo && b < nbits) v = wht_place_stage(v, b, place);
  return v;
}

// a lane's value and that of lane ^ 16 (b = 4) or lane ^ 32 (5), the lower lane's first
__device__ __forceinline__ float2 lane_pair(float v, int b) {
  const uint32_t u = __builtin_bit_cast(uint32_t, v);
  auto sw = b == 4 ? __builtin_amdgcn_permlane16_swap(u, u, false, false) : __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return float2{__builtin_bit_cast(float, (uint32_t)sw[0]), __builtin_bit_cast(float, (uint32_t)sw[1])};
}
__device__ __forceinline__ float lane_add(float v, int b) {
  const float2 s = lane_pair(v, b);
  return s.x + s.y;
}

// the sum over the lanes of a wave (four lanes hold the same sum when eight are mirrored)
__device__ __forceinline__ float wave_sum(float v) {
  v += lane_xor(v, 0);
  v += lane_xor(v, 1);
  v += half_mirror(v);
  v += lane_xor(v, 3);
  return lane_add(lane_add(v, 4), 5);
}
// the sum of values that a workgroup's 16 waves left in LDS, the same in every lane
__device__ __forceinline__ float waves16_sum(const float* w, int lane) {
  float v = w[lane & 15];
  v += lane_xor(v, 0);
  v += lane_xor(v, 1);
  v += half_mirror(v);
  return v + lane_xor(v, 3);
}

// EPT consecutive elements as floats, with the widest loads the alignment (EPT elements) allows
template <int EPT>
__device__ __forceinline__ void ld_f32(const float* p, float v[EPT]) {
  if constexpr (EPT == 2) {
    const float2 t = *reinterpret_cast<const float2*>(p);
    v[0] = t.x;
    v[1] = t.y;
  } else {
#pragma unroll
    for (int q = 0; q < EPT / 4; ++q) {
      const float4w t = *reinterpret_cast<const float4w*>(p + 4 * q);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[4 * q + e] = t[e];
    }
  }
}
template <int EPT>
__device__ __forceinline__ void st_f32(float* p, const float v[EPT]) {
  if constexpr (EPT == 2) {
    *reinterpret_cast<float2*>(p) = float2{v[0], v[1]};
  } else {
#pragma unroll
    for (int q = 0; q < EPT / 4; ++q)
      *reinterpret_cast<float4w*>(p + 4 * q) = float4w{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
  }
}
template <int EPT>
__device__ __forceinline__ void ld_f16(const _Float16* p, float v[EPT]) {
  typedef _Float16 hvec __attribute__((ext_vector_type(EPT)));
  const hvec t = *reinterpret_cast<const hvec*>(p);
#pragma unroll
  for (int e = 0; e < EPT; ++e) v[e] = (float)t[e];
}
template <int EPT>
__device__ __forceinline__ void st_f16(_Float16* p, const _Float16 v[EPT]) {
  typedef _Float16 hvec __attribute__((ext_vector_type(EPT)));
  hvec t;
#pragma unroll
  for (int e = 0; e < EPT; ++e) t[e] = v[e];
  *reinterpret_cast<hvec*>(p) = t;
}

template <int EPT>
__device__ __forceinline__ void wht_regs(float v[EPT]) {
#pragma unroll
  for (int h = 1; h < EPT; h <<= 1)
#pragma unroll
    for (int i = 0; i < EPT; ++i)
      if (!(i & h)) {
        const float a = v[i], b = v[i + h];
        v[i] = a + b;
        v[i + h] = a - b;
      }
}

// exchange buffer index of element e: one pad block of EPT floats per 64 lanes keeps the strided reads apart
template <int EPT>
__device__ __forceinline__ int xidx(int e) {
  return e + EPT * (e / (64 * EPT));
}


}  // namespace qtip_wht
