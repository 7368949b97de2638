// The boundary between two linear layers of a decoder in one workgroup of 1024 threads:
//   x_new = residual + fp16(scale_out * post * H_k (sum of the previous layer's partial results)),
//   x_t   = fp16(scale_in * H_k (su * RMSNorm(x_new) * norm_w))
// for k = 1024 * EPT, shared by the matvec prologue and the boundary's own launch (all of it) and the token head (x_new
// and its norm).
// Bound by latency: one cold round trip for the operands, three barriers, and between them some 70 vector instructions on
// four waves a SIMD.  Nothing in it waits for the LDS crossbar (wht_place), no load waits for another, and no conversion
// for a load.  us, a 2-bit launch of 12288 or 22016 rows of 4096 with the boundary in front, on average: 13.45 -> 12.33, past
// the barrier behind its table after 5.8 -> 4.1; 57344 and 10240 rows of 8192 at 4 bits 51.9 -> 48.4 and
// 21.2 -> 18.3.  A token of 8 layers of 4096 496 -> 473, of 4 layers of 8192 594 -> 584.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "qtip_wht.h"

#ifndef QTIP_STAMP_SV
#define QTIP_STAMP_SV(i)
#endif

namespace qtip_chain {

constexpr int kThreads = 1024;  // of the workgroup
constexpr int kWaves = kThreads / 64;

struct ChainArgs {
  const float* parts;        // [in_parts][k] fp32 partial results of the previous linear layer
  const float* post;         // its output sign vector times its scale (SV), k fp32
  const _Float16* residual;  // the residual stream, k fp16
  const _Float16* norm_w;    // RMSNorm weight, k fp16
  _Float16* x_out;           // the new residual stream, k fp16 (NULL: nobody reads it)
  size_t part_stride;        // floats between partial results
  float scale_out, eps;
  int in_parts;
};

template <int EPT>
struct ChainRegs {  // a thread's operands, EPT consecutive elements each
  typedef _Float16 hvec __attribute__((ext_vector_type(EPT)));
  float v[EPT], v1[EPT];  // the first two partial results, where the first transform takes them
  float pv[EPT];          // of the middle part
  hvec rv, wv, sv;        // (as loaded: a conversion would wait for the load)
};

// A thread holds EPT consecutive elements, those of thread index t (ten bits, e = t * EPT) of one of two layouts:
//   natural   t = [wave 4 | place 6]
//   swapped   t = [place 3..0 | wave 4 | place 5..4]
// with place = wht_place(lane).  A transform does its register and place bits in one of them, changes over to the other
// through LDS, and finds the bits that were the wave's among its places.  The boundary runs swapped -> natural -> swapped:
// the partial results are read in runs of 4 * EPT floats, and the four operands of the middle part and the new residual
// stream, which are fp16 but for one, whole cache lines at a time.  (The other way round they had to change over in LDS as well.)
template <int EPT>
__device__ __forceinline__ int nat_index(int place, int wave) {
  return (wave * 64 + place) * EPT;
}
template <int EPT>
__device__ __forceinline__ int swp_index(int place, int wave) {
  return (((place & 15) << 6) | ((wave & 15) << 2) | (place >> 4)) * EPT;
}

// All loads of the boundary but the partial results past the second, without a wait between them (SU: the sign vector too).
template <int EPT, bool SU = true>
__device__ __forceinline__ void chain_load(const ChainArgs& c, const _Float16* su, int place, int wave, ChainRegs<EPT>& r) {
  using namespace qtip_wht;
  const int e_nat = nat_index<EPT>(place, wave), e_swp = swp_index<EPT>(place, wave);
  ld_f32<EPT>(c.parts + e_swp, r.v);
  ld_f32<EPT>(c.parts + (c.in_parts > 1 ? c.part_stride : 0) + e_swp, r.v1);
  ld_f32<EPT>(c.post + e_nat, r.pv);
  typedef typename ChainRegs<EPT>::hvec hvec;
  r.rv = *reinterpret_cast<const hvec*>(c.residual + e_nat);
  r.wv = *reinterpret_cast<const hvec*>(c.norm_w + e_nat);
  if constexpr (SU) r.sv = *reinterpret_cast<const hvec*>(su + e_nat);
}

// floats of LDS: the exchange buffer and, behind it, the waves' sums
constexpr int chain_floats(int k) { return k + k / 64 + kWaves; }

// x_new in v (natural layout) and the reciprocal of its RMS.  xbuf: chain_floats(k) floats; the exchange buffer in
// it is free again afterwards.
template <int EPT>
__device__ __forceinline__ float chain_residual(const ChainRegs<EPT>& r, const ChainArgs& c, float* xbuf, float (&v)[EPT], int lane, int place,
                                                int wave, bool write_x, unsigned long long* sv = nullptr) {
  using namespace qtip_wht;
  constexpr int N = kThreads * EPT;
  (void)sv;
  QTIP_STAMP_SV(6)
  const int e_nat = nat_index<EPT>(place, wave), e_swp = swp_index<EPT>(place, wave);
  float* wsum = xbuf + N + N / 64;
#pragma unroll
  for (int i = 0; i < EPT; ++i) v[i] = r.v[i];
  if (c.in_parts > 1) {
#pragma unroll
    for (int i = 0; i < EPT; ++i) v[i] += r.v1[i];
    for (int w = 2; w < c.in_parts; ++w) {
      float t[EPT];
      ld_f32<EPT>(c.parts + w * c.part_stride + e_swp, t);
#pragma unroll
      for (int i = 0; i < EPT; ++i) v[i] += t[i];
    }
  }
  // ---- first transform (swapped -> natural layout)
  wht_regs<EPT>(v);
  wht_places<EPT>(v, 6, place);
  st_f32<EPT>(xbuf + xidx<EPT>(e_swp), v);
  __syncthreads();
  QTIP_STAMP_SV(7)
  ld_f32<EPT>(xbuf + xidx<EPT>(e_nat), v);
  wht_places<EPT>(v, 6, place, 2);
  // ---- residual, RMSNorm
  float ss = 0.f;
  _Float16 xn[EPT];
#pragma unroll
  for (int i = 0; i < EPT; ++i) {
    const float o = v[i] * c.scale_out * r.pv[i];
    xn[i] = (_Float16)((float)r.rv[i] + (float)(_Float16)o);
    v[i] = (float)xn[i];
    ss += v[i] * v[i];
  }
  if (write_x) st_f16<EPT>(c.x_out + e_nat, xn);
  ss = wave_sum(ss);
  if (lane == 0) wsum[wave] = ss;
  __syncthreads();  // also: every read of xbuf above is done
  QTIP_STAMP_SV(8)
  return __builtin_amdgcn_rsqf(waves16_sum(wsum, lane) / (float)N + c.eps);
}

// The whole boundary; x_t in the swapped layout, scaled and rounded, in xo.
template <int EPT>
__device__ __forceinline__ void chain_compute(const ChainRegs<EPT>& r, const ChainArgs& c, float scale_in, float* xbuf, _Float16 (&xo)[EPT],
                                              int lane, int place, int wave, bool write_x, unsigned long long* sv = nullptr) {
  using namespace qtip_wht;
  float v[EPT];
  const float rs = chain_residual<EPT>(r, c, xbuf, v, lane, place, wave, write_x, sv);
#pragma unroll
  for (int i = 0; i < EPT; ++i) v[i] = (float)(_Float16)((float)r.wv[i] * (float)(_Float16)(v[i] * rs)) * (float)r.sv[i];
  // ---- second transform (natural -> swapped layout)
  wht_regs<EPT>(v);
  wht_places<EPT>(v, 6, place);
  st_f32<EPT>(xbuf + xidx<EPT>(nat_index<EPT>(place, wave)), v);
  __syncthreads();
  QTIP_STAMP_SV(9)
  ld_f32<EPT>(xbuf + xidx<EPT>(swp_index<EPT>(place, wave)), v);
  wht_places<EPT>(v, 4, place);
#pragma unroll
  for (int i = 0; i < EPT; ++i) xo[i] = (_Float16)(v[i] * scale_in);
}

}  // namespace qtip_chain
