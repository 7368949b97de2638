// The boundary between two linear layers of a decoder in one workgroup of 1024 threads:
//   x_new = residual + fp16(scale_out * post * H_k (sum of the previous layer's partial results)),
//   x_t   = fp16(scale_in * H_k (su * RMSNorm(x_new) * norm_w))
// for k = 1024 * EPT, shared by the matvec prologue (all of it) and the token head (x_new and its norm).
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

struct ChainRegs {  // a thread's operands, k / 1024 <= 8 consecutive elements each
  float v[8], pv[8], rv[8], wv[8], sv[8];
};

// Where the operands of the boundary's middle part are read.  It works in the swapped layout, in which
// the lanes of a wave hold 16 runs of 4 * EPT consecutive elements: with eight elements a thread a
// run is 64 bytes of fp16 and the operands are read there, with two or four it is half that or less
// and a load touches four to eight times the cache lines it needs, so that they are read in the
// natural layout and change over in LDS.  A token of 8 layers of 4096 (16 boundaries): 583 -> 565 us;
// of layers of 8192, with the change-over in LDS or without, the same.
template <int EPT>
constexpr bool kChainStaged = EPT < 8;

// the operands but for the partial results past the first
template <int EPT>
__device__ __forceinline__ void chain_load_first(const ChainArgs& c, const _Float16* su, int tid, int lane,
                                                 int wave, ChainRegs& r) {
  using namespace qtip_wht;
  const int e_nat = tid * EPT;
  const int e_mid = kChainStaged<EPT> ? e_nat : (((lane & 15) << 6) | ((wave & 15) << 2) | (lane >> 4)) * EPT;
  ld_f32<EPT>(c.post + e_mid, r.pv);
  ld_f16<EPT>(c.residual + e_mid, r.rv);
  ld_f16<EPT>(c.norm_w + e_mid, r.wv);
  ld_f16<EPT>(su + e_mid, r.sv);
  ld_f32<EPT>(c.parts + e_nat, r.v);
}

// adds the partial results from `w` on
template <int EPT>
__device__ __forceinline__ void chain_load_parts(const ChainArgs& c, int w, int tid, ChainRegs& r) {
  for (; w < c.in_parts; ++w) {
    float t[EPT];
    qtip_wht::ld_f32<EPT>(c.parts + w * c.part_stride + tid * EPT, t);
#pragma unroll
    for (int i = 0; i < EPT; ++i) r.v[i] += t[i];
  }
}

template <int EPT>
__device__ __forceinline__ void chain_load(const ChainArgs& c, const _Float16* su, int tid, int lane,
                                           int wave, ChainRegs& r) {
  chain_load_first<EPT>(c, su, tid, lane, wave, r);
  chain_load_parts<EPT>(c, 1, tid, r);
}

// index of element e of an operand that changes over in LDS: a pad of four lanes per 64 puts the 16
// runs of a read on banks of their own
template <int EPT>
__device__ __forceinline__ int sidx(int e) {
  return e + 4 * EPT * (e / (64 * EPT));
}
// the floats of LDS behind xbuf and wsum that the operands take: one of fp32, three of fp16
template <int EPT>
constexpr int kChainStage = (kThreads + 64) * EPT * 5 / 2;

// floats of LDS behind xbuf: k + k/64 of exchange buffer, the waves' sums, the operands that change over
template <int EPT>
constexpr int kChainFloats = kThreads * EPT + kThreads * EPT / 64 + kWaves + (kChainStaged<EPT> ? kChainStage<EPT> : 0);

// x_new in v (swapped layout: element e_swp + i of thread tid) and the reciprocal of its RMS.  xbuf: k + k/64 floats of
// exchange buffer, wsum behind it: 16 floats and kChainStage of operands; xbuf and the operands are free again, the sums
// are not.  Leaves the norm weights (and the sign vector) of the layout in r.
template <int EPT>
__device__ __forceinline__ float chain_residual(ChainRegs& r, const ChainArgs& c, float* xbuf, float* wsum, float (&v)[EPT],
                                                int tid, int lane, int wave, bool write_x, unsigned long long* sv = nullptr) {
  using namespace qtip_wht;
  constexpr int N = kThreads * EPT;
  (void)sv;
  QTIP_STAMP_SV(6)
  const int e_nat = tid * EPT;
  const int e_swp = (((lane & 15) << 6) | ((wave & 15) << 2) | (lane >> 4)) * EPT;
#pragma unroll
  for (int i = 0; i < EPT; ++i) v[i] = r.v[i];
  // ---- first transform (natural -> swapped layout)
  wht_regs<EPT>(v);
#pragma unroll
  for (int i = 0; i < EPT; ++i) v[i] = wht_lanes(v[i], 6, lane);
#pragma unroll
  for (int i = 0; i < EPT; ++i) xbuf[xidx<EPT>(e_nat + i)] = v[i];
  float* post_s = wsum + kWaves;
  _Float16* half_s = reinterpret_cast<_Float16*>(post_s + sidx<EPT>(N));  // residual, norm weight, sign vector
  if constexpr (kChainStaged<EPT>) {
    _Float16 h[EPT];
#pragma unroll
    for (int i = 0; i < EPT; ++i) post_s[sidx<EPT>(e_nat) + i] = r.pv[i];
#pragma unroll
    for (int i = 0; i < EPT; ++i) h[i] = (_Float16)r.rv[i];
    st_f16<EPT>(half_s + sidx<EPT>(e_nat), h);
#pragma unroll
    for (int i = 0; i < EPT; ++i) h[i] = (_Float16)r.wv[i];
    st_f16<EPT>(half_s + sidx<EPT>(N) + sidx<EPT>(e_nat), h);
#pragma unroll
    for (int i = 0; i < EPT; ++i) h[i] = (_Float16)r.sv[i];
    st_f16<EPT>(half_s + 2 * sidx<EPT>(N) + sidx<EPT>(e_nat), h);
  }
  __syncthreads();
  QTIP_STAMP_SV(7)
  if constexpr (kChainStaged<EPT>) {
    ld_f32<EPT>(post_s + sidx<EPT>(e_swp), r.pv);
    ld_f16<EPT>(half_s + sidx<EPT>(e_swp), r.rv);
    ld_f16<EPT>(half_s + sidx<EPT>(N) + sidx<EPT>(e_swp), r.wv);
    ld_f16<EPT>(half_s + 2 * sidx<EPT>(N) + sidx<EPT>(e_swp), r.sv);
  }
#pragma unroll
  for (int i = 0; i < EPT; ++i) v[i] = wht_lanes(xbuf[xidx<EPT>(e_swp + i)], 4, lane);
  // ---- residual, RMSNorm, sign vector of this layer
  float ss = 0.f;
  _Float16 xn[EPT];
#pragma unroll
  for (int i = 0; i < EPT; ++i) {
    const float o = v[i] * c.scale_out * r.pv[i];
    xn[i] = (_Float16)(r.rv[i] + (float)(_Float16)o);
    v[i] = (float)xn[i];
    ss += v[i] * v[i];
  }
  if (write_x) st_f16<EPT>(c.x_out + e_swp, xn);
  ss = wave_sum(ss);
  if (lane == 0) wsum[wave] = ss;
  __syncthreads();  // also: every read of xbuf above is done
  QTIP_STAMP_SV(8)
  float tot = 0.f;
#pragma unroll
  for (int w = 0; w < 16; ++w) tot += wsum[w];
  return __builtin_amdgcn_rsqf(tot / (float)N + c.eps);
}

// xbuf, wsum: as in chain_residual; xs: the k fp16 activations of the matvec
template <int EPT>
__device__ __forceinline__ void chain_compute(ChainRegs& r, const ChainArgs& c, float scale_in, float* xbuf,
                                              float* wsum, _Float16* xs, int tid, int lane, int wave,
                                              bool write_x, unsigned long long* sv = nullptr) {
  using namespace qtip_wht;
  const int e_nat = tid * EPT;
  const int e_swp = (((lane & 15) << 6) | ((wave & 15) << 2) | (lane >> 4)) * EPT;
  float v[EPT];
  const float rs = chain_residual<EPT>(r, c, xbuf, wsum, v, tid, lane, wave, write_x, sv);
#pragma unroll
  for (int i = 0; i < EPT; ++i) v[i] = (float)(_Float16)(r.wv[i] * (float)(_Float16)(v[i] * rs)) * r.sv[i];
  // ---- second transform (swapped -> natural layout)
  wht_regs<EPT>(v);
#pragma unroll
  for (int i = 0; i < EPT; ++i) v[i] = wht_lanes(v[i], 6, lane);
#pragma unroll
  for (int i = 0; i < EPT; ++i) xbuf[xidx<EPT>(e_swp + i)] = v[i];
  __syncthreads();
  QTIP_STAMP_SV(9)
  // the bits still missing are the top four of the element's lane field = lane bits 2..5 here
  _Float16 xo[EPT];
#pragma unroll
  for (int i = 0; i < EPT; ++i) {
    float y = xbuf[xidx<EPT>(e_nat + i)];
    y = wht_lanes(y, 6, lane, 2);
    xo[i] = (_Float16)(y * scale_in);
  }
  st_f16<EPT>(xs + e_nat, xo);
  __syncthreads();  // the exchange buffer is free for the table, xs is complete
  QTIP_STAMP_SV(10)
}

}  // namespace qtip_chain
