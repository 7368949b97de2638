// The end of a decoded token: output transform of the last layer's `down`, residual addition, final RMSNorm and the
// dense fp16 output matrix (model/llama.py:1466-1467), one launch.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/qtip_hip.h"
#include "qtip_chain.h"
#include "qtip_setup.h"

namespace {

using namespace qtip_chain;
typedef uint32_t u32x4h __attribute__((ext_vector_type(4)));
typedef _Float16 half8h __attribute__((ext_vector_type(8)));

constexpr int kMaxLoads = 16;  // 16-byte loads of a lane per matrix row: n <= 8192

// logits[v] = fp16(head[v][:] . xn), xn = norm_w * fp16(x * rsqrt(mean(x^2) + eps)), with x the residual stream as it is
// (EPT = 0) or behind the layer boundary of 1024 * EPT elements.
//
// Bound by the stream of the matrix.  256 persistent workgroups of 16 waves; a wave takes a row at a time, 1 KiB a load
// instruction, and asks for a piece of the next row where it has used one of the present row, so that NL KiB a wave (128 KiB
// a CU at n = 4096) are in flight from before the norm on: what the workgroup computes in front of the product, which every
// workgroup repeats, hides behind its first rows.  A workgroup's 16 rows lie side by side.
// us from cold memory, norm and library product / here / with the boundary in front: 32000 x 4096 62.9 / 43.3 / 43.3 (6.1 TB/s),
// 32000 x 8192 103 / 84 / 86, 128256 x 8192 367 / 318 / 319, 32000 x 5120 69 / 54, 32000 x 512 15.7 / 9.2, 1000 x 256
// 5.5 / 2.2: faster at every size, so there is no line.  A token of 8 layers of 4096, in which it takes the place of four
// launches, 551 -> 497; of 4 layers of 8192 617 -> 596.
template <int EPT, int NL, typename TOut>
__global__ __launch_bounds__(kThreads, 1) void token_head_kernel(TOut* __restrict__ out, const _Float16* __restrict__ head,
                                                                 int vocab, int n, const ChainArgs c) {
  __shared__ __align__(16) float smem[EPT ? chain_floats(kThreads * EPT) : kMaxLoads * 256 + kWaves];
  _Float16* xs = reinterpret_cast<_Float16*>(smem);  // n values, padded with zeros to whole loads
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int step = (int)gridDim.x * kWaves;
  int row = (int)blockIdx.x * kWaves + wave;

  // the operands of the norm first: a CU's requests return in order
  const int place = qtip_wht::wht_place(lane);
  half8h px = {}, pw = {};
  constexpr int E = EPT ? EPT : 2;
  ChainRegs<E> r;
  if constexpr (EPT != 0) {
    chain_load<E, false>(c, nullptr, place, wave, r);
  } else if (tid * 8 < n) {
    px = *reinterpret_cast<const half8h*>(c.residual + tid * 8);
    pw = *reinterpret_cast<const half8h*>(c.norm_w + tid * 8);
  }
  u32x4h buf[NL];
  const bool live = lane * 8 + (NL - 1) * 512 < n;  // the last load of a row may be ragged
  auto fetch = [&](int i, int rw) {
    const _Float16* p = head + (size_t)rw * n;
    const int e = i < NL - 1 || live ? lane * 8 + i * 512 : 0;
    buf[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4h*>(p + e));
  };
  const int first = row < vocab ? row : vocab - 1;
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    fetch(i, first);
    __builtin_amdgcn_sched_barrier(0);
  }

  if constexpr (EPT != 0) {
    float v[E];
    const float rs = chain_residual<E>(r, c, smem, v, lane, place, wave, false);
    _Float16 h[E];
#pragma unroll
    for (int i = 0; i < E; ++i) h[i] = (_Float16)((float)r.wv[i] * (float)(_Float16)(v[i] * rs));
    qtip_wht::st_f16<E>(xs + nat_index<E>(place, wave), h);
  } else {
    float ss = 0.f;
#pragma unroll
    for (int q = 0; q < 8; ++q) ss += (float)px[q] * (float)px[q];
    ss = qtip_wht::wave_sum(ss);
    float* wsum = smem + kMaxLoads * 256;
    if (lane == 0) wsum[wave] = ss;
    __syncthreads();
    const float rs = __builtin_amdgcn_rsqf(qtip_wht::waves16_sum(wsum, lane) / (float)n + c.eps);
    half8h y;
#pragma unroll
    for (int q = 0; q < 8; ++q) y[q] = (_Float16)((float)pw[q] * (float)(_Float16)((float)px[q] * rs));
    if (tid * 8 < NL * 512) *reinterpret_cast<half8h*>(xs + tid * 8) = tid * 8 < n ? y : half8h{};
  }
  __syncthreads();

  uint32_t xo = lane * 8;
  auto dot = [&](int i, float acc) {
    const half8h x = *reinterpret_cast<const half8h*>(xs + xo + i * 512);
    half8h w = __builtin_bit_cast(half8h, buf[i]);
    if (i == NL - 1 && !live) w = half8h{};
#pragma unroll
    for (int q = 0; q < 8; ++q) acc += (float)x[q] * (float)w[q];
    return acc;
  };
  auto store = [&](float acc, int rw) {
    acc = qtip_wht::wave_sum(acc);
    if (lane == 0) out[rw] = (TOut)(_Float16)acc;
  };
  if (row >= vocab) return;
  for (; row + step < vocab; row += step) {
    float acc = 0.f;
    asm("" : "+v"(xo));  // (xn stays in LDS: kept in registers over the rows it would spill)
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      acc = dot(i, acc);
      fetch(i, row + step);
      __builtin_amdgcn_sched_barrier(0);  // (a load goes out as soon as its register is free)
    }
    store(acc, row);
  }
  float acc = 0.f;
#pragma unroll
  for (int i = 0; i < NL; ++i) acc = dot(i, acc);
  store(acc, row);
}

template <int EPT, int NL>
void launch_head(int grid, void* out, int out_dtype, const void* head, int vocab, int n, const ChainArgs& c, hipStream_t st) {
  if (out_dtype == QTIP_F16)
    token_head_kernel<EPT, NL><<<grid, kThreads, 0, st>>>((_Float16*)out, (const _Float16*)head, vocab, n, c);
  else
    token_head_kernel<EPT, NL><<<grid, kThreads, 0, st>>>((float*)out, (const _Float16*)head, vocab, n, c);
}

}  // namespace

extern "C" int qtip_token_head(void* out, int out_dtype, const void* head_f16, int vocab, int n, const void* x_f16,
                               const float* parts, int in_parts, size_t part_stride, const float* post_f32, float scale_out,
                               const void* norm_weight_f16, float eps, void* stream) {
  if (!out || !head_f16 || !x_f16 || !norm_weight_f16) return QTIP_E_NULL;
  if (out_dtype != QTIP_F16 && out_dtype != QTIP_F32) return QTIP_E_DTYPE;
  if (vocab < 1 || vocab > (1 << 30) || n < 8 || n > 512 * kMaxLoads || (n & 7)) return QTIP_E_SHAPE;
  if (!aligned16(head_f16) || !aligned16(x_f16) || !aligned16(norm_weight_f16)) return QTIP_E_ALIGN;
  ChainArgs c = {};
  c.residual = (const _Float16*)x_f16;
  c.norm_w = (const _Float16*)norm_weight_f16;
  c.eps = eps;
  if (parts) {
    if (!post_f32) return QTIP_E_NULL;
    if ((n != 2048 && n != 4096 && n != 8192) || in_parts < 1 || in_parts > 16) return QTIP_E_SHAPE;
    if (!aligned16(parts) || !aligned16(post_f32) || ((part_stride * sizeof(float)) & 15u)) return QTIP_E_ALIGN;
    c.parts = parts;
    c.post = post_f32;
    c.part_stride = part_stride;
    c.scale_out = scale_out;
    c.in_parts = in_parts;
  }
  int cus = 0;
  if (const int rc = qtip_device_ready(stream, &cus)) return rc;
  const int want = (vocab + kWaves - 1) / kWaves, grid = want < cus ? want : cus;
  hipStream_t st = (hipStream_t)stream;
  if (parts) {
    switch (n >> 10) {
      case 2: launch_head<2, 4>(grid, out, out_dtype, head_f16, vocab, n, c, st); break;
      case 4: launch_head<4, 8>(grid, out, out_dtype, head_f16, vocab, n, c, st); break;
      default: launch_head<8, 16>(grid, out, out_dtype, head_f16, vocab, n, c, st); break;
    }
    return (int)hipGetLastError();
  }
  switch ((n + 511) >> 9) {
#define QTIP_HEAD(NL) case NL: launch_head<0, NL>(grid, out, out_dtype, head_f16, vocab, n, c, st); break;
    QTIP_HEAD(1) QTIP_HEAD(2) QTIP_HEAD(3) QTIP_HEAD(4) QTIP_HEAD(5) QTIP_HEAD(6) QTIP_HEAD(7) QTIP_HEAD(8)
    QTIP_HEAD(9) QTIP_HEAD(10) QTIP_HEAD(11) QTIP_HEAD(12) QTIP_HEAD(13) QTIP_HEAD(14) QTIP_HEAD(15) QTIP_HEAD(16)
#undef QTIP_HEAD
  }
  return (int)hipGetLastError();
}
