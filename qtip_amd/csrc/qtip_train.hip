// Backward of a per-column scale (qtip_scale_columns_grad): what a fine-tuning step adds to the forward's kernels.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/qtip_hip.h"
#include "qtip_setup.h"

namespace {

typedef float float4v __attribute__((ext_vector_type(4)));
typedef _Float16 half4v __attribute__((ext_vector_type(4)));

constexpr int kBlock = 256, kLanes = 64, kRowLanes = kBlock / kLanes;
constexpr int kCols = 4 * kLanes;  // columns of a workgroup

// y = x * s over the columns of a (rows, n) matrix: gx = g * s and gs[c] = sum over rows of g * x.
// Bound by memory traffic: g and x are read once, gx written once, and the column sums are taken on the way
// (as separate passes: a product written out, read again by a reduction over the rows that ran at 0.6 TB/s, and a
// second product).  A workgroup takes 256 columns by `chunk` rows, one row per wave at a time, 16 bytes per lane; its
// four waves' sums meet in LDS and leave as one row of partial sums, which the second kernel adds in order:
// the result does not depend on the schedule.  2048 rows of 11008 / 4096, fp32: 221 -> 44 + 6 (6.2 TB/s) / 47 -> 20 + 6 us.
template <typename TS>
__global__ __launch_bounds__(kBlock) void scale_grad_kernel(float* __restrict__ gx, float* __restrict__ parts,
                                                            const float* __restrict__ g, const float* __restrict__ x,
                                                            const TS* __restrict__ s, int rows, int n, int chunk) {
  __shared__ __align__(16) float4v sums[kRowLanes][kLanes];
  const int lane = threadIdx.x & (kLanes - 1), wave = threadIdx.x / kLanes;
  const int c = blockIdx.x * kCols + 4 * lane;
  const int r0 = blockIdx.y * chunk, r1 = r0 + chunk < rows ? r0 + chunk : rows;
  float4v acc = {0.f, 0.f, 0.f, 0.f};
  if (c < n) {  // (n is a multiple of 4)
    float4v sv;
    if constexpr (sizeof(TS) == 2) {
      const half4v h = *reinterpret_cast<const half4v*>(s + c);
#pragma unroll
      for (int e = 0; e < 4; ++e) sv[e] = (float)h[e];
    } else {
      sv = *reinterpret_cast<const float4v*>(s + c);
    }
#pragma unroll 4
    for (int r = r0 + wave; r < r1; r += kRowLanes) {
      const size_t o = (size_t)r * n + c;
      const float4v gv = *reinterpret_cast<const float4v*>(g + o);
      acc += gv * *reinterpret_cast<const float4v*>(x + o);
      *reinterpret_cast<float4v*>(gx + o) = gv * sv;
    }
  }
  sums[wave][lane] = acc;
  __syncthreads();
  if (wave == 0 && c < n)
    *reinterpret_cast<float4v*>(parts + (size_t)blockIdx.y * n + c) =
        (sums[0][lane] + sums[1][lane]) + (sums[2][lane] + sums[3][lane]);
}

// gs[c] = the sum of `count` rows of partial sums: a workgroup takes 64 columns, its waves every fourth row
__global__ __launch_bounds__(kBlock) void sum_rows_kernel(float* __restrict__ gs, const float* __restrict__ parts, int n,
                                                          int count) {
  __shared__ float sums[kRowLanes][kLanes];
  const int lane = threadIdx.x & (kLanes - 1), wave = threadIdx.x / kLanes;
  const int c = blockIdx.x * kLanes + lane;
  float acc = 0.f;
  if (c < n)
    for (int i = wave; i < count; i += kRowLanes) acc += parts[(size_t)i * n + c];
  sums[wave][lane] = acc;
  __syncthreads();
  if (wave == 0 && c < n) gs[c] = (sums[0][lane] + sums[1][lane]) + (sums[2][lane] + sums[3][lane]);
}

// Rows of a workgroup: about 1024 workgroups (four a CU) where there are enough rows, at least four rows per wave,
// so that the partial sums are a sixteenth of what is read at most from 8 rows on (one row of n for fewer).
int chunk_rows(int rows, int n) {
  const int colb = (n + kCols - 1) / kCols;
  const int chunks = (1024 + colb - 1) / colb;
  const int chunk = ((rows + chunks - 1) / chunks + kRowLanes - 1) / kRowLanes * kRowLanes;
  return chunk < 4 * kRowLanes ? 4 * kRowLanes : chunk;
}
int chunk_count(int rows, int n) {
  const int chunk = chunk_rows(rows, n);
  return (rows + chunk - 1) / chunk;
}

}  // namespace

extern "C" {

size_t qtip_scale_columns_grad_workspace_bytes(int rows, int n) {
  if (rows < 1 || n < 4 || (n & 3)) return 0;
  return (size_t)chunk_count(rows, n) * n * sizeof(float);
}

int qtip_scale_columns_grad(float* gx, float* gs, const float* g, const float* x, const void* s, int s_dtype, int rows,
                            int n, void* workspace, size_t workspace_bytes, void* stream) {
  if (!gx || !gs || !g || !x || !s || !workspace) return QTIP_E_NULL;
  if (rows < 1 || n < 4 || (n & 3)) return QTIP_E_SHAPE;
  if (s_dtype != QTIP_F16 && s_dtype != QTIP_F32) return QTIP_E_DTYPE;
  if (!aligned16(gx) || !aligned16(g) || !aligned16(x) || !aligned16(workspace) ||
      (reinterpret_cast<uintptr_t>(s) & (s_dtype == QTIP_F16 ? 7u : 15u)) || (reinterpret_cast<uintptr_t>(gs) & 3u))
    return QTIP_E_ALIGN;
  if (workspace_bytes < qtip_scale_columns_grad_workspace_bytes(rows, n)) return QTIP_E_WORKSPACE;
  const int chunk = chunk_rows(rows, n), count = chunk_count(rows, n);
  const dim3 grid((unsigned)((n + kCols - 1) / kCols), (unsigned)count);
  hipStream_t st = (hipStream_t)stream;
  auto* parts = (float*)workspace;
  if (s_dtype == QTIP_F16)
    scale_grad_kernel<_Float16><<<grid, kBlock, 0, st>>>(gx, parts, g, x, (const _Float16*)s, rows, n, chunk);
  else
    scale_grad_kernel<float><<<grid, kBlock, 0, st>>>(gx, parts, g, x, (const float*)s, rows, n, chunk);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return (int)e;
  sum_rows_kernel<<<(n + kLanes - 1) / kLanes, kBlock, 0, st>>>(gs, parts, n, count);
  return (int)hipGetLastError();
}

}  // extern "C"
