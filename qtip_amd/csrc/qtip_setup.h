// Per-device set-up shared by the library's source files (not part of the C ABI).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/qtip_hip.h"

#define QTIP_INTERNAL __attribute__((visibility("hidden")))

// Set-up of the current device on its first use (see qtip_init): 0 and the CU count, QTIP_E_NOT_INIT
// inside a stream capture, or the hipError_t of a failed set-up.
QTIP_INTERNAL int qtip_device_ready(void* stream, int* cus);

// CU count of the current device without any set-up (size queries), 0 when there is none
QTIP_INTERNAL int qtip_device_cus();

// LDS opt-in of the transform and batched kernels, called by the set-up
QTIP_INTERNAL hipError_t qtip_rht_allow_lds();
QTIP_INTERNAL hipError_t qtip_gemm_allow_lds();

// A product cut along k that leaves its partial sums, and the transform that adds them on load (qtip_linear): the number of
// ranges of the one launch of such a product (1: it is not cut, or runs in several launches), the launch, whether the transform
// takes them, and its launch.
QTIP_INTERNAL int qtip_gemm_ranges(int m, int k, int bits, int batch, bool fine);
QTIP_INTERNAL int qtip_gemm_parts(float* parts, int nparts, const void* packed, const void* x_f16, const void* tlut, int m,
                                  int k, int bits, int batch, bool fine, void* stream);
QTIP_INTERNAL bool qtip_rht_takes_parts(int n, int order, int rows, int nparts, bool residual);
QTIP_INTERNAL int qtip_rht_from_parts(void* out, int out_dtype, const float* parts, int nparts, int rows, int n, int order,
                                      const uint32_t* had_bits, const float* post, float scale, const void* residual_f16, void* stream);

// Scratch of a batched product with fine or with long sums (qtip_decompress_gemm, qtip_decompress_gemm_long_f16)
QTIP_INTERNAL size_t qtip_gemm_scratch(int m, int k, int bits, int batch, bool fine);

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

inline int check_common(const void* a, const void* b, const void* c, const void* d, int m, int k,
                 int bits) {
  if (!a || !b || !c || !d) return QTIP_E_NULL;
  if (bits < 2 || bits > 4) return QTIP_E_SHAPE;
  if (m <= 0 || k <= 0 || (m & 31) || (k & 31)) return QTIP_E_SHAPE;
  if ((long)m * k * bits / 8 >= (1L << 31)) return QTIP_E_SHAPE;  // 32-bit buffer offsets
  return QTIP_OK;
}
