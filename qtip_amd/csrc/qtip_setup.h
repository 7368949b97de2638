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

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

inline int check_common(const void* a, const void* b, const void* c, const void* d, int m, int k,
                 int bits) {
  if (!a || !b || !c || !d) return QTIP_E_NULL;
  if (bits < 2 || bits > 4) return QTIP_E_SHAPE;
  if (m <= 0 || k <= 0 || (m & 31) || (k & 31)) return QTIP_E_SHAPE;
  if ((long)m * k * bits / 8 >= (1L << 31)) return QTIP_E_SHAPE;  // 32-bit buffer offsets
  return QTIP_OK;
}
