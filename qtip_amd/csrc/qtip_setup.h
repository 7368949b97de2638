// Per-device set-up shared by the library's source files (not part of the C ABI).
#pragma once
#include <hip/hip_runtime.h>

#define QTIP_INTERNAL __attribute__((visibility("hidden")))

// Set-up of the current device on its first use (see qtip_init): 0 and the CU count, QTIP_E_NOT_INIT
// inside a stream capture, or the hipError_t of a failed set-up.
QTIP_INTERNAL int qtip_device_ready(void* stream, int* cus);

// LDS opt-in of the transform kernels, called by the set-up
QTIP_INTERNAL hipError_t qtip_rht_allow_lds();
