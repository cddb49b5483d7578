// sidon_host.h -- host-side helpers shared by the library's translation units
// (error text, device check).  Not part of the C ABI: every symbol here has
// hidden visibility.
#pragma once

#include <stdint.h>

#include "sidon_flexrel.h"

namespace sidon {

// Record a printf-style message as the thread's last error; returns `code`.
int fail(int code, const char* fmt, ...);
// Clear the thread's last error (start of every entry point).
void clear_error();
// SIDON_OK when the current HIP device is a gfx950, else SIDON_E_DEVICE.
int check_device();
// Compute units of the current device (after a successful check_device).
int compute_units();

// The tiled GEMM kernel's fp16-output form (gemm.hip): y = act(x . w^T + bias)
// with one rounding, act 1 = SiLU of the fp32 sum.  gemm_half_takes: the
// operands fit it and it is expected to beat the library; gemm_half launches
// it on operands that fit.
bool gemm_half_preferred(int M, int N, int K);
bool gemm_half_takes(const void* x, int ldx, const void* w, int ldw, const void* bias, const void* y, int ldy, int M,
                     int N, int K);
int gemm_half(const void* x, int ldx, const void* w, int ldw, const void* bias, void* y, int ldy, int M, int N, int K,
              int act, void* stream);

inline bool aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15u) == 0; }

}  // namespace sidon
