// stage.hip -- a bucketed call's inputs into the fixed buffers its captured
// graph reads (MI355X / gfx950): the chunk zero-padded to its bucket and the
// items' true lengths, in one launch (src/sidon_triton/runtime.py:374-401 does
// it with a copy per buffer).
//
// The lengths travel as kernel arguments.  As a copy from host memory they
// made the host wait for the previous call's graph, so every call paid its
// launches (60 us) with the GPU idle; the data copy is bound by HBM (a 96 s item
// is 6 MB of samples or 3 MB of features, read and written) and far below that.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include "sidon_encoder.h"
#include "sidon_host.h"

#define SIDON_API extern "C" __attribute__((visibility("default")))

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int kItems = 64;     // items per launch (their values are arguments)
constexpr int kThreads = 256;

struct StageParams {
  const float* src;
  float* dst;
  int* out[2];
  int64_t src_stride, dst_stride;  // elements per item
  bool vec;                        // 16-byte loads: src and its items 16-byte aligned
  int64_t count[kItems];           // elements copied; zeros up to dst_stride
  int value[2][kItems];
};

// Block (x, item): 4 elements per thread.
__global__ void __launch_bounds__(kThreads) stage_kernel(const StageParams p) {
  const int b = blockIdx.y;
  if (blockIdx.x == 0 && threadIdx.x < 2 && p.out[threadIdx.x] != nullptr) p.out[threadIdx.x][b] = p.value[threadIdx.x][b];
  if (p.src == nullptr) return;
  const int64_t i = 4 * ((int64_t)blockIdx.x * kThreads + threadIdx.x);
  if (i >= p.dst_stride) return;  // a multiple of 4
  const int64_t n = p.count[b];
  const float* s = p.src + b * p.src_stride + i;
  f4 v = {0.f, 0.f, 0.f, 0.f};
  if (p.vec && i + 3 < n) {
    v = *reinterpret_cast<const f4*>(s);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (i + e < n) v[e] = s[e];
  }
  *reinterpret_cast<f4*>(p.dst + b * p.dst_stride + i) = v;
}

}  // namespace

SIDON_API int sidon_stage_items(const float* src, int64_t src_stride, float* dst, int64_t dst_stride,
                                const int64_t* counts, int* out0, const int* values0, int* out1, const int* values1,
                                int B, sidon_stream_t stream) {
  using sidon::fail;
  sidon::clear_error();
  if ((src == nullptr) != (dst == nullptr) || (src != nullptr && counts == nullptr))
    return fail(SIDON_E_NULL, "src needs dst and counts");
  if ((out0 != nullptr && values0 == nullptr) || (out1 != nullptr && values1 == nullptr))
    return fail(SIDON_E_NULL, "an output needs its values");
  if (!src && !out0 && !out1) return fail(SIDON_E_NULL, "nothing to write");
  if (B < 1) return fail(SIDON_E_SHAPE, "B=%d must be >= 1", B);
  if (src) {
    if (dst_stride < 4 || dst_stride % 4 != 0 || dst_stride / 4 > (int64_t)kThreads * INT32_MAX)
      return fail(SIDON_E_SHAPE, "dst_stride=%lld must be a positive multiple of 4", (long long)dst_stride);
    for (int b = 0; b < B; ++b)
      if (counts[b] < 0 || counts[b] > dst_stride || counts[b] > src_stride)
        return fail(SIDON_E_SHAPE, "counts[%d]=%lld outside [0, min(%lld, %lld)]", b, (long long)counts[b],
                    (long long)src_stride, (long long)dst_stride);
    if (!sidon::aligned16(dst)) return fail(SIDON_E_ALIGN, "dst must be 16-byte aligned");
    if ((reinterpret_cast<uintptr_t>(src) & 3u) != 0) return fail(SIDON_E_ALIGN, "src must be 4-byte aligned");
  }
  int rc;
  if ((rc = sidon::check_device())) return rc;
  for (int b0 = 0; b0 < B; b0 += kItems) {
    const int nb = B - b0 < kItems ? B - b0 : kItems;
    StageParams p{};
    p.src = src ? src + b0 * src_stride : nullptr;
    p.dst = dst ? dst + b0 * dst_stride : nullptr;
    p.out[0] = out0 ? out0 + b0 : nullptr;
    p.out[1] = out1 ? out1 + b0 : nullptr;
    p.src_stride = src_stride;
    p.dst_stride = dst_stride;
    p.vec = src && sidon::aligned16(src) && src_stride % 4 == 0;
    for (int b = 0; b < nb; ++b) {
      p.count[b] = src ? counts[b0 + b] : 0;
      p.value[0][b] = out0 ? values0[b0 + b] : 0;
      p.value[1][b] = out1 ? values1[b0 + b] : 0;
    }
    const unsigned blocks = src ? (unsigned)((dst_stride / 4 + kThreads - 1) / kThreads) : 1u;
    hipLaunchKernelGGL(stage_kernel, dim3(blocks, nb), dim3(kThreads), 0, reinterpret_cast<hipStream_t>(stream), p);
  }
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return fail(SIDON_E_LAUNCH, "stage launch failed: %s", hipGetErrorString(err));
  return SIDON_OK;
}
