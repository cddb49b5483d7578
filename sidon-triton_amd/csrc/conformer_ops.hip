// conformer_ops.hip -- the conformer layer's elementwise and convolution
// kernels around its GEMMs (MI355X / gfx950):
//
//   glu              g = h[:, :C] * sigmoid(h[:, C:])                  fp16 -> fp16
//   silu (in place)  h = h * sigmoid(h)                                 fp16
//   causal_dw_norm   out[t] = silu(LN(sum_k w[k] * g[t + k - (K-1)]))   fp16 -> fp16
//
// They replace _glu_kernel / glu and _causal_dw_norm_kernel / causal_dw_norm
// of src/sidon_triton/triton_encoder.py:113-181, and the in-place F.silu of
// the feed-forward modules (:498-499, :507-508).  causal_dw_norm can also read
// the pointwise conv's output h [R, 2C] and form g = GLU(h) on the fly (g is
// rounded to fp16 exactly as glu stores it), which saves the g round trip
// through HBM.
//
// causal_dw_norm maps one thread to a channel pair and one block to BT
// consecutive frames of one batch item over all C channels.  The thread
// keeps its 2 K taps, its channels of the BT + K - 1 source frames and BT
// accumulator pairs in registers: each g element is read once per block (plus
// the K - 1 frames of left context the block shares with its neighbour), and
// every output frame sums its taps in order k = 0 .. K-1.  LayerNorm reduces
// the block's BT rows at once.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <initializer_list>

#include "sidon_encoder.h"
#include "sidon_host.h"
#include "sidon_wave.h"

#define SIDON_API extern "C" __attribute__((visibility("default")))

namespace {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef float f8 __attribute__((ext_vector_type(8)));

constexpr int kMaxC = 2048;      // channels: one thread per pair, <= 1024 threads
constexpr int kEwThreads = 256;  // glu / silu block size
constexpr int kXcds = 8;         // accelerator complex dies of an MI355X

// sigmoid(x) = 1 / (1 + e^-x) with the hardware exponential and reciprocal
// (each within about 1 ulp in fp32; the results are rounded to fp16).
__device__ __forceinline__ float sigmoid(float x) { return __builtin_amdgcn_rcpf(1.f + __expf(-x)); }

// GLU of one element as glu stores it: the fp32 product rounded to fp32,
// then to fp16.  The empty asm keeps the compiler from fusing the product and
// the conversion into one mixed-precision instruction, whose single rounding
// can differ from the two.
__device__ __forceinline__ _Float16 glu1(float a, float b) {
  float prod = a * sigmoid(b);
  asm volatile("" : "+v"(prod));
  return (_Float16)prod;
}

// SiLU of one element, rounded the same way (fp32, then fp16).
__device__ __forceinline__ _Float16 silu1(float x) {
  float y = x * sigmoid(x);
  asm volatile("" : "+v"(y));
  return (_Float16)y;
}

// ---- glu / silu -------------------------------------------------------------

// kVec chunks of 8 columns per thread (loads first, then math); requires
// C % 8 == 0 and 16-byte aligned rows.
constexpr int kVec = 4;
__global__ void __launch_bounds__(kEwThreads) glu_vec_kernel(const _Float16* __restrict__ h, _Float16* __restrict__ g,
                                                             int64_t n8, int c8) {
  const int64_t i0 = ((int64_t)blockIdx.x * kEwThreads * kVec) + threadIdx.x;
  h8 a[kVec], b[kVec];
#pragma unroll
  for (int v = 0; v < kVec; ++v) {
    const int64_t i = i0 + (int64_t)v * kEwThreads;
    if (i < n8) {
      const int64_t row = i / c8;
      const int64_t col = i - row * c8;
      a[v] = reinterpret_cast<const h8*>(h)[row * 2 * c8 + col];
      b[v] = reinterpret_cast<const h8*>(h)[row * 2 * c8 + c8 + col];
    }
  }
#pragma unroll
  for (int v = 0; v < kVec; ++v) {
    const int64_t i = i0 + (int64_t)v * kEwThreads;
    if (i < n8) {
      h8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = glu1((float)a[v][j], (float)b[v][j]);
      reinterpret_cast<h8*>(g)[i] = o;
    }
  }
}

__global__ void __launch_bounds__(kEwThreads) glu_scalar_kernel(const _Float16* __restrict__ h,
                                                                _Float16* __restrict__ g, int64_t n, int C) {
  const int64_t i = (int64_t)blockIdx.x * kEwThreads + threadIdx.x;
  if (i >= n) return;
  const int64_t row = i / C;
  const int64_t col = i - row * C;
  const float a = (float)h[row * 2 * C + col];
  const float b = (float)h[row * 2 * C + C + col];
  g[i] = glu1(a, b);
}

__global__ void __launch_bounds__(kEwThreads) silu_vec_kernel(_Float16* __restrict__ h, int64_t n8) {
  const int64_t i0 = ((int64_t)blockIdx.x * kEwThreads * kVec) + threadIdx.x;
  h8 x[kVec];
#pragma unroll
  for (int v = 0; v < kVec; ++v) {
    const int64_t i = i0 + (int64_t)v * kEwThreads;
    if (i < n8) x[v] = reinterpret_cast<const h8*>(h)[i];
  }
#pragma unroll
  for (int v = 0; v < kVec; ++v) {
    const int64_t i = i0 + (int64_t)v * kEwThreads;
    if (i < n8) {
#pragma unroll
      for (int j = 0; j < 8; ++j) x[v][j] = silu1((float)x[v][j]);
      reinterpret_cast<h8*>(h)[i] = x[v];
    }
  }
}

__global__ void __launch_bounds__(kEwThreads) silu_scalar_kernel(_Float16* __restrict__ h, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kEwThreads + threadIdx.x;
  if (i >= n) return;
  h[i] = silu1((float)h[i]);
}

// ---- causal depthwise conv + LayerNorm + SiLU --------------------------------

struct DwParams {
  const _Float16* src;  // g [B*T, C] or h [B*T, 2C] (kGlu)
  const float* dwt;     // [K, C] taps
  const float* ln_w;
  const float* ln_b;
  _Float16* out;        // [B*T, C]
  float eps;
  int T, C;
};

using sidon::wave_sum;

// Sums v[t] over the block's threads for every t < BT (result in every
// thread), in wavefront order: wavefront sums to LDS, then lane t of every
// wavefront adds the block's for row t and hands the total to the others as a
// scalar -- one barrier, and NW LDS reads instead of BT NW per thread.
template <int BT, int NW>
__device__ __forceinline__ void block_sums(float (&v)[BT], float (*red)[NW], int nwaves) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
#pragma unroll
  for (int t = 0; t < BT; ++t) v[t] = wave_sum(v[t]);
  if (lane == 0) {
#pragma unroll
    for (int t = 0; t < BT; ++t) red[t][wave] = v[t];
  }
  __syncthreads();
  float s = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w)
    if (w < nwaves) s += red[min(lane, BT - 1)][w];
#pragma unroll
  for (int t = 0; t < BT; ++t)
    v[t] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, s), t));
}

// One block: output frames [t0, t0 + BT) of one item, all C channels (tiles
// numbered item-major over a 1-D grid).  Thread i owns channels 2i, 2i + 1.
//   1. It loads its 2 K taps, norm weights and its channels of the BT + K - 1
//      source frames (256 bytes per wavefront and frame) straight into
//      registers, all in flight at once up to 1024 channels, and forms g; no
//      other thread needs its channels, so nothing is staged.
//   2. It walks the frames once, adding frame j into output i through tap
//      k = j - i, so every output sums its taps in order k = 0 .. K-1.
//   3. LayerNorm over the C channels of the BT rows (two passes, block
//      reductions), SiLU, fp16 store.
// Bound by the memory round trip and the reductions at few frames per block
// and by vector instructions at many (20 frames: 1240 FMAs, 40 SiLUs).
// C = 1024, K = 31, us per launch from g (from h in brackets), before with a
// tile staged in LDS, its own wait for the taps and 8 BT LDS reads per thread
// and reduction -> now: 150 frames 7.6 -> 5.5 (9.8 -> 7.5), 750 8.7 -> 7.3 (10.7 ->
// 9.8), 1600 11.6 -> 9.4 (14.1 -> 12.5), 3000 18.2 -> 12.0 (20.9 -> 16.1), 4800
// 21.7 -> 17.3 (25.1 -> 22.8).
template <int K, int BT, bool kGlu, int kMaxThreads>
__global__ void __launch_bounds__(kMaxThreads) causal_dw_norm_kernel(const DwParams p) {
  constexpr int NW = kMaxThreads / 64;
  constexpr int kRows = BT + K - 1;
  __shared__ float red[2][BT][NW];
  const int C = p.C;
  const int nwaves = blockDim.x >> 6;
  // Workgroups go to the 8 XCDs round-robin; give each XCD a contiguous run
  // of tiles, so the K - 1 frames a tile shares with its left neighbour are
  // usually in the same L2.
  const int ntiles = (p.T + BT - 1) / BT;
  const int nblk = gridDim.x;
  const int xcd = blockIdx.x % kXcds;
  const int tile_id = xcd * (nblk / kXcds) + min(xcd, nblk % kXcds) + blockIdx.x / kXcds;
  const int b = tile_id / ntiles;
  const int t0 = (tile_id - b * ntiles) * BT;
  const int s0 = t0 - (K - 1);
  const int64_t row0 = (int64_t)b * p.T;
  const int64_t stride = kGlu ? 2 * (int64_t)C : (int64_t)C;

  // 1. loads (threads past C load its last channels and are left out of the
  // sums; frames outside [0, T) load the nearest one)
  const bool on = 2 * (int)threadIdx.x < C;
  const int c = on ? 2 * threadIdx.x : C - 2;
  const _Float16* src = p.src + row0 * stride + c;
  // Up to 8 wavefronts per block every frame is in flight at once.  More leave
  // each 168 or 128 registers: 8 frames at a time up to 8 output frames, past
  // that kFlight ahead of the products, each refilled as it is taken.
  constexpr bool kRing = kMaxThreads > 512 && BT > 8;
  constexpr int kFlight = kMaxThreads <= 512 ? kRows : !kRing || kMaxThreads <= 768 ? 8 : kGlu ? 4 : 6;
  h2 a[kFlight], gate[kGlu ? kFlight : 1];
  auto load = [&](int j) {
    const _Float16* at = src + min(max(s0 + j, 0), p.T - 1) * stride;
    a[j % kFlight] = *reinterpret_cast<const h2*>(at);
    if constexpr (kGlu) gate[j % kFlight] = *reinterpret_cast<const h2*>(at + C);
  };
  auto load_from = [&](int j0) {
#pragma unroll
    for (int j = j0; j < min(j0 + kFlight, kRows); ++j) load(j);
  };
  load_from(0);
  f2 w[K];
#pragma unroll
  for (int k = 0; k < K; ++k) w[k] = *reinterpret_cast<const f2*>(p.dwt + (int64_t)k * C + c);
  const f2 lw = *reinterpret_cast<const f2*>(p.ln_w + c);
  const f2 lb = *reinterpret_cast<const f2*>(p.ln_b + c);
  __builtin_amdgcn_sched_barrier(0);  // every load so far in front of the first product

  // 2. conv
  f2 acc[BT];
#pragma unroll
  for (int t = 0; t < BT; ++t) acc[t] = f2{0.f, 0.f};
#pragma unroll
  for (int j = 0; j < kRows; ++j) {
    if (!kRing && j > 0 && j % kFlight == 0) {
      load_from(j);
      __builtin_amdgcn_sched_barrier(0);
    }
    const int u = j % kFlight;
    f2 g = {(float)a[u][0], (float)a[u][1]};
    if constexpr (kGlu) g = f2{(float)glu1(g[0], (float)gate[u][0]), (float)glu1(g[1], (float)gate[u][1])};
    if constexpr (kRing) {
      if (j + kFlight < kRows) load(j + kFlight);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (j < K - 1 && s0 + j < 0) g = f2{0.f, 0.f};  // uniform: left of the item
#pragma unroll
    for (int i = 0; i < BT; ++i) {
      const int k = j - i;
      if (k >= 0 && k < K) {
        acc[i][0] = fmaf(g[0], w[k][0], acc[i][0]);
        acc[i][1] = fmaf(g[1], w[k][1], acc[i][1]);
      }
    }
  }

  // 3. LayerNorm over the C channels of every row (two passes), then SiLU.
  float v[BT];
#pragma unroll
  for (int t = 0; t < BT; ++t) v[t] = on ? acc[t][0] + acc[t][1] : 0.f;
  block_sums<BT, NW>(v, red[0], nwaves);
  const float inv_c = 1.f / (float)C;
#pragma unroll
  for (int t = 0; t < BT; ++t) {
    const float mean = v[t] * inv_c;
    acc[t][0] -= mean;
    acc[t][1] -= mean;
    v[t] = on ? acc[t][0] * acc[t][0] + acc[t][1] * acc[t][1] : 0.f;
  }
  block_sums<BT, NW>(v, red[1], nwaves);
  if (!on) return;
#pragma unroll
  for (int t = 0; t < BT; ++t) {
    if (t0 + t >= p.T) continue;
    const float rstd = rsqrtf(v[t] * inv_c + p.eps);
    const float y0 = acc[t][0] * rstd * lw[0] + lb[0];
    const float y1 = acc[t][1] * rstd * lw[1] + lb[1];
    *reinterpret_cast<h2*>(p.out + (row0 + t0 + t) * C + c) = h2{silu1(y0), silu1(y1)};
  }
}

// Frames per block: the candidate that minimises (blocks per compute unit,
// rounded up) x (source frames per block).  Blocks are counted per CU, not per
// resident slot: two blocks sharing a CU run no faster than one after the
// other (1600 frames: 400 blocks of 4 10.3 us, 200 of 8 9.4; 150 frames: 38 of
// 4 6.9, 150 of 1 5.5).
int pick_bt(std::initializer_list<int> frames, int K, int B, int T) {
  int best = 0;
  long best_cost = 0;
  const int cus = sidon::compute_units();
  for (int bt : frames) {
    const long blocks = (long)((T + bt - 1) / bt) * B;
    const long cost = ((blocks + cus - 1) / cus) * (bt + K - 1);
    if (best == 0 || cost < best_cost) {
      best = bt;
      best_cost = cost;
    }
  }
  return best;
}

template <int K, int BT, int kMaxThreads>
hipError_t launch_dw_bt(const DwParams& p, int B, bool glu_input, hipStream_t stream) {
  const dim3 grid((unsigned)(((p.T + BT - 1) / BT) * B)), block(64 * ((p.C / 2 + 63) / 64));
  if (glu_input) {
    hipLaunchKernelGGL((causal_dw_norm_kernel<K, BT, true, kMaxThreads>), grid, block, 0, stream, p);
  } else {
    hipLaunchKernelGGL((causal_dw_norm_kernel<K, BT, false, kMaxThreads>), grid, block, 0, stream, p);
  }
  return hipGetLastError();
}

// Past 1024 channels.  Many frames per block pay from 15 taps on, where the K - 1
// frames in front of a block are most of its work (us from h, at most 8 frames |
// up to 20: K = 31, C = 1536 3000 frames 31.5 | 23.8, 4800 45.3 | 28.1; C = 1600 4800
// 54.6 | 33.6; K = 15, C = 2048 4800 38.6 | 28.4; K = 3, C = 2048 3000 16.3 | 19.1).
template <int K, int kMaxThreads>
hipError_t launch_dw_wide(const DwParams& p, int B, bool glu_input, hipStream_t stream) {
  if constexpr (K >= 15) {
    const int bt = pick_bt({20, 16, 8, 4}, K, B, p.T);
    if (bt == 20) return launch_dw_bt<K, 20, kMaxThreads>(p, B, glu_input, stream);
    if (bt == 16) return launch_dw_bt<K, 16, kMaxThreads>(p, B, glu_input, stream);
    if (bt == 8) return launch_dw_bt<K, 8, kMaxThreads>(p, B, glu_input, stream);
    return launch_dw_bt<K, 4, kMaxThreads>(p, B, glu_input, stream);
  }
  return pick_bt({8, 4}, K, B, p.T) == 8 ? launch_dw_bt<K, 8, kMaxThreads>(p, B, glu_input, stream)
                                         : launch_dw_bt<K, 4, kMaxThreads>(p, B, glu_input, stream);
}

template <int K>
hipError_t launch_dw(const DwParams& p, int B, bool glu_input, hipStream_t stream) {
  if (p.C > 1536) return launch_dw_wide<K, 1024>(p, B, glu_input, stream);
  if (p.C > 1024) return launch_dw_wide<K, 768>(p, B, glu_input, stream);
  switch (pick_bt({20, 16, 12, 8, 6, 4, 2, 1}, K, B, p.T)) {
    case 20: return launch_dw_bt<K, 20, 512>(p, B, glu_input, stream);
    case 16: return launch_dw_bt<K, 16, 512>(p, B, glu_input, stream);
    case 12: return launch_dw_bt<K, 12, 512>(p, B, glu_input, stream);
    case 8: return launch_dw_bt<K, 8, 512>(p, B, glu_input, stream);
    case 6: return launch_dw_bt<K, 6, 512>(p, B, glu_input, stream);
    case 4: return launch_dw_bt<K, 4, 512>(p, B, glu_input, stream);
    case 2: return launch_dw_bt<K, 2, 512>(p, B, glu_input, stream);
    default: return launch_dw_bt<K, 1, 512>(p, B, glu_input, stream);
  }
}

bool aligned(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

}  // namespace

SIDON_API int sidon_glu(const void* h, void* g, int R, int C, sidon_stream_t stream) {
  using sidon::fail;
  sidon::clear_error();
  if (!h || !g) return fail(SIDON_E_NULL, "h and g must be non-NULL");
  if (R < 1 || C < 1) return fail(SIDON_E_SHAPE, "R=%d and C=%d must be >= 1", R, C);
  if (!aligned(h, 2) || !aligned(g, 2)) return fail(SIDON_E_ALIGN, "fp16 tensors must be 2-byte aligned");
  int rc;
  if ((rc = sidon::check_device())) return rc;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const auto* hp = static_cast<const _Float16*>(h);
  auto* gp = static_cast<_Float16*>(g);
  if (C % 8 == 0 && aligned(h, 16) && aligned(g, 16)) {
    const int64_t n8 = (int64_t)R * (C / 8);
    const int64_t per_block = (int64_t)kEwThreads * kVec;
    hipLaunchKernelGGL(glu_vec_kernel, dim3((unsigned)((n8 + per_block - 1) / per_block)), dim3(kEwThreads), 0, s, hp,
                       gp, n8, C / 8);
  } else {
    const int64_t n = (int64_t)R * C;
    hipLaunchKernelGGL(glu_scalar_kernel, dim3((unsigned)((n + kEwThreads - 1) / kEwThreads)), dim3(kEwThreads), 0, s,
                       hp, gp, n, C);
  }
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return fail(SIDON_E_LAUNCH, "glu launch failed: %s", hipGetErrorString(err));
  return SIDON_OK;
}

SIDON_API int sidon_silu(void* h, int64_t n, sidon_stream_t stream) {
  using sidon::fail;
  sidon::clear_error();
  if (!h) return fail(SIDON_E_NULL, "h must be non-NULL");
  if (n < 1) return fail(SIDON_E_SHAPE, "n=%lld must be >= 1", (long long)n);
  if (!aligned(h, 2)) return fail(SIDON_E_ALIGN, "fp16 tensors must be 2-byte aligned");
  int rc;
  if ((rc = sidon::check_device())) return rc;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  auto* hp = static_cast<_Float16*>(h);
  if (n % 8 == 0 && aligned(h, 16)) {
    const int64_t n8 = n / 8;
    const int64_t per_block = (int64_t)kEwThreads * kVec;
    hipLaunchKernelGGL(silu_vec_kernel, dim3((unsigned)((n8 + per_block - 1) / per_block)), dim3(kEwThreads), 0, s, hp,
                       n8);
  } else {
    hipLaunchKernelGGL(silu_scalar_kernel, dim3((unsigned)((n + kEwThreads - 1) / kEwThreads)), dim3(kEwThreads), 0, s,
                       hp, n);
  }
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return fail(SIDON_E_LAUNCH, "silu launch failed: %s", hipGetErrorString(err));
  return SIDON_OK;
}

SIDON_API int sidon_causal_dw_norm(const void* src, int glu_input, const float* dwt, const float* ln_w,
                                   const float* ln_b, float eps, void* out, int B, int T, int C, int K,
                                   sidon_stream_t stream) {
  using sidon::fail;
  sidon::clear_error();
  if (!src || !dwt || !ln_w || !ln_b || !out) return fail(SIDON_E_NULL, "every pointer must be non-NULL");
  if (B < 1 || T < 1 || C < 2 || C > kMaxC || (C & 1) != 0)
    return fail(SIDON_E_SHAPE, "B=%d and T=%d must be >= 1 and C=%d even in [2, %d]", B, T, C, kMaxC);
  if (K != 3 && K != 7 && K != 15 && K != 31)
    return fail(SIDON_E_SHAPE, "K=%d: supported kernel sizes are 3, 7, 15 and 31", K);
  if ((int64_t)B * T > INT32_MAX / 2) return fail(SIDON_E_SHAPE, "B*T=%lld rows is too large", (long long)B * T);
  if (!aligned(src, 4) || !aligned(out, 4)) return fail(SIDON_E_ALIGN, "fp16 tensors must be 4-byte aligned");
  if (!aligned(dwt, 8) || !aligned(ln_w, 8) || !aligned(ln_b, 8))
    return fail(SIDON_E_ALIGN, "fp32 tensors must be 8-byte aligned");
  int rc;
  if ((rc = sidon::check_device())) return rc;
  const DwParams p{static_cast<const _Float16*>(src), dwt, ln_w, ln_b, static_cast<_Float16*>(out), eps, T, C};
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const bool g = glu_input != 0;
  hipError_t err;
  switch (K) {
    case 3: err = launch_dw<3>(p, B, g, s); break;
    case 7: err = launch_dw<7>(p, B, g, s); break;
    case 15: err = launch_dw<15>(p, B, g, s); break;
    default: err = launch_dw<31>(p, B, g, s); break;
  }
  if (err != hipSuccess) return fail(SIDON_E_LAUNCH, "causal_dw_norm launch failed: %s", hipGetErrorString(err));
  return SIDON_OK;
}
