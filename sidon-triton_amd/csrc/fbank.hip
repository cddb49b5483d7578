// fbank.hip -- the encoder's fbank front end (MI355X / gfx950), the work of
// src/sidon_triton/frontend.py:218-240:
//
//   spectrum   chunk [B, S] -> log(max(power . mel, 1.19e-7)) [B, F, 80]: framing, DC removal,
//              pre-emphasis, window, 512-point real FFT, power, mel and log in one kernel
//   normalize  per (item, mel bin) over the item's true frames:
//              (x - mean) / sqrt(var_ddof1 + 1e-7); the frame after an odd
//              count of true frames is 1.0; later frames 0.  [B, F, 80] is
//              also the stride-2 stacked [B, F / 2, 160] layout.
//
// normalize: statistics are per-tile two-pass sums (fixed tiles of frames,
// one block per (tile, item)); the blocks that apply them first merge the
// tiles by a fixed tree -- deterministic, no atomics -- through a
// caller-provided workspace.  frames and logmel (around a framing GEMM with the
// [400, 514] transform matrix) are the same spectrum in parts.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <mutex>

#include "sidon_encoder.h"
#include "sidon_host.h"
#include "sidon_wave.h"

#define SIDON_API extern "C" __attribute__((visibility("default")))

namespace {

constexpr int kBins = 257;
constexpr int kSpecWidth = 2 * kBins;
constexpr int kMel = 80;
constexpr int kFrameShift = 160;
constexpr int kFrameSize = 400;
constexpr int kEdgePad = 160;
constexpr float kMelFloor = 1.192092955078125e-07f;
constexpr float kVarEps = 1e-7f;
constexpr float kPadValue = 1.0f;
constexpr int kLmFrames = 12;        // logmel: frames per block
constexpr int kLmLanes = 3;          // logmel: threads per mel bin (each kLmFrames / kLmLanes frames)
constexpr int kLmThreads = 256;      // logmel: threads per block (kMel * kLmLanes = 240 sum)
constexpr int kLanes = 4;            // normalize: frame lanes x 80 bins per block
constexpr int kApplyFrames = 32;     // normalize: frames per apply block
constexpr int kMaxTiles = 64;
constexpr int kTileFloats = 2 * kMel;  // a statistics tile in the workspace: means, squared deviations
constexpr int kStatsCache = 40;      // statistics: frames per lane held in registers
constexpr int kSpWaves = 4;          // spectrum: wavefronts per block
// Frames per wavefront and block: with 8 per block a 96 s chunk's 1200 blocks
// give the busiest CU 7% more than the mean, with 12 28%.
constexpr int kSpFrames = 2;
constexpr int kSpBlock = kSpWaves * kSpFrames;
constexpr int kSpLanes = 2;          // spectrum: threads per mel bin
constexpr int kPoints = 256;         // spectrum: complex points of a 512-point real FFT
constexpr double kPreemph = 0.97;

// frames[b, f, i] = chunk[b, 160 f + i - 160] (zero outside [0, S)): the
// (160, 160) edge padding and the 400 / 160 framing in one pass, 4 samples
// per thread.
// Block (x, item b): 256 of the item's F * 100 16-byte frame chunks; 32-bit
// index math within the item (F * 100 < 2^32; the division by 100 is a
// multiply).
__global__ void __launch_bounds__(256) frames_kernel(const float* __restrict__ chunk, float* __restrict__ frames,
                                                    int S, int F, bool vec4) {
  constexpr uint32_t kPerRow = kFrameSize / 4;  // 100 chunks of 4 samples
  const uint32_t q = blockIdx.x * 256u + threadIdx.x;
  if (q >= (uint32_t)F * kPerRow) return;
  const uint32_t f = q / kPerRow;
  const int i = (int)(q - f * kPerRow) * 4;     // 0, 4, ..., 396
  const int t0 = (int)f * kFrameShift + i - kEdgePad;
  const float* src = chunk + (int64_t)blockIdx.y * S;
  float4 v;
  if (t0 >= 0 && t0 + 3 < S && vec4) {
    v = *reinterpret_cast<const float4*>(src + t0);  // t0 % 4 == 0; rows 16-byte aligned
  } else {
    v.x = (t0 >= 0 && t0 < S) ? src[t0] : 0.f;
    v.y = (t0 + 1 >= 0 && t0 + 1 < S) ? src[t0 + 1] : 0.f;
    v.z = (t0 + 2 >= 0 && t0 + 2 < S) ? src[t0 + 2] : 0.f;
    v.w = (t0 + 3 >= 0 && t0 + 3 < S) ? src[t0 + 3] : 0.f;
  }
  *reinterpret_cast<float4*>(frames + ((int64_t)blockIdx.y * F + f) * kFrameSize + i) = v;
}

// The block's kFrames power spectra -> log mel rows f0, f0 + 1, ... < R.
// Thread (mel m, lane fl) sums frames fl, fl + kLanesPer, ...: each weight
// is loaded once for kFrames / kLanesPer frames.  Every sum keeps the
// order i = 0 .. n - 1.
template <int kFrames, int kLanesPer>
__device__ __forceinline__ void mel_log(const float (*power)[kBins + 3], const float* __restrict__ mel_w,
                                        const int* __restrict__ mel_lo, const int* __restrict__ mel_len, int max_len,
                                        float* __restrict__ out, int f0, int R) {
  const int t = threadIdx.x;
  if (t >= kMel * kLanesPer) return;
  const int m = t % kMel;
  const int fl = t / kMel;
  const int lo = mel_lo[m];
  const int n = mel_len[m];
  const float* wm = mel_w + m * max_len;
  constexpr int kPerLane = kFrames / kLanesPer;
  float acc[kPerLane] = {};
#pragma unroll 4
  for (int i = 0; i < n; ++i) {
    const float wv = wm[i];
#pragma unroll
    for (int j = 0; j < kPerLane; ++j) acc[j] = fmaf(wv, power[fl + kLanesPer * j][lo + i], acc[j]);
  }
#pragma unroll
  for (int j = 0; j < kPerLane; ++j) {
    const int r = f0 + fl + kLanesPer * j;
    if (r < R) out[(int64_t)r * kMel + m] = logf(fmaxf(acc[j], kMelFloor));
  }
}

__global__ void __launch_bounds__(kLmThreads) logmel_kernel(const float* __restrict__ spec,
                                                          const float* __restrict__ mel_w,
                                                          const int* __restrict__ mel_lo,
                                                          const int* __restrict__ mel_len, int max_len,
                                                          float* __restrict__ out, int R) {
  __shared__ float power[kLmFrames][kBins + 3];
  const int f0 = blockIdx.x * kLmFrames;
  // Power spectra of the block's frames, every load of a thread in flight
  // together (consecutive threads read consecutive bins of a frame).
  {
    constexpr int kPer = (kLmFrames * kBins + kLmThreads - 1) / kLmThreads;
    float re[kPer], im[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int idx = threadIdx.x + kLmThreads * j;
      const int f = idx / kBins;
      const int k = idx - f * kBins;
      const bool ok = idx < kLmFrames * kBins && f0 + f < R;
      const float* row = spec + (int64_t)(f0 + f) * kSpecWidth;
      re[j] = ok ? row[k] : 0.f;
      im[j] = ok ? row[kBins + k] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int idx = threadIdx.x + kLmThreads * j;
      const int f = idx / kBins;
      if (idx < kLmFrames * kBins) power[f][idx - f * kBins] = re[j] * re[j] + im[j] * im[j];
    }
  }
  __syncthreads();
  mel_log<kLmFrames, kLmLanes>(power, mel_w, mel_lo, mel_len, max_len, out, f0, R);
}

// Spectrum.  A block owns kSpBlock frames, each wavefront kSpFrames of them.
// A frame's 400 samples, DC removed, pre-emphasised and windowed, are the 256
// complex points z[n] = y[2n] + i y[2n + 1] (zero from n = 200); lane l holds
// points l + 64 r.  Four radix-4 passes of the Stockham form (Ns = 1, 4, 16,
// 64; inputs l + 64 r, outputs (l / Ns) 4 Ns + l % Ns + r Ns, twiddles
// exp(-2 pi i (l % Ns) r / 4 Ns)) transform them, with the points exchanged
// through the wavefront's own LDS between passes (no block barrier: a
// wavefront's LDS accesses are in order); then X[k], conj(X[256 - k]) = E +- T
// with E, O the even and odd parts of (Z[k], conj(Z[256 - k])) and T = -i
// exp(-2 pi i k / 512) O.
//
// In float64 up to the powers, which are rounded to fp32: an fp32 FFT carries
// the loud bins' rounding into the quiet ones (a frame of 115 dB range: 9e-3
// off in log mel; the framing GEMM, whose sums are each bin's own, 1e-4).  The
// vector unit's float64 rate is its unpacked fp32 rate, so this costs LDS
// traffic and registers only.
//
// The framing GEMM that this replaces multiplied each frame by a dense [400,
// 514] matrix: 4.0 GFLOP and 41 MB of frames and spectra per 96 s chunk, on
// fp32 matrix instructions, against 0.13 GFLOP and 9 MB here.  Bound by vector
// instructions and LDS exchanges.
// 96 s chunk: 7.0 + 41 + 8.1 us for frames, GEMM and logmel -> 14.4
// us; 9.8 of it without the three inner passes.
struct Complex {
  double x, y;
};

__device__ __forceinline__ Complex cmul(Complex a, Complex b) {
  return {fma(-a.y, b.y, a.x * b.x), fma(a.x, b.y, a.y * b.x)};
}

__device__ __forceinline__ void radix4(Complex (&v)[4]) {
  const Complex a = {v[0].x + v[2].x, v[0].y + v[2].y}, b = {v[0].x - v[2].x, v[0].y - v[2].y};
  const Complex c = {v[1].x + v[3].x, v[1].y + v[3].y}, d = {v[1].x - v[3].x, v[1].y - v[3].y};
  v[0] = {a.x + c.x, a.y + c.y};
  v[1] = {b.x + d.y, b.y - d.x};
  v[2] = {a.x - c.x, a.y - c.y};
  v[3] = {b.x - d.y, b.y + d.x};
}

__device__ __forceinline__ float power_of(Complex a, bool infinite) {
  return infinite ? __builtin_inff() : (float)fma(a.x, a.x, a.y * a.y);
}

// LDS position of point i: one spare point per 16 spreads the strided writes.
__device__ __forceinline__ int spread(int i) { return i + (i >> 4); }

// The wavefront's LDS writes before are read after (other lanes' data).
__device__ __forceinline__ void lds_in_order() { asm volatile("" ::: "memory"); }

__global__ void __launch_bounds__(64 * kSpWaves) spectrum_kernel(const float* __restrict__ chunk,
                                                               const double* __restrict__ window,
                                                               const Complex* __restrict__ roots,
                                                               const float* __restrict__ mel_w,
                                                               const int* __restrict__ mel_lo,
                                                               const int* __restrict__ mel_len, int max_len,
                                                               float* __restrict__ out, int S, int F, int R) {
  __shared__ float power[kSpBlock][kBins + 3];
  __shared__ __attribute__((aligned(16))) Complex points[kSpWaves][kPoints + kPoints / 16];
  const int lane = threadIdx.x & 63;
  const int w = threadIdx.x >> 6;
  const int f0 = blockIdx.x * kSpBlock;
  float in[kSpFrames][4][3];  // samples 2n - 1, 2n, 2n + 1 of points n = lane + 64 r
#pragma unroll
  for (int q = 0; q < kSpFrames; ++q) {
    const int row = __builtin_amdgcn_readfirstlane(min(f0 + w * kSpFrames + q, R - 1));
    const int b = row / F;
    const int t0 = (row - b * F) * kFrameShift - kEdgePad;
    const float* src = chunk + (int64_t)b * S;
    if (t0 > 0 && t0 + kFrameSize <= S) {  // wave-uniform: all but an item's first and last frames
      const float* at = src + t0 + 2 * lane;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool ok = r < 3 || lane < kFrameSize / 2 - 192;
        in[q][r][1] = ok ? at[128 * r] : 0.f;
        in[q][r][2] = ok ? at[128 * r + 1] : 0.f;
        in[q][r][0] = ok ? at[128 * r - 1] : 0.f;
      }
      if (lane == 0) in[q][0][0] = in[q][0][1];  // the first sample is its own predecessor
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          const int n = max(2 * (lane + 64 * r) + i - 1, 0);
          const int t = t0 + n;
          in[q][r][i] = n < kFrameSize && t >= 0 && t < S ? src[t] : 0.f;
        }
    }
  }
  // Per lane: window of its samples, twiddles of passes 2-4, roots of its bins.
  Complex win[4], tw[3][3], root[2];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int n = 2 * (lane + 64 * r);
    win[r] = n < kFrameSize ? Complex{window[n], window[n + 1]} : Complex{0., 0.};
  }
#pragma unroll
  for (int p = 0; p < 3; ++p)
#pragma unroll
    for (int r = 1; r < 4; ++r) tw[p][r - 1] = roots[(lane & ((4 << (2 * p)) - 1)) * r * (128 >> (2 * p + 2))];
#pragma unroll
  for (int r = 0; r < 2; ++r) root[r] = roots[lane + 64 * r];

  Complex* own = points[w];
  Complex v[kSpFrames][4];
  // An infinite sample makes every power infinite, and so the item's features NaN,
  // as in a product with the transform matrix; the FFT alone gives NaN powers, which
  // the floor of the log would take for silence.
  bool infinite[kSpFrames];
#pragma unroll
  for (int q = 0; q < kSpFrames; ++q) {
    double s = 0.;
#pragma unroll
    for (int r = 0; r < 4; ++r) s += (double)in[q][r][1] + (double)in[q][r][2];
    const double mean = sidon::wave_sum(s) * (1. / kFrameSize);
    infinite[q] = __builtin_isinf(mean);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const double before = in[q][r][0] - mean, x0 = in[q][r][1] - mean, x1 = in[q][r][2] - mean;
      v[q][r] = {fma(-kPreemph, before, x0) * win[r].x, fma(-kPreemph, x0, x1) * win[r].y};
    }
    radix4(v[q]);
  }
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    const int ns = 1 << (2 * p);
    const int to = (lane / ns) * 4 * ns + (lane & (ns - 1));
#pragma unroll
    for (int q = 0; q < kSpFrames; ++q) {
#pragma unroll
      for (int r = 0; r < 4; ++r) own[spread(to + r * ns)] = v[q][r];
      lds_in_order();
#pragma unroll
      for (int r = 0; r < 4; ++r) v[q][r] = own[spread(lane + 64 * r)];
      lds_in_order();
    }
#pragma unroll
    for (int q = 0; q < kSpFrames; ++q) {
#pragma unroll
      for (int r = 1; r < 4; ++r) v[q][r] = cmul(v[q][r], tw[p][r - 1]);
      radix4(v[q]);
    }
  }
  // Z[lane + 64 r] = v[r]; the partners Z[256 - k] of k = lane, lane + 64 lie
  // in lane (64 - lane) % 64, registers 3 and 2 (lane 0: Z[0] and Z[192]).
  const int mirror = (64 - lane) & 63;
#pragma unroll
  for (int q = 0; q < kSpFrames; ++q) {
    own[lane] = v[q][3];
    own[64 + lane] = v[q][2];
    lds_in_order();
    const Complex p3 = own[mirror], p2 = own[64 + mirror];
    lds_in_order();
    float* dst = power[w * kSpFrames + q];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const Complex z = v[q][r];
      const Complex c = lane == 0 ? (r == 0 ? z : p3) : (r == 0 ? p3 : p2);
      const Complex e = {0.5 * (z.x + c.x), 0.5 * (z.y - c.y)}, o = {0.5 * (z.x - c.x), 0.5 * (z.y + c.y)};
      const Complex u = cmul(o, root[r]);
      const Complex lo = {e.x + u.y, e.y - u.x}, hi = {e.x - u.y, e.y + u.x};
      dst[lane + 64 * r] = power_of(lo, infinite[q]);
      dst[kPoints - lane - 64 * r] = power_of(hi, infinite[q]);
    }
    if (lane == 0) dst[128] = power_of(v[q][2], infinite[q]);
  }
  __syncthreads();
  mel_log<kSpBlock, kSpLanes>(power, mel_w, mel_lo, mel_len, max_len, out, f0, R);
}

// True frames of the exact-length extractor for `samples` valid samples:
// 1 + (samples + 2 * 160 - 400) / 160 (floor), clamped to [0, F].
__device__ __forceinline__ int true_frames(int samples, int F) {
  const int t = samples + 2 * kEdgePad - kFrameSize;
  const int n = t < 0 ? 0 : t / kFrameShift + 1;
  return min(n, F);
}

// Block (tile g, item b): two-pass sums over the true frames of tile g.
__global__ void __launch_bounds__(kLanes * kMel) stats_kernel(const float* __restrict__ x,
                                                             const int* __restrict__ valid,
                                                             float* __restrict__ part, int F, int G) {
  __shared__ float red[kLanes][kMel];
  const int b = blockIdx.y;
  const int g = blockIdx.x;
  const int m = threadIdx.x % kMel;
  const int fl = threadIdx.x / kMel;
  const int tf = true_frames(valid[b], F);
  const int per = (F + G - 1) / G;
  const int f0 = g * per;
  const int f1 = min(f0 + per, tf);
  const int n = max(f1 - f0, 0);
  const float* xb = x + (int64_t)b * F * kMel;
  // Tiles of up to kLanes * kStatsCache frames are held in registers, loaded
  // in one round (one memory latency for both passes); longer tiles stream.
  // Either way the sums run over f = f0 + fl, f0 + fl + kLanes, ... in order.
  // (The loads cover the tile's frames, true or not: they do not wait for valid.)
  const int nl = f1 > f0 + fl ? (f1 - f0 - fl + kLanes - 1) / kLanes : 0;
  const int tile = min(f0 + per, F) - f0 - fl;
  float xv[kStatsCache];
  const bool cached = per <= kLanes * kStatsCache;
  if (cached) {
#pragma unroll
    for (int j = 0; j < kStatsCache; ++j)
      xv[j] = kLanes * j < tile ? xb[(int64_t)(f0 + fl + kLanes * j) * kMel + m] : 0.f;
  }
  float s = 0.f;
  if (cached) {
#pragma unroll
    for (int j = 0; j < kStatsCache; ++j)
      if (j < nl) s += xv[j];
  } else {
#pragma unroll 8
    for (int f = f0 + fl; f < f1; f += kLanes) s += xb[(int64_t)f * kMel + m];
  }
  red[fl][m] = s;
  __syncthreads();
  const float mean = n > 0 ? ((red[0][m] + red[1][m]) + (red[2][m] + red[3][m])) / (float)n : 0.f;
  __syncthreads();
  float q = 0.f;
  if (cached) {
#pragma unroll
    for (int j = 0; j < kStatsCache; ++j) {
      if (j < nl) {
        const float d = xv[j] - mean;
        q = fmaf(d, d, q);
      }
    }
  } else {
#pragma unroll 8
    for (int f = f0 + fl; f < f1; f += kLanes) {
      const float d = xb[(int64_t)f * kMel + m] - mean;
      q = fmaf(d, d, q);
    }
  }
  red[fl][m] = q;
  __syncthreads();
  if (fl == 0) {
    float* dst = part + ((int64_t)b * G + g) * kTileFloats + m;
    dst[0] = mean;
    dst[kMel] = (red[0][m] + red[1][m]) + (red[2][m] + red[3][m]);
  }
}

// (count, mean, sum of squared deviations) of the union of two sets of frames
// (Chan et al.'s update).
struct Moments {
  float n, mean, m2;
};

__device__ __forceinline__ Moments join(const Moments& a, const Moments& b) {
  const float n = a.n + b.n;
  const float d = b.mean - a.mean;
  const float share = b.n > 0.f ? b.n / n : 0.f;   // an empty set's m2 is 0
  const float mean = a.n > 0.f ? a.mean + d * share : b.mean;
  return {n, mean, a.m2 + b.m2 + d * d * (a.n * share)};
}

// Block (frame range, item b): merge the item's tile sums, then normalize the
// range's frames.  Every block merges for itself (41 KB out of L2, all loads in
// flight at once) instead of waiting for a launch that does it (5.5 us); a
// branch around each tile's loads cost 1.8 us.
// Thread (m, fl) joins tiles 16 fl .. 16 fl + 15 of bin m pairwise, LDS the
// four results: the same tree in every block and call.
__global__ void __launch_bounds__(kLanes * kMel) apply_kernel(const float* __restrict__ x,
                                                             const int* __restrict__ valid,
                                                             const float* __restrict__ part,
                                                             float* __restrict__ out, int F, int G) {
  constexpr int kOwn = kMaxTiles / kLanes;
  __shared__ Moments quarter[kLanes][kMel];
  const int b = blockIdx.y;
  const int m = threadIdx.x % kMel;
  const int fl = threadIdx.x / kMel;
  const int tf = true_frames(valid[b], F);
  const float* xb = x + (int64_t)b * F * kMel;
  float* ob = out + (int64_t)b * F * kMel;
  const int fbase = blockIdx.x * kApplyFrames;
  // All of the thread's loads first (one memory latency), then the stores.
  constexpr int kPer = kApplyFrames / kLanes;
  float x_in[kPer];
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int f = fbase + fl + kLanes * j;
    x_in[j] = f < F ? xb[(int64_t)f * kMel + m] : 0.f;  // not waiting for valid: frames past tf are dropped below
  }
  Moments own[kOwn];
  const int per = (F + G - 1) / G;  // frames of a tile, as in stats_kernel
#pragma unroll
  for (int j = 0; j < kOwn; ++j) {
    const int g = kOwn * fl + j;
    const float* src = part + ((int64_t)b * G + min(g, G - 1)) * kTileFloats + m;  // no branch between the loads
    own[j] = Moments{g < G ? (float)max(min(per, tf - g * per), 0) : 0.f, src[0], g < G ? src[kMel] : 0.f};
  }
#pragma unroll
  for (int stride = 1; stride < kOwn; stride *= 2)
#pragma unroll
    for (int j = 0; j + stride < kOwn; j += 2 * stride) own[j] = join(own[j], own[j + stride]);
  quarter[fl][m] = own[0];
  __syncthreads();
  const Moments all = join(join(quarter[0][m], quarter[1][m]), join(quarter[2][m], quarter[3][m]));
  const float denom = sqrtf(all.m2 / (float)(tf - 1) + kVarEps);
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int f = fbase + fl + kLanes * j;
    if (f < F) {
      const float v = f < tf ? (x_in[j] - all.mean) / denom : ((f == tf && (tf & 1)) ? kPadValue : 0.f);
      ob[(int64_t)f * kMel + m] = v;
    }
  }
}

int tiles_for(int F) { return F / 128 < 1 ? 1 : (F / 128 > kMaxTiles ? kMaxTiles : F / 128); }

// Scratch of sidon_fbank_normalize_noalloc: the normalize workspace of up
// to kScratchItems items of any length (tiles_for() caps the tiles at
// kMaxTiles), 1.3 MiB in all, one copy per device for the life of the
// process.  Every word a call reads was written earlier in the same call, so
// nothing needs clearing between calls.
constexpr int kScratchItems = 32;
constexpr size_t kScratchFloats = (size_t)kScratchItems * kMaxTiles * kTileFloats;
static __device__ __align__(256) float scratch[kScratchFloats];

// Device address of `scratch` per device, taken once per device with that
// device current (host code must never pass the symbol itself to a kernel).
constexpr int kMaxDevices = 64;
std::once_flag g_scratch_once[kMaxDevices];
float* g_scratch[kMaxDevices] = {};
hipError_t g_scratch_err[kMaxDevices] = {};

int normalize_launch(const float* logmel, const int* valid, float* workspace, float* feats, int B, int F,
                     hipStream_t s) {
  using sidon::fail;
  const int G = tiles_for(F);
  hipLaunchKernelGGL(stats_kernel, dim3(G, B), dim3(kLanes * kMel), 0, s, logmel, valid, workspace, F, G);
  hipError_t err = hipGetLastError();
  if (err == hipSuccess) {
    hipLaunchKernelGGL(apply_kernel, dim3((F + kApplyFrames - 1) / kApplyFrames, B), dim3(kLanes * kMel), 0, s,
                       logmel, valid, workspace, feats, F, G);
    err = hipGetLastError();
  }
  if (err != hipSuccess) return fail(SIDON_E_LAUNCH, "fbank normalize launch failed: %s", hipGetErrorString(err));
  return SIDON_OK;
}

}  // namespace

SIDON_API int sidon_fbank_logmel(const float* spec, const float* mel_w, const int* mel_lo, const int* mel_len,
                                 int max_len, float* logmel, int R, sidon_stream_t stream) {
  using sidon::fail;
  sidon::clear_error();
  if (!spec || !mel_w || !mel_lo || !mel_len || !logmel) return fail(SIDON_E_NULL, "every pointer must be non-NULL");
  if (R < 1 || max_len < 1 || max_len > kBins) return fail(SIDON_E_SHAPE, "R=%d must be >= 1 and max_len=%d in [1, %d]", R, max_len, kBins);
  int rc;
  if ((rc = sidon::check_device())) return rc;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(logmel_kernel, dim3((unsigned)((R + kLmFrames - 1) / kLmFrames)), dim3(kLmThreads), 0, s, spec,
                     mel_w, mel_lo, mel_len, max_len, logmel, R);
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return fail(SIDON_E_LAUNCH, "fbank logmel launch failed: %s", hipGetErrorString(err));
  return SIDON_OK;
}

SIDON_API int sidon_fbank_frames(const float* chunk, float* frames, int B, int S, sidon_stream_t stream) {
  using sidon::fail;
  sidon::clear_error();
  if (!chunk || !frames) return fail(SIDON_E_NULL, "chunk and frames must be non-NULL");
  if (B < 1 || S < 2 * kFrameShift || S % (2 * kFrameShift) != 0)
    return fail(SIDON_E_SHAPE, "B=%d must be >= 1 and S=%d a positive multiple of %d", B, S, 2 * kFrameShift);
  if (!sidon::aligned16(frames)) return fail(SIDON_E_ALIGN, "frames must be 16-byte aligned");
  int rc;
  if ((rc = sidon::check_device())) return rc;
  const int F = S / kFrameShift;
  // 16-byte source loads when every item's row starts 16-byte aligned (S is a
  // multiple of 320, so that holds when the chunk pointer is aligned).
  const bool vec4 = sidon::aligned16(chunk);
  const unsigned blocks = (unsigned)(((int64_t)F * (kFrameSize / 4) + 255) / 256);
  for (int b0 = 0; b0 < B; b0 += 65535) {  // items on grid y, at most 65535 per launch
    const int nb = B - b0 < 65535 ? B - b0 : 65535;
    hipLaunchKernelGGL(frames_kernel, dim3(blocks, (unsigned)nb), dim3(256), 0, reinterpret_cast<hipStream_t>(stream),
                       chunk + (int64_t)b0 * S, frames + (int64_t)b0 * F * kFrameSize, S, F, vec4);
  }
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return fail(SIDON_E_LAUNCH, "fbank frames launch failed: %s", hipGetErrorString(err));
  return SIDON_OK;
}

SIDON_API int sidon_fbank_features(const float* chunk, const int* valid, const double* window, const double* roots,
                                   const float* mel_w, const int* mel_lo, const int* mel_len, int max_len,
                                   float* logmel, float* workspace, size_t workspace_bytes, float* feats, int B,
                                   int S, sidon_stream_t stream) {
  using sidon::fail;
  sidon::clear_error();
  if (!chunk || !valid || !window || !roots || !mel_w || !mel_lo || !mel_len || !logmel || !workspace || !feats)
    return fail(SIDON_E_NULL, "every pointer must be non-NULL");
  if (B < 1 || S < 2 * kFrameShift || S % (2 * kFrameShift) != 0)
    return fail(SIDON_E_SHAPE, "B=%d must be >= 1 and S=%d a positive multiple of %d", B, S, 2 * kFrameShift);
  if (max_len < 1 || max_len > kBins) return fail(SIDON_E_SHAPE, "max_len=%d in [1, %d]", max_len, kBins);
  const int F = S / kFrameShift;
  if ((int64_t)B * F > INT32_MAX - kSpBlock) return fail(SIDON_E_SHAPE, "B=%d items of %d frames are too many", B, F);
  if (workspace_bytes < sidon_fbank_workspace_bytes(B, F))
    return fail(SIDON_E_SHAPE, "workspace of %zu bytes is smaller than the %zu needed", workspace_bytes,
                sidon_fbank_workspace_bytes(B, F));
  if (logmel == feats) return fail(SIDON_E_SHAPE, "feats must not alias logmel");
  if (!sidon::aligned16(roots) || !sidon::aligned16(window))
    return fail(SIDON_E_ALIGN, "window and roots must be 16-byte aligned");
  int rc;
  if ((rc = sidon::check_device())) return rc;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int R = B * F;
  hipLaunchKernelGGL(spectrum_kernel, dim3((unsigned)((R + kSpBlock - 1) / kSpBlock)), dim3(64 * kSpWaves), 0, s,
                     chunk, window, reinterpret_cast<const Complex*>(roots), mel_w, mel_lo, mel_len, max_len, logmel,
                     S, F, R);
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return fail(SIDON_E_LAUNCH, "fbank spectrum launch failed: %s", hipGetErrorString(err));
  return normalize_launch(logmel, valid, workspace, feats, B, F, s);
}

SIDON_API size_t sidon_fbank_workspace_bytes(int B, int F) {
  if (B < 1 || F < 1) return 0;
  return (size_t)B * tiles_for(F) * kTileFloats * sizeof(float);
}

SIDON_API int sidon_fbank_normalize(const float* logmel, const int* valid, float* workspace, size_t workspace_bytes,
                                    float* feats, int B, int F, sidon_stream_t stream) {
  using sidon::fail;
  sidon::clear_error();
  if (!logmel || !valid || !workspace || !feats) return fail(SIDON_E_NULL, "every pointer must be non-NULL");
  if (B < 1 || F < 2 || (F & 1) != 0) return fail(SIDON_E_SHAPE, "B=%d must be >= 1 and F=%d even and >= 2", B, F);
  if (workspace_bytes < sidon_fbank_workspace_bytes(B, F))
    return fail(SIDON_E_SHAPE, "workspace of %zu bytes is smaller than the %zu needed", workspace_bytes,
                sidon_fbank_workspace_bytes(B, F));
  if (logmel == feats) return fail(SIDON_E_SHAPE, "feats must not alias logmel");
  int rc;
  if ((rc = sidon::check_device())) return rc;
  return normalize_launch(logmel, valid, workspace, feats, B, F, reinterpret_cast<hipStream_t>(stream));
}

SIDON_API int sidon_fbank_normalize_noalloc(const float* logmel, const int* valid, float* feats, int B, int F,
                                            sidon_stream_t stream) {
  using sidon::fail;
  sidon::clear_error();
  if (!logmel || !valid || !feats) return fail(SIDON_E_NULL, "every pointer must be non-NULL");
  if (B < 1 || F < 2 || (F & 1) != 0) return fail(SIDON_E_SHAPE, "B=%d must be >= 1 and F=%d even and >= 2", B, F);
  if (B > kScratchItems || sidon_fbank_workspace_bytes(B, F) > sizeof(scratch))
    return fail(SIDON_E_SHAPE, "B=%d items exceed the %d the static scratch holds (use sidon_fbank_normalize)", B,
                kScratchItems);
  if (logmel == feats) return fail(SIDON_E_SHAPE, "feats must not alias logmel");
  int rc;
  if ((rc = sidon::check_device())) return rc;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return fail(SIDON_E_DEVICE, "no usable HIP device");
  std::call_once(g_scratch_once[dev], [dev]() {
    void* ptr = nullptr;
    g_scratch_err[dev] = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    g_scratch[dev] = g_scratch_err[dev] == hipSuccess ? static_cast<float*>(ptr) : nullptr;
  });
  if (g_scratch[dev] == nullptr)
    return fail(SIDON_E_DEVICE, "hipGetSymbolAddress(scratch) failed on device %d: %s", dev,
                hipGetErrorString(g_scratch_err[dev]));
  return normalize_launch(logmel, valid, g_scratch[dev], feats, B, F, reinterpret_cast<hipStream_t>(stream));
}
