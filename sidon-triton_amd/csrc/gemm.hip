// gemm.hip -- the encoder's fp16 projections on the tiled GEMM kernel of
// gemm_tile.h (MI355X / gfx950): the host side that checks arguments, picks
// the tile shape and the K split, and launches.
//
//   sidon_gemm_bias_act   y = act(fp16(x . w^T + bias))            feed-forward input, two roundings
//   sidon_gemm_lt_act     y = act(x . w^T + bias), one rounding    (blaslt.hip calls gemm_half below)
//   sidon_gemm_glu        y = a . sigmoid(b), (a | b) = x . w^T    pointwise conv 1 + GLU
//   sidon_gemm_res        y += x . w^T, fp32 in place              residual projections
//   sidon_gemm_part       partial sums of x . w^T, K split         the same, summed by the next norm
//
// These are the GEMMs of src/sidon_triton/triton_encoder.py:491-510 (with the
// F.silu_ of :499 / :508 and the GLU of :505 taken in the epilogue).
//
// Tile choice.  A launch of n tiles takes about
//
//   3.0 + load (0.062 nk mm + 0.031 nk + e mm) + 0.065 (n / CUs) nk cp   us
//
// with load = ceil(n / CUs) tiles on the busiest CU, nk 64-wide K slices per
// tile, mm = BM BN / 4096 its MFMA work, cp = (BM + BN) / 64 its copy
// traffic and e = 0.39 (fp16 out) or 0.48 (fp32 out): fitted to 1400 timings
// of the encoder's five projections at M = 25-4800 with weights from HBM
// (rms 9%).  The tile with the least estimate is taken; it is 0-3% (mean per
// projection) slower than the best one measured.  A K split costs the norm
// behind it its partial tiles and the stream's write on top, at 7-11 TB/s
// (N = 1024: 4 splits at M = 750 1.4 us, 2 at 1600 2.3, 2 at 3000 5.7).
//
// Measured on MI355X (weights from HBM, graph replays, us), own | library:
//   M =                          150          750          1600         4800
//   4096 x 1024 + bias + SiLU    7.5 | 12.0+  12.3 | 14.3+ 20.4 | 22.3+ 47.0 | 47.0+  (library without SiLU)
//   3072 x 1024 + bias           6.2 |  9.7    9.7 | 12.8  15.0 | 17.7  35.4 | 30.9
//   2048 x 1024 + GLU            5.3 |  8.6+   6.8 |  9.7+ 10.3 | 13.2+ 23.3 | 30.6+  (library without GLU)
//   1024 x 4096 fp32, split K    6.9 | 12.3   12.3 | 20.8  19.7 | 27.5  45.4 | 48.7 (4800: in place)
//   1024 x 1024 fp32             4.0 |  8.1    6.1 |  9.0   8.0 | 11.0  17.3 | 18.4 (split at 150, else in place)
#include "gemm_tile.h"

#include "sidon_encoder.h"
#include "sidon_host.h"

#define SIDON_API extern "C" __attribute__((visibility("default")))

namespace {

using namespace sidon_gemm;
using sidon::fail;

typedef void (*KernelFn)(TileParams);

struct TileKernel {
  int bm, bn, threads;
  KernelFn fn[4];  // by epilogue; null where that epilogue has no use for the shape
};

#define SIDON_TILE(BM, BN, WM, WN, MF, ST, GLU, F32)                                       \
  {BM, BN, 64 * WM * WN,                                                                   \
   {gemm_tile_kernel<BM, BN, WM, WN, MF, ST, kHalf>, GLU(BM, BN, WM, WN, MF, ST, kGlu),    \
    F32(BM, BN, WM, WN, MF, ST, kPart), F32(BM, BN, WM, WN, MF, ST, kAdd)}}
#define SIDON_HAS(BM, BN, WM, WN, MF, ST, MODE) gemm_tile_kernel<BM, BN, WM, WN, MF, ST, MODE>
#define SIDON_NOT(BM, BN, WM, WN, MF, ST, MODE) nullptr

// The shapes that some measured (M, N, K) needs: a mean of 0.3% over the best
// of 22 shapes.  One workgroup of the larger ones fills a CU's LDS.  256 wide
// ones only where an fp16 output is wide enough to need them.
const TileKernel kTiles[] = {
    SIDON_TILE(32, 64, 2, 2, 16, 6, SIDON_HAS, SIDON_HAS),
    SIDON_TILE(64, 64, 2, 2, 16, 4, SIDON_HAS, SIDON_HAS),
    SIDON_TILE(96, 64, 2, 2, 16, 4, SIDON_HAS, SIDON_HAS),
    SIDON_TILE(128, 64, 4, 2, 16, 4, SIDON_HAS, SIDON_HAS),
    SIDON_TILE(160, 64, 2, 2, 16, 4, SIDON_HAS, SIDON_HAS),
    SIDON_TILE(64, 128, 2, 4, 16, 4, SIDON_HAS, SIDON_HAS),
    SIDON_TILE(96, 128, 2, 2, 16, 4, SIDON_HAS, SIDON_HAS),
    SIDON_TILE(128, 128, 2, 4, 16, 4, SIDON_HAS, SIDON_HAS),
    SIDON_TILE(160, 128, 2, 2, 16, 3, SIDON_HAS, SIDON_HAS),
    SIDON_TILE(192, 128, 2, 4, 16, 3, SIDON_HAS, SIDON_HAS),
    SIDON_TILE(128, 256, 2, 4, 16, 3, SIDON_HAS, SIDON_NOT),
    SIDON_TILE(160, 256, 1, 4, 32, 3, SIDON_HAS, SIDON_NOT),
    SIDON_TILE(192, 256, 2, 4, 16, 2, SIDON_NOT, SIDON_NOT),
    SIDON_TILE(256, 256, 2, 4, 16, 2, SIDON_NOT, SIDON_NOT),
    SIDON_TILE(320, 256, 2, 4, 32, 2, SIDON_NOT, SIDON_NOT),
};

constexpr int kMaxSplits = 8;        // what the norm sums in one pass
constexpr int kGroupM = 8;           // row tiles walked together (level with 4, better from M = 1600 on)
// The partial tiles of a split projection hold at most this many rows in
// all (splits x M), so that a caller's workspace is bounded.
constexpr int64_t kMaxPartRows = 8192;

struct Choice {
  const TileKernel* tile = nullptr;
  int splits = 1;
  double us = 0;
};

Choice search(int M, int N, int K, int mode, int max_splits, int cus) {
  const int slices = K / 64;
  Choice best;
  for (const TileKernel& t : kTiles) {
    if (t.fn[mode] == nullptr || N % t.bn != 0) continue;
    const int64_t tiles = (int64_t)((M + t.bm - 1) / t.bm) * (N / t.bn);
    const double mm = t.bm * t.bn / 4096.0, cp = (t.bm + t.bn) / 64.0;
    for (int s = 1; s <= max_splits; ++s) {
      // At least two slices per split, and the splits of one round of CUs.
      if (s > 1 && (2 * s > slices || tiles * s > cus || (int64_t)s * M > kMaxPartRows)) break;
      const double n = (double)tiles * s;
      const double load = (double)((tiles * s + cus - 1) / cus);
      const double nk = (double)slices / s;
      double us = 3.0 + load * (0.062 * nk * mm + 0.031 * nk + (mode <= kGlu ? 0.39 : 0.48) * mm) +
                  0.065 * (n / cus) * nk * cp;
      if (s > 1) us += (s + 1.0) * M * N * 4.0 / 8e6;  // partial tiles read back, the stream written by the norm
      if (best.tile == nullptr || us < best.us) best = Choice{&t, s, us};
    }
  }
  return best;
}

// The search (a few microseconds) once per shape: an encoder call asks for the
// same few again and again.  One table per thread, the newest shape kept.
Choice choose(int M, int N, int K, int mode, int max_splits) {
  struct Entry {
    int M, N, K, mode, max_splits, cus;
    Choice choice;
  };
  constexpr unsigned kEntries = 32;
  static thread_local Entry table[kEntries] = {};
  const int cus = sidon::compute_units();
  const unsigned hash = ((unsigned)M * 2654435761u ^ (unsigned)N * 40503u ^ (unsigned)K * 97u ^ (unsigned)mode) >> 7;
  Entry& e = table[hash % kEntries];
  if (e.M != M || e.N != N || e.K != K || e.mode != mode || e.max_splits != max_splits || e.cus != cus)
    e = Entry{M, N, K, mode, max_splits, cus, search(M, N, K, mode, max_splits, cus)};
  return e.choice;
}

// Operands as the kernel's 16-byte copies and 32-bit offsets need them.
bool operands_fit(int64_t M, int64_t N, int ldx, int ldw, const void* x, const void* w) {
  return ldx % 8 == 0 && ldw % 8 == 0 && M * ldx * 2 < (int64_t(1) << 32) && N * ldw * 2 < (int64_t(1) << 32) &&
         sidon::aligned16(x) && sidon::aligned16(w);
}

int launch(const Choice& c, int mode, TileParams p, hipStream_t stream, const char* what) {
  p.tiles_m = (p.M + c.tile->bm - 1) / c.tile->bm;
  p.tiles_n = p.N / c.tile->bn;
  p.splits = c.splits;
  p.group = p.tiles_m < kGroupM ? p.tiles_m : kGroupM;
  const int64_t wgs = (int64_t)p.tiles_m * p.tiles_n * p.splits;
  if (wgs >= (int64_t(1) << 31)) return fail(SIDON_E_SHAPE, "too many tiles");
  hipLaunchKernelGGL(c.tile->fn[mode], dim3((unsigned)wgs), dim3(c.tile->threads), 0, stream, p);
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return fail(SIDON_E_LAUNCH, "%s launch failed: %s", what, hipGetErrorString(err));
  return SIDON_OK;
}

TileParams params(const void* x, int ldx, const void* w, int ldw, const void* bias, void* y, int ldy, int M, int N,
                  int K, int act) {
  TileParams p{};
  p.x = static_cast<const _Float16*>(x);
  p.w = static_cast<const _Float16*>(w);
  p.bias = static_cast<const _Float16*>(bias);
  p.y = y;
  p.ldx = ldx;
  p.ldw = ldw;
  p.ldy = ldy;
  p.M = M;
  p.N = N;
  p.K = K;
  p.act = act;
  return p;
}

bool res_fits(int M, int N, int K) { return M >= 1 && N >= 64 && N % 64 == 0 && K >= 128 && K % 128 == 0; }

// Whether the byte ranges of x [M, K] or w [N, K] and of y (rows of
// `y_row` bytes, ldy_bytes apart) overlap: workgroups read X and W while
// others already write Y.
bool overlaps(const void* x, int ldx, const void* w, int ldw, const void* y, int64_t ldy_bytes, int64_t y_row, int M,
              int N, int K) {
  const uintptr_t xb = reinterpret_cast<uintptr_t>(x), wb = reinterpret_cast<uintptr_t>(w);
  const uintptr_t yb = reinterpret_cast<uintptr_t>(y);
  const uintptr_t xe = xb + (uintptr_t)(((int64_t)(M - 1) * ldx + K) * 2);
  const uintptr_t we = wb + (uintptr_t)(((int64_t)(N - 1) * ldw + K) * 2);
  const uintptr_t ye = yb + (uintptr_t)((int64_t)(M - 1) * ldy_bytes + y_row);
  return (xb < ye && yb < xe) || (wb < ye && yb < we);
}

// Few outputs of a long K: a handful of workgroups that walk all of it, where the
// library's kernels are faster (us, this kernel | library: 150 x 256 x 4096 11.7 |
// 8.3, 150 x 1024 x 4096 15.2 | 12.3, x 8192 26.3 | 20.2, but 400 x 1024 x 4096 level).
bool few_of_long_k(int M, int N, int K) { return (int64_t)M * N <= 1 << 18 && K > 2048; }

}  // namespace

namespace sidon {

// Up to here the kernel is faster than hipBLASLt at every measured shape;
// past it the library's 256 x 256 kernels win (M x 3072 x 1024: M = 3000 23.9
// against 30.8 us, 3600 30.5 against 27.6; M x 4096: 2000 23.0 against 24.1
// without its SiLU, 3000 32.9 against 28.7).
bool gemm_half_preferred(int M, int N, int K) {
  return M >= 1 && N >= 64 && N % 64 == 0 && K >= 64 && K % 64 == 0 && (int64_t)M * N <= (int64_t)9 << 20 &&
         !few_of_long_k(M, N, K);
}

bool gemm_half_takes(const void* x, int ldx, const void* w, int ldw, const void* bias, const void* y, int ldy, int M,
                     int N, int K) {
  return gemm_half_preferred(M, N, K) && operands_fit(M, N, ldx, ldw, x, w) && ldy % 8 == 0 && aligned16(y) &&
         (reinterpret_cast<uintptr_t>(bias) & 7u) == 0 &&
         !overlaps(x, ldx, w, ldw, y, (int64_t)ldy * 2, (int64_t)N * 2, M, N, K);
}

int gemm_half(const void* x, int ldx, const void* w, int ldw, const void* bias, void* y, int ldy, int M, int N, int K,
              int act, void* stream) {
  return launch(choose(M, N, K, kHalf, 1), kHalf,
                params(x, ldx, w, ldw, bias, y, ldy, M, N, K, act == 1 ? kSilu : kNone),
                reinterpret_cast<hipStream_t>(stream), "gemm");
}

}  // namespace sidon

SIDON_API int sidon_gemm_choice(int M, int N, int K, int epilogue, int max_splits, int cus, int* bm, int* bn) {
  if (M < 1 || N < 64 || N % 64 != 0 || K < 64 || K % 64 != 0 || epilogue < kHalf || epilogue > kAdd || cus < 1) return 0;
  if (max_splits < 1 || max_splits > kMaxSplits || (epilogue != kPart && max_splits != 1)) return 0;
  const Choice c = search(M, N, K, epilogue, max_splits, cus);
  if (bm != nullptr) *bm = c.tile->bm;
  if (bn != nullptr) *bn = c.tile->bn;
  return c.splits;
}

SIDON_API int sidon_gemm_bias_act_fits(int M, int N, int K) {
  return M >= 1 && N >= 256 && N % 256 == 0 && K >= 64 && K % 64 == 0 ? 1 : 0;
}

// Past gemm_half_preferred's range, where 320 x 256 tiles would keep four fifths
// of the CUs busy in every round (the tile that then runs is the cost rule's: 256 x
// 256 up to 4096 rows).  M x 4096 x 1024, us, own | the library with the SiLU in
// its epilogue: 3400 35.0 | 32.2, 3700 36.3 | 34.2, 4097 42.3 | 47.3, 4200 43.7 | 63.0,
// 4800 46.1 | 50.4.  From 3841 to 4096 rows the line is generous (37.5 | 33.9).
SIDON_API int sidon_gemm_bias_act_preferred(int M, int N, int K) {
  if (!sidon_gemm_bias_act_fits(M, N, K)) return 0;
  if (sidon::check_device() != SIDON_OK) return 0;
  const int64_t tiles = (int64_t)((M + 319) / 320) * (N / 256);
  const int64_t cus = sidon::compute_units();
  const int64_t rounds = (tiles + cus - 1) / cus;
  return !sidon::gemm_half_preferred(M, N, K) && 5 * tiles >= 4 * rounds * cus ? 1 : 0;
}

SIDON_API int sidon_gemm_bias_act(const void* x, int ldx, const void* w, int ldw, const void* bias, void* y, int ldy,
                                  int M, int N, int K, int act, sidon_stream_t stream) {
  sidon::clear_error();
  if (!x || !w || !y) return fail(SIDON_E_NULL, "x, w and y must be non-NULL");
  if (!sidon_gemm_bias_act_fits(M, N, K))
    return fail(SIDON_E_SHAPE, "M=%d N=%d K=%d: need M >= 1, N a multiple of 256, K a multiple of 64", M, N, K);
  if (ldx < K || ldw < K || ldy < N || (ldx | ldw | ldy) % 8 != 0)
    return fail(SIDON_E_STRIDE, "row strides ldx=%d ldw=%d ldy=%d must be multiples of 8 and >= K, K, N", ldx, ldw,
                ldy);
  if ((int64_t)M * ldx * 2 >= (int64_t(1) << 32) || (int64_t)N * ldw * 2 >= (int64_t(1) << 32))
    return fail(SIDON_E_SHAPE, "X and W must each span less than 4 GiB");
  if (act != 0 && act != 1) return fail(SIDON_E_SHAPE, "act=%d: 0 (none) or 1 (SiLU)", act);
  if (!sidon::aligned16(x) || !sidon::aligned16(w) || !sidon::aligned16(y) || (bias && ((uintptr_t)bias & 7) != 0))
    return fail(SIDON_E_ALIGN, "x, w, y must be 16-byte aligned and bias 8-byte aligned");
  int rc;
  if ((rc = sidon::check_device())) return rc;
  return launch(choose(M, N, K, kHalf, 1), kHalf,
                params(x, ldx, w, ldw, bias, y, ldy, M, N, K, act == 1 ? kSiluHalf : kNone),
                reinterpret_cast<hipStream_t>(stream), "gemm");
}

SIDON_API int sidon_gemm_half_preferred(int M, int N, int K) {
  if (!sidon::gemm_half_preferred(M, N, K)) return 0;
  return sidon::check_device() == SIDON_OK ? 1 : 0;
}

SIDON_API int sidon_gemm_half_takes(const void* x, int ldx, const void* w, int ldw, const void* bias, const void* y,
                                    int ldy, int M, int N, int K) {
  return ldx >= K && ldw >= K && ldy >= N && sidon::gemm_half_takes(x, ldx, w, ldw, bias, y, ldy, M, N, K) ? 1 : 0;
}

SIDON_API int sidon_gemm_glu(const void* x, int ldx, const void* w, int ldw, void* y, int ldy, int M, int C, int K,
                             sidon_stream_t stream) {
  sidon::clear_error();
  if (!x || !w || !y) return fail(SIDON_E_NULL, "x, w and y must be non-NULL");
  if (M < 1 || C < 32 || C % 32 != 0 || C > (1 << 29) || K < 64 || K % 64 != 0)
    return fail(SIDON_E_SHAPE, "M=%d C=%d K=%d: need M >= 1, C a multiple of 32, K a multiple of 64", M, C, K);
  if (ldx < K || ldw < K || ldy < C || (ldx | ldw | ldy) % 8 != 0)
    return fail(SIDON_E_STRIDE, "row strides ldx=%d ldw=%d ldy=%d must be multiples of 8 and >= K, K, C", ldx, ldw,
                ldy);
  if (!sidon::aligned16(x) || !sidon::aligned16(w) || !sidon::aligned16(y))
    return fail(SIDON_E_ALIGN, "x, w and y must be 16-byte aligned");
  const int N = 2 * C;
  if (!operands_fit(M, N, ldx, ldw, x, w)) return fail(SIDON_E_SHAPE, "X and W must each span less than 4 GiB");
  if (overlaps(x, ldx, w, ldw, y, (int64_t)ldy * 2, (int64_t)C * 2, M, N, K))
    return fail(SIDON_E_SHAPE, "x and w must not overlap y");
  int rc;
  if ((rc = sidon::check_device())) return rc;
  return launch(choose(M, N, K, kGlu, 1), kGlu, params(x, ldx, w, ldw, nullptr, y, ldy, M, N, K, 0),
                reinterpret_cast<hipStream_t>(stream), "gemm + GLU");
}

SIDON_API int sidon_gemm_res_fits(int M, int N, int K) { return res_fits(M, N, K) ? 1 : 0; }

// The library's kernels were slower at the encoder's two residual shapes up to
// 4800 rows of N = 1024, but for few outputs of a long K (1024 x 4096, us, in place |
// library: 150 rows 15.0 | 12.3, 225 13.3 | 12.1, 257 13.5 | 14.9).  There torch.addmm's
// host side outweighs that for a call launched on its own (a feed-forward step of
// 150 rows, 32.0 us a pass against 42.2; in a graph 24.0 against 22.4), and a caller with
// a buffer splits K.  Past the measured range the library is kept.
SIDON_API int sidon_gemm_res_preferred(int M, int N, int K) {
  if (!res_fits(M, N, K) || (int64_t)M * N > (int64_t)5 << 20) return 0;
  return sidon::check_device() == SIDON_OK ? 1 : 0;
}

SIDON_API int sidon_gemm_res(const void* x, int ldx, const void* w, int ldw, float* y, int ldy, int M, int N, int K,
                             sidon_stream_t stream) {
  sidon::clear_error();
  if (!x || !w || !y) return fail(SIDON_E_NULL, "x, w and y must be non-NULL");
  if (!res_fits(M, N, K))
    return fail(SIDON_E_SHAPE, "M=%d N=%d K=%d: need M >= 1, N a multiple of 64, K a multiple of 128", M, N, K);
  if (ldx < K || ldw < K || ldy < N || ldx % 8 != 0 || ldw % 8 != 0 || ldy % 4 != 0)
    return fail(SIDON_E_STRIDE, "row strides ldx=%d ldw=%d (multiples of 8, >= K) ldy=%d (multiple of 4, >= N)", ldx,
                ldw, ldy);
  if ((int64_t)M * ldx * 2 >= (int64_t(1) << 32) || (int64_t)N * ldw * 2 >= (int64_t(1) << 32))
    return fail(SIDON_E_SHAPE, "X and W must each span less than 4 GiB");
  if (!sidon::aligned16(x) || !sidon::aligned16(w) || !sidon::aligned16(y))
    return fail(SIDON_E_ALIGN, "x, w and y must be 16-byte aligned");
  if (overlaps(x, ldx, w, ldw, y, (int64_t)ldy * 4, (int64_t)N * 4, M, N, K))
    return fail(SIDON_E_SHAPE, "x and w must not overlap y (the kernel reads them while adding into y)");
  int rc;
  if ((rc = sidon::check_device())) return rc;
  return launch(choose(M, N, K, kAdd, 1), kAdd, params(x, ldx, w, ldw, nullptr, y, ldy, M, N, K, 0),
                reinterpret_cast<hipStream_t>(stream), "residual gemm");
}

SIDON_API int sidon_gemm_part_splits(int M, int N, int K) {
  if (!res_fits(M, N, K) || sidon::check_device() != SIDON_OK) return 0;
  return choose(M, N, K, kPart, kMaxSplits).splits;
}

SIDON_API int64_t sidon_gemm_part_rows(int M) { return M > kMaxPartRows ? M : kMaxPartRows; }

SIDON_API int sidon_gemm_part(const void* x, int ldx, const void* w, int ldw, float* part, int64_t part_elems, int M,
                              int N, int K, sidon_stream_t stream) {
  sidon::clear_error();
  if (!x || !w || !part) return fail(SIDON_E_NULL, "x, w and part must be non-NULL");
  if (!res_fits(M, N, K))
    return fail(SIDON_E_SHAPE, "M=%d N=%d K=%d: need M >= 1, N a multiple of 64, K a multiple of 128", M, N, K);
  if (ldx < K || ldw < K || ldx % 8 != 0 || ldw % 8 != 0)
    return fail(SIDON_E_STRIDE, "row strides ldx=%d ldw=%d must be multiples of 8 and >= K", ldx, ldw);
  if (!sidon::aligned16(x) || !sidon::aligned16(w) || !sidon::aligned16(part))
    return fail(SIDON_E_ALIGN, "x, w and part must be 16-byte aligned");
  if (!operands_fit(M, N, ldx, ldw, x, w)) return fail(SIDON_E_SHAPE, "X and W must each span less than 4 GiB");
  int rc;
  if ((rc = sidon::check_device())) return rc;
  const Choice c = choose(M, N, K, kPart, kMaxSplits);
  if (part_elems < (int64_t)c.splits * M * N)
    return fail(SIDON_E_SHAPE, "part holds %lld values, %d splits of %d x %d need more", (long long)part_elems,
                c.splits, M, N);
  // The splits' tiles lie one after another: `splits` times M rows of N.
  if (overlaps(x, ldx, w, ldw, part, (int64_t)N * 4, (int64_t)N * 4 + (int64_t)(c.splits - 1) * M * N * 4, M, N, K))
    return fail(SIDON_E_SHAPE, "x and w must not overlap part");
  TileParams p = params(x, ldx, w, ldw, nullptr, part, N, M, N, K, 0);
  p.split_stride = (int64_t)M * N;
  return launch(c, kPart, p, reinterpret_cast<hipStream_t>(stream), "partial gemm");
}
