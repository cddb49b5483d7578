// gemm_tile.h -- the tiled fp16 GEMM kernel behind the encoder's projections
// (MI355X / gfx950):  acc[m, n] = sum_k X[m, k] . W[n, k], X [M, K] and
// W [N, K] fp16 with K contiguous, fp32 sums, and an epilogue per use.
//
// A workgroup owns a BM x BN tile (of one K range, when K is split over
// workgroups) and runs WM x WN wavefronts, each TM x TN of it in MF x MF MFMA
// blocks, Y^T = W . X^T, so a lane holds four consecutive columns of one row.
// 64-wide K slices (whole 128-byte lines: 32-wide slices fetched every line
// twice from L2 and were 10-20% slower) go global -> LDS with
// global_load_lds_dwordx4 into a ring of ST buffers.  16-byte chunk c of the
// 128-byte LDS row r sits at chunk c ^ ((r >> 1) & 7): conflict-free operand
// reads (a read loop measured 240 of the 256 B/clock per CU).
//
// What bounds it: the copies and the MFMAs nearly add up unless they are
// interleaved, because a wavefront stalls at a copy instruction whose queue
// is full (96 x 128 tile, per 1024 of K: copies alone 4.9 us, MFMAs alone 4.3,
// together 9.6 when a slice's copies were issued at once).  So every step
// issues its share of the copies and of the next step's operand reads between
// its MFMAs (7.6 us), operands are read one step ahead across the slice
// boundary, and one barrier per slice, in front of the slice's last step,
// both publishes slice k + 1 and frees the buffer of slice k.  At large M the
// board's power limit holds the clock at 1.65-1.8 GHz (2.3 without copies).
// MF = 16 gives small tiles four independent accumulator chains per 32 x 32
// (a 64 x 64 tile at K = 1024: 8.2 -> 7.8 us); 32 reads fewer registers per flop.
#pragma once

#include <hip/hip_runtime.h>

#include <stdint.h>

#define SIDON_INLINE __attribute__((always_inline))

namespace sidon_gemm {

typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));

// Epilogues.
enum : int {
  kHalf = 0,   // fp16 Y = act(acc + bias)
  kGlu = 1,    // fp16 Y [M, N / 2] = a . sigmoid(b), a / b the two halves of the columns
  kPart = 2,   // fp32 partial sums of the K range: Y + split * split_stride
  kAdd = 3,    // fp32 Y += acc in place
};
// Activations of kHalf.
enum : int {
  kNone = 0,       // one rounding
  kSilu = 1,       // SiLU of the fp32 acc + bias, one rounding
  kSiluHalf = 2,   // acc + bias rounded to fp16, then SiLU rounded to fp16
};

struct TileParams {
  const _Float16* x;
  const _Float16* w;
  const _Float16* bias;
  void* y;
  int64_t split_stride;
  int ldx, ldw, ldy;  // row strides (elements)
  int M, N, K;
  int tiles_m, tiles_n;
  int splits;   // K ranges (1 unless kPart)
  int group;    // row tiles walked together (tile order)
  int act;
};

struct Yes { static constexpr bool value = true; };
struct No { static constexpr bool value = false; };
template <int N>
struct Int { static constexpr int value = N; };

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// Copy of 1 KB (8 rows of 128 bytes) global -> LDS; lane l's 16 bytes land at
// lds_addr + 16 l.  Completion is awaited with wait_vmcnt.
__device__ __forceinline__ void copy_1k(uint32_t lds_addr, const char* gbase, uint32_t voff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :: "s"(lds_addr), "v"(voff), "s"(gbase) : "memory", "m0");
}
#pragma clang diagnostic pop

template <int N>
__device__ __forceinline__ void wait_vmcnt() { asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory"); }

// Wait until all but the `newer` (<= kMax) youngest slices of kPer copies
// each have landed.
template <int kPer, int kMax>
__device__ __forceinline__ void wait_newer(int newer) {
  if constexpr (kMax > 0) {
    if (newer >= kMax) {
      wait_vmcnt<kPer * kMax>();
      return;
    }
    wait_newer<kPer, kMax - 1>(newer);
  } else {
    (void)newer;
    wait_vmcnt<0>();
  }
}

// This wavefront's LDS accesses have retired, then the workgroup's barrier
// (copies of later slices stay in flight).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

__device__ __forceinline__ float sigmoid(float x) { return __builtin_amdgcn_rcpf(1.f + __expf(-x)); }

// fp32 value rounded to fp16 on its own: the empty asm keeps a product and
// its conversion from fusing into one mixed-precision rounding.
__device__ __forceinline__ _Float16 to_half(float y) {
  asm volatile("" : "+v"(y));
  return (_Float16)y;
}

template <int BM, int BN, int WM, int WN, int MF, int ST, int kMode>
struct Tile {
  static constexpr int kWaves = WM * WN;
  static constexpr int kThreads = 64 * kWaves;
  static constexpr int TM = BM / WM, TN = BN / WN;
  static constexpr int kStage = (BM + BN) * 128;
  static constexpr int kCopies = kStage / 1024;
  // Per wavefront: the fp16 tile (kHalf; half of it for kGlu) or MF rows of fp32.
  static constexpr int kOutCols = kMode == kGlu ? TN / 2 : TN;
  static constexpr int kEpiWave = kMode <= kGlu ? TM * kOutCols * 2 : MF * (TN + 4) * 4;
  static constexpr int kLds = ST * kStage > kWaves * kEpiWave ? ST * kStage : kWaves * kEpiWave;
  static_assert(kLds <= 160 * 1024, "LDS of one CU");
  static_assert(ST >= 2 && (MF == 16 || MF == 32) && TM % MF == 0 && TN % MF == 0, "tile shape");
  static_assert(kCopies % kWaves == 0 && kCopies / kWaves * ST < 64, "even split of the copies, vmcnt range");
  static_assert(kMode != kGlu || (TN / MF) % 2 == 0, "a GLU wavefront holds pairs of blocks");
};

template <int BM, int BN, int WM, int WN, int MF, int ST, int kMode>
__global__ void __launch_bounds__(64 * WM * WN) gemm_tile_kernel(const TileParams p) {
  using T = Tile<BM, BN, WM, WN, MF, ST, kMode>;
  constexpr int NW = T::kWaves, TM = T::TM, TN = T::TN;
  constexpr int IM = TM / MF, IN = TN / MF;      // MFMA blocks per wavefront
  constexpr int NG = 64 / MF;                    // lane groups along K
  constexpr int AR = MF * MF / 64, Q = AR / 4;   // accumulator registers per block
  constexpr int KS = 64 / (8 * NG);              // steps per slice
  constexpr int kPer = T::kCopies / NW;          // copies per wavefront and slice
  constexpr int kFirst = kPer / KS;              // copies issued in a slice's last step
  typedef float acc_t __attribute__((ext_vector_type(AR)));
  __shared__ __attribute__((aligned(16))) char smem[T::kLds];

  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = w / WN;
  const int wn = w % WN;

  // Each XCD (workgroups go round-robin over the 8) takes a contiguous range
  // of tile numbers: K range slowest, then groups of p.group row tiles, then
  // columns, the group's row tiles fastest -- what runs on an XCD at once
  // shares a few row blocks of X and of W in its L2.
  const int nwg = gridDim.x;
  const int xcd = blockIdx.x & 7;
  const int per = nwg >> 3;
  const int rem = nwg & 7;
  int lin = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + ((int)blockIdx.x >> 3);
  const int tiles = p.tiles_m * p.tiles_n;
  const int split = lin / tiles;
  lin -= split * tiles;
  const int gsize = p.group * p.tiles_n;
  const int g = lin / gsize;
  const int gm = min(p.tiles_m - g * p.group, p.group);
  const int in_group = lin - g * gsize;
  const int m0 = (g * p.group + in_group % gm) * BM;
  const int tn = in_group / gm;
  const int slices = p.K / 64;
  const int kb = (int)((int64_t)slices * split / p.splits);
  const int nk = (int)((int64_t)slices * (split + 1) / p.splits) - kb;   // >= 1: the host keeps splits <= slices

  // Copy instruction i of a slice (wavefront w issues i = w + NW j): rows
  // 8 i + lane / 8 of the tile's X part, then of its W part.  X rows >= M
  // re-read row M - 1 (their results are never stored).  GLU tiles pair
  // column blocks: of a wavefront's TN columns the first half are values and
  // the second half their gates, N / 2 further on.
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  uint32_t voff[kPer];
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int i = w + NW * j;
    const bool xi = i < BM / 8;
    const int r = 8 * (xi ? i : i - BM / 8) + (lane >> 3);
    const int c = (lane & 7) ^ ((r >> 1) & 7);
    if (xi) {
      voff[j] = (uint32_t)min(m0 + r, p.M - 1) * (uint32_t)p.ldx * 2u + (uint32_t)c * 16u;
    } else {
      int col;
      if constexpr (kMode == kGlu) {
        const int q = r % TN;
        col = tn * (BN / 2) + (r / TN) * (TN / 2) + (q < TN / 2 ? q : (p.N >> 1) + q - TN / 2);
      } else {
        col = tn * BN + r;
      }
      voff[j] = (uint32_t)col * (uint32_t)p.ldw * 2u + (uint32_t)c * 16u;
    }
  }
  const char* xg = reinterpret_cast<const char*>(p.x) + (int64_t)kb * 128;
  const char* wg = reinterpret_cast<const char*>(p.w) + (int64_t)kb * 128;
  auto copy = [&](int kt, int slot, int j) SIDON_INLINE {
    const int i = w + NW * j;
    copy_1k(lds0 + (uint32_t)(slot * T::kStage + i * 1024), (i < BM / 8 ? xg : wg) + (int64_t)kt * 128, voff[j]);
  };
  // Operand reads: lane (ln, lg) reads LDS row MF b + ln, chunk NG s + lg.
  const int ln = lane & (MF - 1);
  const int lg = lane / MF;
  const int swz = (ln >> 1) & 7;  // rows MF b + ln share the swizzle of row ln
  const char* xrow = smem + (TM * wm + ln) * 128;
  const char* wrow = smem + (BM + TN * wn + ln) * 128;

  acc_t acc[IM][IN];
#pragma unroll
  for (int i = 0; i < IM; ++i)
#pragma unroll
    for (int j = 0; j < IN; ++j) acc[i][j] = acc_t{};
  h8 xa[2][IM], wb[2][IN];
  constexpr int R = IM + IN;  // operand reads per step, the first MFMA's two first
  auto read = [&](int slot, int s, int set, int r) SIDON_INLINE {
    const int off = slot * T::kStage + (((NG * s + lg) ^ swz) << 4);
    if (r == 0) {
      wb[set][0] = *reinterpret_cast<const h8*>(wrow + off);
    } else if (r == 1) {
      xa[set][0] = *reinterpret_cast<const h8*>(xrow + off);
    } else if (r < 1 + IN) {
      wb[set][r - 1] = *reinterpret_cast<const h8*>(wrow + off + (r - 1) * MF * 128);
    } else {
      xa[set][r - IN] = *reinterpret_cast<const h8*>(xrow + off + (r - IN) * MF * 128);
    }
  };

  // Slice kt: its MFMAs, and between them the operand reads of the next step,
  // the rest of the copies of slice kt - 1 + ST (kRest) and, after the
  // barrier, the first copies of slice kt + ST (kAhead) into the buffer that
  // the barrier freed.  kNext: there is a slice kt + 1.
  int slot = 0;
  auto body = [&](int kt, auto rest, auto ahead, auto next) SIDON_INLINE {
    constexpr bool kRest = decltype(rest)::value, kAhead = decltype(ahead)::value, kNext = decltype(next)::value;
    const int prev = slot == 0 ? ST - 1 : slot - 1;
    const int succ = slot == ST - 1 ? 0 : slot + 1;
    constexpr int TT = IM * IN;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const bool last = s == KS - 1;
      const int c0 = last ? 0 : kFirst + (kPer - kFirst) * s / (KS - 1);
      const int c1 = last ? kFirst : kFirst + (kPer - kFirst) * (s + 1) / (KS - 1);
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        const int i = t / IN, j = t % IN;
        if constexpr (MF == 32) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wb[s & 1][j], xa[s & 1][i], acc[i][j], 0, 0, 0);
        } else {
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wb[s & 1][j], xa[s & 1][i], acc[i][j], 0, 0, 0);
        }
#pragma unroll
        for (int r = R * t / TT; r < R * (t + 1) / TT; ++r) {
          if (!last) {
            read(slot, s + 1, (s + 1) & 1, r);
          } else if (kNext) {
            read(succ, 0, 0, r);
          }
        }
#pragma unroll
        for (int c = c0 + (c1 - c0) * t / TT; c < c0 + (c1 - c0) * (t + 1) / TT; ++c) {
          if (!last && kRest) copy(kt - 1 + ST, prev, c);
          if (last && kAhead) copy(kt + ST, slot, c);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (s == KS - 2 && kNext) {
        // Slice kt + 1 has landed for every wavefront; slice kt is in
        // registers everywhere, so its buffer may be refilled.
        if constexpr (kAhead) {
          wait_vmcnt<kPer * (ST - 2)>();
        } else {
          wait_newer<kPer, ST - 2>(min(ST - 2, nk - 2 - kt));
        }
        lds_barrier();
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    slot = succ;
  };

#pragma unroll
  for (int kt = 0; kt < ST; ++kt) {
    if (kt < nk) {
#pragma unroll
      for (int j = 0; j < kPer; ++j)
        if (kt < ST - 1 || j < kFirst) copy(kt, kt, j);
    }
  }
  if (nk >= ST) {
    wait_vmcnt<kPer * (ST - 2) + kFirst>();
  } else {
    wait_newer<kPer, ST - 2>(min(ST - 2, nk - 1));
  }
  lds_barrier();
#pragma unroll
  for (int r = 0; r < R; ++r) read(0, 0, 0, r);
  int kt = 0;
  for (; kt < nk - ST; ++kt) body(kt, Yes{}, Yes{}, Yes{});
  if (nk >= ST) {  // ST >= 2, so a slice follows
    body(kt, Yes{}, No{}, Yes{});
    ++kt;
  }
  for (; kt < nk - 1; ++kt) body(kt, No{}, No{}, Yes{});
  // kAdd: the rows of Y that this lane will add to, loaded under the last
  // slice's products.
  constexpr int kFLanes = TN / 4, kFRows = 64 / kFLanes;    // fp32 epilogue: lanes per row, rows per store
  constexpr int kOld = kMode == kAdd ? TM / kFRows : 1;
  f4 old[kOld];
  if constexpr (kMode == kAdd) {
    const float* yb = static_cast<const float*>(p.y) + tn * BN + TN * wn + 4 * (lane % kFLanes);
#pragma unroll
    for (int t = 0; t < kOld; ++t)
      old[t] = *reinterpret_cast<const f4*>(yb + (int64_t)min(m0 + TM * wm + kFRows * t + lane / kFLanes, p.M - 1) * p.ldy);
  }
  body(kt, No{}, No{}, No{});
  lds_barrier();  // every wavefront is done with the ring, which the epilogue reuses

  // acc[i][j]: row MF i + ln, columns MF j + 8 (e / 4) + 4 lg + e % 4 of the
  // wavefront's tile.
  if constexpr (kMode <= kGlu) {
    // The fp16 tile through the wavefront's own LDS, whole row pieces out:
    // 8-byte unit u of row r sits at u ^ (r & kUnitMask).
    constexpr int OC = T::kOutCols;
    constexpr int kRow = OC * 2;
    constexpr int kUnits = OC / 4;
    constexpr int kUnitMask = kUnits < 16 ? kUnits - 1 : 15;
    static_assert((kUnits & (kUnits - 1)) == 0, "power of two columns per wavefront");
    char* ep = smem + w * T::kEpiWave;
    auto put = [&](int i, int col, h4 v) SIDON_INLINE {
      const int row = MF * i + ln;
      *reinterpret_cast<h4*>(ep + row * kRow + (((col >> 2) ^ (row & kUnitMask)) << 3)) = v;
    };
    if constexpr (kMode == kGlu) {
#pragma unroll
      for (int j = 0; j < IN / 2; ++j)
#pragma unroll
        for (int q = 0; q < Q; ++q)
#pragma unroll
          for (int i = 0; i < IM; ++i) {
            h4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              // Both halves rounded to fp16 first, as the projection stores them.
              const float a = (float)to_half(acc[i][j][4 * q + e]);
              const float b = (float)to_half(acc[i][j + IN / 2][4 * q + e]);
              v[e] = to_half(a * sigmoid(b));
            }
            put(i, MF * j + 8 * q + 4 * lg, v);
          }
    } else {
      auto fill = [&](auto act) SIDON_INLINE {
        constexpr int kAct = decltype(act)::value;
#pragma unroll
        for (int j = 0; j < IN; ++j)
#pragma unroll
          for (int q = 0; q < Q; ++q) {
            const int col = MF * j + 8 * q + 4 * lg;
            h4 bv = {};
            if (p.bias != nullptr) bv = *reinterpret_cast<const h4*>(p.bias + tn * BN + TN * wn + col);
#pragma unroll
            for (int i = 0; i < IM; ++i) {
              h4 v;
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                float s = acc[i][j][4 * q + e] + (float)bv[e];
                if constexpr (kAct == kSiluHalf) s = (float)to_half(s);
                if constexpr (kAct != kNone) s = s * sigmoid(s);
                v[e] = to_half(s);
              }
              put(i, col, v);
            }
          }
      };
      if (p.act == kSilu) {
        fill(Int<kSilu>{});
      } else if (p.act == kSiluHalf) {
        fill(Int<kSiluHalf>{});
      } else {
        fill(Int<kNone>{});
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // own LDS writes done (wave-private region)
    constexpr int kLanes = OC / 8, kRows = 64 / kLanes;  // 16 bytes per lane
    const int c = lane % kLanes;
#pragma unroll
    for (int t = 0; t < (TM + kRows - 1) / kRows; ++t) {
      const int row = kRows * t + lane / kLanes;
      const int gmr = m0 + TM * wm + row;
      if ((TM % kRows == 0 || row < TM) && gmr < p.M) {
        const h4 lo = *reinterpret_cast<const h4*>(ep + row * kRow + (((2 * c) ^ (row & kUnitMask)) << 3));
        const h4 hi = *reinterpret_cast<const h4*>(ep + row * kRow + (((2 * c + 1) ^ (row & kUnitMask)) << 3));
        const h8 v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        *reinterpret_cast<h8*>(static_cast<_Float16*>(p.y) + (int64_t)gmr * p.ldy +
                               tn * (kMode == kGlu ? BN / 2 : BN) + OC * wn + 8 * c) = v;
      }
    }
  } else {
    // fp32 rows through the wavefront's own LDS, MF at a time.
    constexpr int kRow = TN + 4;
    constexpr int kLanes = kFLanes, kRows = kFRows;
    static_assert(64 % kLanes == 0 && MF % kRows == 0, "whole rows per store instruction");
    float* ep = reinterpret_cast<float*>(smem + w * T::kEpiWave);
    float* yb = static_cast<float*>(p.y) + split * p.split_stride + tn * BN + TN * wn + 4 * (lane % kLanes);
#pragma unroll
    for (int i = 0; i < IM; ++i) {
#pragma unroll
      for (int j = 0; j < IN; ++j)
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          const f4 v = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
          *reinterpret_cast<f4*>(ep + ln * kRow + MF * j + 8 * q + 4 * lg) = v;
        }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int t = 0; t < MF / kRows; ++t) {
        const int row = kRows * t + lane / kLanes;
        const int gmr = m0 + TM * wm + MF * i + row;
        f4 v = *reinterpret_cast<const f4*>(ep + row * kRow + 4 * (lane % kLanes));
        if (gmr < p.M) {
          f4* dst = reinterpret_cast<f4*>(yb + (int64_t)gmr * p.ldy);
          if constexpr (kMode == kAdd) v += old[i * (MF / kRows) + t];
          *dst = v;
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
  }
}

}  // namespace sidon_gemm
