// Dense GEMM C = beta * C + alpha * op(A) * op(B), row-major (bclx_gemm): the tile multiply BCL's dense gemm
// calls through cblas_gemm_wrapper_ (bcl/containers/algorithms/cblas_wrapper.hpp:16-40, called with
// alpha = beta = 1 from gemm_cowns, bcl/containers/algorithms/gemm.hpp:86-107).
//
// Three arithmetic modes on the matrix cores for fp32 operands (bclx_gemm), and an fp64 product (bclx_gemm_f64):
//   0  FP32: fp32 inputs, v_mfma_f32_32x32x2f32 (exact fp32 products, fp32 accumulation)
//   1  BF16: inputs rounded to bf16 (round to nearest even), v_mfma_f32_32x32x16_bf16, fp32 accumulation
//   2  split-BF16 3-term: x = x_hi + x_lo with x_hi = bf16(x), x_lo = bf16(x - x_hi); a*b is taken as
//      a_lo*b_hi + a_hi*b_lo + a_hi*b_hi (the a_lo*b_lo term, below 2^-16 relative, is dropped), fp32 accumulation
//
// Two pipelines (gemm_impl chooses by predicted time):
//   packed, for large fp32-operand products: a pack pass writes op(A) as Ap[M'][K'] and op(B) as Bp[N'][K'] (K
//     contiguous, zero-padded to the block tile, converted / split for the bf16 modes), then the MFMA kernel runs on
//     the packed operands with no bounds checks in its main loop. Block tile 128 x 128, four wavefronts of 64 x 64 (2 x
//     2 MFMA tiles of 32 x 32);
//   direct, for the others and for fp64: one kernel reads the caller's arrays, 64 x 64 tiles, K split over blocks
//     where the tiles alone leave CUs idle.
// In both the next K tile is loaded into registers while the current one is multiplied out of LDS, and blocks are
// ordered so that each XCD
// (blocks are dealt round-robin over the 8 XCDs) works on a compact patch of C tiles and shares their A and B panels
// in its L2.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "internal.hpp"

namespace bclx {

// Compile-time loop: f(std::integral_constant<int, I>) for I in [B, E), so register arrays get constant indices.
template <int B, int E, typename F>
__device__ inline void static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));

constexpr int kGThreads = 256;

// C tile of block b. XCD-aware: block b runs on XCD b % 8, so each XCD is given a contiguous run of the order below.
// The order walks groups of kTileGroup tile rows column by column, so the blocks an XCD runs at one time cover a
// near-square patch of C and share their A and B panels in that XCD's L2 (a row-major order would share one A
// panel and stream every B panel through L2; measured 8% slower on the BF16 8192^3 product).
constexpr int kTileGroup = 4;
__device__ inline void gemm_tile_of(int b, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int T = tiles_m * tiles_n;
  if (T % 8 == 0) b = (b % 8) * (T / 8) + (b / 8);
  const int per_group = kTileGroup * tiles_n;
  const int first = (b / per_group) * kTileGroup;
  const int rows = tiles_m - first < kTileGroup ? tiles_m - first : kTileGroup;
  const int r = b % per_group;
  tm = first + r % rows;
  tn = r / rows;
}

__device__ inline uint16_t f32_to_bf16_rne(float x) {
  uint32_t u = __float_as_uint(x);
  if ((u & 0x7FFFFFFFu) > 0x7F800000u) return (uint16_t)((u >> 16) | 0x40u);  // NaN stays a (quiet) NaN
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ inline float bf16_bits_to_f32(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// dst[r * Kp + c] for r < Rp, c < Kp from src[r * rs + c * cs] (r < R, c < K), zero padding outside.
// MODE 0: fp32 copy; 1: bf16 (hi only); 2: bf16 hi and lo. 64 x 64 tiles staged through LDS: the reads run along
// the source's contiguous direction and each lane writes 8
// consecutive k of one row (16 bytes of bf16, 32 of fp32). Kp is a multiple of 32, so a chunk of 8 is wholly inside.
// Bound by HBM: whole tiles of 16-byte aligned sources (vec: base and leading dimension) are read 16 bytes per lane, four loads in
// flight per thread; others 4 bytes at a time (8192^2 to bf16: 119 -> 97 us).
template <int MODE>
__global__ __launch_bounds__(256) void k_pack(const float* __restrict__ src, int64_t R, int64_t K, int64_t rs,
                                              int64_t cs, void* dst_hi, uint16_t* dst_lo, int64_t Rp, int64_t Kp,
                                              int vec) {
  __shared__ float tile[64][65];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int64_t r0 = (int64_t)blockIdx.y * 64, c0 = (int64_t)blockIdx.x * 64;
  const bool rows_contig = cs != 1;  // source contiguous along r (a transposed operand)
  if (vec && r0 + 64 <= R && c0 + 64 <= K) {  // whole tile, 16-byte loads, all four of a thread in flight
    const int x = (tid & 15) * 4, y = tid >> 4;  // x along the contiguous index
    const float* p = src + (rows_contig ? r0 + c0 * cs : r0 * rs + c0) + x;
    const int64_t step = rows_contig ? cs : rs;
    u32x4 v[4];
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = *reinterpret_cast<const u32x4*>(p + (y + 16 * i) * step);
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const float f = __uint_as_float(v[i][j]);
        if (rows_contig) tile[x + j][y + 16 * i] = f;
        else tile[y + 16 * i][x + j] = f;
      }
  } else {
    for (int q = w; q < 64; q += 4) {
      int64_t r, c;
      if (rows_contig) { r = r0 + lane; c = c0 + q; }
      else { r = r0 + q; c = c0 + lane; }
      const float v = (r < R && c < K) ? src[r * rs + c * cs] : 0.f;
      if (rows_contig) tile[lane][q] = v;
      else tile[q][lane] = v;
    }
  }
  __syncthreads();
  for (int ch = tid; ch < 512; ch += 256) {
    const int rr = ch >> 3, cc = (ch & 7) * 8;
    const int64_t r = r0 + rr, c = c0 + cc;
    if (r >= Rp || c >= Kp) continue;
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = tile[rr][cc + i];
    if constexpr (MODE == 0) {
      u32x4* d = reinterpret_cast<u32x4*>(static_cast<float*>(dst_hi) + r * Kp + c);
      d[0] = u32x4{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])};
      d[1] = u32x4{__float_as_uint(v[4]), __float_as_uint(v[5]), __float_as_uint(v[6]), __float_as_uint(v[7])};
    } else {
      uint16_t hi[8], lo[8];
#pragma unroll
      for (int i = 0; i < 8; i++) {
        hi[i] = f32_to_bf16_rne(v[i]);
        if constexpr (MODE == 2) lo[i] = f32_to_bf16_rne(v[i] - bf16_bits_to_f32(hi[i]));
      }
      auto pk = [](const uint16_t* x) {
        return u32x4{(uint32_t)x[0] | ((uint32_t)x[1] << 16), (uint32_t)x[2] | ((uint32_t)x[3] << 16),
                     (uint32_t)x[4] | ((uint32_t)x[5] << 16), (uint32_t)x[6] | ((uint32_t)x[7] << 16)};
      };
      *reinterpret_cast<u32x4*>(static_cast<uint16_t*>(dst_hi) + r * Kp + c) = pk(hi);
      if constexpr (MODE == 2) *reinterpret_cast<u32x4*>(dst_lo + r * Kp + c) = pk(lo);
    }
  }
}

template <int MODE>
struct GemmCfg;
template <>
struct GemmCfg<0> {
  using E = float;
  static constexpr int BK = 32, PAD = 4, KSTEP = 2;
};
template <>
struct GemmCfg<1> {
  using E = uint16_t;
  static constexpr int BK = 64, PAD = 8, KSTEP = 16;
};
template <>
struct GemmCfg<2> {
  using E = uint16_t;
  static constexpr int BK = 64, PAD = 8, KSTEP = 16;
};

// Block tile (64 * TM) x (64 * TN): four wavefronts in a 2 x 2 arrangement, each owning TM x TN MFMA tiles of
// 32 x 32. Larger wavefront tiles reuse each LDS fragment for more MFMAs (TM + TN fragment loads per k step feed
// TM * TN MFMAs).
template <int MODE, int TM, int TN>
__global__ __launch_bounds__(kGThreads, TM * TN > 4 ? 2 : 1) void k_gemm(const typename GemmCfg<MODE>::E* __restrict__ Ahi,
                                                    const typename GemmCfg<MODE>::E* __restrict__ Alo,
                                                    const typename GemmCfg<MODE>::E* __restrict__ Bhi,
                                                    const typename GemmCfg<MODE>::E* __restrict__ Blo, int64_t M,
                                                    int64_t N, int64_t Kp, float alpha, float beta, float* C,
                                                    int64_t ldc, int tiles_m, int tiles_n) {
  using E = typename GemmCfg<MODE>::E;
  constexpr int BK = GemmCfg<MODE>::BK, PAD = GemmCfg<MODE>::PAD, KSTEP = GemmCfg<MODE>::KSTEP;
  constexpr int BM = 64 * TM, BN = 64 * TN;
  constexpr int LDK = BK + PAD;
  constexpr int NSPLIT = MODE == 2 ? 2 : 1;
  constexpr int VPR = BK * (int)sizeof(E) / 16;   // 16-byte vectors per tile row
  constexpr int VPA = BM * VPR / kGThreads;       // vectors per thread, A tile
  constexpr int VPB = BN * VPR / kGThreads;       // vectors per thread, B tile
  __shared__ __align__(16) E As[NSPLIT][BM * LDK];
  __shared__ __align__(16) E Bs[NSPLIT][BN * LDK];

  int tm, tn;
  gemm_tile_of(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;

  const E* __restrict__ Ag0 = Ahi + m0 * Kp;
  const E* __restrict__ Bg0 = Bhi + n0 * Kp;
  const E* __restrict__ Ag1 = MODE == 2 ? Alo + m0 * Kp : Ag0;
  const E* __restrict__ Bg1 = MODE == 2 ? Blo + n0 * Kp : Bg0;
  constexpr int EPV = 16 / (int)sizeof(E);  // elements per 16-byte vector
  // per-thread vector slots: row = (tid + i * 256) / VPR, column vector = (tid + i * 256) % VPR
  u32x4 ra0[VPA], rb0[VPB], ra1[VPA], rb1[VPB];
  auto gload = [&](int64_t k0) {
    static_for<0, VPA>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      const int v = tid + i * kGThreads;
      const int64_t o = (int64_t)(v / VPR) * Kp + k0 + (v % VPR) * EPV;
      ra0[i] = *reinterpret_cast<const u32x4*>(Ag0 + o);
      if constexpr (MODE == 2) ra1[i] = *reinterpret_cast<const u32x4*>(Ag1 + o);
    });
    static_for<0, VPB>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      const int v = tid + i * kGThreads;
      const int64_t o = (int64_t)(v / VPR) * Kp + k0 + (v % VPR) * EPV;
      rb0[i] = *reinterpret_cast<const u32x4*>(Bg0 + o);
      if constexpr (MODE == 2) rb1[i] = *reinterpret_cast<const u32x4*>(Bg1 + o);
    });
  };
  auto lstore = [&]() {
    static_for<0, VPA>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      const int v = tid + i * kGThreads;
      const int o = (v / VPR) * LDK + (v % VPR) * EPV;
      *reinterpret_cast<u32x4*>(&As[0][o]) = ra0[i];
      if constexpr (MODE == 2) *reinterpret_cast<u32x4*>(&As[NSPLIT - 1][o]) = ra1[i];
    });
    static_for<0, VPB>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      const int v = tid + i * kGThreads;
      const int o = (v / VPR) * LDK + (v % VPR) * EPV;
      *reinterpret_cast<u32x4*>(&Bs[0][o]) = rb0[i];
      if constexpr (MODE == 2) *reinterpret_cast<u32x4*>(&Bs[NSPLIT - 1][o]) = rb1[i];
    });
  };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; a++)
#pragma unroll
    for (int c = 0; c < TN; c++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[a][c][v] = 0.f;

  const int nk = (int)(Kp / BK);
  gload(0);
  lstore();
  __syncthreads();
  const int fr = lane & 31, fk = lane >> 5;
  for (int kt = 0; kt < nk; kt++) {
    if (kt + 1 < nk) gload((int64_t)(kt + 1) * BK);
#pragma unroll
    for (int ks = 0; ks < BK; ks += KSTEP) {
      if constexpr (MODE == 0) {
        float af[TM], bf[TN];
#pragma unroll
        for (int t = 0; t < TM; t++) af[t] = As[0][(wm * 32 * TM + t * 32 + fr) * LDK + ks + fk];
#pragma unroll
        for (int t = 0; t < TN; t++) bf[t] = Bs[0][(wn * 32 * TN + t * 32 + fr) * LDK + ks + fk];
#pragma unroll
        for (int a = 0; a < TM; a++)
#pragma unroll
          for (int c = 0; c < TN; c++) acc[a][c] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[a], bf[c], acc[a][c], 0, 0, 0);
      } else {
        bf16x8 ah[TM], bh[TN], al[TM], bl[TN];
#pragma unroll
        for (int t = 0; t < TM; t++) {
          ah[t] = *reinterpret_cast<const bf16x8*>(&As[0][(wm * 32 * TM + t * 32 + fr) * LDK + ks + fk * 8]);
          if constexpr (MODE == 2)
            al[t] = *reinterpret_cast<const bf16x8*>(&As[NSPLIT - 1][(wm * 32 * TM + t * 32 + fr) * LDK + ks + fk * 8]);
        }
#pragma unroll
        for (int t = 0; t < TN; t++) {
          bh[t] = *reinterpret_cast<const bf16x8*>(&Bs[0][(wn * 32 * TN + t * 32 + fr) * LDK + ks + fk * 8]);
          if constexpr (MODE == 2)
            bl[t] = *reinterpret_cast<const bf16x8*>(&Bs[NSPLIT - 1][(wn * 32 * TN + t * 32 + fr) * LDK + ks + fk * 8]);
        }
#pragma unroll
        for (int a = 0; a < TM; a++)
#pragma unroll
          for (int c = 0; c < TN; c++) {
            if constexpr (MODE == 2) {
              acc[a][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[a], bh[c], acc[a][c], 0, 0, 0);
              acc[a][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[a], bl[c], acc[a][c], 0, 0, 0);
            }
            acc[a][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[a], bh[c], acc[a][c], 0, 0, 0);
          }
      }
    }
    __syncthreads();
    if (kt + 1 < nk) {
      lstore();
      __syncthreads();
    }
  }
  // accumulator layout of a 32 x 32 MFMA tile: lane l holds column l % 32, rows 8 * (v / 4) + 4 * (l / 32) + v % 4
#pragma unroll
  for (int a = 0; a < TM; a++)
#pragma unroll
    for (int c = 0; c < TN; c++) {
      const int64_t col = n0 + wn * 32 * TN + c * 32 + fr;
      if (col >= N) continue;
#pragma unroll
      for (int v = 0; v < 16; v++) {
        const int64_t row = m0 + wm * 32 * TM + a * 32 + 8 * (v / 4) + 4 * fk + (v % 4);
        if (row < M) {
          float* p = C + row * ldc + col;
          *p = beta == 0.f ? alpha * acc[a][c][v] : fmaf(beta, *p, alpha * acc[a][c][v]);
        }
      }
    }
}

// ---- direct kernels: operands read from the caller's arrays ----------------------------------------------------
// Sizes at which a pack pass (two more launches, each operand read and written once more) costs more than it saves,
// and every fp32 and fp64 product: the block reads its A and B tiles straight from the caller's row-major arrays into
// registers (bounds-checked at the edges, the next K tile while the current one is multiplied), converts / splits them
// for the bf16 modes and stores them to LDS with K contiguous. A thread moves micro-tiles of 4 x 4 (fp32) or 2 x 2
// (fp64) elements: one 16-byte load per source line of the micro-tile, along K or along the rows, whichever the source
// has contiguous, and one K-contiguous LDS store per row. Loads need only the element's own alignment.
// K is split over gridDim.z where the C tiles alone leave CUs idle: each split writes its partial sums to a workspace
// and k_gemm_reduce adds them in order.

// Micro-tiles of one operand's block tile, and their way to LDS. Operand element (r, k), r < R, k < K, at
// src[r * ld + k] (KC: contiguous along K) or src[k * ld + r].
template <typename T, int Q, int ROWS, int BK, bool KC>
struct MicroTiles {
  static constexpr int COUNT = ROWS * BK / (Q * Q) / kGThreads;  // per thread
  static constexpr int KQ = BK / Q;                              // micro-tiles along K
  static_assert(ROWS * BK % (Q * Q * kGThreads) == 0, "whole micro-tiles per thread");
  typedef T line_t __attribute__((ext_vector_type(Q)));
  typedef T line_u __attribute__((ext_vector_type(Q), aligned(sizeof(T))));  // element-aligned in memory
  line_t x[COUNT][Q];  // [micro-tile][source line]
  int row[COUNT];      // first row of each micro-tile within the block tile
  bool inside;         // every micro-tile lies inside the operand's rows

  // Neighbouring lanes run along the contiguous direction (all of a K row of the tile, or 8 micro-tiles of rows). A
  // micro-tile that would reach past the operand's last row is moved back to end there: it stores the rows it shares
  // with its neighbour a second time (the same values), and the block's rows past the end stay unset (their products
  // are not stored). Fewer than Q rows left in the whole block: the guarded path.
  __device__ inline void init(int64_t r0, int64_t R) {
    const int last = (int)(R - r0 < ROWS ? R - r0 - Q : ROWS - Q);
    inside = last >= 0;
    static_for<0, COUNT>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      const int q = (int)threadIdx.x + i * kGThreads;
      const int r = KC ? q / KQ * Q : (q % 8 + q / (8 * KQ) * 8) * Q;
      row[i] = inside && r > last ? last : r;
    });
  }
  static __device__ inline int k_of(int i) {
    const int q = (int)threadIdx.x + i * kGThreads;
    return (KC ? q % KQ : q / 8 % KQ) * Q;
  }
  // rows r0.. and K positions k0.. of the operand; k_whole: the K tile lies wholly inside it
  __device__ inline void load(const T* src, int64_t ld, int64_t r0, int64_t k0, int64_t R, int64_t K, bool k_whole) {
    const bool whole = inside && k_whole;
    static_for<0, COUNT>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      const int64_t line0 = KC ? r0 + row[i] : k0 + k_of(i), elem0 = KC ? k0 + k_of(i) : r0 + row[i];
      const T* p = src + line0 * ld + elem0;
      if (whole) {
        static_for<0, Q>([&](auto jc) {
          constexpr int j = decltype(jc)::value;
          x[i][j] = *reinterpret_cast<const line_u*>(p + j * ld);
        });
      } else {
        const int64_t nl = (KC ? R : K) - line0, ne = (KC ? K : R) - elem0;
        static_for<0, Q>([&](auto jc) {
          constexpr int j = decltype(jc)::value;
          static_for<0, Q>([&](auto ec) {
            constexpr int e = decltype(ec)::value;
            x[i][j][e] = (j < nl && e < ne) ? p[j * ld + e] : T(0);
          });
        });
      }
    });
  }
  // f(row, k, values of k .. k + Q - 1) for each row of each micro-tile
  template <typename F>
  __device__ inline void rows(F&& f) const {
    static_for<0, COUNT>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      static_for<0, Q>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        line_t v;
        static_for<0, Q>([&](auto ec) {
          constexpr int e = decltype(ec)::value;
          v[e] = x[i][KC ? j : e][KC ? e : j];
        });
        f(row[i] + j, k_of(i), v);
      });
    });
  }
};

// C tile of this block, its K tiles, and where its result goes.
struct DirectArgs {
  int64_t M, N, K, lda, ldb, ldc;
  int32_t tiles_m, tiles_n;
  int32_t kt_per_split;      // K tiles per split
  int64_t split_stride;      // elements between the splits' copies of C
};

constexpr int kDirectTile = 64;   // C tile of a block: 64 x 64, four wavefronts (2 x 2) of 32 x 32 each
constexpr int kDirectBK = 64;     // K per LDS tile (fp32 operands)
constexpr int kDirectBK64 = 16;   // K per LDS tile (fp64)

template <int MODE, bool AKC, bool BKC>
__global__ __launch_bounds__(kGThreads, 2) void k_gemm_direct(DirectArgs D, const float* __restrict__ A,
                                                              const float* __restrict__ B, float alpha, float beta,
                                                              float* C) {
  using E = typename GemmCfg<MODE>::E;
  constexpr int BK = kDirectBK, LDK = BK + GemmCfg<MODE>::PAD;
  constexpr int BM = kDirectTile, BN = kDirectTile;
  constexpr int NSPLIT = MODE == 2 ? 2 : 1;
  __shared__ __align__(16) E As[NSPLIT][BM * LDK];
  __shared__ __align__(16) E Bs[NSPLIT][BN * LDK];
  int tm, tn;
  gemm_tile_of(blockIdx.x, D.tiles_m, D.tiles_n, tm, tn);
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int nk = (int)((D.K + BK - 1) / BK);
  const int kt0 = (int)blockIdx.z * D.kt_per_split;
  const int kt1 = min(nk, kt0 + D.kt_per_split);
  C += (int64_t)blockIdx.z * D.split_stride;
  MicroTiles<float, 4, BM, BK, AKC> ma;
  MicroTiles<float, 4, BN, BK, BKC> mb;
  ma.init(m0, D.M);
  mb.init(n0, D.N);
  auto gload = [&](int kt) {
    const int64_t k0 = (int64_t)kt * BK;
    const bool k_whole = k0 + BK <= D.K;
    ma.load(A, D.lda, m0, k0, D.M, D.K, k_whole);
    mb.load(B, D.ldb, n0, k0, D.N, D.K, k_whole);
  };
  auto put = [&](E* hi, E* lo, int r, int k, f32x4 v) {
    if constexpr (MODE == 0) {
      *reinterpret_cast<f32x4*>(hi + r * LDK + k) = v;
    } else {
      typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
      uint32_t h[4], l[4];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        h[e] = f32_to_bf16_rne(v[e]);
        if constexpr (MODE == 2) l[e] = f32_to_bf16_rne(v[e] - bf16_bits_to_f32((uint16_t)h[e]));
      }
      *reinterpret_cast<u32x2*>(hi + r * LDK + k) = u32x2{h[0] | h[1] << 16, h[2] | h[3] << 16};
      if constexpr (MODE == 2) *reinterpret_cast<u32x2*>(lo + r * LDK + k) = u32x2{l[0] | l[1] << 16, l[2] | l[3] << 16};
    }
  };
  auto lstore = [&]() {
    ma.rows([&](int r, int k, f32x4 v) { put(As[0], As[NSPLIT - 1], r, k, v); });
    mb.rows([&](int r, int k, f32x4 v) { put(Bs[0], Bs[NSPLIT - 1], r, k, v); });
  };

  f32x16 acc;
#pragma unroll
  for (int v = 0; v < 16; v++) acc[v] = 0.f;

  const int fr = lane & 31, fk = lane >> 5;
  const int oa = (wm * 32 + fr) * LDK, ob = (wn * 32 + fr) * LDK;
  if (kt0 < kt1) {
    gload(kt0);
    lstore();
  }
  __syncthreads();
  for (int kt = kt0; kt < kt1; kt++) {
    if (kt + 1 < kt1) gload(kt + 1);
    if constexpr (MODE == 0) {
      // a lane's fragments of four K steps are one 16-byte read: half fk takes k = ks + 4 fk + q at step q
#pragma unroll
      for (int ks = 0; ks < BK; ks += 8) {
        const f32x4 af = *reinterpret_cast<const f32x4*>(&As[0][oa + ks + 4 * fk]);
        const f32x4 bf = *reinterpret_cast<const f32x4*>(&Bs[0][ob + ks + 4 * fk]);
#pragma unroll
        for (int q = 0; q < 4; q++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(af[q], bf[q], acc, 0, 0, 0);
      }
    } else {
#pragma unroll
      for (int ks = 0; ks < BK; ks += 16) {
        const bf16x8 ah = *reinterpret_cast<const bf16x8*>(&As[0][oa + ks + fk * 8]);
        const bf16x8 bh = *reinterpret_cast<const bf16x8*>(&Bs[0][ob + ks + fk * 8]);
        if constexpr (MODE == 2) {
          const bf16x8 al = *reinterpret_cast<const bf16x8*>(&As[NSPLIT - 1][oa + ks + fk * 8]);
          const bf16x8 bl = *reinterpret_cast<const bf16x8*>(&Bs[NSPLIT - 1][ob + ks + fk * 8]);
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, bh, acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bl, acc, 0, 0, 0);
        }
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bh, acc, 0, 0, 0);
      }
    }
    __syncthreads();
    if (kt + 1 < kt1) {
      lstore();
      __syncthreads();
    }
  }
  // accumulator layout of a 32 x 32 MFMA tile: lane l holds column l % 32, rows 8 * (v / 4) + 4 * (l / 32) + v % 4
  const int64_t col = n0 + wn * 32 + fr;
  if (col >= D.N) return;
#pragma unroll
  for (int v = 0; v < 16; v++) {
    const int64_t row = m0 + wm * 32 + 8 * (v / 4) + 4 * fk + (v % 4);
    if (row < D.M) {
      float* p = C + row * D.ldc + col;
      *p = beta == 0.f ? alpha * acc[v] : fmaf(beta, *p, alpha * acc[v]);
    }
  }
}

// fp64 (cblas_gemm_wrapper_'s double overload -> cblas_dgemm, bcl/containers/algorithms/cblas_wrapper.hpp:29-40):
// each wavefront owns 2 x 2 tiles of 16 x 16 computed by v_mfma_f64_16x16x4f64 (fp64 products and sums). Blocks of
// 128 x 128 (two per CU at most) were slower at every size from 64 to 4096 (4096^3: 2.47 ms against 2.27).
template <bool AKC, bool BKC>
__global__ __launch_bounds__(kGThreads, 3) void k_gemm_f64_direct(DirectArgs D, const double* __restrict__ A,
                                                               const double* __restrict__ B, double alpha, double beta,
                                                               double* C) {
  constexpr int TT = 2, BK = kDirectBK64, LDK = BK + 2, BM = kDirectTile;
  __shared__ __align__(16) double As[BM * LDK];
  __shared__ __align__(16) double Bs[BM * LDK];
  int tm, tn;
  gemm_tile_of(blockIdx.x, D.tiles_m, D.tiles_n, tm, tn);
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BM;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int nk = (int)((D.K + BK - 1) / BK);
  const int kt0 = (int)blockIdx.z * D.kt_per_split;
  const int kt1 = min(nk, kt0 + D.kt_per_split);
  C += (int64_t)blockIdx.z * D.split_stride;
  MicroTiles<double, 2, BM, BK, AKC> ma;
  MicroTiles<double, 2, BM, BK, BKC> mb;
  ma.init(m0, D.M);
  mb.init(n0, D.N);
  auto gload = [&](int kt) {
    const int64_t k0 = (int64_t)kt * BK;
    const bool k_whole = k0 + BK <= D.K;
    ma.load(A, D.lda, m0, k0, D.M, D.K, k_whole);
    mb.load(B, D.ldb, n0, k0, D.N, D.K, k_whole);
  };
  auto lstore = [&]() {
    ma.rows([&](int r, int k, f64x2 v) { *reinterpret_cast<f64x2*>(&As[r * LDK + k]) = v; });
    mb.rows([&](int r, int k, f64x2 v) { *reinterpret_cast<f64x2*>(&Bs[r * LDK + k]) = v; });
  };
  f64x4 acc[TT][TT];
#pragma unroll
  for (int a = 0; a < TT; a++)
#pragma unroll
    for (int c = 0; c < TT; c++) acc[a][c] = f64x4{0.0, 0.0, 0.0, 0.0};
  const int fr = lane & 15, fk = lane >> 4;  // operand lane layout: row (or column) fr, k offset fk
  if (kt0 < kt1) {
    gload(kt0);
    lstore();
  }
  __syncthreads();
  for (int kt = kt0; kt < kt1; kt++) {
    if (kt + 1 < kt1) gload(kt + 1);
    // a lane's fragments of two K steps are one 16-byte read: lane group fk takes k = ks + 2 fk + q at step q
#pragma unroll
    for (int ks = 0; ks < BK; ks += 8) {
      f64x2 af[TT], bf[TT];
#pragma unroll
      for (int t = 0; t < TT; t++) {
        af[t] = *reinterpret_cast<const f64x2*>(&As[(wm * 16 * TT + t * 16 + fr) * LDK + ks + 2 * fk]);
        bf[t] = *reinterpret_cast<const f64x2*>(&Bs[(wn * 16 * TT + t * 16 + fr) * LDK + ks + 2 * fk]);
      }
#pragma unroll
      for (int q = 0; q < 2; q++)
#pragma unroll
        for (int a = 0; a < TT; a++)
#pragma unroll
          for (int c = 0; c < TT; c++)
            acc[a][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[a][q], bf[c][q], acc[a][c], 0, 0, 0);
    }
    __syncthreads();
    if (kt + 1 < kt1) {
      lstore();
      __syncthreads();
    }
  }
  // accumulator layout of a 16 x 16 fp64 tile: lane l holds column l % 16, rows l / 16 + 4 * v
  static_for<0, TT>([&](auto ac) {
    constexpr int a = decltype(ac)::value;
    static_for<0, TT>([&](auto cc) {
      constexpr int c = decltype(cc)::value;
      const int64_t col = n0 + wn * 16 * TT + c * 16 + fr;
      static_for<0, 4>([&](auto vc) {
        constexpr int v = decltype(vc)::value;
        const int64_t row = m0 + wm * 16 * TT + a * 16 + fk + 4 * v;
        if (row < D.M && col < D.N) {
          double* p = C + row * D.ldc + col;
          *p = beta == 0.0 ? alpha * acc[a][c][v] : fma(beta, *p, alpha * acc[a][c][v]);
        }
      });
    });
  });
}

// C = beta * C + alpha * (sum of the splits' partial products, in order)
template <typename T>
__global__ __launch_bounds__(256) void k_gemm_reduce(const T* ws, int splits, int64_t M, int64_t N, T alpha, T beta,
                                                     T* C, int64_t ldc) {
  const int64_t total = M * N;
  for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < total; t += (int64_t)gridDim.x * 256) {
    T sum = ws[t];
    for (int z = 1; z < splits; z++) sum += ws[(int64_t)z * total + t];
    T* p = C + t / N * ldc + t % N;
    *p = beta == T(0) ? alpha * sum : fma(beta, *p, alpha * sum);
  }
}

template <typename T>
static void reduce_splits(bclx_handle* h, const T* ws, int splits, int64_t M, int64_t N, T alpha, T beta, T* C,
                          int64_t ldc) {
  const unsigned g = (unsigned)std::min<int64_t>(div_up(M * N, 256), (int64_t)h->num_cus * 8);
  hipLaunchKernelGGL((k_gemm_reduce<T>), dim3(g), dim3(256), 0, h->stream, ws, splits, M, N, alpha, beta, C, ldc);
  BCLX_HIP(hipGetLastError());
}

// Do the rows x cols elements of C (leading dimension ldc) share memory with an operand's?
template <typename T>
static bool overlaps(const T* C, int64_t rows, int64_t cols, int64_t ldc, const T* X, int64_t xrows, int64_t xcols,
                     int64_t ldx) {
  if (xrows <= 0 || xcols <= 0) return false;
  const uintptr_t c0 = reinterpret_cast<uintptr_t>(C), c1 = c0 + sizeof(T) * (size_t)((rows - 1) * ldc + cols);
  const uintptr_t x0 = reinterpret_cast<uintptr_t>(X), x1 = x0 + sizeof(T) * (size_t)((xrows - 1) * ldx + xcols);
  return c0 < x1 && x0 < c1;
}

// K tiles of bk in about `splits` equal parts, one grid layer each; launch(D, grid, alpha, beta, C). `apart`: C may
// share memory with an operand, so no block may write it while others read.
template <typename T, typename LAUNCH>
static void direct_run(bclx_handle* h, DirectArgs D, int bk, int splits, bool apart, T alpha, T beta, T* C,
                       LAUNCH&& launch) {
  D.tiles_m = (int)((D.M + kDirectTile - 1) / kDirectTile);
  D.tiles_n = (int)((D.N + kDirectTile - 1) / kDirectTile);
  const int64_t nk = (D.K + bk - 1) / bk;
  D.kt_per_split = (int)std::max<int64_t>(1, (nk + splits - 1) / splits);
  splits = (int)std::max<int64_t>(1, (nk + D.kt_per_split - 1) / D.kt_per_split);
  const dim3 grid((unsigned)(D.tiles_m * D.tiles_n), 1, (unsigned)splits);
  if (splits > 1 || apart) {  // partial products into the workspace, scaled and added to C afterwards
    T* ws = reinterpret_cast<T*>(dense_scratch(h, sizeof(T) * (size_t)splits * (size_t)(D.M * D.N)));
    const int64_t ldc = D.ldc;
    D.ldc = D.N;
    D.split_stride = D.M * D.N;
    launch(D, grid, T(1), T(0), ws);
    BCLX_HIP(hipGetLastError());
    reduce_splits<T>(h, ws, splits, D.M, D.N, alpha, beta, C, ldc);
  } else {
    launch(D, grid, alpha, beta, C);
    BCLX_HIP(hipGetLastError());
  }
}

// f(A contiguous along K, B contiguous along K) as compile-time constants
template <typename F>
static void with_layout(bool ta, bool tb, F&& f) {
  if (!ta && !tb) f(std::true_type{}, std::false_type{});
  else if (!ta) f(std::true_type{}, std::true_type{});
  else if (!tb) f(std::false_type{}, std::false_type{});
  else f(std::false_type{}, std::true_type{});
}

template <int MODE>
static void gemm_direct(bclx_handle* h, const DirectArgs& D, bool ta, bool tb, int splits, float alpha, const float* A,
                        const float* B, float beta, float* C) {
  direct_run<float>(h, D, kDirectBK, splits, false, alpha, beta, C,
                    [&](const DirectArgs& d, dim3 grid, float al, float be, float* out) {
    with_layout(ta, tb, [&](auto ac, auto bc) {
      hipLaunchKernelGGL((k_gemm_direct<MODE, decltype(ac)::value, decltype(bc)::value>), grid, dim3(kGThreads), 0,
                         h->stream, d, A, B, al, be, out);
    });
  });
}

static void gemm_f64_direct(bclx_handle* h, const DirectArgs& D, bool ta, bool tb, int splits, bool apart, double alpha,
                            const double* A, const double* B, double beta, double* C) {
  direct_run<double>(h, D, kDirectBK64, splits, apart, alpha, beta, C,
                     [&](const DirectArgs& d, dim3 grid, double al, double be, double* out) {
    with_layout(ta, tb, [&](auto ac, auto bc) {
      hipLaunchKernelGGL((k_gemm_f64_direct<decltype(ac)::value, decltype(bc)::value>), grid, dim3(kGThreads), 0,
                         h->stream, d, A, B, al, be, out);
    });
  });
}

// FP64 reference: C += A * B (fp32 inputs widened exactly), 16 x 16 tiles, row-major. Error oracle only.
__global__ __launch_bounds__(256) void k_gemm_f64_ref(int64_t M, int64_t N, int64_t K, const float* A, int64_t lda,
                                                      const float* B, int64_t ldb, double* C, int64_t ldc) {
  __shared__ double as[16][17], bs[16][17];
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int64_t row = (int64_t)blockIdx.y * 16 + ty, col = (int64_t)blockIdx.x * 16 + tx;
  double s = 0.0;
  for (int64_t k0 = 0; k0 < K; k0 += 16) {
    as[ty][tx] = (row < M && k0 + tx < K) ? (double)A[row * lda + k0 + tx] : 0.0;
    bs[ty][tx] = (k0 + ty < K && col < N) ? (double)B[(k0 + ty) * ldb + col] : 0.0;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 16; q++) s = fma(as[ty][q], bs[q][tx], s);
    __syncthreads();
  }
  if (row < M && col < N) C[row * ldc + col] += s;
}

// Can k_pack read an operand 16 bytes at a time?
static int pack_vec(const float* p, int64_t ld) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0 && ld % 4 == 0; }

// Pack both operands, then the packed kernel.
template <int MODE, int TM, int TN>
static void gemm_run(bclx_handle* h, bool ta, bool tb, int64_t m, int64_t n, int64_t k, float alpha, const float* A,
                     int64_t lda, const float* B, int64_t ldb, float beta, float* C, int64_t ldc) {
  using E = typename GemmCfg<MODE>::E;
  constexpr int BK = GemmCfg<MODE>::BK, BM = 64 * TM, BN = 64 * TN;
  const int64_t Mp = (m + BM - 1) / BM * BM, Np = (n + BN - 1) / BN * BN;
  const int64_t Kp = std::max<int64_t>(BK, (k + BK - 1) / BK * BK);
  const size_t a_bytes = (size_t)Mp * Kp * sizeof(E), b_bytes = (size_t)Np * Kp * sizeof(E);
  const size_t lo_a = MODE == 2 ? (size_t)Mp * Kp * 2 : 0, lo_b = MODE == 2 ? (size_t)Np * Kp * 2 : 0;
  const size_t off_b = (a_bytes + 255) / 256 * 256, off_la = off_b + (b_bytes + 255) / 256 * 256;
  const size_t off_lb = off_la + (lo_a + 255) / 256 * 256, total = off_lb + lo_b + 256;
  char* ws = dense_scratch(h, total);
  E* Ap = reinterpret_cast<E*>(ws);
  E* Bp = reinterpret_cast<E*>(ws + off_b);
  uint16_t* Al = MODE == 2 ? reinterpret_cast<uint16_t*>(ws + off_la) : nullptr;
  uint16_t* Bl = MODE == 2 ? reinterpret_cast<uint16_t*>(ws + off_lb) : nullptr;
  // op(A)[i][kk] = ta ? A[kk * lda + i] : A[i * lda + kk]; Bp[j][kk] = op(B)[kk][j] = tb ? B[j * ldb + kk] : B[kk * ldb + j]
  dim3 blk(256);
  hipLaunchKernelGGL(k_pack<MODE>, dim3((unsigned)div_up(Kp, 64), (unsigned)div_up(Mp, 64)), blk, 0, h->stream, A, m, k,
                     ta ? (int64_t)1 : lda, ta ? lda : (int64_t)1, (void*)Ap, Al, Mp, Kp, pack_vec(A, lda));
  BCLX_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_pack<MODE>, dim3((unsigned)div_up(Kp, 64), (unsigned)div_up(Np, 64)), blk, 0, h->stream, B, n, k,
                     tb ? ldb : (int64_t)1, tb ? (int64_t)1 : ldb, (void*)Bp, Bl, Np, Kp, pack_vec(B, ldb));
  BCLX_HIP(hipGetLastError());
  const int tiles_m = (int)(Mp / BM), tiles_n = (int)(Np / BN);
  hipLaunchKernelGGL((k_gemm<MODE, TM, TN>), dim3((unsigned)(tiles_m * tiles_n)), dim3(kGThreads), 0, h->stream, Ap,
                     (const E*)Al, Bp, (const E*)Bl, m, n, Kp, alpha, beta, C, ldc, tiles_m, tiles_n);
  BCLX_HIP(hipGetLastError());
}

// Predicted microseconds of a kernel: `packed` (with its two pack passes) or direct, C tiles of bm x bn, `per` and
// `per_block` = a K tile of 64 on one CU: fixed and for each block that shares the CU. The constants are fitted to
// square, ragged, flat and deep products from 64 to 8192 (within about 15%): what decides is how many blocks a CU
// gets, what a K tile costs a block alone (its load latency) and what the pack passes or the K splits' sum cost.
struct GemmCost {
  bool packed;
  int bm, bn;
  double per, per_block;
};
struct GemmPlan {
  double us;
  int splits;
};
// w: bytes of an element of C; pack_bytes: read and written per packed element
static GemmPlan gemm_cost(const bclx_handle* h, const GemmCost& c, int64_t m, int64_t n, int64_t k, int w,
                          int pack_bytes) {
  const double nk = std::max<double>(1.0, std::ceil((double)k / 64));
  const double tiles = std::ceil((double)m / c.bm) * std::ceil((double)n / c.bn);
  GemmPlan best{0, 0};
  for (int s = 1; s <= 64 && (s == 1 || (!c.packed && 2 * s <= nk)); s *= 2) {
    const double load = tiles * s / h->num_cus;
    // the fullest CU decides; the packed bf16 kernels wait more for memory, which the emptier CUs leave to them
    const double blocks = c.packed ? 0.5 * (std::ceil(load) + std::max(1.0, load)) : std::ceil(load);
    double us = 3 + std::ceil(nk / s) * (c.per + c.per_block * blocks);
    if (s > 1) us += 3 + (2 * s + 2) * (double)m * (double)n * w / 5e6;
    if (c.packed) us += 6 + (double)(m + n) * (double)k * pack_bytes / 4e6;
    if (best.splits == 0 || us < 0.95 * best.us) best = {us, s};
  }
  return best;
}

// Direct kernels where they are predicted faster, and smaller packed tiles where 128 x 128 leave CUs idle. The
// 128 x 128 (bf16: 256 x 128) packed kernel is the one for large products; the others have to beat it by 10%.
// Measured, us, packed 128 x 128 against the choice made here: fp32 2000 x 1500 x 3001 255 -> 174 (direct), 489 x 93 x
// 3552 268 -> 16 (direct, K split), 4096^3 1108 (packed; direct 1200); bf16 1500^3 46 -> 39 (packed 64 x 64), 512^3
// 24 -> 11 (direct); split-bf16 947 x 1486 x 2519 102 -> 61 (packed 64 x 64).
template <int MODE>
static void gemm_impl(bclx_handle* h, bool ta, bool tb, int64_t m, int64_t n, int64_t k, float alpha, const float* A,
                      int64_t lda, const float* B, int64_t ldb, float beta, float* C, int64_t ldc) {
  constexpr int pack_bytes = MODE == 1 ? 6 : 8;
  constexpr GemmCost large{true, 128, 128, MODE == 0 ? 0.6 : MODE == 1 ? 0.55 : 0.35,
                           MODE == 0 ? 3.9 : MODE == 1 ? 0.56 : 1.45};
  constexpr GemmCost small{true, 64, 64, MODE == 1 ? 0.3 : 0.1, MODE == 1 ? 0.225 : 0.46};
  constexpr GemmCost direct{false, 64, 64, MODE == 0 ? 0.4 : MODE == 1 ? 0.85 : 1.45,
                            MODE == 0 ? 1.1 : MODE == 1 ? 0.5 : 0.95};
  const DirectArgs D{m, n, k, lda, ldb, ldc, 0, 0, 0, 0};
  const double us_large = gemm_cost(h, large, m, n, k, 4, pack_bytes).us;
  GemmPlan d = gemm_cost(h, direct, m, n, k, 4, pack_bytes);
  // the packed kernels read only their copies of A and B, so C may share memory with them
  if (overlaps(C, m, n, ldc, A, ta ? k : m, ta ? m : k, lda) || overlaps(C, m, n, ldc, B, tb ? n : k, tb ? k : n, ldb))
    d.us = HUGE_VAL;
  if constexpr (MODE == 0) {
    if (d.us < 0.98 * us_large) gemm_direct<0>(h, D, ta, tb, d.splits, alpha, A, B, beta, C);
    else gemm_run<0, 2, 2>(h, ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
  } else {
    const bool big = MODE == 1 && ((m + 255) / 256) * ((n + 127) / 128) >= 2 * (int64_t)h->num_cus;
    const double us_small = gemm_cost(h, small, m, n, k, 4, pack_bytes).us;
    if (big) gemm_run<1, 4, 2>(h, ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
    else if (d.us < 0.9 * us_large && d.us < us_small) gemm_direct<MODE>(h, D, ta, tb, d.splits, alpha, A, B, beta, C);
    else if (us_small < 0.9 * us_large) gemm_run<MODE, 1, 1>(h, ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
    else gemm_run<MODE, 2, 2>(h, ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
  }
}

// fp64, us, against packed operands and 128 x 128 blocks: 512^3 103 -> 17, 1234 x 2048 x 1777 355 -> 181, 4096^3 2940 ->
// 2175 (63 TFLOP/s of the 72.6 that the vendor library reaches at 8192^3).
static void gemm_f64_run(bclx_handle* h, bool ta, bool tb, int64_t m, int64_t n, int64_t k, double alpha,
                         const double* A, int64_t lda, const double* B, int64_t ldb, double beta, double* C,
                         int64_t ldc) {
  constexpr GemmCost direct{false, 64, 64, 1.56, 1.72};
  const GemmPlan d = gemm_cost(h, direct, m, n, k, 8, 0);
  const bool apart = overlaps(C, m, n, ldc, A, ta ? k : m, ta ? m : k, lda) ||
                     overlaps(C, m, n, ldc, B, tb ? n : k, tb ? k : n, ldb);
  gemm_f64_direct(h, DirectArgs{m, n, k, lda, ldb, ldc, 0, 0, 0, 0}, ta, tb, d.splits, apart, alpha, A, B, beta, C);
}

}  // namespace bclx

using namespace bclx;

extern "C" {

bclx_status bclx_gemm(bclx_handle* h, int32_t trans_a, int32_t trans_b, int64_t m, int64_t n, int64_t k, float alpha,
                      const float* d_A, int64_t lda, const float* d_B, int64_t ldb, float beta, float* d_C,
                      int64_t ldc, int32_t mode) {
  return guarded([&] {
    BCLX_REQUIRE(h && d_C, BCLX_ERR_INVALID, "null handle or C");
    BCLX_REQUIRE(m >= 0 && n >= 0 && k >= 0, BCLX_ERR_INVALID, "negative size");
    BCLX_REQUIRE(mode >= 0 && mode <= 2, BCLX_ERR_INVALID, "mode must be 0 (fp32), 1 (bf16) or 2 (split-bf16)");
    BCLX_REQUIRE(ldc >= n, BCLX_ERR_INVALID, "ldc < n");
    BCLX_REQUIRE(lda >= (trans_a ? m : k) && ldb >= (trans_b ? k : n), BCLX_ERR_INVALID, "lda / ldb too small");
    BCLX_REQUIRE(k == 0 || (d_A && d_B), BCLX_ERR_INVALID, "null A or B");
    set_device(h);
    if (m == 0 || n == 0) return;  // k == 0 packs zeros, so C = beta * C
    const bool ta = trans_a != 0, tb = trans_b != 0;
    switch (mode) {
      case 0: gemm_impl<0>(h, ta, tb, m, n, k, alpha, d_A, lda, d_B, ldb, beta, d_C, ldc); break;
      case 1: gemm_impl<1>(h, ta, tb, m, n, k, alpha, d_A, lda, d_B, ldb, beta, d_C, ldc); break;
      default: gemm_impl<2>(h, ta, tb, m, n, k, alpha, d_A, lda, d_B, ldb, beta, d_C, ldc); break;
    }
  });
}

bclx_status bclx_gemm_f64(bclx_handle* h, int32_t trans_a, int32_t trans_b, int64_t m, int64_t n, int64_t k,
                          double alpha, const double* d_A, int64_t lda, const double* d_B, int64_t ldb, double beta,
                          double* d_C, int64_t ldc) {
  return guarded([&] {
    BCLX_REQUIRE(h && d_C, BCLX_ERR_INVALID, "null handle or C");
    BCLX_REQUIRE(m >= 0 && n >= 0 && k >= 0, BCLX_ERR_INVALID, "negative size");
    BCLX_REQUIRE(ldc >= n, BCLX_ERR_INVALID, "ldc < n");
    BCLX_REQUIRE(lda >= (trans_a ? m : k) && ldb >= (trans_b ? k : n), BCLX_ERR_INVALID, "lda / ldb too small");
    BCLX_REQUIRE(k == 0 || (d_A && d_B), BCLX_ERR_INVALID, "null A or B");
    set_device(h);
    if (m == 0 || n == 0) return;
    gemm_f64_run(h, trans_a != 0, trans_b != 0, m, n, k, alpha, d_A, lda, d_B, ldb, beta, d_C, ldc);
  });
}

bclx_status bclx_gemm_f64_ref(bclx_handle* h, int64_t m, int64_t n, int64_t k, const float* d_A, int64_t lda,
                              const float* d_B, int64_t ldb, double* d_C, int64_t ldc) {
  return guarded([&] {
    BCLX_REQUIRE(h && d_A && d_B && d_C && m >= 0 && n >= 0 && k >= 0, BCLX_ERR_INVALID, "bad argument");
    set_device(h);
    if (m == 0 || n == 0) return;
    hipLaunchKernelGGL(k_gemm_f64_ref, dim3(div_up(n, 16), div_up(m, 16)), dim3(256), 0, h->stream, m, n, k, d_A,
                       lda, d_B, ldb, d_C, ldc);
    BCLX_HIP(hipGetLastError());
  });
}

}  // extern "C"
