// SpMM: C[i*ldc + j] = beta * C + alpha * sum_k A[i,k] * B[k*ldb + j], j < n (bclx_spmm).
//
// The reference's spmm_wrapper (bcl/containers/algorithms/spgemm.hpp:78-96, :140-149) is alpha = beta = 1 with
// row-major B and C and explicit ldb / ldc (DMatrix tiles padded to the full tile width).
//
// Work split: a block takes consecutive entries of A (2048, or 512: spmm_launch) and one slice of C's
// columns; groups of LPE lanes, each lane 16 bytes of a B row, share the entries out, each walking its run in order. A
// wavefront so gathers the B rows of 64 / LPE entries with one load instruction, and narrow products use fewer lanes
// per entry instead of leaving them idle.
// The block stages its entries in LDS: columns and values, and each entry's row, found from row_ptr by marking the
// first entry of every row and a running maximum.
// What bounds it is how C is written, then the gathers: a row whose entries lie in one block and are no more than a
// group's run belongs to one group, which adds it with a plain load (issued with the gathers) and store. Only rows that
// are cut (long ones, and those at a block's ends) are added with atomics. With atomics for every row the same kernel
// takes 1707 us on R-MAT scale 20 x 128 fp32 columns and 2825 us with bf16 B; 899 and 578 us this way (a wavefront per
// 256 entries, whole rows of 128 columns, atomics: 1486 and 1541). (Rows and columns rotated; with the hubs at row and
// column 0, where R-MAT puts them, 1061 and 659 us.)
// B is fp32 or bf16 (converted on load) with fp32 accumulation, or, for the fp64 product (bclx_spmm_f64, the
// reference's double spmm_wrapper, spgemm.hpp:119-149), fp64 throughout.
#include <algorithm>
#include <type_traits>

#include "internal.hpp"

namespace bclx {

constexpr int kSpmmThreads = 256;

// Largest r in [0, m) with rp[r] <= e, 0 if there is none: one wavefront, 64 probes a round.
template <typename RP>
__device__ inline int64_t spmm_row_of(const RP* rp, int64_t m, int64_t e, int lane) {
  int64_t lo = 0, len = m;
  while (len > 1) {
    const int64_t step = (len + 63) / 64;
    const int64_t q = lo + lane * step;
    const bool le = q < lo + len && (int64_t)rp[q] <= e;
    const int hits = (int)__popcll(__ballot(le)), k = hits > 0 ? hits - 1 : 0;  // rp is monotone: hits come first
    const int64_t end = lo + len;
    lo += k * step;
    len = step < end - lo ? step : end - lo;
  }
  return lo;
}

// VT: A's values, the accumulation and C (float, or double for the fp64 product); BT: B (VT, or bf16 under float).
// LPE lanes of VEC columns per entry; slice y (from slice0) covers columns [y * LPE * VEC, ...). Needs n >= VEC: a lane
// whose columns would pass n starts at n - VEC. EPB: entries per block. FRESH: C's rows that other blocks share hold
// zeros and the others anything (beta 0), so a row's sum is stored without reading C.
template <typename RP, typename VT, typename BT, int LPE, int VEC, int EPB, bool FRESH>
__global__ __launch_bounds__(kSpmmThreads) void k_spmm(const RP* __restrict__ rp, const int* __restrict__ col,
                                                       const VT* __restrict__ val, int64_t m, int64_t nnz,
                                                       const BT* __restrict__ B, int64_t ldb, VT* C, int64_t ldc, int n,
                                                       int slice0, VT alpha) {
  constexpr int GROUPS = kSpmmThreads / LPE;
  constexpr int RUN = EPB / GROUPS;  // consecutive entries of a group
  constexpr int PER = EPB / kSpmmThreads;
  constexpr int COLS = LPE * VEC;
  constexpr int kUnroll = VEC == 8 && !FRESH ? 4 : 8;      // (8 with eight fp32 columns of C per lane spill occupancy)
  constexpr int U = RUN < kUnroll ? RUN : kUnroll;          // gathers in flight per group
  constexpr int PADDED = EPB + GROUPS + U;  // one word between the groups' runs: they start on different banks
  typedef BT vec_t __attribute__((ext_vector_type(VEC), aligned(sizeof(BT))));
  typedef VT cvec_t __attribute__((ext_vector_type(VEC), aligned(sizeof(VT))));
  __shared__ int s_col[PADDED];
  __shared__ VT s_val[PADDED];
  // per entry: first slot of its row in the block << 1 | shared. Entries of no row (rp may start above 0 or end below nnz)
  // count as a shared row that is not listed in s_shared.
  __shared__ uint16_t s_row[PADDED];
  __shared__ int s_id[EPB];           // at a row's first slot: the row, relative to the block's first
  __shared__ VT s_sum[GROUPS + 1][COLS];  // sums of the rows that several groups share
  __shared__ int s_shared[GROUPS + 1];    // those rows << 1 | crosses the block's ends, or -1
  __shared__ int64_t s_first;
  __shared__ int s_scan[kSpmmThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int64_t e0 = (int64_t)blockIdx.x * EPB;
  const int cnt = (int)(nnz - e0 < EPB ? nnz - e0 : EPB);
  auto slot = [](int q) { return q + q / RUN; };
  // a shared row's place in s_sum: two such rows start more than RUN apart, but for the row that the block starts in
  auto place = [](int first) { return first == 0 ? 0 : 1 + first / RUN; };
#pragma unroll
  for (int q = 0; q < PER; q++) {
    const int x = q * kSpmmThreads + tid;
    s_col[slot(x)] = x < cnt ? col[e0 + x] : 0;
    s_val[slot(x)] = x < cnt ? val[e0 + x] : VT(0);
    s_row[slot(x)] = x == 0 ? 1 : 0;
  }
  if (tid < U) s_col[PADDED - U + tid] = 0;  // read, not used, by the last group
  for (int x = tid; x < (GROUPS + 1) * COLS; x += kSpmmThreads) s_sum[x / COLS][x % COLS] = VT(0);
  for (int x = tid; x <= GROUPS; x += kSpmmThreads) s_shared[x] = -1;
  if (tid < 64) {
    const int64_t r = spmm_row_of(rp, m, e0, lane);
    if (lane == 0) s_first = r;
  }
  __syncthreads();
  // rows of the entries: shared when the row has entries in another block or more than one group's run here
  const int64_t r0 = s_first;
  for (int64_t w = r0; w <= m; w += kSpmmThreads) {
    const int64_t r = w + tid;  // row m: the entries after the last row, which are not listed
    const int64_t b = r <= m ? (int64_t)rp[r] - e0 : cnt, e = r < m ? (int64_t)rp[r + 1] - e0 : cnt;
    if (b < cnt && e > b && e > 0) {
      const int first = b > 0 ? (int)b : 0;
      const bool cross = b < 0 || e > cnt, sh = cross || e - b > RUN || r == m;
      s_row[slot(first)] = (uint16_t)(first << 1 | (sh ? 1 : 0));
      s_id[first] = (int)(r - r0);
      if (sh && r < m) s_shared[place(first)] = (int)(r - r0) << 1 | (cross ? 1 : 0);
    }
    if (__syncthreads_or(r < m && e >= cnt)) break;
  }
  {
    int run = 0;
#pragma unroll
    for (int q = 0; q < PER; q++) run = max(run, (int)s_row[slot(tid * PER + q)]);
    int inc = run;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int t = __shfl_up(inc, d, 64);
      if (lane >= d) inc = max(inc, t);
    }
    if (lane == 63) s_scan[tid >> 6] = inc;
    int before = __shfl_up(inc, 1, 64);
    if (lane == 0) before = 0;
    __syncthreads();
    for (int w = 0; w < (tid >> 6); w++) before = max(before, s_scan[w]);
#pragma unroll
    for (int q = 0; q < PER; q++) {
      const int x = slot(tid * PER + q);
      before = max(before, (int)s_row[x]);
      s_row[x] = (uint16_t)before;
    }
  }
  __syncthreads();
  const int g = tid / LPE, l = tid % LPE;
  // where the group whose run starts at q begins: past a row of its own that an earlier group began
  auto begin_of = [&](int q) {
    if (q >= cnt) return cnt;
    const int v = s_row[slot(q)];
    if (q == 0 || (v & 1) || s_row[slot(q - 1)] != v) return q;
    int lo = q, hi = q + RUN < cnt ? q + RUN : cnt;  // the row ends within one run of its start
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (s_row[slot(mid)] == v) lo = mid + 1;
      else hi = mid;
    }
    return lo;
  };
  const int q0 = begin_of(g * RUN), q1 = begin_of((g + 1) * RUN);
  const int cs = (slice0 + (int)blockIdx.y) * COLS;       // the slice's first column
  const int c_own = cs + l * VEC;                         // the lane's first column
  const int c0 = c_own < n - VEC ? c_own : n - VEC;       // where it reads
  const int skip = c_own - c0;                            // columns read to end at n, not its own
  const BT* Bc = B + c0;
  VT* Cc = C + r0 * ldc + c0;
  if (skip < VEC && q0 < q1) {
    VT acc[VEC];
#pragma unroll
    for (int v = 0; v < VEC; v++) acc[v] = VT(0);
    for (int j = q0; j < q1; j += U) {
      vec_t b[U];
      cvec_t c[U];
      VT a[U];
      int r[U + 1];
#pragma unroll
      for (int u = 0; u <= U; u++) r[u] = j + u < q1 ? (int)s_row[slot(j + u)] : -1;
      // entries past the run load too (their columns are valid, or 0): what they add to acc after the run's last row
      // is not used
#pragma unroll
      for (int u = 0; u < U; u++) {
        a[u] = s_val[slot(j + u)];
        b[u] = *reinterpret_cast<const vec_t*>(Bc + (int64_t)s_col[slot(j + u)] * ldb);
      }
      if (!FRESH) {  // the C rows that end in this batch
#pragma unroll
        for (int u = 0; u < U; u++)
          if (r[u] != r[u + 1] && !(r[u] & 1))
            c[u] = *reinterpret_cast<const cvec_t*>(Cc + (int64_t)s_id[r[u] >> 1] * ldc);
      }
      // one wait for the batch: a wait at each use would also wait for the stores in between (they share the counter)
      __builtin_amdgcn_s_waitcnt(0x0f70);
#pragma unroll
      for (int u = 0; u < U; u++) {
#pragma unroll
        for (int v = 0; v < VEC; v++) {
          if constexpr (sizeof(BT) == 2) acc[v] = fmaf(a[u], __uint_as_float((uint32_t)b[u][v] << 16), acc[v]);
          else acc[v] = fma(a[u], b[u][v], acc[v]);
        }
        if (r[u] != r[u + 1]) {  // the row's last entry in this run
          if (r[u] & 1) {
            VT* sum = s_sum[place(r[u] >> 1)] + (l * VEC - skip);
#pragma unroll
            for (int v = 0; v < VEC; v++)
              if (v >= skip) atomicAdd(&sum[v], acc[v]);
          } else {
            VT* cr = Cc + (int64_t)s_id[r[u] >> 1] * ldc;
            cvec_t o;
#pragma unroll
            for (int v = 0; v < VEC; v++) o[v] = FRESH ? alpha * acc[v] : fma(alpha, acc[v], c[u][v]);
            if (skip == 0) {
              *reinterpret_cast<cvec_t*>(cr) = o;
            } else {  // the first columns belong to another lane, perhaps of another block
#pragma unroll
              for (int v = 1; v < VEC; v++)
                if (v >= skip) cr[v] = o[v];
            }
          }
#pragma unroll
          for (int v = 0; v < VEC; v++) acc[v] = VT(0);
        }
      }
    }
  }
  __syncthreads();
  // the shared rows: a row that crosses the block's ends is added with atomics, the others are the block's own
  for (int x = tid; x < (GROUPS + 1) * COLS; x += kSpmmThreads) {
    const int id = s_shared[x / COLS], c = cs + x % COLS;
    if (id < 0 || c >= n) continue;
    VT* p = C + (r0 + (id >> 1)) * ldc + c;
    const VT v = alpha * s_sum[x / COLS][x % COLS];
    if (id & 1) __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else *p = FRESH ? v : *p + v;
  }
}

// C's rows that no block of EPB entries stores whole: empty rows, and rows with entries in two blocks (which are added
// to). One block of 256 rows lists them, then clears them together.
template <typename RP, typename VT>
__global__ __launch_bounds__(256) void k_spmm_clear(const RP* __restrict__ rp, int64_t m, int64_t nnz, int epb, VT* C,
                                                    int64_t ldc, int64_t n) {
  __shared__ int s_list[256];
  __shared__ int s_n;
  if (threadIdx.x == 0) s_n = 0;
  __syncthreads();
  const int64_t r0 = (int64_t)blockIdx.x * 256, r = r0 + threadIdx.x;
  if (r < m) {
    const int64_t b = (int64_t)rp[r], e = (int64_t)rp[r + 1];
    if (e <= b || e > nnz || b / epb != (e - 1) / epb) s_list[atomicAdd(&s_n, 1)] = threadIdx.x;
  }
  __syncthreads();
  for (int q = threadIdx.x >> 6; q < s_n; q += 4)
    for (int64_t c = threadIdx.x & 63; c < n; c += 64) C[(r0 + s_list[q]) * ldc + c] = VT(0);
}

template <typename VT>
__global__ void k_scale_rows(VT* C, int64_t m, int64_t n, int64_t ldc, VT beta) {
  const int64_t total = m * n;
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i = t / n, j = t % n;
    VT* p = C + i * ldc + j;
    *p = beta == VT(0) ? VT(0) : beta * *p;
  }
}

template <typename VT>
static void scale_rows(bclx_handle* h, VT* C, int64_t m, int64_t n, int64_t ldc, VT beta) {
  if (beta == VT(1) || m == 0 || n == 0) return;
  const int64_t total = m * n;
  hipLaunchKernelGGL((k_scale_rows<VT>), dim3((unsigned)std::min<int64_t>((total + 255) / 256, 65536)), dim3(256), 0,
                     h->stream, C, m, n, ldc, beta);
  BCLX_HIP(hipGetLastError());
}

template <typename RP, typename VT, typename BT, int LPE, int VEC>
static void spmm_launch(bclx_handle* h, const bclx_csr* A, const BT* B, int64_t ldb, VT* C, int64_t ldc, int64_t n,
                        VT alpha, bool fresh, bool whole_lines) {
  const RP* rp = static_cast<const RP*>(A->row_ptr);
  const int64_t slices = (n + LPE * VEC - 1) / (LPE * VEC);
  constexpr int64_t kMaxY = 32768;  // grid rows of one launch
  // 2048 entries per block (fp64: 1024, the same LDS) where that gives every CU four blocks (one, for narrow products,
  // whose groups' runs are short), else 512. Measured, us, 512 against 2048: 200 K rows of 9, fp32, 1 column 21.6 / 15.3,
  // 64 columns 72 / 68; 20 K rows of 9, 64 columns 15 / 34. Always 512 where wide rows of B are not whole lines
  // (100 K rows of 32, fp32, 33 columns 95 / 115, 129 columns 393 / 411; fp64, 33 columns 162 / 169).
  constexpr int kLarge = sizeof(VT) == 8 ? 1024 : 2048;
  const bool large = whole_lines && (A->nnz / kLarge) * slices >= (LPE <= 4 ? 1 : 4) * (int64_t)h->num_cus;
  const int epb = large ? kLarge : 512;
  if (fresh) {
    hipLaunchKernelGGL((k_spmm_clear<RP, VT>), dim3(div_up(A->m, 256)), dim3(256), 0, h->stream, rp, A->m, A->nnz, epb, C,
                       ldc, n);
    BCLX_HIP(hipGetLastError());
  }
  for (int64_t s0 = 0; s0 < slices; s0 += kMaxY) {
    const dim3 grid(div_up(A->nnz, epb), (unsigned)std::min(kMaxY, slices - s0));
    auto go = [&](auto e, auto fr) {
      hipLaunchKernelGGL((k_spmm<RP, VT, BT, LPE, VEC, decltype(e)::value, decltype(fr)::value>), grid,
                         dim3(kSpmmThreads), 0, h->stream, rp, A->col_idx, static_cast<const VT*>(A->vals), A->m, A->nnz,
                         B, ldb, C, ldc, (int)n, (int)s0, alpha);
      BCLX_HIP(hipGetLastError());
    };
    using L = std::integral_constant<int, kLarge>;
    using S = std::integral_constant<int, 512>;
    if (large) fresh ? go(L{}, std::true_type{}) : go(L{}, std::false_type{});
    else fresh ? go(S{}, std::true_type{}) : go(S{}, std::false_type{});
  }
}

// fresh: beta is 0, C is written anew
template <typename RP, typename VT, typename BT>
static void spmm_impl(bclx_handle* h, const bclx_csr* A, const void* Bv, int64_t ldb, VT* C, int64_t ldc, int64_t n,
                      VT alpha, bool fresh) {
  const BT* B = static_cast<const BT*>(Bv);
  if (n == 0 || A->m == 0) return;
  if (A->nnz == 0) {
    if (fresh) scale_rows<VT>(h, C, A->m, n, ldc, VT(0));
    return;
  }
#define BCLX_SPMM(LPE, VEC) spmm_launch<RP, VT, BT, LPE, VEC>(h, A, B, ldb, C, ldc, n, alpha, fresh, true)
#define BCLX_SPMM_LINES(LPE, VEC) spmm_launch<RP, VT, BT, LPE, VEC>(h, A, B, ldb, C, ldc, n, alpha, fresh, lines)
  // Slices of 256 bytes of a B row where rows are whole 128-byte lines: half as many lanes idle at odd widths and a
  // smaller B to gather from at a time (fp32 x 128 columns: 899 us against 1036 with 512-byte slices). Where rows are
  // not, a slice's ends share lines with its neighbours, and 512-byte slices gather fewer lines (fp32 x 100 columns, 200 K
  // rows of 9: 158 us against 203). Lanes of 16 bytes, but of 8 where fp32 rows are not 16-byte aligned (x 17 columns: 61 us
  // against 73) or are that narrow (more lanes per entry mean longer runs: x 16 columns 51 us against 64).
  const bool lines = n * (int64_t)sizeof(BT) % 128 == 0 && ldb * (int64_t)sizeof(BT) % 128 == 0 &&
                     reinterpret_cast<uintptr_t>(B) % 128 == 0;
  const bool vec16 = ldb * (int64_t)sizeof(BT) % 16 == 0 && reinterpret_cast<uintptr_t>(B) % 16 == 0;
  if constexpr (sizeof(BT) == 2) {
    if (n > 128 && !lines) BCLX_SPMM(32, 8);
    else if (n > 64) BCLX_SPMM(16, 8);
    else if (n > 32) BCLX_SPMM(8, 8);
    else if (n > 16) BCLX_SPMM(8, 4);
    else if (n > 8) BCLX_SPMM(4, 4);
    else if (n >= 4) BCLX_SPMM(2, 4);
    else if (n > 2) BCLX_SPMM(4, 1);
    else if (n > 1) BCLX_SPMM(2, 1);
    else BCLX_SPMM(1, 1);
  } else if constexpr (sizeof(BT) == 4) {
    if (n > 64 && !lines) BCLX_SPMM_LINES(32, 4);
    else if (n > 32 && !vec16) BCLX_SPMM_LINES(32, 2);
    else if (n > 32) BCLX_SPMM(16, 4);
    else if (n > 16 && !vec16) BCLX_SPMM(16, 2);
    else if (n > 16) BCLX_SPMM(8, 4);
    else if (n > 8) BCLX_SPMM(8, 2);
    else if (n > 4) BCLX_SPMM(4, 2);
    else if (n > 1) BCLX_SPMM(2, 2);
    else BCLX_SPMM(1, 1);
  } else {
    // fp64 rows that are not whole lines: slices of 1024 bytes where the last one is more than half used, else of 512
    // (200 K rows of 9, x 127 columns 361 us against 415, x 145 columns 506 against 478)
    if (n > 64 && !lines && (n - 1) % 128 >= 64) BCLX_SPMM_LINES(32, 4);
    else if (n > 32 && !lines) BCLX_SPMM_LINES(32, 2);
    else if (n > 16) BCLX_SPMM(16, 2);
    else if (n > 8) BCLX_SPMM(8, 2);
    else if (n > 4) BCLX_SPMM(4, 2);
    else if (n > 1) BCLX_SPMM(2, 2);
    else BCLX_SPMM(1, 1);
  }
#undef BCLX_SPMM_LINES
#undef BCLX_SPMM
}

}  // namespace bclx

using namespace bclx;

extern "C" {

bclx_status bclx_spmm(bclx_handle* h, const bclx_csr* A, const void* d_B, int32_t b_dtype, int64_t ldb, float* d_C,
                      int64_t ldc, int64_t n, float alpha, float beta) {
  return guarded([&] {
    BCLX_REQUIRE(h && A && d_C, BCLX_ERR_INVALID, "null argument");
    BCLX_REQUIRE(A->dtype == BCLX_F32, BCLX_ERR_INVALID, "A must hold fp32 values");
    BCLX_REQUIRE(A->ptr_width == 4 || A->ptr_width == 8, BCLX_ERR_INVALID, "A->ptr_width must be 4 or 8");
    BCLX_REQUIRE(b_dtype == BCLX_F32 || b_dtype == BCLX_BF16, BCLX_ERR_INVALID, "B must be fp32 or bf16");
    BCLX_REQUIRE(n >= 0 && ldb >= n && ldc >= n, BCLX_ERR_INVALID, "need ldb >= n and ldc >= n");
    BCLX_REQUIRE(A->nnz == 0 || (A->col_idx && A->vals && d_B), BCLX_ERR_INVALID, "null A arrays or B");
    set_device(h);
    if (beta != 0.f) scale_rows<float>(h, d_C, A->m, n, ldc, beta);
    if (A->ptr_width == 8) {
      if (b_dtype == BCLX_F32) spmm_impl<int64_t, float, float>(h, A, d_B, ldb, d_C, ldc, n, alpha, beta == 0);
      else spmm_impl<int64_t, float, uint16_t>(h, A, d_B, ldb, d_C, ldc, n, alpha, beta == 0);
    } else {
      if (b_dtype == BCLX_F32) spmm_impl<int32_t, float, float>(h, A, d_B, ldb, d_C, ldc, n, alpha, beta == 0);
      else spmm_impl<int32_t, float, uint16_t>(h, A, d_B, ldb, d_C, ldc, n, alpha, beta == 0);
    }
  });
}

bclx_status bclx_spmm_f64(bclx_handle* h, const bclx_csr* A, const double* d_B, int64_t ldb, double* d_C, int64_t ldc,
                          int64_t n, double alpha, double beta) {
  return guarded([&] {
    BCLX_REQUIRE(h && A && d_C, BCLX_ERR_INVALID, "null argument");
    BCLX_REQUIRE(A->dtype == BCLX_F64, BCLX_ERR_INVALID, "A must hold fp64 values");
    BCLX_REQUIRE(A->ptr_width == 4 || A->ptr_width == 8, BCLX_ERR_INVALID, "A->ptr_width must be 4 or 8");
    BCLX_REQUIRE(n >= 0 && ldb >= n && ldc >= n, BCLX_ERR_INVALID, "need ldb >= n and ldc >= n");
    BCLX_REQUIRE(A->nnz == 0 || (A->col_idx && A->vals && d_B), BCLX_ERR_INVALID, "null A arrays or B");
    set_device(h);
    if (beta != 0.0) scale_rows<double>(h, d_C, A->m, n, ldc, beta);
    if (A->ptr_width == 8) spmm_impl<int64_t, double, double>(h, A, d_B, ldb, d_C, ldc, n, alpha, beta == 0);
    else spmm_impl<int32_t, double, double>(h, A, d_B, ldb, d_C, ldc, n, alpha, beta == 0);
  });
}

}  // extern "C"
