// Tile ingest and dense tile arithmetic on the GPU (bclx_csr_split_grid, bclx_dense_binary_op).
//
// bclx_csr_split_grid cuts one CSR matrix resident in HBM into the tiles of a grid, the way SPMatrix's constructor
// slices a matrix read from a file into its tiles (SPMatrix::init_, bcl/containers/SPMatrix.hpp:212-266, through
// CSRMatrix::get_slice_impl_, bcl/containers/sequential/CSRMatrix.hpp:238-276): tile (ti, tj) holds rows
// [ti * tile_m, (ti + 1) * tile_m) and columns [tj * tile_n, (tj + 1) * tile_n) of A, columns shifted to start at 0,
// entries in their order in A. With 288 GB of HBM a whole matrix fits next to its tiles, so the cut is two passes over
// A on the GPU instead of one host slice per tile:
//   1. count: one thread per (row, tile column) finds where the tile column's segment of the row starts (binary
//      search; A's columns are sorted within each row) and writes that start and the segment length;
//   2. one scan over the lengths of all tile columns, one column after the other, turns them into offsets; a tile's
//      row_ptr is that scan restricted to its rows, minus the value at its first row;
//   3. copy: work is split by entries plus rows (kSplitChunk per workgroup), so hub, short and empty rows cost the same; a lane
//      finds its entry's row in a window of row offsets in LDS, its tile column by a division, and writes the entry to
//      its tile at (row offset + position in the segment).
// Bytes: A's row_ptr and col_idx are read twice (count, copy) and its values once; every tile is written once. Measured
// on R-MAT scale 20 (16.1 M entries, 4 x 4 tiles), sizes and copy together: 1.82 ms with one wavefront per row and
// one scan per tile column, 0.43 ms this way.
//
// bclx_dense_binary_op is DMatrix's elementwise arithmetic on a tile (DMatrix::binary_op / binary_op_inplace,
// bcl/containers/DMatrix.hpp:319-366, with operator+, -, *, / and += at :368-386): C = A op B per element, rows of
// ld-strided row-major tiles; C may be A (in place). HBM-bound streaming: 16-byte loads and stores where the rows
// are aligned, one pass.
#include <algorithm>
#include <vector>

#include "internal.hpp"
#include "spgemm.hpp"

namespace bclx {

constexpr int kSplitMaxGridN = 256;            // tile columns of one split
constexpr int kSplitChunk = 4096;              // entries plus rows of A per copying workgroup
constexpr int kSplitWindow = 1024;             // rows whose offsets a copying workgroup holds at a time

// Row i's segment of tile column tj: seg[tj * stride + i] = its first position within the row, cnt[...] its length.
// A block takes 256 / gn whole rows, so a segment's end is its neighbour's start. Also clears the counts that pad a
// tile column to the stride.
template <typename RP>
__global__ __launch_bounds__(256) void k_split_count(const RP* rp, const int32_t* col, int64_t m, int64_t tile_n,
                                                     int gn, int32_t* cnt, int32_t* seg, int64_t stride,
                                                     int32_t* bad) {
  __shared__ int s_lo[257];
  const int rows = 256 / gn;
  const int r = (int)threadIdx.x / gn, tj = (int)threadIdx.x - r * gn;
  const int64_t i = (int64_t)blockIdx.x * rows + r;
  const bool live = r < rows && i < m;
  if (blockIdx.x == 0 && threadIdx.x == 0) *bad = 0;
  int len = 0;
  if (live) {
    const int64_t a0 = (int64_t)rp[i], a1 = (int64_t)rp[i + 1];
    len = (int)(a1 - a0);
    int lo = 0, hi = tj == 0 ? 0 : len;  // first position with column >= tj * tile_n
    const int64_t bound = (int64_t)tj * tile_n;
    while (lo < hi) {
      const int mid = lo + (hi - lo) / 2;
      if ((int64_t)col[a0 + mid] < bound) lo = mid + 1;
      else hi = mid;
    }
    s_lo[threadIdx.x] = lo;
  }
  __syncthreads();
  if (live) {
    const int lo = s_lo[threadIdx.x], end = tj + 1 < gn ? s_lo[threadIdx.x + 1] : len;
    seg[(int64_t)tj * stride + i] = lo;
    cnt[(int64_t)tj * stride + i] = end > lo ? end - lo : 0;  // shorter than 0 only when the row is not sorted
    if (i == m - 1)
      for (int64_t q = m; q < stride; q++) cnt[(int64_t)tj * stride + q] = 0;
  }
}

struct SplitTile {
  void* rp;      // tile rows + 1 entries of ptr_width
  int32_t* col;
  void* val;
  int64_t nnz;   // entries the tile holds (from the counting pass)
  int32_t ptr_width;
};

struct SplitChunk {
  int64_t row, entry;  // where a chunk of A starts
};

// i / d, in 32 bits where the rows fit them
__device__ inline int64_t row_div(int64_t i, int64_t d, int64_t m) {
  return m <= (int64_t)UINT32_MAX && d <= (int64_t)UINT32_MAX ? (int64_t)((uint32_t)i / (uint32_t)d) : i / d;
}

// The tiles' row_ptrs from the scanned offsets: one thread per (tile column, row). The threads of tile column 0 also
// cut A into chunks of kSplitChunk entries plus rows: row i weighs its entries and one more; chunk[c] is the row
// that weight c * kSplitChunk falls in and the entry it stands for. The entries are counted from rp[0] on: A may be rows
// of a larger matrix, with its col_idx and vals.
template <typename RP>
__global__ __launch_bounds__(256) void k_split_rowptr(const RP* rp, const int64_t* off, int64_t stride, int64_t m,
                                                      int64_t tile_m, int gn, const SplitTile* tiles,
                                                      SplitChunk* chunk, int64_t nchunks) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int tj = blockIdx.y;
  if (i >= m) return;
  if (tj == 0) {
    const int64_t e0 = (int64_t)rp[0], a0 = (int64_t)rp[i] - e0, a1 = (int64_t)rp[i + 1] - e0;
    for (int64_t c = (a0 + i + kSplitChunk - 1) / kSplitChunk; c < nchunks && c * kSplitChunk <= a1 + i; c++)
      chunk[c] = SplitChunk{i, e0 + (c * kSplitChunk - i < a1 ? c * kSplitChunk - i : a1)};
  }
  const int64_t ti = row_div(i, tile_m, m), first = ti * tile_m, li = i - first;
  const int64_t rows = (m - first) < tile_m ? (m - first) : tile_m;
  const int64_t* o = off + (int64_t)tj * stride;
  const SplitTile t = tiles[ti * gn + tj];
  const int64_t base = o[first], v = o[i] - base;
  if (t.ptr_width == 8) static_cast<int64_t*>(t.rp)[li] = v;
  else static_cast<int32_t*>(t.rp)[li] = (int32_t)v;
  if (li == rows - 1) {  // the row that closes its tile row also writes the tile's last row_ptr entry
    const int64_t e = o[first + rows] - base;
    if (t.ptr_width == 8) static_cast<int64_t*>(t.rp)[rows] = e;
    else static_cast<int32_t*>(t.rp)[rows] = (int32_t)e;
  }
}

// Copies a chunk of A's entries to their tiles, walking windows of its row offsets; unit-stride loads, four entries in flight
// per thread. An entry that would land outside its tile (columns
// of A not sorted within the row, or not below n) is not written and sets *bad.
// Bound by the latency of a window (offsets, then entries, then stores): chunks of 4096 entries alone and windows of 256 rows
// gave the workgroups on the sparse rows of an R-MAT matrix up to a hundred windows one after the other (16 M entries at
// scale 20 into 4 x 4 tiles: 218 -> 120 us; 4 M rows with an entry in every 20th, 2 x 2 tiles, sizes and copy 1030 ->
// 260 us). Staging each segment's place in LDS instead of reading it per entry
// made no difference.
template <typename RP, typename T>
__global__ __launch_bounds__(256) void k_split_copy(const RP* rp, const int32_t* col, const T* val, int64_t m,
                                                    int64_t n, int64_t tile_m, uint32_t tile_n, int gn,
                                                    const int64_t* off, const int32_t* seg, int64_t stride,
                                                    const SplitTile* tiles, const SplitChunk* chunk, int64_t nchunks,
                                                    int32_t* bad) {
  __shared__ int s_rp[kSplitWindow + 1];  // offsets less the window's first entry, from -1 (before it) to kSplitChunk
  __shared__ int64_t s_first, s_end;      // first and last offset
  const int tid = threadIdx.x;
  const int64_t b = blockIdx.x;
  // the chunk's rows [r0, r1] and entries [e, c1)
  const SplitChunk from = chunk[b], to = b + 1 < nchunks ? chunk[b + 1] : SplitChunk{m - 1, (int64_t)rp[m]};
  int64_t r0 = from.row, e = from.entry;
  const int64_t r1 = to.row, c1 = to.entry;
  while (e < c1 && r0 <= r1) {
    const int rows = (int)(r1 - r0 + 1 < kSplitWindow ? r1 - r0 + 1 : kSplitWindow);
    int top = 1;  // the largest power of two below the number of rows, or 0
    while (top < rows) top <<= 1;
    for (int r = tid; r <= top; r += 256) {
      const int64_t p = (int64_t)rp[r0 + (r < rows ? r : rows)], d = p - e;
      s_rp[r] = r >= rows || d > kSplitChunk ? kSplitChunk : d < -1 ? -1 : (int)d;
      if (r == 0) s_first = p;
      if (r == rows) s_end = p;
    }
    __syncthreads();
    const int64_t we = s_end < c1 ? s_end : c1, p0 = s_first;
    top >>= 1;
    for (int64_t x0 = e; x0 < we; x0 += 4 * 256) {
      int a[4];  // largest a with s_rp[a] <= x - e: four branchless searches in lockstep
#pragma unroll
      for (int q = 0; q < 4; q++) a[q] = 0;
#pragma unroll
      for (int step = kSplitWindow / 2; step > 0; step >>= 1) {
        if (step > top) continue;  // uniform
#pragma unroll
        for (int q = 0; q < 4; q++)
          if (s_rp[a[q] + step] <= (int)(x0 - e) + q * 256 + tid) a[q] += step;
      }
      int c[4];
      T v[4];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int64_t x = x0 + q * 256 + tid;
        c[q] = x < we ? __builtin_nontemporal_load(&col[x]) : 0;
        v[q] = x < we ? __builtin_nontemporal_load(&val[x]) : T(0);
      }
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int64_t x = x0 + q * 256 + tid;
        if (x >= we) continue;
        const uint32_t tj = (uint32_t)c[q] / tile_n;
        if (c[q] < 0 || (int64_t)c[q] >= n || tj >= (uint32_t)gn) {
          *bad = 1;
          continue;
        }
        const int64_t i = r0 + a[q], ti = row_div(i, tile_m, m);
        const int64_t* o = off + (int64_t)tj * stride;
        const int64_t row = a[q] > 0 ? e + s_rp[a[q]] : p0;  // only the first row starts before the window's entries
        const int64_t at = x - row - seg[(int64_t)tj * stride + i];  // position within the segment
        const int64_t oi = o[i], dst = oi - o[ti * tile_m] + at;
        const SplitTile& t = tiles[ti * gn + tj];
        if (at < 0 || oi + at >= o[i + 1] || dst < 0 || dst >= t.nnz) {
          *bad = 1;
          continue;
        }
        t.col[dst] = (int32_t)((uint32_t)c[q] - tj * tile_n);
        static_cast<T*>(t.val)[dst] = v[q];
      }
    }
    e = we > e ? we : e;
    r0 += kSplitWindow;
    __syncthreads();
  }
}

// tot[ti * gn + tj] = entries of tile (ti, tj); tot[gm * gn] = entries of A.
template <typename RP>
__global__ void k_split_totals(const RP* rp, const int64_t* off, int64_t ostride, int64_t m, int64_t tile_m, int gm,
                               int gn, int64_t* tot) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t == gm * gn) tot[t] = (int64_t)rp[m] - (int64_t)rp[0];
  if (t >= gm * gn) return;
  const int ti = t / gn, tj = t - ti * gn;
  const int64_t r0 = (int64_t)ti * tile_m, r1 = (r0 + tile_m) < m ? (r0 + tile_m) : m;
  const int64_t* o = off + (int64_t)tj * ostride;
  tot[t] = o[r1] - o[r0];
}

template <typename RP, typename T>
void split_grid(bclx_handle* h, const bclx_csr* A, int64_t tile_m, int64_t tile_n, int gm, int gn, bclx_csr* tiles) {
  hipStream_t s = h->stream;
  const int64_t m = A->m;
  const int64_t stride = m / 4 * 4 + 4;  // a tile column's counts, padded with zeros: off[tj * stride + m] is its end
  const int64_t L = stride * gn;
  Arena ws;  // in a CallWorkspace: this call waits for the stream before it returns
  const size_t o_cnt = ws.reserve(sizeof(int32_t) * (size_t)L), o_seg = ws.reserve(sizeof(int32_t) * (size_t)L),
               o_off = ws.reserve(sizeof(int64_t) * (size_t)(L + 4)),
               o_part = ws.reserve(sizeof(long long) * (size_t)scan_partials(L)),
               o_tot = ws.reserve(sizeof(int64_t) * (size_t)(gm * gn + 1)),
               o_chunk = ws.reserve(sizeof(SplitChunk) * (size_t)((A->nnz + m) / kSplitChunk + 1)),
               o_tile = ws.reserve(sizeof(SplitTile) * (size_t)(gm * gn)), o_bad = ws.reserve(sizeof(int32_t));
  CallWorkspace use(h, ws);
  int32_t* cnt = ws.at<int32_t>(o_cnt);
  int32_t* seg = ws.at<int32_t>(o_seg);
  int64_t* off = ws.at<int64_t>(o_off);
  int64_t* tot = ws.at<int64_t>(o_tot);
  int32_t* bad = ws.at<int32_t>(o_bad);
  const RP* rp = static_cast<const RP*>(A->row_ptr);
  std::vector<int64_t> nnz((size_t)gm * gn + 1);
  if (m > 0) {
    hipLaunchKernelGGL((k_split_count<RP>), dim3(div_up(m, 256 / gn)), dim3(256), 0, s, rp, A->col_idx, m, tile_n, gn,
                       cnt, seg, stride, bad);
    BCLX_HIP(hipGetLastError());
    scan_counts(s, cnt, L, off, ws.at<long long>(o_part), nullptr);
    hipLaunchKernelGGL((k_split_totals<RP>), dim3(div_up((int64_t)gm * gn + 1, 256)), dim3(256), 0, s, rp, off, stride, m,
                       tile_m, gm, gn, tot);
    BCLX_HIP(hipGetLastError());
    BCLX_HIP(hipMemcpyAsync(nnz.data(), tot, sizeof(int64_t) * nnz.size(), hipMemcpyDeviceToHost, s));
    BCLX_HIP(hipStreamSynchronize(s));
  }
  bool sizes_only = true;
  for (int t = 0; t < gm * gn; t++) sizes_only = sizes_only && tiles[t].row_ptr == nullptr;
  for (int t = 0; t < gm * gn; t++) {
    const int ti = t / gn, tj = t % gn;
    const int64_t r0 = (int64_t)ti * tile_m, c0 = (int64_t)tj * tile_n;
    bclx_csr& d = tiles[t];
    d.m = std::min<int64_t>(tile_m, m - r0);
    d.n = std::min<int64_t>(tile_n, A->n - c0);
    d.dtype = A->dtype;
    if (sizes_only) {
      d.nnz = nnz[t];
      continue;
    }
    BCLX_REQUIRE(d.nnz == nnz[t], BCLX_ERR_INVALID,
                 "tile " + std::to_string(t) + ": nnz " + std::to_string(d.nnz) + " given, " + std::to_string(nnz[t]) +
                     " needed (sizes come from a call with every row_ptr NULL)");
    BCLX_REQUIRE(d.ptr_width == 4 || d.ptr_width == 8, BCLX_ERR_INVALID, "tile ptr_width must be 4 or 8");
    BCLX_REQUIRE(d.ptr_width == 8 || nnz[t] <= INT32_MAX, BCLX_ERR_OVERFLOW,
                 "tile " + std::to_string(t) + " has more than 2^31 - 1 entries: use ptr_width 8");
    BCLX_REQUIRE(d.row_ptr != nullptr && (nnz[t] == 0 || (d.col_idx != nullptr && d.vals != nullptr)),
                 BCLX_ERR_INVALID, "null tile array");
  }
  if (sizes_only) return;
  std::vector<SplitTile> st((size_t)gm * gn);
  for (int t = 0; t < gm * gn; t++)
    st[t] = SplitTile{tiles[t].row_ptr, tiles[t].col_idx, tiles[t].vals, nnz[t], tiles[t].ptr_width};
  int32_t h_bad = 0;
  const int64_t entries = nnz.back();
  DevBuf more_chunks;
  if (m > 0) {
    SplitChunk* chunk = ws.at<SplitChunk>(o_chunk);
    if (entries > A->nnz) {  // the descriptor's nnz is not what row_ptr says
      more_chunks.alloc(sizeof(SplitChunk) * (size_t)((entries + m) / kSplitChunk + 1));
      chunk = more_chunks.as<SplitChunk>();
    }
    const int64_t nchunks = (entries + m + kSplitChunk - 1) / kSplitChunk;
    SplitTile* dt = ws.at<SplitTile>(o_tile);
    BCLX_HIP(hipMemcpyAsync(dt, st.data(), sizeof(SplitTile) * st.size(), hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL((k_split_rowptr<RP>), dim3(div_up(m, 256), (unsigned)gn), dim3(256), 0, s, rp, off, stride, m,
                       tile_m, gn, dt, chunk, nchunks);
    BCLX_HIP(hipGetLastError());
    if (entries > 0) {
      hipLaunchKernelGGL((k_split_copy<RP, T>), dim3((unsigned)nchunks), dim3(256), 0, s, rp, A->col_idx,
                         static_cast<const T*>(A->vals), m, A->n, tile_m, (uint32_t)std::min<int64_t>(tile_n, UINT32_MAX),
                         gn, off, seg, stride, dt, chunk, nchunks, bad);
      BCLX_HIP(hipGetLastError());
    }
    BCLX_HIP(hipMemcpyAsync(&h_bad, bad, sizeof(int32_t), hipMemcpyDeviceToHost, s));
  } else {  // one row of tiles with no rows: each row_ptr is {0}
    for (int t = 0; t < gm * gn; t++) BCLX_HIP(hipMemsetAsync(tiles[t].row_ptr, 0, (size_t)tiles[t].ptr_width, s));
  }
  BCLX_HIP(hipStreamSynchronize(s));  // the tiles are complete, and the workspace free, on return
  BCLX_REQUIRE(h_bad == 0, BCLX_ERR_INVALID, "A's columns must be sorted within each row and below A->n");
}

// ---- dense elementwise ---------------------------------------------------------------------------------------

template <int OP, typename T>
__device__ inline T apply_op(T a, T b) {
  if (OP == 0) return a + b;
  if (OP == 1) return a - b;
  if (OP == 2) return a * b;
  return a / b;
}

// Rows of VEC-element vectors: block (x, y) covers vectors [x * 256, x * 256 + 256) of rows y, y + gridDim.y, ...
template <int OP, typename T, int VEC>
__global__ __launch_bounds__(256) void k_binary_op(int64_t m, int64_t nvec, const T* A, int64_t lda, const T* B,
                                                   int64_t ldb, T* C, int64_t ldc) {
  typedef T vec_t __attribute__((ext_vector_type(VEC)));
  const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (v >= nvec) return;
  for (int64_t i = blockIdx.y; i < m; i += gridDim.y) {
    const vec_t a = *reinterpret_cast<const vec_t*>(A + i * lda + v * VEC);
    const vec_t b = *reinterpret_cast<const vec_t*>(B + i * ldb + v * VEC);
    vec_t c;
#pragma unroll
    for (int q = 0; q < VEC; q++) c[q] = apply_op<OP, T>(a[q], b[q]);
    *reinterpret_cast<vec_t*>(C + i * ldc + v * VEC) = c;
  }
}

template <int OP, typename T>
void binary_op(hipStream_t s, int64_t m, int64_t n, const T* A, int64_t lda, const T* B, int64_t ldb, T* C,
               int64_t ldc) {
  constexpr int V = 16 / sizeof(T);
  auto aligned = [](const void* p, int64_t ld) {
    return (reinterpret_cast<uintptr_t>(p) % 16) == 0 && (ld * (int64_t)sizeof(T)) % 16 == 0;
  };
  // a full tile (ld == n for all three) is one long row
  if (lda == n && ldb == n && ldc == n) {
    n *= m;
    lda = ldb = ldc = n;
    m = 1;
  }
  const bool vec = n % V == 0 && aligned(A, lda) && aligned(B, ldb) && aligned(C, ldc);
  const int64_t nvec = vec ? n / V : n;
  const unsigned gx = div_up(nvec, 256);
  const unsigned gy = (unsigned)std::max<int64_t>(1, std::min<int64_t>(m, std::max<int64_t>(1, 4096 / (int64_t)gx)));
  if (vec)
    hipLaunchKernelGGL((k_binary_op<OP, T, V>), dim3(gx, gy), dim3(256), 0, s, m, nvec, A, lda, B, ldb, C, ldc);
  else
    hipLaunchKernelGGL((k_binary_op<OP, T, 1>), dim3(gx, gy), dim3(256), 0, s, m, nvec, A, lda, B, ldb, C, ldc);
  BCLX_HIP(hipGetLastError());
}

template <typename T>
void binary_op_t(hipStream_t s, int op, int64_t m, int64_t n, const void* A, int64_t lda, const void* B, int64_t ldb,
                 void* C, int64_t ldc) {
  const T* a = static_cast<const T*>(A);
  const T* b = static_cast<const T*>(B);
  T* c = static_cast<T*>(C);
  switch (op) {
    case 0: binary_op<0, T>(s, m, n, a, lda, b, ldb, c, ldc); break;
    case 1: binary_op<1, T>(s, m, n, a, lda, b, ldb, c, ldc); break;
    case 2: binary_op<2, T>(s, m, n, a, lda, b, ldb, c, ldc); break;
    default: binary_op<3, T>(s, m, n, a, lda, b, ldb, c, ldc); break;
  }
}

}  // namespace bclx

using namespace bclx;

extern "C" {

bclx_status bclx_csr_split_grid(bclx_handle* h, const bclx_csr* A, int64_t tile_m, int64_t tile_n, int32_t ntiles,
                                bclx_csr* tiles) {
  return guarded([&] {
    BCLX_REQUIRE(h && A && tiles, BCLX_ERR_INVALID, "null argument");
    BCLX_REQUIRE(tile_m > 0 && tile_n > 0, BCLX_ERR_INVALID, "tile sizes must be positive");
    BCLX_REQUIRE(A->m >= 0 && A->n >= 0 && A->nnz >= 0, BCLX_ERR_INVALID, "bad matrix shape");
    BCLX_REQUIRE(A->ptr_width == 4 || A->ptr_width == 8, BCLX_ERR_INVALID, "A->ptr_width must be 4 or 8");
    BCLX_REQUIRE(A->dtype == BCLX_F32 || A->dtype == BCLX_F64, BCLX_ERR_INVALID, "A->dtype must be fp32 or fp64");
    BCLX_REQUIRE(A->row_ptr && (A->nnz == 0 || (A->col_idx && A->vals)), BCLX_ERR_INVALID, "null array in A");
    const int64_t gm = std::max<int64_t>(1, (A->m + tile_m - 1) / tile_m);
    const int64_t gn = std::max<int64_t>(1, (A->n + tile_n - 1) / tile_n);
    BCLX_REQUIRE(gn <= kSplitMaxGridN, BCLX_ERR_UNSUPPORTED,
                 "more than " + std::to_string(kSplitMaxGridN) + " tile columns in one split");
    BCLX_REQUIRE((int64_t)ntiles == gm * gn, BCLX_ERR_INVALID,
                 "tiles must hold ceil(m / tile_m) * ceil(n / tile_n) = " + std::to_string(gm * gn) + " descriptors");
    set_device(h);
    const bool w8 = A->ptr_width == 8, f64 = A->dtype == BCLX_F64;
    if (!w8 && !f64) split_grid<int32_t, float>(h, A, tile_m, tile_n, (int)gm, (int)gn, tiles);
    else if (!w8) split_grid<int32_t, double>(h, A, tile_m, tile_n, (int)gm, (int)gn, tiles);
    else if (!f64) split_grid<int64_t, float>(h, A, tile_m, tile_n, (int)gm, (int)gn, tiles);
    else split_grid<int64_t, double>(h, A, tile_m, tile_n, (int)gm, (int)gn, tiles);
  });
}

bclx_status bclx_dense_binary_op(bclx_handle* h, int32_t op, int32_t dtype, int64_t m, int64_t n, const void* d_A,
                                 int64_t lda, const void* d_B, int64_t ldb, void* d_C, int64_t ldc) {
  return guarded([&] {
    BCLX_REQUIRE(h != nullptr, BCLX_ERR_INVALID, "null handle");
    BCLX_REQUIRE(op >= 0 && op <= 3, BCLX_ERR_INVALID, "op must be 0 (+), 1 (-), 2 (*) or 3 (/)");
    BCLX_REQUIRE(dtype == BCLX_F32 || dtype == BCLX_F64, BCLX_ERR_INVALID, "dtype must be fp32 or fp64");
    BCLX_REQUIRE(m >= 0 && n >= 0 && lda >= n && ldb >= n && ldc >= n, BCLX_ERR_INVALID, "bad shape or ld");
    if (m == 0 || n == 0) return;
    BCLX_REQUIRE(d_A && d_B && d_C, BCLX_ERR_INVALID, "null array");
    set_device(h);
    if (dtype == BCLX_F32) binary_op_t<float>(h->stream, op, m, n, d_A, lda, d_B, ldb, d_C, ldc);
    else binary_op_t<double>(h->stream, op, m, n, d_A, lda, d_B, ldb, d_C, ldc);
  });
}

}  // extern "C"
