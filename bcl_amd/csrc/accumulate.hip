// Cross-stage accumulation (bclx_accumulate_tiles): C = sum of K partial m x n tiles, the GPU counterpart of
// SparseHashAccumulator::get_matrix (bcl/containers/sequential/SparseHashAccumulator.hpp:101-182) and of the
// pairwise sum_tiles_cusparse fold (bcl/containers/experimental/cuda/sequential/cusparse_util.cuh:251-265).
//
// The tiles' rows are sorted, so the sum is a K-way merge. The rows are cut into pieces of at most kAccCap entries
// (whole short rows, or a column range of a long row); one workgroup loads a piece into LDS, merges its K sorted runs
// as a tree of merge-path merges, and equal (row, column) pairs, now adjacent and in tile order, are summed in
// float64 and rounded once. A counting merge sizes the rows, a scan places them, a second merge writes them.
//
// Measured: eight R-MAT scale 16 tiles (11.2 M entries, fp32) 11.0 ms through the general path, 0.81 ms here.
//
// Tiles whose columns are not strictly increasing within each row, and sums of more than kAccMaxTiles tiles (one lane
// per tile sets a piece up), and sums written over their own tiles, take the general path: one SpGEMM
// [T_1 T_2 ... T_K] * [I; I; ...; I], where the left operand stacks copies of the tiles side by side
// (row i of it is the concatenation of row i of every tile, tile t's columns shifted by t * n) and the right operand
// stacks K identities. Every product is x * 1 (exact), so the two-phase SpGEMM returns exactly the union pattern,
// sorted, with each entry summed in float64 and rounded once.
#include <algorithm>

#include "spgemm.hpp"

namespace bclx {

template <typename T, typename RP>
struct TileIn {
  const RP* rp;
  const int* col;
  const T* val;
};

template <typename T, typename RP>
__global__ void k_stack_count(const TileIn<T, RP>* tiles, int K, int64_t m, int32_t* cnt) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m) return;
  long long c = 0;
  for (int t = 0; t < K; t++) c += (long long)(tiles[t].rp[i + 1] - tiles[t].rp[i]);
  cnt[i] = (int32_t)c;
}

// one wavefront per row: copies row i of every tile into the stacked row, columns shifted by t * n
template <typename T, typename RP>
__global__ void k_stack_fill(const TileIn<T, RP>* tiles, int K, int64_t m, int64_t n, const int64_t* srp,
                             int* scol, T* sval) {
  const int64_t i = (int64_t)blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (i >= m) return;
  int64_t pos = srp[i];
  for (int t = 0; t < K; t++) {
    const RP a0 = tiles[t].rp[i], a1 = tiles[t].rp[i + 1];
    for (RP p = a0 + lane; p < a1; p += 64) {
      scol[pos + (p - a0)] = tiles[t].col[p] + (int)(t * n);
      sval[pos + (p - a0)] = tiles[t].val[p];
    }
    pos += (int64_t)(a1 - a0);
  }
}

template <typename T>
__global__ void k_ident_stack(int64_t rows, int64_t n, int64_t* rp, int* col, T* val) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r <= rows) rp[r] = r;
  if (r < rows) {
    col[r] = (int)(r % n);
    val[r] = (T)1;
  }
}

template <typename T, typename RP>
static void accumulate_spgemm(bclx_handle* h, int K, const bclx_csr* tiles, bclx_csr* C) {
  const int64_t m = tiles[0].m, n = tiles[0].n;
  hipStream_t s = h->stream;
  std::vector<TileIn<T, RP>> tin(K);
  for (int t = 0; t < K; t++)
    tin[t] = {static_cast<const RP*>(tiles[t].row_ptr), tiles[t].col_idx, static_cast<const T*>(tiles[t].vals)};
  int64_t total_in = 0;
  for (int t = 0; t < K; t++) total_in += tiles[t].nnz;
  // workspace: tile table, counts, stacked A (int64 row_ptr), stacked identity B
  DevBuf tin_d(sizeof(TileIn<T, RP>) * K), cnt(sizeof(int32_t) * (m + 1)), srp(sizeof(int64_t) * (m + 1));
  DevBuf scol(sizeof(int) * std::max<int64_t>(total_in, 1)), sval(sizeof(T) * std::max<int64_t>(total_in, 1));
  const int64_t brows = (int64_t)K * n;
  DevBuf brp(sizeof(int64_t) * (brows + 1)), bcol(sizeof(int) * std::max<int64_t>(brows, 1)),
      bval(sizeof(T) * std::max<int64_t>(brows, 1));
  BCLX_HIP(hipMemcpyAsync(tin_d.p, tin.data(), sizeof(TileIn<T, RP>) * K, hipMemcpyHostToDevice, s));
  if (m > 0) {
    hipLaunchKernelGGL((k_stack_count<T, RP>), dim3(div_up(m, 256)), dim3(256), 0, s, tin_d.as<TileIn<T, RP>>(), K, m,
                       cnt.as<int32_t>());
    BCLX_HIP(hipGetLastError());
  }
  DevBuf part(sizeof(long long) * scan_partials(m));
  scan_counts(s, cnt.as<int32_t>(), m, srp.as<int64_t>(), part.as<long long>(), nullptr);
  if (m > 0) {
    hipLaunchKernelGGL((k_stack_fill<T, RP>), dim3(div_up(m, 4)), dim3(256), 0, s, tin_d.as<TileIn<T, RP>>(), K, m, n,
                       srp.as<int64_t>(), scol.as<int>(), sval.as<T>());
    BCLX_HIP(hipGetLastError());
  }
  hipLaunchKernelGGL((k_ident_stack<T>), dim3(div_up(brows + 1, 256)), dim3(256), 0, s, brows, n, brp.as<int64_t>(),
                     bcol.as<int>(), bval.as<T>());
  BCLX_HIP(hipGetLastError());
  bclx_csr A{m, brows, total_in, 8, tiles[0].dtype, srp.p, scol.as<int>(), sval.p};
  bclx_csr B{brows, n, brows, 8, tiles[0].dtype, brp.p, bcol.as<int>(), bval.p};
  TwoPhase<T, int64_t> tp(h, make_tile<T, int64_t>(&A, &B), BinTuning{});
  const int64_t nnz = tp.symbolic();
  if (C->col_idx == nullptr) {
    C->m = m;
    C->n = n;
    C->nnz = nnz;
    if (C->row_ptr) {
      BCLX_REQUIRE(C->ptr_width == 8 || nnz <= INT32_MAX, BCLX_ERR_OVERFLOW, "nnz does not fit an int32 row_ptr");
      const unsigned g = div_up(m + 1, 256);
      if (C->ptr_width == 8)
        hipLaunchKernelGGL(k_rowptr<int64_t>, dim3(g), dim3(256), 0, s, tp.F.R.off, (int64_t)0, m,
                           static_cast<int64_t*>(C->row_ptr));
      else
        hipLaunchKernelGGL(k_rowptr<int32_t>, dim3(g), dim3(256), 0, s, tp.F.R.off, (int64_t)0, m,
                           static_cast<int32_t*>(C->row_ptr));
      BCLX_HIP(hipGetLastError());
    }
  } else {
    BCLX_REQUIRE(C->row_ptr && C->vals, BCLX_ERR_INVALID, "C->row_ptr / C->vals are null");
    BCLX_REQUIRE(C->dtype == tiles[0].dtype, BCLX_ERR_INVALID, "C dtype must match the tiles");
    tp.numeric(C->col_idx, static_cast<T*>(C->vals), C->nnz, C->row_ptr, C->ptr_width);
    C->m = m;
    C->n = n;
    C->nnz = nnz;
  }
  BCLX_HIP(hipStreamSynchronize(s));  // the workspace above is released on return
}

// ------------------------------------------------------------------------------------------------------------
// merge path
// ------------------------------------------------------------------------------------------------------------

constexpr int kAccThreads = 256;
constexpr int kAccItems = 9;                       // merged entries per thread (odd: LDS bank spread)
constexpr int kAccCap = kAccThreads * kAccItems;   // 2304 entries per piece
constexpr int kAccTarget = 1024;                   // a piece holds the rows whose weight offset lies in one such span
constexpr int kAccMaxTiles = 64;                   // one lane per tile in the setup of a piece
constexpr int kAccSlotBits = 12;                   // key = local row << 43 | column << 12 | slot
static_assert(kAccCap <= (1 << kAccSlotBits) && 2 * kAccTarget <= kAccCap && kAccTarget + kAccMaxTiles + 1 <= kAccCap,
              "a piece fits its slots");
static_assert(kAccTarget <= 1024, "a local row fits 10 bits beside the tile number in a mark");

// A piece of a long row: entries q of its npieces; bounds of piece p at bound[p * K + t].
struct AccPiece {
  int32_t row, q, npieces;
};

template <typename T, typename RP>
struct AccDev {
  TileIn<T, RP> tile[kAccMaxTiles];
  int32_t K;
  int64_t m, n;
  int64_t* woff;         // m + 1: offset of each row in units of entries + 1 per row
  int32_t* cnt;          // m: row weights, then entries of each row of C
  int64_t* off;          // m + 1: row offsets of C
  int64_t nchunks;       // spans of kAccTarget weight
  int32_t* chunk;        // 2 * nchunks: first row and end row of the short rows that start in each span
  AccPiece* piece;       // pieces of rows longer than kAccTarget
  int32_t max_pieces;
  int64_t* bound;        // max_pieces * K: first position of each piece in each tile
  int32_t* piece_cnt;    // entries of C per piece
  int32_t* npieces;      // pieces in use
  int32_t* bad;          // [0] set by the cut (descriptors disagree with the row_ptrs: nothing may use the pieces),
                         // [1] set by the cut and the merge (columns not strictly increasing): the general path
                         // takes the sum
};

// row weights: entries over all tiles, plus one (so a span of weights holds a bounded number of empty rows too)
template <typename T, typename RP>
__global__ __launch_bounds__(256) void k_acc_weight(AccDev<T, RP> D) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i == 0) {
    *D.npieces = 0;
    D.bad[0] = D.bad[1] = 0;
  }
  for (int64_t c = i; c < 2 * D.nchunks; c += (int64_t)gridDim.x * 256) D.chunk[c] = 0;
  if (i >= D.m) return;
  long long c = 1;
  for (int t = 0; t < D.K; t++) c += (long long)(D.tile[t].rp[i + 1] - D.tile[t].rp[i]);
  D.cnt[i] = (int32_t)c;
}

// Cuts the rows into pieces: span c of weights [c * kAccTarget, (c + 1) * kAccTarget) owns the rows that start in it
// (together at most 2 * kAccTarget - 1 entries: all but the last end inside the span), except a last row of more than
// kAccTarget entries, which is listed as pieces of its own. One thread per row.
template <typename T, typename RP>
__global__ __launch_bounds__(256) void k_acc_chunks(AccDev<T, RP> D) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i > D.m) return;
  const int64_t w = D.woff[i];
  const int64_t c = w / kAccTarget;
  if (i > 0) {
    const int64_t pw = D.woff[i - 1], pc = pw / kAccTarget;
    if ((i == D.m || pc != c) && pc < D.nchunks) D.chunk[2 * pc + 1] = (int32_t)(w - pw - 1 > kAccTarget ? i - 1 : i);
  }
  if (i == D.m) return;
  D.cnt[i] = 0;
  if (i == 0 || D.woff[i - 1] / kAccTarget != c) {
    if (c < D.nchunks) D.chunk[2 * c] = (int32_t)i;
    else D.bad[0] = 1;  // more entries than the descriptors say
  }
  const int64_t len = D.woff[i + 1] - w - 1;
  if (len > kAccTarget) {
    const int P = (int)((len + kAccTarget - 1) / kAccTarget);
    const int base = atomicAdd(D.npieces, P);
    if (base < 0 || base + P > D.max_pieces) {
      D.bad[0] = 1;
      return;
    }
    for (int q = 0; q < P; q++) D.piece[base + q] = AccPiece{(int32_t)i, q, P};
  }
}

// First positions of a long row's pieces: piece q starts at the largest column c before which the row has at most
// q * ceil(len / P) entries. One wavefront per piece, one tile per lane: a binary search over the columns, each step
// a binary search of every tile's row within the bounds the earlier steps left. A piece then holds at most
// ceil(len / P) + K entries.
template <typename T, typename RP>
__global__ __launch_bounds__(256) void k_acc_split(AccDev<T, RP> D) {
  const int lane = threadIdx.x & 63;
  if (D.bad[0]) return;
  const int np = *D.npieces;
  for (int p = blockIdx.x * 4 + (threadIdx.x >> 6); p < np; p += gridDim.x * 4) {  // wave-uniform
    const AccPiece pc = D.piece[p];
    const bool live = lane < D.K;
    const int* col = live ? D.tile[lane].col : nullptr;
    int64_t lo = live ? (int64_t)D.tile[lane].rp[pc.row] : 0;
    int64_t hi = live ? (int64_t)D.tile[lane].rp[pc.row + 1] : 0;
    const int64_t first = lo, last = hi;
    const int64_t len = wave_sum<long long>(hi - lo);
    const int64_t want = pc.q * ((len + pc.npieces - 1) / pc.npieces);
    int64_t clo = 0, chi = pc.q == 0 ? 1 : D.n;
    while (chi - clo > 1) {
      const int64_t mid = (clo + chi) >> 1;
      int64_t a = lo, b = hi;  // first position with column >= mid
      while (a < b) {
        const int64_t x = (a + b) >> 1;
        if ((int64_t)col[x] < mid) a = x + 1;
        else b = x;
      }
      if (wave_sum<long long>(a - first) <= want) {
        clo = mid;
        lo = a;
      } else {
        chi = mid;
        hi = a;
      }
    }
    if (live) {
      D.bound[(int64_t)p * D.K + lane] = lo;
      // the merge looks at the order inside a piece: here, at the seam to the piece before
      if (lo > first && lo < last && col[lo - 1] >= col[lo]) D.bad[1] = 1;
    }
  }
}

// One workgroup per piece (blocks below nlong: long-row pieces, strided; then one block per span of short rows).
// NUM false: entries of C per row (cnt) and per long-row piece; NUM true: the entries, at off[].
// Bound by VALU instructions, a third of them in the merge tree (log2 K levels, about two 8-byte LDS reads per entry and
// level), with five workgroups per CU (fp32; four for the writing pass, three in fp64) to cover each other's loads: counting
// pass of eight R-MAT scale 16 tiles 195 -> 157 us and writing pass 251 -> 231 us when the loads of a piece were put
// in one batch.
template <bool NUM, typename T, typename RP>
__global__ __launch_bounds__(kAccThreads, NUM ? (sizeof(T) == 8 ? 3 : 4) : 5) void k_acc_merge(AccDev<T, RP> D, int nlong,
                                                                                               int* c_col, T* c_val) {
  __shared__ unsigned long long s_key[kAccCap];
  __shared__ T s_val[NUM ? kAccCap : 1];
  __shared__ unsigned s_mark[kAccCap];  // tile << 10 | local row of each slot; then entries per local row
  __shared__ int s_seg[kAccMaxTiles + 1];
  __shared__ int64_t s_beg[kAccMaxTiles];
  __shared__ const int* s_tcol[kAccMaxTiles];
  __shared__ const T* s_tval[kAccMaxTiles];
  __shared__ unsigned s_scan[kAccThreads / 64 + 1];
  __shared__ long long s_base;
  const int tid = threadIdx.x, K = D.K;
  const bool is_long = (int)blockIdx.x < nlong;
  const int bad = D.bad[0];  // written by an earlier kernel only
  const int np = is_long ? *D.npieces : 1;
  int row0 = 0, nrows = 1;
  if (!is_long) {
    const int64_t c = (int64_t)blockIdx.x - nlong;
    row0 = D.chunk[2 * c];
    nrows = D.chunk[2 * c + 1] - row0;
  }
  TileIn<T, RP> mine{};  // of tile tid
  if (tid < K) mine = D.tile[tid];
  if (bad || nrows <= 0) return;
  for (int p = is_long ? (int)blockIdx.x : 0; p < np; p += nlong > 0 && is_long ? nlong : 1) {
    // the piece's K runs: [beg, beg + len) of each tile, laid out one after the other in the slots
    AccPiece pc{0, 0, 0};
    if (is_long) {
      pc = D.piece[p];
      row0 = pc.row;
    }
    if (tid < 64) {
      int64_t beg = 0, end = 0;
      if (tid < K) {
        if (is_long) {
          beg = D.bound[(int64_t)p * K + tid];
          // the next piece is the row's, or another row's (or past the last): read with the rest, not after it
          const int64_t next = D.bound[(int64_t)(p + 1 < np ? p + 1 : p) * K + tid];
          end = (int64_t)mine.rp[row0 + 1];
          if (pc.q + 1 < pc.npieces) end = next;
        } else {
          beg = (int64_t)mine.rp[row0];
          end = (int64_t)mine.rp[row0 + nrows];
        }
        s_beg[tid] = beg;
        s_tcol[tid] = mine.col;
        if (NUM) s_tval[tid] = mine.val;
      }
      // only possible when the row is not sorted or a row_ptr changed meanwhile (a run cut short would pass every check
      // that follows, so it is refused here)
      const bool refused = end < beg || end - beg > kAccCap;
      const int len = refused ? 0 : (int)(end - beg);
      const int inc = wave_incl_scan(len);
      if (__ballot(refused) != 0ull && tid == 0) D.bad[1] = 1;
      if (tid < K) s_seg[tid] = inc - len;
      if (tid == 63) s_seg[K] = inc;
      if (NUM && is_long) {  // entries of the row's earlier pieces
        long long before = 0;
        for (int q = tid; q < pc.q; q += 64) before += D.piece_cnt[p - pc.q + q];
        before = wave_sum<long long>(before);
        if (tid == 0) s_base = D.off[row0] + before;
      } else if (NUM && tid == 0) {
        s_base = D.off[row0];
      }
    }
    for (int s = tid; s < kAccCap; s += kAccThreads) s_mark[s] = 0;
    __syncthreads();
    const int E = s_seg[K];
    if (E > kAccCap) {  // likewise: runs that fit one by one, but not together
      if (tid == 0) D.bad[1] = 1;
      return;
    }
    // the first slot of every (tile, row) run is marked; a running maximum gives each slot its tile and row
    for (int x = tid; x < K * nrows; x += kAccThreads) {
      const int t = x / nrows, r = x - t * nrows;
      if (is_long) {
        if (s_seg[t + 1] > s_seg[t]) s_mark[s_seg[t]] = (unsigned)t << 10;
      } else {
        const RP* rp = D.tile[t].rp + row0 + r;
        const int64_t a = (int64_t)rp[0] - s_beg[t], b = (int64_t)rp[1] - s_beg[t];
        if (b > a && a >= 0 && s_seg[t] + a < E) s_mark[s_seg[t] + a] = (unsigned)t << 10 | (unsigned)r;
      }
    }
    __syncthreads();
    int vt = (E + kAccThreads - 1) / kAccThreads;
    vt |= 1;
    const int s0 = tid * vt;
    {
      unsigned run = 0;
      for (int v = 0; v < vt; v++) run = max(run, s_mark[s0 + v]);
      unsigned inc = run;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const unsigned t = __shfl_up(inc, d, 64);
        if ((tid & 63) >= d) inc = max(inc, t);
      }
      if ((tid & 63) == 63) s_scan[tid >> 6] = inc;
      unsigned before = __shfl_up(inc, 1, 64);
      if ((tid & 63) == 0) before = 0;
      __syncthreads();
      for (int w = 0; w < (tid >> 6); w++) before = max(before, s_scan[w]);
      for (int v = 0; v < vt; v++) {
        before = max(before, s_mark[s0 + v]);
        s_mark[s0 + v] = before;
      }
    }
    __syncthreads();
    // every load of the piece is issued before the first is used
    int64_t at[kAccItems];
    int tile[kAccItems], col[kAccItems];
    T val[NUM ? kAccItems : 1];
#pragma unroll
    for (int v = 0; v < kAccItems; v++) {
      const int s = v * kAccThreads + tid;
      tile[v] = s < E ? (int)(s_mark[s] >> 10) : 0;
      at[v] = s_beg[tile[v]] + (s - s_seg[tile[v]]);
    }
#pragma unroll
    for (int v = 0; v < kAccItems; v++) {
      if (v * kAccThreads + tid < E) {
        col[v] = glob(s_tcol[tile[v]])[at[v]];
        if (NUM) val[v] = glob(s_tval[tile[v]])[at[v]];
      }
    }
#pragma unroll
    for (int v = 0; v < kAccItems; v++) {
      const int s = v * kAccThreads + tid;
      if (s < E) {
        s_key[s] = (unsigned long long)(s_mark[s] & 1023u) << (31 + kAccSlotBits) |
                   (unsigned long long)((unsigned)col[v] & 0x7fffffffu) << kAccSlotBits | (unsigned)s;
        if (NUM) s_val[s] = val[v];
      }
    }
    __syncthreads();
    if (!NUM) {  // each run must be strictly increasing in (row, column)
#pragma unroll
      for (int v = 0; v < kAccItems; v++) {
        const int s = v * kAccThreads + tid;
        if (s > 0 && s < E && (s_mark[s] >> 10) == (s_mark[s - 1] >> 10) &&
            (s_key[s] >> kAccSlotBits) <= (s_key[s - 1] >> kAccSlotBits))
          D.bad[1] = 1;
      }
    }
    // merge tree: at width w, runs of w tiles are merged pairwise; thread tid produces slots [s0, s0 + vt)
    for (int w = 1; w < K; w *= 2) {
      unsigned long long out[kAccItems];
      int a = 0, a1 = 0, b = 0, b1 = -1;  // next positions and ends of the two runs being merged
#pragma unroll
      for (int v = 0; v < kAccItems; v++) {
        const int s = s0 + v;
        if (v < vt && s < E) {
          if (s >= b1) {  // the pair of runs holding slot s, and how much of each comes before s (merge path)
            int t = 0;    // last tile whose first slot is at or before s
            for (int step = kAccMaxTiles / 2; step > 0; step >>= 1)
              if (t + step < K && s_seg[t + step] <= s) t += step;
            const int t0 = t / (2 * w) * (2 * w);
            const int a0 = s_seg[t0];
            a1 = s_seg[t0 + w < K ? t0 + w : K];
            b1 = s_seg[t0 + 2 * w < K ? t0 + 2 * w : K];
            const int d = s - a0;
            int lo = d > b1 - a1 ? d - (b1 - a1) : 0, hi = d < a1 - a0 ? d : a1 - a0;
            while (lo < hi) {
              const int mid = (lo + hi) >> 1;
              if (s_key[a0 + mid] < s_key[a1 + d - 1 - mid]) lo = mid + 1;
              else hi = mid;
            }
            a = a0 + lo;
            b = a1 + d - lo;
          }
          const unsigned long long ka = a < a1 ? s_key[a] : ~0ull, kb = b < b1 ? s_key[b] : ~0ull;
          out[v] = ka < kb ? ka : kb;
          if (ka < kb) a++;
          else b++;
        }
      }
      __syncthreads();
#pragma unroll
      for (int v = 0; v < kAccItems; v++)
        if (v < vt && s0 + v < E) s_key[s0 + v] = out[v];
      __syncthreads();
    }
    // compress: an entry of C starts where the (row, column) changes
    unsigned heads = 0;
#pragma unroll
    for (int v = 0; v < kAccItems; v++) {
      const int s = s0 + v;
      if (v < vt && s < E && (s == 0 || (s_key[s - 1] >> kAccSlotBits) != (s_key[s] >> kAccSlotBits))) heads |= 1u << v;
    }
    unsigned total;
    const unsigned before = block_excl_scan<kAccThreads, unsigned>((unsigned)__popc(heads), &total, s_scan);
    if constexpr (!NUM) {
      if (is_long) {
        if (tid == 0) {
          D.piece_cnt[p] = (int)total;
          atomicAdd(&D.cnt[row0], (int)total);
        }
      } else {
        for (int r = tid; r < nrows; r += kAccThreads) s_mark[r] = 0;
        __syncthreads();
        int r = -1, c = 0;
#pragma unroll
        for (int v = 0; v < kAccItems; v++) {
          if (heads >> v & 1u) {
            const int rr = (int)(s_key[s0 + v] >> (31 + kAccSlotBits));
            if (rr != r) {
              if (c) atomicAdd(&s_mark[r], (unsigned)c);
              r = rr;
              c = 0;
            }
            c++;
          }
        }
        if (c) atomicAdd(&s_mark[r], (unsigned)c);
        __syncthreads();
        for (int x = tid; x < nrows; x += kAccThreads) D.cnt[row0 + x] = (int)s_mark[x];
      }
    } else {
      double sum[kAccItems];
      int col[kAccItems];
#pragma unroll
      for (int v = 0; v < kAccItems; v++) {
        if (heads >> v & 1u) {
          const unsigned long long k = s_key[s0 + v];
          const unsigned long long rc = k >> kAccSlotBits;
          col[v] = (int)(rc & 0x7fffffffu);
          sum[v] = (double)s_val[k & ((1u << kAccSlotBits) - 1u)];
          for (int q = s0 + v + 1; q < E; q++) {  // the same entry in later tiles, in tile order
            const unsigned long long kq = s_key[q];
            if ((kq >> kAccSlotBits) != rc) break;
            sum[v] += (double)s_val[kq & ((1u << kAccSlotBits) - 1u)];
          }
        }
      }
      __syncthreads();
      // staged by rank in LDS, then stored with unit stride
      int* s_col = reinterpret_cast<int*>(s_key);
      int r = (int)before;
#pragma unroll
      for (int v = 0; v < kAccItems; v++)
        if (heads >> v & 1u) {
          s_col[r] = col[v];
          s_val[r] = (T)sum[v];
          r++;
        }
      __syncthreads();
      const long long base = s_base;
      for (int x = tid; x < (int)total; x += kAccThreads) {
        __builtin_nontemporal_store(s_col[x], &c_col[base + x]);
        __builtin_nontemporal_store(s_val[x], &c_val[base + x]);
      }
    }
    __syncthreads();  // the next piece reuses the LDS
  }
}

// row_ptr of C from the row offsets
static void write_rowptr(hipStream_t s, const int64_t* off, int64_t m, void* row_ptr, int ptr_width) {
  const unsigned g = div_up(m + 1, 256);
  if (ptr_width == 8)
    hipLaunchKernelGGL(k_rowptr<int64_t>, dim3(g), dim3(256), 0, s, off, (int64_t)0, m, static_cast<int64_t*>(row_ptr));
  else
    hipLaunchKernelGGL(k_rowptr<int32_t>, dim3(g), dim3(256), 0, s, off, (int64_t)0, m, static_cast<int32_t*>(row_ptr));
  BCLX_HIP(hipGetLastError());
}

// The merge path; false when the tiles need the general path (nothing of C is written then).
template <typename T, typename RP>
static bool accumulate_merge(bclx_handle* h, int K, const bclx_csr* tiles, bclx_csr* C) {
  const int64_t m = tiles[0].m, n = tiles[0].n;
  if (K > kAccMaxTiles || m == 0) return false;
  int64_t total_in = 0;
  for (int t = 0; t < K; t++) total_in += tiles[t].nnz;
  const int64_t max_pieces = 2 * (total_in / kAccTarget) + 1;
  if (m >= INT32_MAX || max_pieces >= INT32_MAX / 2) return false;
  hipStream_t s = h->stream;
  AccDev<T, RP> D;
  for (int t = 0; t < K; t++)
    D.tile[t] = {static_cast<const RP*>(tiles[t].row_ptr), tiles[t].col_idx, static_cast<const T*>(tiles[t].vals)};
  D.K = K;
  D.m = m;
  D.n = n;
  D.nchunks = (total_in + m) / kAccTarget + 1;
  D.max_pieces = (int32_t)max_pieces;
  Arena ws;  // in a CallWorkspace: this call waits for the stream before it returns
  const size_t o_woff = ws.reserve(sizeof(int64_t) * (m + 4)), o_cnt = ws.reserve(sizeof(int32_t) * (m + 4)),
               o_off = ws.reserve(sizeof(int64_t) * (m + 4)), o_chunk = ws.reserve(sizeof(int32_t) * 2 * D.nchunks),
               o_piece = ws.reserve(sizeof(AccPiece) * max_pieces), o_bound = ws.reserve(sizeof(int64_t) * max_pieces * K),
               o_pcnt = ws.reserve(sizeof(int32_t) * max_pieces), o_part = ws.reserve(sizeof(long long) * scan_partials(m)),
               o_flag = ws.reserve(2 * sizeof(int64_t) + sizeof(int32_t));
  CallWorkspace use(h, ws);
  D.woff = ws.at<int64_t>(o_woff);
  D.cnt = ws.at<int32_t>(o_cnt);
  D.off = ws.at<int64_t>(o_off);
  D.chunk = ws.at<int32_t>(o_chunk);
  D.piece = ws.at<AccPiece>(o_piece);
  D.bound = ws.at<int64_t>(o_bound);
  D.piece_cnt = ws.at<int32_t>(o_pcnt);
  long long* part = ws.at<long long>(o_part);
  int64_t* total = ws.at<int64_t>(o_flag);  // nnz(C), and beside it the two flags: the host reads them together
  D.bad = reinterpret_cast<int32_t*>(total + 1);
  D.npieces = D.bad + 2;
  const unsigned grow = div_up(m + 1, 256);
  hipLaunchKernelGGL((k_acc_weight<T, RP>), dim3(grow), dim3(256), 0, s, D);
  scan_counts(s, D.cnt, m, D.woff, part, nullptr);
  hipLaunchKernelGGL((k_acc_chunks<T, RP>), dim3(grow), dim3(256), 0, s, D);
  const int nlong = total_in > kAccTarget ? (int)std::min<int64_t>(max_pieces, (int64_t)h->num_cus * 8) : 0;
  if (nlong > 0) hipLaunchKernelGGL((k_acc_split<T, RP>), dim3(nlong), dim3(256), 0, s, D);
  const unsigned grid = (unsigned)(D.nchunks + nlong);
  hipLaunchKernelGGL((k_acc_merge<false, T, RP>), dim3(grid), dim3(kAccThreads), 0, s, D, nlong, (int*)nullptr,
                     (T*)nullptr);
  BCLX_HIP(hipGetLastError());
  scan_counts(s, D.cnt, m, D.off, part, total);
  int64_t got[2] = {0, 0};
  BCLX_HIP(hipMemcpyAsync(got, total, sizeof(got), hipMemcpyDeviceToHost, s));
  BCLX_HIP(hipStreamSynchronize(s));
  if (got[1] != 0) return false;
  const int64_t nnz = got[0];
  if (C->col_idx == nullptr) {
    if (C->row_ptr) {
      BCLX_REQUIRE(C->ptr_width == 8 || nnz <= INT32_MAX, BCLX_ERR_OVERFLOW, "nnz does not fit an int32 row_ptr");
      write_rowptr(s, D.off, m, C->row_ptr, C->ptr_width);
    }
  } else {
    BCLX_REQUIRE(C->row_ptr && C->vals, BCLX_ERR_INVALID, "C->row_ptr / C->vals are null");
    BCLX_REQUIRE(C->dtype == tiles[0].dtype, BCLX_ERR_INVALID, "C dtype must match the tiles");
    BCLX_REQUIRE(C->nnz >= nnz, BCLX_ERR_INVALID, "C arrays smaller than the sum's entries");
    BCLX_REQUIRE(C->ptr_width == 8 || nnz <= INT32_MAX, BCLX_ERR_OVERFLOW,
                 "nnz(C) = " + std::to_string(nnz) + " does not fit an int32 row_ptr; request ptr_width 8");
    // pieces are written while others still read their tiles
    auto over = [&](const void* out, size_t bytes) {
      return std::any_of(tiles, tiles + K, [&](const bclx_csr& x) {
        return share_memory(out, bytes, x.row_ptr, sizeof(RP) * (m + 1)) ||
               share_memory(out, bytes, x.col_idx, sizeof(int) * x.nnz) || share_memory(out, bytes, x.vals, sizeof(T) * x.nnz);
      });
    };
    if (over(C->col_idx, sizeof(int) * nnz) || over(C->vals, sizeof(T) * nnz)) return false;
    hipLaunchKernelGGL((k_acc_merge<true, T, RP>), dim3(grid), dim3(kAccThreads), 0, s, D, nlong, C->col_idx,
                       static_cast<T*>(C->vals));
    BCLX_HIP(hipGetLastError());
    write_rowptr(s, D.off, m, C->row_ptr, C->ptr_width);
  }
  C->m = m;
  C->n = n;
  C->nnz = nnz;
  BCLX_HIP(hipStreamSynchronize(s));  // C is complete, and the workspace free, on return
  return true;
}

template <typename T, typename RP>
static void accumulate_impl(bclx_handle* h, int K, const bclx_csr* tiles, bclx_csr* C) {
  BCLX_REQUIRE(K * tiles[0].n < INT32_MAX, BCLX_ERR_OVERFLOW, "K * n must fit int32 (stacked column index)");
  if (!accumulate_merge<T, RP>(h, K, tiles, C)) accumulate_spgemm<T, RP>(h, K, tiles, C);
}

}  // namespace bclx

using namespace bclx;

extern "C" {

bclx_status bclx_accumulate_tiles(bclx_handle* h, int ntiles, const bclx_csr* tiles, bclx_csr* C) {
  return guarded([&] {
    BCLX_REQUIRE(h && tiles && C && ntiles > 0, BCLX_ERR_INVALID, "null argument or ntiles <= 0");
    for (int t = 0; t < ntiles; t++) {
      const bclx_csr& x = tiles[t];
      BCLX_REQUIRE(x.m == tiles[0].m && x.n == tiles[0].n, BCLX_ERR_INVALID, "tiles must share their shape");
      BCLX_REQUIRE(x.dtype == tiles[0].dtype && x.ptr_width == tiles[0].ptr_width, BCLX_ERR_INVALID,
                   "tiles must share dtype and ptr_width");
      BCLX_REQUIRE(x.dtype == BCLX_F32 || x.dtype == BCLX_F64, BCLX_ERR_INVALID, "dtype must be fp32 or fp64");
      BCLX_REQUIRE(x.ptr_width == 4 || x.ptr_width == 8, BCLX_ERR_INVALID, "ptr_width must be 4 or 8");
      BCLX_REQUIRE(x.row_ptr && (x.nnz == 0 || (x.col_idx && x.vals)), BCLX_ERR_INVALID, "null tile arrays");
    }
    set_device(h);
    const bool f64 = tiles[0].dtype == BCLX_F64, w8 = tiles[0].ptr_width == 8;
    if (!f64 && !w8) accumulate_impl<float, int32_t>(h, ntiles, tiles, C);
    else if (!f64 && w8) accumulate_impl<float, int64_t>(h, ntiles, tiles, C);
    else if (f64 && !w8) accumulate_impl<double, int32_t>(h, ntiles, tiles, C);
    else accumulate_impl<double, int64_t>(h, ntiles, tiles, C);
  });
}

}  // extern "C"
