// SpGEMM device kernels: row analysis, binning, LDS-hash accumulators (symbolic / numeric / predicted / one-pass),
// heavy-row global accumulators, scans and compaction. Shared by the per-product two-phase path and the batched
// stage pipeline: every kernel works on a "flat row" space that concatenates the rows of all products of a batch,
// each product padded to a multiple of 256 rows, so one 256-row block never straddles two products.
#pragma once

#include <hip/hip_runtime.h>

#include <climits>
#include <cstdint>
#include <type_traits>

namespace bclx {

constexpr int kEmptyKey = 0x7fffffff;  // larger than any column index
// 0: empty row; 1..9: LDS hash tables; 10: heavy (global accumulator); 11..17: sort-based (ESC) rows of up to
// 64 * 2^(b - 11) products (bin 11: sorted in registers by 16 lanes per row; 12..14: one wavefront per row; 15..17:
// 2, 4 or 8 wavefronts per row); 18: rows of at most 32 products, sorted in registers by eight lanes per row
constexpr int kNumBins = 19;
constexpr int kHeavyBin = 10;
constexpr int kCountStride = 32;  // bin counters sit 128 bytes apart
constexpr int kEscBin0 = 11;
constexpr int kEscBins = 7;
constexpr int kEscWaveBins = 4;                         // bins 11..14 sort within one wavefront (or less)
constexpr int kEscMaxProducts = 64 << (kEscBins - 1);  // 4096
constexpr int kEscColBits = 19;                         // sort keys pack column (< 2^19) and product index (13 bits)
constexpr int kSmallBin = 18;
constexpr int kSmallMax = 32;       // products per row in the small bin
constexpr int kSmallColBits = 27;   // small-bin keys pack column (< 2^27 - 1) and product index (5 bits)
constexpr int kSmallGroup = 8;      // lanes per small-bin row (four products per lane; 16 and 4 measured slower)
constexpr int kRowBlock = 256;         // flat-row padding and analysis block size
constexpr int kHeavyThreads = 1024;

// Table geometry of LDS bins 1..9: TS = 2^(b+4) slots holds up to TS/2 keys (load <= 1/2); G lanes per row.
// Groups are either part of one wavefront (G <= 64, several rows per block) or the whole block (G >= 256).
__host__ __device__ constexpr int bin_table(int b) { return 1 << (b + 4); }
__host__ __device__ constexpr int bin_group(int b) {
  return b == 1 ? 16 : b == 2 ? 32 : b <= 5 ? 64 : b == 6 ? 256 : b <= 8 ? 512 : 1024;
}

// Where every tile of the batch is at most 2^19 columns wide: rows of more than 4096 products that need more entries than
// this run in the rank-slice kernel of the heavy bin, whatever heavy_need allows to hash. (One wider tile gives the batch's
// heavy rows to the wide-tile kernel, whose accumulator is in HBM.) 20000 rows of 6400 products: 3190 entries
// 2.1 ms there and 7.8 ms hashed, 1918 entries 2.1 and 4.3 ms, 998 entries 2.1 and 1.95 ms; rows of 90000 products with
// 1500 entries 2.3 and 3.3 ms; R-MAT square at scale 16 1.79 and 2.34 ms.
constexpr int kRankNeed = 1024;

// Tunable binning knobs (chosen by the autotuner; these are the defaults).
struct BinTuning {
  int32_t work_per_lane = 64;     // a row's group must have >= products / work_per_lane lanes
  int32_t heavy_need = 4096;      // rows needing more table entries than this use the global accumulator
  int32_t load_shift = 1;         // table slots >= need << load_shift (1: load <= 1/2)
  int32_t esc_min = 32;           // rows with esc_min < products <= esc_max sort instead of hashing (when the
  int32_t esc_max = 4096;         //   tile is at most 2^19 columns wide); esc_max 0 turns sorting off
};

// ESC bin of a row with `work` products: the smallest 64 * 2^e >= work.
__host__ __device__ inline int esc_bin(int64_t work) {
  int e = 0;
  while ((64LL << e) < work) e++;
  return kEscBin0 + e;
}

// n: the tile's width. Rows of at most 32 products sort in registers (tiles narrower than 2^27 - 1 columns); longer
// rows sort in the ESC bins when the columns fit their packed key (n <= 2^19). esc_max = 0 turns both off. rank_kernel: the
// batch's heavy rows run in the rank-slice kernel.
__host__ __device__ inline int bin_for(int64_t need, int64_t work, const BinTuning& tn, int64_t n, bool rank_kernel) {
  if (work <= 0) return 0;
  if (tn.esc_max > 0 && work <= kSmallMax && n < ((int64_t)1 << kSmallColBits) - 1) return kSmallBin;
  const bool esc_ok = n <= (1 << kEscColBits);
  if (esc_ok && work > tn.esc_min && work <= tn.esc_max && work <= kEscMaxProducts) return esc_bin(work);
  const bool rank = rank_kernel && work > kEscMaxProducts;  // the rank-slice kernel takes it from kRankNeed on
  if (need > (rank && tn.heavy_need > kRankNeed ? kRankNeed : tn.heavy_need)) return kHeavyBin;
  int64_t slots = need << tn.load_shift;
  int bn = 1;
  while (bn < 9 && bin_table(bn) < slots) bn++;
  if (bin_table(bn) < slots) return kHeavyBin;
  int bw = bn;
  while (bw < 9 && (int64_t)bin_group(bw) * tn.work_per_lane < work) bw++;
  return bw;
}

// Home slot of column j in a table of TS = 2^b slots: Fibonacci hashing (top b bits of j * 2^32 / phi), so every
// bit of j moves the slot. (A multiplier-and-mask hash keeps only j's low bits; R-MAT columns have biased bits, so
// their low bits take few distinct values and linear probing would chain.)
template <int TS>
__device__ inline unsigned slot_hash(int j) {
  constexpr int b = __builtin_ctz(TS);
  return ((unsigned)j * 0x9E3779B1u) >> (32 - b);
}

template <typename T, typename RP>
struct TileDev {
  const RP* a_rp;
  const int* a_col;
  const T* a_val;
  const RP* b_rp;
  const int* b_col;
  const T* b_val;
  // output base (positions come from off[]). The kernels write it with nontemporal (streaming) stores, except those
  // of rows of at most 64 products: an entry is written once and not read by this launch, so it need not displace
  // the B rows held in L2.
  int* c_col;
  T* c_val;
  int64_t flat0;  // first flat row of this product
  int32_t m, n;
  float avg_a, avg_b;      // average row lengths of A and B (predictor features)
  int64_t krows;           // rows of B
};

// A column range of a heavy row (split rows: see k_heavy_split). Bounds are multiples of kHRGroup words of columns.
struct HeavyPart {
  int32_t fr, lo, hi;  // row, columns [lo, hi)
  int32_t parts;       // of a row's first part: its number of parts
  int32_t nnz;         // the part's output entries
  int32_t bad;         // of a row's first part: a B row's columns are not sorted, the row runs whole
  int32_t split_row;   // entry q: first part of the q-th split row
  int32_t pad;
  int64_t off;         // output offset: in the row (symbolic), in C (modes 2 and 3; < 0: refused)
};
struct HeavyHead {
  int32_t parts, split_rows;
  int32_t ordered;  // whole rows in the heavy bin's list
  int32_t rows;     // with the split rows found bad, appended to the list
};
// Products of a part: about an eighth of a compute unit's share of all heavy products, so the last one to finish is short,
// between 8192 (below, staging a part costs as much as its products) and 2^18, and never so few that more than
// kMaxHeavyParts parts would be made (a row of P gives ceil(P / size) parts and only rows with more than size are
// split, so total / (kMaxHeavyParts / 2) is enough).
constexpr int kMaxHeavyParts = 16384;
constexpr int kMaxRowParts = 256;
__host__ __device__ inline long long heavy_part_size(long long total) {
  const long long share = total / 2048, most = (total + kMaxHeavyParts / 2 - 1) / (kMaxHeavyParts / 2);
  long long size = share < (1 << 18) ? share : (1 << 18);
  size = size > 8192 ? size : 8192;
  return size > most ? size : most;
}

template <typename T, typename RP>
struct RowsDev {
  const TileDev<T, RP>* tiles;
  const uint16_t* blk_tile;  // (flat row >> 8) -> product index
  int64_t* prod;             // products per flat row
  int32_t* nnz;              // nnz(C_i): symbolic count, or measured count
  int32_t* cap;              // predicted capacity (learned path)
  int64_t* off;              // output offset per flat row (nflat + 1 entries)
  int32_t* bin_count;        // kNumBins counters, kCountStride ints apart (one cache line each: no false sharing of
                             // the atomics that fill them)
  __host__ __device__ int32_t* count_of(int b) const { return bin_count + b * kCountStride; }
  int32_t* bin_items;        // kNumBins lists of flat rows, bin_stride apart
  int64_t bin_stride;
  int32_t* ovf_count;        // overflow list (learned path)
  int32_t* ovf_items;
  int32_t* pred_count;       // rows whose capacity the predictor sets (learned path)
  int32_t* long_count;       // rows of more than 32 A entries, listed by the analysis in tmp_items
  int32_t* pred_items;
  float* pred_val;             // the network's raw prediction per listed row (learned path; pred_val_cap entries)
  int32_t pred_val_cap;
  unsigned long long* cursor;  // bump allocator for rows placed outside their predicted slot
  unsigned long long* heavy_queue;  // next heavy row to take (rows are handed out largest first)
  int32_t* tmp_items;               // scratch list for ordering the heavy bin
  HeavyHead* heavy_head;
  HeavyPart* heavy_parts;           // kMaxHeavyParts
  int32_t* heavy_first;             // per row of the heavy bin: its first part, -1 if it is not split
  unsigned long long* stats;   // [0] products [1] heavy rows [2] overflow rows [3] capacity exceeded [4] predicted
  bool rank_kernel;            // every tile fits the rank-slice kernel (k_heavy_rank), which then runs the heavy bin
  long long out_limit;         // entries available in the output arrays; writes beyond it are refused
  BinTuning tn;
};

// A pointer read from device memory, as one to global memory: the compiler then emits global loads and stores. Flat ones also
// count as LDS operations, so that each LDS wait waits for them.
template <typename P>
__device__ inline __attribute__((address_space(1))) P* glob(P* p) {
  return (__attribute__((address_space(1))) P*)p;
}

// ------------------------------------------------------------------------------------------------------------
// reductions / scans
// ------------------------------------------------------------------------------------------------------------

template <typename V>
__device__ inline V wave_sum(V v) {
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d, 64);
  return v;
}

// Inclusive scan within a wave.
template <typename V>
__device__ inline V wave_incl_scan(V v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    V t = __shfl_up(v, d, 64);
    if (lane >= d) v += t;
  }
  return v;
}

// Block-wide exclusive scan (BLOCK a multiple of 64, <= 1024). Returns exclusive prefix; *total = block sum.
template <int BLOCK, typename V>
__device__ inline V block_excl_scan(V v, V* total, V* smem /* >= BLOCK/64 + 1 */) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  constexpr int NW = BLOCK / 64;
  V inc = wave_incl_scan(v);
  if (lane == 63) smem[w] = inc;
  __syncthreads();
  if (threadIdx.x == 0) {
    V run = 0;
    for (int q = 0; q < NW; q++) {
      V t = smem[q];
      smem[q] = run;
      run += t;
    }
    smem[NW] = run;
  }
  __syncthreads();
  V r = smem[w] + inc - v;
  *total = smem[NW];
  __syncthreads();
  return r;
}

template <int BLOCK, typename V>
__device__ inline V block_sum(V v, V* smem) {
  V t;
  (void)block_excl_scan<BLOCK, V>(v, &t, smem);
  return t;
}

// Inclusive scan of one int per lane of a wavefront, by DPP: six VALU instructions, no LDS.
__device__ inline int wave_scan_dpp(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, true);   // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);  // row_bcast:15 into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);  // row_bcast:31 into rows 2 and 3
  return v;
}

// Block-wide exclusive scan of one int per thread with one barrier. `smem` (BLOCK / 64 ints) may be written again only
// after another barrier.
template <int BLOCK>
__device__ inline int block_scan_dpp(int v, int* total, int* smem) {
  constexpr int NW = BLOCK / 64;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int inc = wave_scan_dpp(v);
  if (lane == 63) smem[w] = inc;
  __syncthreads();
  const int waves = wave_scan_dpp(lane < NW ? smem[lane] : 0);
  *total = __builtin_amdgcn_readlane(waves, NW - 1);
  const int before = w > 0 ? __builtin_amdgcn_readlane(waves, w - 1) : 0;
  return before + inc - v;
}

// ------------------------------------------------------------------------------------------------------------
// row analysis: products per row, optional binning by upper bound min(products, n) (symbolic bins)
// ------------------------------------------------------------------------------------------------------------

// 256-row blocks of flat rows per analysis workgroup: each thread analyzes one row of each, with the loads of its
// rows issued together, and the workgroup takes its bin and list positions with one global atomic per bin.
// Four blocks where that still fills the GPU; one where it does not (16384 rows of 8 entries: 18 us with four, 8 us with
// one).
constexpr int kAnaSubLarge = 4;

template <int kAnaSub, typename T, typename RP>
__global__ __launch_bounds__(kRowBlock) void k_analyze(RowsDev<T, RP> R, int64_t nblocks, int do_bin,
                                                       long long pred_min, int with_stats) {
  __shared__ int s_nlong, s_lbase;
  __shared__ int s_bcount[kNumBins], s_bbase[kNumBins];
  __shared__ int s_npred, s_pbase;
  __shared__ long long s_red[kRowBlock / 64 + 1];
  const int tid = threadIdx.x;
  const int64_t sb0 = (int64_t)blockIdx.x * kAnaSub;
  if (tid == 0) {
    s_nlong = 0;
    s_npred = 0;
  }
  if (tid < kNumBins) s_bcount[tid] = 0;
  __syncthreads();
  const TileDev<T, RP>* tp[kAnaSub];
  bool in[kAnaSub], valid[kAnaSub];
  int64_t i[kAnaSub];
  RP a0[kAnaSub], a1[kAnaSub];
  long long prod[kAnaSub];
  bool lng[kAnaSub];
#pragma unroll
  for (int s = 0; s < kAnaSub; s++) {
    in[s] = sb0 + s < nblocks;
    tp[s] = R.tiles + (in[s] ? R.blk_tile[sb0 + s] : 0);
    i[s] = (sb0 + s) * kRowBlock + tid - tp[s]->flat0;
    valid[s] = in[s] && i[s] >= 0 && i[s] < tp[s]->m;
    a0[s] = valid[s] ? tp[s]->a_rp[i[s]] : 0;
    a1[s] = valid[s] ? tp[s]->a_rp[i[s] + 1] : 0;
    prod[s] = 0;
  }
  // rows of up to 32 entries: four entries of every row at a time, their column loads and then their B-row-pointer
  // loads issued together. Longer rows (R-MAT hubs cluster in a few workgroups) go on a global list that
  // k_analyze_long spreads over the whole GPU, so they do not hold their workgroup.
  bool more = false;
  int lpos[kAnaSub];
#pragma unroll
  for (int s = 0; s < kAnaSub; s++) {
    lng[s] = a1[s] - a0[s] > 32;
    lpos[s] = lng[s] ? atomicAdd(&s_nlong, 1) : 0;
    if (lng[s]) a1[s] = a0[s];
    more = more || a1[s] > a0[s];
  }
  for (RP p0 = 0; more; p0 += 4) {
    int k[kAnaSub][4];
    more = false;
#pragma unroll
    for (int s = 0; s < kAnaSub; s++)
#pragma unroll
      for (int u = 0; u < 4; u++) k[s][u] = a0[s] + p0 + u < a1[s] ? tp[s]->a_col[a0[s] + p0 + u] : -1;
#pragma unroll
    for (int s = 0; s < kAnaSub; s++) {
#pragma unroll
      for (int u = 0; u < 4; u++)
        if (k[s][u] >= 0) prod[s] += (long long)(tp[s]->b_rp[k[s][u] + 1] - tp[s]->b_rp[k[s][u]]);
      more = more || a0[s] + p0 + 4 < a1[s];
    }
  }
  __syncthreads();
  if (tid == 0 && s_nlong > 0) s_lbase = atomicAdd(R.long_count, s_nlong);
  __syncthreads();
  int b0[kAnaSub];
  bool pr[kAnaSub];
  long long ub0[kAnaSub];
#pragma unroll
  for (int s = 0; s < kAnaSub; s++) {
    const int64_t fr = (sb0 + s) * kRowBlock + tid;
    if (lng[s]) {  // finished by k_analyze_long
      R.tmp_items[s_lbase + lpos[s]] = (int32_t)fr;
      valid[s] = false;
      in[s] = false;
    }
    if (in[s]) R.prod[fr] = valid[s] ? prod[s] : 0;
    ub0[s] = prod[s] < (long long)tp[s]->n ? prod[s] : (long long)tp[s]->n;
    b0[s] = valid[s] ? bin_for(ub0[s], prod[s], R.tn, tp[s]->n, R.rank_kernel) : 0;
    if (with_stats && b0[s] == kHeavyBin) atomicAdd(&R.stats[5], 1ull);
    pr[s] = false;
  }
  if (pred_min >= 0) {
    // learned path: every row starts at the exact bound min(prod, n); rows with more than pred_min products that
    // hash (sorted rows are exact in one pass and keep the bound) go on the list whose capacities the predictor
    // then lowers, and are binned after the prediction
    int ppos[kAnaSub];
#pragma unroll
    for (int s = 0; s < kAnaSub; s++) {
      const int64_t fr = (sb0 + s) * kRowBlock + tid;
      if (in[s]) R.cap[fr] = valid[s] ? (int32_t)ub0[s] : 0;
      pr[s] = valid[s] && prod[s] > pred_min && b0[s] < kEscBin0;
      ppos[s] = pr[s] ? atomicAdd(&s_npred, 1) : 0;
    }
    __syncthreads();
    if (tid == 0 && s_npred > 0) s_pbase = atomicAdd(R.pred_count, s_npred);
    __syncthreads();
#pragma unroll
    for (int s = 0; s < kAnaSub; s++)
      if (pr[s]) R.pred_items[s_pbase + ppos[s]] = (int32_t)((sb0 + s) * kRowBlock + tid);
  }
  if (do_bin) {
    int b[kAnaSub], pos[kAnaSub];
#pragma unroll
    for (int s = 0; s < kAnaSub; s++) {
      b[s] = pr[s] ? 0 : b0[s];
      pos[s] = b[s] > 0 ? atomicAdd(&s_bcount[b[s]], 1) : 0;
    }
    __syncthreads();
    if (tid > 0 && tid < kNumBins && s_bcount[tid] > 0) s_bbase[tid] = atomicAdd(R.count_of(tid), s_bcount[tid]);
    __syncthreads();
#pragma unroll
    for (int s = 0; s < kAnaSub; s++) {
      const int64_t fr = (sb0 + s) * kRowBlock + tid;
      if (b[s] > 0) R.bin_items[b[s] * R.bin_stride + s_bbase[b[s]] + pos[s]] = (int)fr;
      if (in[s] && b[s] == 0 && !pr[s]) R.nnz[fr] = 0;  // empty and padding rows
    }
  }
  if (with_stats) {  // one global atomic per block: only when asked (a plan counts products once)
    long long mine = 0;
#pragma unroll
    for (int s = 0; s < kAnaSub; s++) mine += prod[s];
    long long tot = block_sum<kRowBlock, long long>(mine, s_red);
    if (tid == 0 && tot) atomicAdd(&R.stats[0], (unsigned long long)tot);
  }
}

// The rows k_analyze listed (more than 32 A entries): one wavefront per row, rows strided over the wavefronts (the
// list holds each workgroup's long rows together, so striding spreads neighbouring hubs), eight entries per lane in
// flight, then the same outputs as k_analyze gives a row (products, capacity, predictor list, bin), with per-row
// atomics.
// The loop control is wave-uniform arithmetic and lane 0's writes are one if-block at the end of the body: no other
// lane-0 region in the loop (a queue pop by lane 0 at the top was merged by the compiler with the writes at the
// bottom, and the other lanes then looped on their own on a stale index).
template <typename T, typename RP>
__global__ __launch_bounds__(kRowBlock) void k_analyze_long(RowsDev<T, RP> R, int do_bin, long long pred_min,
                                                            int with_stats) {
  const int lane = threadIdx.x & 63;
  const int nwaves = (int)gridDim.x * (kRowBlock / 64);
  const int cnt = R.long_count[0];
  for (int q = (int)blockIdx.x * (kRowBlock / 64) + (int)(threadIdx.x >> 6); q < cnt; q += nwaves) {
    const int fr = R.tmp_items[q];
    const TileDev<T, RP>* t = R.tiles + R.blk_tile[fr >> 8];
    const int64_t i = fr - t->flat0;
    const RP a0 = t->a_rp[i], a1 = t->a_rp[i + 1];
    long long prod = 0;
    for (RP p = a0 + lane; p < a1; p += 8 * 64) {
      int kk[8];
#pragma unroll
      for (int u = 0; u < 8; u++) kk[u] = p + 64 * u < a1 ? t->a_col[p + 64 * u] : -1;
#pragma unroll
      for (int u = 0; u < 8; u++)
        if (kk[u] >= 0) prod += (long long)(t->b_rp[kk[u] + 1] - t->b_rp[kk[u]]);
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) prod += __shfl_xor(prod, d);
    if (lane == 0) {
      R.prod[fr] = prod;
      const long long ub0 = prod < (long long)t->n ? prod : (long long)t->n;
      const int b0 = bin_for(ub0, prod, R.tn, t->n, R.rank_kernel);
      if (with_stats) {
        atomicAdd(&R.stats[0], (unsigned long long)prod);
        if (b0 == kHeavyBin) atomicAdd(&R.stats[5], 1ull);
      }
      bool pr = false;
      if (pred_min >= 0) {
        R.cap[fr] = (int32_t)ub0;
        pr = prod > pred_min && b0 < kEscBin0;
        if (pr) R.pred_items[atomicAdd(R.pred_count, 1)] = fr;
      }
      if (do_bin) {
        const int b = pr ? 0 : b0;
        if (b > 0) R.bin_items[b * R.bin_stride + atomicAdd(R.count_of(b), 1)] = fr;
        if (b == 0 && !pr) R.nnz[fr] = 0;
      }
    }
  }
}

// Bin rows by `need` (src 0: nnz, 1: cap) and products. Padded / empty rows go nowhere.
template <typename T, typename RP>
__global__ __launch_bounds__(kRowBlock) void k_bin(RowsDev<T, RP> R, int src) {
  __shared__ int s_bcount[kNumBins], s_bbase[kNumBins];
  const int tid = threadIdx.x;
  const int64_t fr = (int64_t)blockIdx.x * kRowBlock + tid;
  const TileDev<T, RP> tile = R.tiles[R.blk_tile[blockIdx.x]];
  const int64_t i = fr - tile.flat0;
  const bool valid = i >= 0 && i < tile.m;
  if (tid < kNumBins) s_bcount[tid] = 0;
  __syncthreads();
  int b = 0;
  if (valid) {
    const long long work = R.prod[fr];
    const long long need = src == 0 ? (long long)R.nnz[fr] : (long long)R.cap[fr];
    b = (need == 0 && src == 0) ? 0 : bin_for(need, work, R.tn, tile.n, R.rank_kernel);
  }
  int pos = 0;
  if (b > 0) pos = atomicAdd(&s_bcount[b], 1);
  __syncthreads();
  if (tid > 0 && tid < kNumBins && s_bcount[tid] > 0) s_bbase[tid] = atomicAdd(R.count_of(tid), s_bcount[tid]);
  __syncthreads();
  if (b > 0) R.bin_items[b * R.bin_stride + s_bbase[b] + pos] = (int)fr;
}

// ------------------------------------------------------------------------------------------------------------
// LDS hash accumulators
//   MODE 0 symbolic: count distinct columns -> nnz[fr]
//   MODE 1 numeric: accumulate, sort, write at off[fr] (nnz known)
//   MODE 2 predicted: table sized by cap[fr]; more than cap distinct columns -> overflow list, else write at off[fr]
//   MODE 3 one-pass exact: table sized by the upper bound; count, bump-allocate from *cursor, write
// Values accumulate in float64 (products of fp32 inputs are exact in float64) and round once on output.
// ------------------------------------------------------------------------------------------------------------

// Synchronise the lanes of one row group: a wavefront-level fence when the group lives inside one wavefront, a
// workgroup barrier when the group is the whole block.
template <int G>
__device__ inline void group_sync() {
  if constexpr (G > 64) {
    __syncthreads();
  } else {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  }
}

// Exclusive scan of one value per lane over a row group; *total = group sum.
template <int G, int BLOCK>
__device__ inline long long group_excl_scan(long long v, long long* total, long long* smem) {
  if constexpr (G > 64) {
    static_assert(G == BLOCK, "multi-wavefront groups must be the whole block");
    return block_excl_scan<BLOCK, long long>(v, total, smem);
  } else {
    const int gl = threadIdx.x & (G - 1);
    long long inc = v;
#pragma unroll
    for (int d = 1; d < G; d <<= 1) {
      const long long t = __shfl_up(inc, d, G);
      if (gl >= d) inc += t;
    }
    *total = __shfl(inc, G - 1, G);
    return inc - v;
  }
}

// The product loop of a staged chunk of A entries: entry e's products are B positions e_start[e] + 0 ..
// e_pre[e + 1] - e_pre[e] - 1 (e_pre holds ne + 1 prefix counts, e_pre[ne] = total). Lane l takes products l,
// l + G, ..., U at a time: the U entry lookups (binary searches over the prefixes) advance in lockstep and the U loads
// are issued together, so their latencies overlap. f(j, v) per product (v = a * b in float64; 0 when !NUM).
template <int G, bool NUM, int U, typename T, typename RP, typename PT, typename F>
__device__ inline void enumerate_staged(const TileDev<T, RP>& tile, int ne, long long total, int lane,
                                        const RP* e_start, const PT* e_pre, const T* e_val,
                                        const volatile int* stop, F&& f) {
  int top = 1;  // largest power of two < ne (0 when ne == 1)
  while (top < ne) top <<= 1;
  top >>= 1;
  for (long long t0 = lane; t0 < total; t0 += (long long)U * G) {
    if (stop && *stop) break;
    int lo[U];
#pragma unroll
    for (int u = 0; u < U; u++) lo[u] = 0;
    for (int step = top; step > 0; step >>= 1) {  // entry e with e_pre[e] <= t < e_pre[e + 1]
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int c = lo[u] + step;
        if (c < ne && e_pre[c] <= t0 + (long long)u * G) lo[u] = c;
      }
    }
    int j[U];
    double v[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const long long t = t0 + (long long)u * G;
      if (t < total) {
        const RP q = e_start[lo[u]] + (RP)(t - e_pre[lo[u]]);
        j[u] = tile.b_col[q];
        v[u] = NUM ? (double)e_val[lo[u]] * (double)tile.b_val[q] : 0.0;
      }
    }
#pragma unroll
    for (int u = 0; u < U; u++)
      if (t0 + (long long)u * G < total) f(j[u], v[u]);
  }
}

// Load-balanced enumeration of the products of one row: the group stages the B-row ranges of up to G entries of
// A's row in LDS, prefix-sums their lengths and runs enumerate_staged over them. `stop` (optional, LDS) ends the
// enumeration early once set.
template <int G, int BLOCK, bool NUM, typename T, typename RP, typename PT, typename F, int U = 4>
__device__ inline void for_each_product(const TileDev<T, RP>& tile, RP a0, RP a1, int lane, RP* e_start,
                                        PT* e_pre, T* e_val, long long* scan_smem, const volatile int* stop,
                                        F&& f) {
  for (RP c0 = a0; c0 < a1; c0 += G) {
    const int ne = (int)((a1 - c0) < (RP)G ? (a1 - c0) : (RP)G);
    long long len = 0;
    if (lane < ne) {
      const int kk = tile.a_col[c0 + lane];
      const RP st = tile.b_rp[kk];
      len = (long long)(tile.b_rp[kk + 1] - st);
      e_start[lane] = st;
      if (NUM) e_val[lane] = tile.a_val[c0 + lane];
    }
    long long total;
    const long long ex = group_excl_scan<G, BLOCK>(len, &total, scan_smem);
    if (lane < ne) e_pre[lane] = (PT)ex;
    if (lane == 0) e_pre[ne] = (PT)total;
    group_sync<G>();
    enumerate_staged<G, NUM, U>(tile, ne, total, lane, e_start, e_pre, e_val, stop, f);
    group_sync<G>();
  }
}

template <int TS, int G, int BLOCK>
__device__ inline void bitonic_sort_groups(int* keys, double* vals, int lane, bool with_vals) {
  // Sort each group's TS-slot table ascending by key; kEmptyKey sorts last. All threads of the block call this.
  for (int k = 2; k <= TS; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int t = lane; t < TS / 2; t += G) {
        const int i = 2 * t - (t & (j - 1));
        const int p = i + j;
        const bool asc = (i & k) == 0;
        const int ki = keys[i], kp = keys[p];
        if ((ki > kp) == asc) {
          keys[i] = kp;
          keys[p] = ki;
          if (with_vals) {
            double vi = vals[i];
            vals[i] = vals[p];
            vals[p] = vi;
          }
        }
      }
      if (G > 64) {
        __syncthreads();
      } else {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
      }
    }
  }
}

// Block-wide min / max of an int (BLOCK <= 1024); smem >= BLOCK/64 ints. Contains barriers.
template <int BLOCK>
__device__ inline int block_min(int v, int* smem) {
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) v = min(v, __shfl_xor(v, d, 64));
  if ((threadIdx.x & 63) == 0) smem[threadIdx.x >> 6] = v;
  __syncthreads();
  int r = smem[0];
  for (int q = 1; q < BLOCK / 64; q++) r = min(r, smem[q]);
  __syncthreads();
  return r;
}
template <int BLOCK>
__device__ inline int block_max(int v, int* smem) {
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) v = max(v, __shfl_xor(v, d, 64));
  if ((threadIdx.x & 63) == 0) smem[threadIdx.x >> 6] = v;
  __syncthreads();
  int r = smem[0];
  for (int q = 1; q < BLOCK / 64; q++) r = max(r, smem[q]);
  __syncthreads();
  return r;
}

// LDS for the bitmap ranking of one row: W words of bits over the row's column span plus one prefix count per
// 8 words. kRankWords words cover spans up to 2^19 columns.
constexpr int kRankWords = 16384;
constexpr int kRankBytes = kRankWords * 4 + (kRankWords / 8 + 16) * 4;

template <int TS, int G, int BLOCK, int MODE, typename T, typename RP>
__global__ __launch_bounds__(BLOCK) void k_hash(RowsDev<T, RP> R, int bin) {
  constexpr int NG = BLOCK / G;
  constexpr bool NUM = MODE != 0;
  // Whole-block rows with large tables: the sorted order comes from ranking every key in a bitmap of the row's
  // column span (prefix popcounts) instead of sorting the table; entries go straight to their output position.
  constexpr bool RANK = NUM && NG == 1 && TS >= 2048;
  constexpr int TBYTES = NG * TS * (NUM ? 12 : 4);
  // entry staging of for_each_product: start (RP), prefix (long long), A value (T) per lane, 16-byte aligned
  constexpr int EPRE = ((NG * (G + 1) * 8) + 15) / 16 * 16;
  constexpr int EST = ((NG * G * (int)sizeof(RP)) + 15) / 16 * 16;
  constexpr int EBYTES = EPRE + EST + ((NG * G * (int)sizeof(T)) + 15) / 16 * 16;
  // the staging lives after the table; the rank bitmap later reuses the whole buffer
  constexpr int LBYTES = (RANK && kRankBytes > TBYTES + EBYTES) ? kRankBytes : TBYTES + EBYTES;
  __shared__ __align__(16) unsigned char s_buf[LBYTES];
  __shared__ int s_cnt[NG];
  __shared__ int s_flag[NG];
  __shared__ long long s_base[NG];
  __shared__ int s_red[BLOCK / 64 + 1];
  __shared__ long long s_lscan[BLOCK / 64 + 1];
  long long* s_epre = reinterpret_cast<long long*>(s_buf + TBYTES);
  RP* s_est = reinterpret_cast<RP*>(s_buf + TBYTES + EPRE);
  T* s_eval = reinterpret_cast<T*>(s_buf + TBYTES + EPRE + EST);
  const int g = threadIdx.x / G, lane = threadIdx.x % G;
  int* keys = reinterpret_cast<int*>(s_buf) + g * TS;
  double* vals = reinterpret_cast<double*>(s_buf + NG * TS * 4) + (NUM ? g * TS : 0);
  const int count = *R.count_of(bin);
  const int* items = R.bin_items + (int64_t)bin * R.bin_stride;
  volatile int* vflag = s_flag;

  for (int base = blockIdx.x * NG; base < count; base += gridDim.x * NG) {
    const int idx = base + g;
    const bool active = idx < count;
    const int fr = active ? items[idx] : 0;
    for (int s = lane; s < TS; s += G) {
      keys[s] = kEmptyKey;
      if (NUM) vals[s] = 0.0;
    }
    if (lane == 0) {
      s_cnt[g] = 0;
      s_flag[g] = 0;
    }
    __syncthreads();
    TileDev<T, RP> tile;
    if (active) {
      tile = R.tiles[R.blk_tile[fr >> 8]];
      const int64_t i = fr - tile.flat0;
      const int limit = MODE == 2 ? R.cap[fr] : INT_MAX;
      const RP a0 = tile.a_rp[i], a1 = tile.a_rp[i + 1];
      auto insert = [&](int j, double pv) {
        unsigned h = slot_hash<TS>(j);
        for (int probe = 0; probe < TS; probe++) {
          const int kcur = keys[h];
          if (kcur == j) {
            if (NUM) atomicAdd(&vals[h], pv);
            return;
          }
          if (kcur == kEmptyKey) {
            const int old = atomicCAS(&keys[h], kEmptyKey, j);
            if (old == kEmptyKey) {
              const int c = atomicAdd(&s_cnt[g], 1);
              if (MODE == 2 && c >= limit) vflag[g] = 1;
              if (NUM) atomicAdd(&vals[h], pv);
              return;
            }
            if (old == j) {
              if (NUM) atomicAdd(&vals[h], pv);
              return;
            }
          }
          h = (h + 1) & (TS - 1);
        }
        if (MODE == 2) vflag[g] = 1;  // table full: only possible after overflow
      };
      for_each_product<G, BLOCK, NUM, T, RP>(tile, a0, a1, lane, s_est + g * G, s_epre + g * (G + 1),
                                              s_eval + (NUM ? g * G : 0), s_lscan, MODE == 2 ? vflag + g : nullptr,
                                              insert);
    }
    __syncthreads();
    if (MODE == 0) {
      if (active && lane == 0) R.nnz[fr] = s_cnt[g];
    } else {
      const int cnt = s_cnt[g];
      const bool ovf = MODE == 2 && s_flag[g];
      // A row refused for lack of output room keeps nnz = 0 (and a harmless offset), so later passes that copy
      // nnz entries from its offset (compaction) stay inside the arrays; the refusal is flagged in stats[3].
      if (active && lane == 0) {
        if (MODE == 2) {
          if (ovf) {
            int slot = atomicAdd(R.ovf_count, 1);
            R.ovf_items[slot] = fr;
            atomicAdd(&R.stats[2], 1ull);
          } else {
            const bool fits = R.off[fr] + cnt <= R.out_limit;
            R.nnz[fr] = fits ? cnt : 0;
            if (!fits) R.stats[3] = 1ull;
          }
        } else if (MODE == 3) {
          s_base[g] = (long long)atomicAdd(R.cursor, (unsigned long long)cnt);
          const bool fits = s_base[g] + cnt <= R.out_limit;
          R.off[fr] = fits ? s_base[g] : 0;
          R.nnz[fr] = fits ? cnt : 0;
          if (!fits) R.stats[3] = 1ull;
        }
      }
      bool ranked = false;
      if constexpr (RANK) {
        constexpr int SPT = TS / BLOCK;
        int rk[SPT];
        double rv[SPT];
        int kmin = INT_MAX, kmax = -1;
#pragma unroll
        for (int q = 0; q < SPT; q++) {
          rk[q] = keys[q * BLOCK + threadIdx.x];
          rv[q] = vals[q * BLOCK + threadIdx.x];
          if (rk[q] != kEmptyKey) {
            kmin = min(kmin, rk[q]);
            kmax = max(kmax, rk[q]);
          }
        }
        kmin = block_min<BLOCK>(kmin, s_red);
        kmax = block_max<BLOCK>(kmax, s_red);
        const long long span = kmax >= kmin ? (long long)kmax - kmin + 1 : 1;
        const int W = (int)((span + 31) / 32);
        if (W <= kRankWords && (W * 4 + ((W + 7) / 8 + 1) * 4) <= LBYTES) {
          ranked = true;
          unsigned* bits = reinterpret_cast<unsigned*>(s_buf);
          int* pre = reinterpret_cast<int*>(s_buf + (size_t)W * 4);
          const int NGR = (W + 7) / 8;
          for (int w = threadIdx.x; w < W; w += BLOCK) bits[w] = 0u;
          __syncthreads();
#pragma unroll
          for (int q = 0; q < SPT; q++)
            if (rk[q] != kEmptyKey) {
              const int rel = rk[q] - kmin;
              atomicOr(&bits[rel >> 5], 1u << (rel & 31));
            }
          __syncthreads();
          const int gpt = (NGR + BLOCK - 1) / BLOCK;
          const int g0 = threadIdx.x * gpt, g1 = min(NGR, g0 + gpt);
          int c = 0;
          for (int gg = g0; gg < g1; gg++)
            for (int w = gg * 8; w < min(gg * 8 + 8, W); w++) c += __popc(bits[w]);
          int tot;
          int run = block_excl_scan<BLOCK, int>(c, &tot, s_red);
          for (int gg = g0; gg < g1; gg++) {
            pre[gg] = run;
            for (int w = gg * 8; w < min(gg * 8 + 8, W); w++) run += __popc(bits[w]);
          }
          __syncthreads();
          const long long o = MODE == 3 ? s_base[0] : (active ? R.off[fr] : 0);
          const bool fits = o + cnt <= R.out_limit;
          if (active && !ovf && !fits && threadIdx.x == 0) R.stats[3] = 1ull;
          if (active && !ovf && fits) {
#pragma unroll
            for (int q = 0; q < SPT; q++) {
              if (rk[q] == kEmptyKey) continue;
              const int rel = rk[q] - kmin;
              const int w = rel >> 5;
              int r = pre[w >> 3];
              for (int w2 = (w >> 3) * 8; w2 < w; w2++) r += __popc(bits[w2]);
              r += __popc(bits[w] & ((1u << (rel & 31)) - 1u));
              __builtin_nontemporal_store(rk[q], &tile.c_col[o + r]);
              __builtin_nontemporal_store((T)rv[q], &tile.c_val[o + r]);
            }
          }
        } else {
          __syncthreads();
#pragma unroll
          for (int q = 0; q < SPT; q++) {
            keys[q * BLOCK + threadIdx.x] = rk[q];
            vals[q * BLOCK + threadIdx.x] = rv[q];
          }
          __syncthreads();
        }
      }
      if (!ranked) {
        bitonic_sort_groups<TS, G, BLOCK>(keys, vals, lane, true);
        __syncthreads();
        const long long o = MODE == 3 ? s_base[g] : (active ? R.off[fr] : 0);
        const bool fits = o + cnt <= R.out_limit;
        if (active && !ovf && !fits && lane == 0) R.stats[3] = 1ull;
        if (active && !ovf && fits) {
          for (int s = lane; s < cnt; s += G) {
            __builtin_nontemporal_store(keys[s], &tile.c_col[o + s]);
            __builtin_nontemporal_store((T)vals[s], &tile.c_val[o + s]);
          }
        }
      }
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------------------------------------------------------
// Sort-based rows (ESC: expand, sort, compress), one wavefront per row, for rows of 64 * K products or fewer.
// Rows of a SUMMA-stage tile product are mostly output-dense (nnz(C_i) close to the products), where a hash table
// costs two LDS slots per output entry plus a rank structure, and caps how many rows a CU holds. Here the products
// of a row are expanded into registers as 32-bit keys (column << 13 | product index), sorted with a bitonic network
// across the wavefront, and equal columns are summed in float64 in a fixed order and rounded once. LDS holds only the float64 products (8 bytes per product) and the sorted
// keys. The count is exact after the sort, so the predicted mode never overflows: a row that outgrows its slot
// is bump-allocated in the same pass.
// Bound by VALU instructions (92 % busy in the kernel of 2048 to 4096 products before the sort kept neighbouring
// positions in a lane).
//   MODE 0 symbolic -> nnz[fr]; MODE 1 numeric at off[fr]; MODE 2 at off[fr] when nnz <= cap[fr], else
//   bump-allocated; MODE 3 bump-allocated.
// ------------------------------------------------------------------------------------------------------------

constexpr int kEscWaves = 4;  // wavefronts per block, each on its own row

constexpr unsigned kEscKeyShift = 32 - kEscColBits;      // key = column << 13 | product index
constexpr unsigned kEscIdxMask = (1u << kEscKeyShift) - 1u;
constexpr unsigned kEscPad = 0xffffffffu;                 // sorts after every real key

// A value moved between the lanes of a 16-lane DPP row, one VALU move (part of the using instruction where that allows
// it): from lane ^ X (X = 1, 2, 3, 7, 8 or 15), or from the lane D below (above); lanes without one get 0.
template <int X>
__device__ inline unsigned dpp_xor(unsigned v) {
  constexpr int ctrl = X == 1 ? 0xB1 : X == 2 ? 0x4E : X == 3 ? 0x1B : X == 7 ? 0x141 : X == 8 ? 0x128 : 0x140;
  static_assert(X == 1 || X == 2 || X == 3 || X == 7 || X == 8 || X == 15, "a quad permutation, a mirror or a rotation");
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, 0xF, 0xF, true);
}
template <int D>
__device__ inline unsigned dpp_below(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x110 + D, 0xF, 0xF, true);
}
template <int D>
__device__ inline unsigned dpp_above(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x100 + D, 0xF, 0xF, true);
}

// min(a, b) where lim is 0, max(a, b) where it is ~0 (the median of the three: one instruction)
__device__ inline unsigned min_or_max(unsigned a, unsigned b, unsigned lim) {
  return max(min(a, b), min(max(a, b), lim));
}

__device__ inline void cx(unsigned& a, unsigned& b) {
  const unsigned lo = min(a, b);
  b = max(a, b);
  a = lo;
}

// Compare-exchange of a wavefront's keys with lane ^ 16 or lane ^ 32 (half-cleaner: the lower lane keeps the minimum), two
// slots at a time: swapping half of one with half of the other brings both keys of each pair into one lane, and swapping
// again takes them home. Two instructions per key, none of them LDS.
template <int X, int K>
__device__ inline void swap_step(unsigned (&key)[K]) {
  static_assert(X == 16 || X == 32, "the distances of the swap instructions");
  auto swap = [](unsigned& a, unsigned& b) {
    if constexpr (X == 16) {
      const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
      a = r[0];
      b = r[1];
    } else {
      const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
      a = r[0];
      b = r[1];
    }
  };
#pragma unroll
  for (int q = 0; q < K; q += 2) {
    swap(key[q], key[q + 1]);
    cx(key[q], key[q + 1]);
    swap(key[q], key[q + 1]);
  }
}

// Half-cleaner at distance X lanes inside a 16-lane row; lim is ~0 in the upper lane of each pair.
template <int X, int K>
__device__ inline void dpp_step(unsigned (&key)[K], unsigned lim) {
#pragma unroll
  for (int q = 0; q < K; q++) {
    // lane ^ 4 is the mirror of eight, then of four
    const unsigned o = X == 4 ? dpp_xor<3>(dpp_xor<7>(key[q])) : dpp_xor<X == 4 ? 1 : X>(key[q]);
    key[q] = min_or_max(key[q], o, lim);
  }
}

// The same against the mirrored position (lane ^ X, slot K - 1 - q), the first stage of a merge of two ascending runs.
template <int X, int K>
__device__ inline void mirror_step(unsigned (&key)[K], unsigned lim) {
  unsigned o[K];
#pragma unroll
  for (int q = 0; q < K; q++) o[q] = dpp_xor<X>(key[K - 1 - q]);
#pragma unroll
  for (int q = 0; q < K; q++) key[q] = min_or_max(key[q], o[q], lim);
}

template <int K>
__device__ inline void lane_merge(unsigned (&key)[K]) {
#pragma unroll
  for (int d = K / 2; d > 0; d >>= 1)
#pragma unroll
    for (int q = 0; q < K; q++)
      if ((q & d) == 0) cx(key[q], key[q + d]);
}

template <int K>
__device__ inline void lane_sort(unsigned (&key)[K]) {
  static_assert(K == 2 || K == 4 || K == 8, "slots per lane");
  if constexpr (K == 2) {
    cx(key[0], key[1]);
  } else {
#pragma unroll
    for (int q = 0; q < K; q += 4) {
      cx(key[q], key[q + 1]);
      cx(key[q + 2], key[q + 3]);
      cx(key[q], key[q + 2]);
      cx(key[q + 1], key[q + 3]);
      cx(key[q + 1], key[q + 2]);
    }
    if constexpr (K == 8) {  // odd-even merge of the two halves
      cx(key[0], key[4]);
      cx(key[1], key[5]);
      cx(key[2], key[6]);
      cx(key[3], key[7]);
      cx(key[2], key[4]);
      cx(key[3], key[5]);
      cx(key[1], key[2]);
      cx(key[3], key[4]);
      cx(key[5], key[6]);
    }
  }
}

// Masks of the lanes that keep the maximum at each distance.
struct LaneLimits {
  unsigned l1, l2, l4, l8;
  __device__ explicit LaneLimits(int lane)
      : l1(lane & 1 ? ~0u : 0u), l2(lane & 2 ? ~0u : 0u), l4(lane & 4 ? ~0u : 0u), l8(lane & 8 ? ~0u : 0u) {}
};

// Sorts a bitonic sequence of the 64 * K keys of a wavefront: position x is slot x % K of lane x / K.
template <int K>
__device__ inline void esc_half_clean(unsigned (&key)[K], const LaneLimits& m) {
  swap_step<32>(key);
  swap_step<16>(key);
  dpp_step<8>(key, m.l8);
  dpp_step<4>(key, m.l4);
  dpp_step<2>(key, m.l2);
  dpp_step<1>(key, m.l1);
  lane_merge(key);
}

// Ascending sort of the 64 * K keys of a wavefront: in, any order; out, position x is slot x % K of lane x / K. Bitonic;
// K neighbours per lane leave 21 of the 45 stages of 512 keys crossing lanes (positions spread over the lanes: 39, in
// LDS exchanges for two of the six distances): 71 instructions per key instead of about 185. Runs up to 16 lanes merge by
// the mirrored position; the odd rows are reversed before runs of 16 lanes merge, and the upper 32 lanes sort
// complemented keys, i.e. descending.
template <int K>
__device__ inline void esc_sort(unsigned (&key)[K], int lane, const LaneLimits& m) {
  const unsigned flip = lane & 32 ? ~0u : 0u;
#pragma unroll
  for (int q = 0; q < K; q++) key[q] ^= flip;
  lane_sort(key);
  mirror_step<1>(key, m.l1);
  lane_merge(key);
  mirror_step<3>(key, m.l2);
  dpp_step<1>(key, m.l1);
  lane_merge(key);
  mirror_step<7>(key, m.l4);
  dpp_step<2>(key, m.l2);
  dpp_step<1>(key, m.l1);
  lane_merge(key);
  mirror_step<15>(key, m.l8);
  dpp_step<4>(key, m.l4);
  dpp_step<2>(key, m.l2);
  dpp_step<1>(key, m.l1);
  lane_merge(key);
  unsigned o[K];
#pragma unroll
  for (int q = 0; q < K; q++) o[q] = key[K - 1 - q];
#pragma unroll
  for (int q = 0; q < K; q++)  // row_mirror in rows 1 and 3
    key[q] = (unsigned)__builtin_amdgcn_update_dpp((int)key[q], (int)o[q], 0x140, 0xA, 0xF, false);
  swap_step<16>(key);
  dpp_step<8>(key, m.l8);
  dpp_step<4>(key, m.l4);
  dpp_step<2>(key, m.l2);
  dpp_step<1>(key, m.l1);
  lane_merge(key);
#pragma unroll
  for (int q = 0; q < K; q++) key[q] ^= flip;
  esc_half_clean(key, m);
}

// Expands a wavefront's share of a row's products, x0 + q * 64 + lane in A-row order, into keys (column << 13 | x), with the
// float64 products in s_val[x]; slots past the row's products keep the pad key. 64 A entries at a time, one per lane. For
// each 64 products the entries that start among them are counted by a ballot: up to eight are broadcast and compared per lane,
// more are searched (a binary search per product took a third of the instructions the sort takes). Every wavefront of a row
// walks the row's entries itself.
template <int K, bool NUM, typename T, typename RP>
__device__ inline void esc_expand(const TileDev<T, RP>& tile, RP a0, RP a1, int x0, int lane, unsigned (&key)[K],
                                  double* s_val) {
#pragma unroll
  for (int q = 0; q < K; q++) key[q] = kEscPad;
  int base = 0;
  for (RP c0 = a0; c0 < a1 && base < x0 + 64 * K; c0 += 64) {
    RP st = 0;
    int len = 0;
    T av = T(0);
    if (c0 + lane < a1) {
      const int kk = glob(tile.a_col)[c0 + lane];
      st = glob(tile.b_rp)[kk];
      len = (int)(glob(tile.b_rp)[kk + 1] - st);
      if (NUM) av = glob(tile.a_val)[c0 + lane];
    }
    const int inc = wave_scan_dpp(len);
    const int total = __builtin_amdgcn_readlane(inc, 63);
    const int ex = inc - len;  // lanes past the row start at `total`: after every product
    const RP delta = st - (RP)ex;
    RP pos[K];
    T a[K];
#pragma unroll
    for (int q = 0; q < K; q++) {
      const int t0 = x0 + q * 64 - base, t = t0 + lane;  // products t of this chunk
      pos[q] = 0;
      a[q] = T(0);
      if (t0 + 63 >= 0 && t0 < total) {  // uniform
        const int before = __popcll(__ballot(ex <= t0));
        const int in = __popcll(__ballot(ex <= t0 + 63)) - before;
        int e = before - 1;  // the last entry that starts at or before t
        if (in <= 8) {
          for (int i = 0; i < in; i++) e += __builtin_amdgcn_readlane(ex, before + i) <= t ? 1 : 0;
        } else {
          e = 0;
#pragma unroll
          for (int step = 32; step > 0; step >>= 1)
            if (__shfl(ex, e + step, 64) <= t) e += step;
        }
        e = e < 0 ? 0 : e;
        pos[q] = (RP)__shfl(delta, e, 64) + (RP)t;
        if (NUM) a[q] = __shfl(av, e, 64);
      }
    }
#pragma unroll
    for (int q = 0; q < K; q++) {
      const int x = x0 + q * 64 + lane, t = x - base;
      if (t >= 0 && t < total) {
        key[q] = ((unsigned)glob(tile.b_col)[pos[q]] << kEscKeyShift) | (unsigned)x;
        if (NUM) s_val[x] = (double)a[q] * (double)glob(tile.b_val)[pos[q]];
      }
    }
    base += total;
  }
}

// What the wavefronts of a row (W of them) tell each other when it is compressed.
template <int W>
struct EscShare {
  unsigned last[W];   // last key
  int count[W];       // output entries
  double lead[W];     // sum of the products before the first output entry (they end the last run of an earlier wavefront)
  int stop[W];        // lead ends inside the wavefront
  int open[W];        // its first position continues a run
  long long o;
};

// Compresses a sorted row (wavefront w of W holds positions [w * 64 * K, ...), slot x % K of lane x / K) and writes it. A position
// starts an output entry when it holds a product whose column differs from the previous position's. The runs of equal columns
// are summed from their end to their start: in the lane, then over the lanes and wavefronts that a run goes on in (a segmented
// suffix scan, skipped when no lane lies inside a run). A loop over each run's products in LDS took as many
// dependent reads as the longest run has products, and all wavefronts of the row waited for the one with the hub
// columns. Entries are staged in LDS by rank and stored with unit stride.
template <int K, int W, int MODE, typename T, typename RP, typename SYNC>
__device__ inline void esc_compress(const RowsDev<T, RP>& R, const TileDev<T, RP>& tile, int fr, unsigned (&key)[K], int w,
                                    int lane, unsigned* s_key, double* s_val, EscShare<W>& sh, SYNC&& sync) {
  constexpr bool NUM = MODE != 0;
  unsigned prev = (unsigned)__shfl_up((int)key[K - 1], 1, 64);
  if constexpr (W > 1) {
    if (lane == 63) sh.last[w] = key[K - 1];
    sync();
    if (lane == 0 && w > 0) prev = sh.last[w - 1];
  }
  bool head[K], pad[K];
  int mine = 0;
#pragma unroll
  for (int q = 0; q < K; q++) {
    pad[q] = key[q] == kEscPad;
    head[q] = !pad[q] && ((q == 0 && w == 0 && lane == 0) || (prev >> kEscKeyShift) != (key[q] >> kEscKeyShift));
    prev = key[q];
    mine += head[q] ? 1 : 0;
  }
  const int inc = wave_scan_dpp(mine);
  const int wcnt = __builtin_amdgcn_readlane(inc, 63);
  double v[NUM ? K : 1];
  double carry = 0.0;       // sum of the lane's products before its first head, and on through later lanes
  bool stop = true;         // carry ends
  const bool open0 = !head[0] && !pad[0];
  if constexpr (NUM) {
#pragma unroll
    for (int q = 0; q < K; q++) v[q] = pad[q] ? 0.0 : s_val[key[q] & kEscIdxMask];
    stop = false;
    bool in = open0;
#pragma unroll
    for (int q = 0; q < K; q++) {
      in = in && !head[q] && !pad[q];
      stop = stop || head[q] || pad[q];
      if (in) carry += v[q];
    }
    for (int d = 1; d < 64; d <<= 1) {
      if (__ballot(!stop) == 0ull) break;
      const double c = __shfl_down(carry, d, 64);
      const bool t = __shfl_down(stop ? 1 : 0, d, 64) != 0;
      if (!stop && lane + d < 64) {
        carry += c;
        stop = t;
      }
    }
  }
  int before = 0, cnt = wcnt;
  if constexpr (W > 1) {
    if (lane == 0) {
      sh.count[w] = wcnt;
      if (NUM) {
        sh.lead[w] = carry;
        sh.stop[w] = stop;
        sh.open[w] = open0;
      }
    }
    sync();
    cnt = 0;
#pragma unroll
    for (int q = 0; q < W; q++) {
      if (q < w) before += sh.count[q];
      cnt += sh.count[q];
    }
  }
  if constexpr (MODE == 0) {
    if (w == 0 && lane == 0) R.nnz[fr] = cnt;
    sync();
    return;
  } else {
    if (w == 0 && lane == 0) {
      long long o;
      if (MODE == 1 || (MODE == 2 && cnt <= R.cap[fr])) {
        o = R.off[fr];
      } else {
        o = (long long)atomicAdd(R.cursor, (unsigned long long)cnt);
        R.off[fr] = o;
      }
      if (o + cnt > R.out_limit) {  // refused: nothing is written and, after this pass, the row holds 0 entries
        R.stats[3] = 1ull;
        o = -1;
        if (MODE != 1) R.off[fr] = 0;
      }
      R.nnz[fr] = (o < 0 && MODE != 1) ? 0 : cnt;
      sh.o = o;
    }
    // what follows the lane's last position: the next lane's carry, or the next wavefronts'
    double next = __shfl_down(carry, 1, 64);
    bool cut = __shfl_down(open0 ? 1 : 0, 1, 64) == 0;
    if (lane == 63) {
      next = 0.0;
      cut = true;
      if constexpr (W > 1) {
        bool go = w + 1 < W && sh.open[w + 1 < W ? w + 1 : w];
        cut = !go;
        for (int q = w + 1; q < W && go; q++) {
          next += sh.lead[q];
          go = !sh.stop[q];
        }
      }
    }
    if constexpr (W > 1) {  // a run through all later lanes of this wavefront continues in the next ones
      const double far = __shfl(next, 63, 64);
      const bool far_cut = __shfl(cut ? 1 : 0, 63, 64) != 0;
      const bool through = __shfl_down(stop ? 1 : 0, 1, 64) == 0;  // the next lane's carry runs off the wavefront
      if (lane < 63 && !cut && through && !far_cut) next += far;
    }
    int r = before + inc;  // one past the lane's last entry
    T* s_out = reinterpret_cast<T*>(s_val);
#pragma unroll
    for (int q = K - 1; q >= 0; q--) {
      next = cut ? v[q] : v[q] + next;
      cut = head[q] || pad[q];
      if (head[q]) {
        r--;
        s_key[r] = key[q] >> kEscKeyShift;
        v[q] = next;
      }
    }
    sync();  // every product is read: s_val takes the entries
    r = before + inc;
#pragma unroll
    for (int q = K - 1; q >= 0; q--)
      if (head[q]) s_out[--r] = (T)v[q];
    sync();
    const long long o = sh.o;
    if (o >= 0) {
      for (int x = w * 64 + lane; x < cnt; x += 64 * W) {
        __builtin_nontemporal_store((int)s_key[x], &glob(tile.c_col)[o + x]);
        __builtin_nontemporal_store(s_out[x], &glob(tile.c_val)[o + x]);
      }
    }
    sync();
  }
}

template <int K, int MODE, typename T, typename RP>
__global__ __launch_bounds__(64 * kEscWaves) void k_esc(RowsDev<T, RP> R, int bin) {
  constexpr int N = 64 * K;
  constexpr bool NUM = MODE != 0;
  __shared__ double s_val[kEscWaves][NUM ? N : 1];    // float64 products by product index, then the entries' values
  __shared__ unsigned s_key[kEscWaves][NUM ? N : 1];  // the entries' columns
  __shared__ EscShare<1> s_share[kEscWaves];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const LaneLimits lim(lane);
  auto wave_sync = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  const int count = *R.count_of(bin);
  const int* items = R.bin_items + (int64_t)bin * R.bin_stride;
  for (int idx = blockIdx.x * kEscWaves + w; idx < count; idx += gridDim.x * kEscWaves) {
    const int fr = items[idx];
    const TileDev<T, RP> tile = R.tiles[R.blk_tile[fr >> 8]];
    const int64_t i = fr - tile.flat0;
    unsigned key[K];
    esc_expand<K, NUM>(tile, glob(tile.a_rp)[i], glob(tile.a_rp)[i + 1], 0, lane, key, s_val[w]);
    esc_sort(key, lane, lim);
    wave_sync();
    esc_compress<K, 1, MODE>(R, tile, fr, key, 0, lane, s_key[w], s_val[w], s_share[w], wave_sync);
  }
}

// ------------------------------------------------------------------------------------------------------------
// Rows of at most 32 (64) products, 8 (16) lanes each. The products are expanded four per lane as 32-bit keys (column
// << 5 (6) | product index), sorted in registers (DPP exchanges: no LDS, no barrier), and equal columns are summed in
// product (A-row) order, in float64, rounded once.
// A hash row of this size costs a table clear, LDS atomics and a sort of its table in LDS; a one-wavefront ESC row
// leaves half the lanes idle. Tiles up to 2^27 - 2 columns wide. Modes as in k_esc.
// ------------------------------------------------------------------------------------------------------------

constexpr int kSmallWaves = 4;  // wavefronts per block

// Ascending sort of the 4 * G keys of each row group (G = 8 or 16 lanes): in, any order; out, element x of the sorted
// sequence is slot x % 4 of lane x / 4. Bitonic, with every comparator ascending (each merge first meets the mirrored
// position). Four neighbours per lane put 10 of the 15 stages of 32 keys (11 of 21 of 64) inside a lane at two instructions a
// pair; the others take a DPP move and a median per key. 82 instructions instead of the 200 that positions
// spread over the lanes (slot * G + lane: 3 stages inside a lane) took.
template <int G>
__device__ inline void grp_sort(unsigned (&key)[4], int gl) {
  cx(key[0], key[1]);
  cx(key[2], key[3]);
  cx(key[0], key[2]);
  cx(key[1], key[3]);
  cx(key[1], key[2]);
  const unsigned l1 = gl & 1 ? ~0u : 0u, l2 = gl & 2 ? ~0u : 0u, l4 = gl & 4 ? ~0u : 0u, l8 = gl & 8 ? ~0u : 0u;
  auto mirror = [&](auto x, unsigned lim) {
    constexpr int X = decltype(x)::value;
    const unsigned o0 = dpp_xor<X>(key[3]), o1 = dpp_xor<X>(key[2]), o2 = dpp_xor<X>(key[1]), o3 = dpp_xor<X>(key[0]);
    key[0] = min_or_max(key[0], o0, lim);
    key[1] = min_or_max(key[1], o1, lim);
    key[2] = min_or_max(key[2], o2, lim);
    key[3] = min_or_max(key[3], o3, lim);
  };
  auto lanes = [&](auto x, unsigned lim) {
    constexpr int X = decltype(x)::value;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      // lane ^ 4 is the mirror of eight, then of four
      const unsigned o = X == 4 ? dpp_xor<3>(dpp_xor<7>(key[q])) : dpp_xor<X == 4 ? 1 : X>(key[q]);
      key[q] = min_or_max(key[q], o, lim);
    }
  };
  auto inside = [&] {
    cx(key[0], key[2]);
    cx(key[1], key[3]);
    cx(key[0], key[1]);
    cx(key[2], key[3]);
  };
  constexpr std::integral_constant<int, 1> x1{};
  constexpr std::integral_constant<int, 2> x2{};
  mirror(x1, l1);
  inside();
  mirror(std::integral_constant<int, 3>{}, l2);
  lanes(x1, l1);
  inside();
  mirror(std::integral_constant<int, 7>{}, l4);
  lanes(x2, l2);
  lanes(x1, l1);
  inside();
  if constexpr (G == 16) {
    mirror(std::integral_constant<int, 15>{}, l8);
    lanes(std::integral_constant<int, 4>{}, l4);
    lanes(x2, l2);
    lanes(x1, l1);
    inside();
  }
}

// One row per group of G lanes, four products per lane (G = 8 for 32 products: eight rows per wavefront): expand, sort,
// compress, write. `next` runs once the row's last global loads are issued (the caller's prefetch of its next row
// overlaps them). Every exchange is executed by all groups of the wavefront.
// Bound by issued instructions: the VALU, and the LDS pipe that lane exchanges and LDS accesses share (all four SIMDs of a CU
// use one). So entries are found by a popcount over a bit mask of their first products instead of a search by lane
// exchanges, prefixes and neighbours move by DPP, runs come from a bit mask of their heads, and products
// are put in sorted order in LDS and summed from there: about 60 LDS operations per row group instead of 300 and, with the
// sort above, 400 VALU instructions instead of 590 (numeric pass of the same square 4.26 -> 2.26 ms, symbolic 1.46 -> 0.99 ms).
template <int MODE, int G, int N, typename T, typename RP, typename NEXT>
__device__ inline void small_row(const RowsDev<T, RP>& R, const TileDev<T, RP>& tile, int fr, bool active, RP a0,
                                 RP a1, int grp, int gl, RP* s_delta, T* s_av, double* s_val, unsigned* s_key,
                                 NEXT&& next) {
  constexpr bool NUM = MODE != 0;
  constexpr int S = N / G;
  constexpr unsigned kShift = N == 32 ? 5 : 6;  // product-index bits of a key
  using Bits = std::conditional_t<N == 32, unsigned, unsigned long long>;  // a bit per product position of the row
  static_assert(S == 4 && (G == 8 || G == 16), "four products per lane, a group inside one 16-lane DPP row");
  auto wave_sync = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  auto group_bits = [&](bool v) { return (unsigned)(__ballot(v) >> (grp * G)) & ((1u << G) - 1u); };
  auto count_bits = [](Bits v) { return N == 32 ? __popc((unsigned)v) : __popcll((unsigned long long)v); };
  const int na = (int)(a1 - a0);
  // expand: product x (A-row order) goes to slot x / G of lane x % G of the group
  unsigned key[S];
#pragma unroll
  for (int q = 0; q < S; q++) key[q] = kEscPad;
  int base = 0;
  for (int c0 = 0; __ballot(c0 < na) != 0ull; c0 += G) {
    int len = 0;
    RP st = 0;
    T av = T(0);
    if (c0 + gl < na) {
      const int kk = glob(tile.a_col)[a0 + c0 + gl];
      st = glob(tile.b_rp)[kk];
      len = (int)(glob(tile.b_rp)[kk + 1] - st);
      if (NUM) av = glob(tile.a_val)[a0 + c0 + gl];
    }
    int inc = len;
    {
      int t = (int)dpp_below<1>((unsigned)inc);
      if (gl >= 1) inc += t;
      t = (int)dpp_below<2>((unsigned)inc);
      if (gl >= 2) inc += t;
      t = (int)dpp_below<4>((unsigned)inc);
      if (gl >= 4) inc += t;
      if constexpr (G == 16) inc += (int)dpp_below<8>((unsigned)inc);
    }
    const int ex = inc - len;
    const int total = __shfl(inc, G - 1, G);
    // the entries that have products, in order, and a bit at each one's first product
    const int rank = __popc(group_bits(len > 0) & ((1u << gl) - 1u));
    if (len > 0) {
      s_delta[rank] = st - (RP)ex;
      if (NUM) s_av[rank] = av;
    }
    auto or_group = [&](unsigned v) {
      v |= dpp_xor<1>(v);
      v |= dpp_xor<2>(v);
      v |= dpp_xor<7>(v);
      if constexpr (G == 16) v |= dpp_xor<15>(v);
      return v;
    };
    const unsigned lo = or_group(len > 0 && ex < 32 ? 1u << ex : 0u);
    unsigned hi = 0;
    if constexpr (N == 64) hi = or_group(len > 0 && ex >= 32 ? 1u << (ex - 32) : 0u);
    wave_sync();
#pragma unroll
    for (int q = 0; q < S; q++) {
      const int t = gl + G * q - base;
      if ((unsigned)t < (unsigned)total) {  // the row has at most N products, so base + total <= N
        int e;  // the entry holding product t
        if constexpr (N == 32) e = __popc(lo & ((2u << t) - 1u)) - 1;
        else e = (t < 32 ? __popc(lo & ((2u << t) - 1u)) : __popc(lo) + __popc(hi & ((2u << (t - 32)) - 1u))) - 1;
        const RP qb = s_delta[e] + (RP)t;
        key[q] = ((unsigned)glob(tile.b_col)[qb] << kShift) | (unsigned)(gl + G * q);
        if (NUM) s_val[gl + G * q] = (double)s_av[e] * (double)glob(tile.b_val)[qb];
      }
    }
    wave_sync();
    base += total;
  }
  next();
  grp_sort<G>(key, gl);
  // compress: a sorted position starts an output entry when its column differs from the previous position's
  if constexpr (MODE == 0) {
    const unsigned up = dpp_below<1>(key[S - 1]);
    unsigned cnt = 0;
#pragma unroll
    for (int q = 0; q < S; q++) {
      const unsigned prev = q > 0 ? key[q > 0 ? q - 1 : 0] : up;
      cnt += key[q] != kEscPad && ((q == 0 && gl == 0) || (prev >> kShift) != (key[q] >> kShift)) ? 1u : 0u;
    }
    cnt += dpp_xor<1>(cnt);
    cnt += dpp_xor<2>(cnt);
    cnt += dpp_xor<7>(cnt);
    if constexpr (G == 16) cnt += dpp_xor<15>(cnt);
    if (active && gl == 0) R.nnz[fr] = (int)cnt;
    return;
  }
  // from here on position x sits in slot x / G of lane x % G: neighbouring lanes take neighbouring outputs and LDS banks
#pragma unroll
  for (int q = 0; q < S; q++) s_key[gl * S + q] = key[q];
  wave_sync();
  Bits heads = 0;
  bool head[S];
  double sum[S];
#pragma unroll
  for (int q = 0; q < S; q++) {
    key[q] = s_key[gl + G * q];
    // the pad keys sort last, so the positions before `base` hold the products
    sum[q] = gl + G * q < base ? s_val[key[q] & (unsigned)(N - 1)] : 0.0;
  }
#pragma unroll
  for (int q = 0; q < S; q++) {
    const unsigned wrap = q > 0 ? dpp_above<G - 1>(key[q > 0 ? q - 1 : 0]) : 0u;  // lane 0's: of lane G - 1
    const unsigned up = dpp_below<1>(key[q]);
    const unsigned prev = gl > 0 ? up : wrap;
    head[q] = gl + G * q < base && (gl + G * q == 0 || (prev >> kShift) != (key[q] >> kShift));
    heads |= (Bits)group_bits(head[q]) << (G * q);
  }
  const int cnt = count_bits(heads);
  wave_sync();
#pragma unroll
  for (int q = 0; q < S; q++)
    if (gl + G * q < base) s_val[gl + G * q] = sum[q];
  long long o = 0;
  if (active && gl == 0) {
    if (MODE == 1 || (MODE == 2 && cnt <= R.cap[fr])) {
      o = R.off[fr];
    } else {
      o = (long long)atomicAdd(R.cursor, (unsigned long long)cnt);
      R.off[fr] = o;
    }
    if (o + cnt > R.out_limit) {  // refused: nothing is written and, after this pass, the row holds 0 entries
      R.stats[3] = 1ull;
      o = -1;
      if (MODE != 1) R.off[fr] = 0;
    }
    R.nnz[fr] = (o < 0 && MODE != 1) ? 0 : cnt;
  }
  o = __shfl(o, 0, G);
  wave_sync();
  // sum each run of equal columns in sorted order, i.e. in product order, by the run's first element
  int len[S];
#pragma unroll
  for (int q = 0; q < S; q++) {
    const int x = gl + G * q;
    const Bits later = heads >> x >> 1;
    len[q] = !head[q] ? 0 : later == 0 ? base - x : (N == 32 ? __ffs((int)later) : __ffsll((long long)later));
  }
  for (int j = 1; __ballot(max(max(len[0], len[1]), max(len[2], len[3])) > j) != 0ull; j++) {
#pragma unroll
    for (int q = 0; q < S; q++)
      if (j < len[q]) sum[q] += s_val[gl + G * q + j];
  }
  if (o >= 0) {
#pragma unroll
    for (int q = 0; q < S; q++) {
      if (head[q]) {
        const long long pos = o + count_bits(heads & (((Bits)1 << (gl + G * q)) - 1));
        // plain stores here: rows this small write a fraction of a cache line each, and L2 merges neighbouring
        // rows' pieces before they reach HBM (streaming stores made a 4096^2-grid Laplacian 6.6 -> 7.2 ms)
        glob(tile.c_col)[pos] = (int)(key[q] >> kShift);
        glob(tile.c_val)[pos] = (T)sum[q];
      }
    }
  }
  wave_sync();  // the next row reuses the LDS
}

// ONE: every row belongs to tiles[0] (a single product): the tile is read once, and the next row's bin item and
// A-row bounds are loaded while the current row runs, so a row waits on three dependent loads (A columns, B-row
// bounds, B entries) instead of five. G: lanes per row (8 or 16), N: its most products (32 or 64).
template <int MODE, bool ONE, int G, int N, typename T, typename RP>
__global__ __launch_bounds__(64 * kSmallWaves, !ONE ? 6 : N == 32 ? 8 : 7) void k_esc_small(RowsDev<T, RP> R, int bin) {
  constexpr int RW = 64 / G;  // rows per wavefront
  constexpr bool NUM = MODE != 0;
  // per row group: the staged A entries (B position of product t of the staged entries, less t), the products' values by
  // product index, the sorted keys. Strides of N + N / 4 put the rows of a wavefront on different banks.
  constexpr int GROUPS = kSmallWaves * RW, STRIDE = N + N / 4;
  __shared__ RP s_delta[GROUPS][G];
  __shared__ T s_av[NUM ? GROUPS : 1][G];
  __shared__ double s_val[NUM ? GROUPS : 1][STRIDE];
  __shared__ __align__(16) unsigned s_key[NUM ? GROUPS : 1][STRIDE];
  const int lane = threadIdx.x & 63, grp = lane / G, gl = lane % G;
  const int gi = (int)(threadIdx.x >> 6) * RW + grp, gn = NUM ? gi : 0;
  const int count = *R.count_of(bin);
  const int* items = R.bin_items + (int64_t)bin * R.bin_stride;
  const int stride = gridDim.x * kSmallWaves * RW;
  int64_t p = (int64_t)(blockIdx.x * kSmallWaves + (threadIdx.x >> 6)) * RW;  // the loop is wave-uniform
  if constexpr (ONE) {
    const TileDev<T, RP> tile = R.tiles[0];
    bool active = p + grp < count;
    int fr = active ? items[p + grp] : 0;
    RP a0 = 0, a1 = 0;
    if (active) {
      a0 = glob(tile.a_rp)[fr - tile.flat0];
      a1 = glob(tile.a_rp)[fr - tile.flat0 + 1];
    }
    for (; p < count; p += stride) {
      const int64_t idx_n = p + stride + grp;
      const bool act_n = idx_n < count;
      const int fr_n = act_n ? items[idx_n] : 0;
      RP a0_n = 0, a1_n = 0;
      small_row<MODE, G, N>(R, tile, fr, active, a0, a1, grp, gl, s_delta[gi], s_av[gn], s_val[gn], s_key[gn], [&] {
        if (act_n) {
          a0_n = glob(tile.a_rp)[fr_n - tile.flat0];
          a1_n = glob(tile.a_rp)[fr_n - tile.flat0 + 1];
        }
      });
      active = act_n;
      fr = fr_n;
      a0 = a0_n;
      a1 = a1_n;
    }
  } else {
    for (; p < count; p += stride) {
      const int64_t idx = p + grp;
      const bool active = idx < count;
      const int fr = active ? items[idx] : 0;
      TileDev<T, RP> tile;
      RP a0 = 0, a1 = 0;
      if (active) {
        tile = R.tiles[R.blk_tile[fr >> 8]];
        const int64_t i = fr - tile.flat0;
        a0 = glob(tile.a_rp)[i];
        a1 = glob(tile.a_rp)[i + 1];
      }
      small_row<MODE, G, N>(R, tile, fr, active, a0, a1, grp, gl, s_delta[gi], s_av[gn], s_val[gn], s_key[gn], [] {});
    }
  }
}

// Sort-based rows of 512 * W products or fewer, W wavefronts per row: each wavefront expands and sorts 512 of the
// row's products in registers (as the single-wavefront kernel does), the sorted runs are merged pairwise by the rest of a
// bitonic network, and the block compresses the sorted row. LDS: 12 bytes per product (key and float64 product). Rows of
// 2048 to 4096 products of an R-MAT square at scale 16 (12 M products): symbolic 131 -> 77 us, numeric
// 175 -> 110 us with the sort, the entry lookup and the compression above.
constexpr int kEscChunk = 512;

template <int W, int MODE, typename T, typename RP>
__global__ __launch_bounds__(64 * W, 6) void k_esc_block(RowsDev<T, RP> R, int bin) {
  constexpr int N = kEscChunk * W;
  constexpr int K = kEscChunk / 64;
  constexpr bool NUM = MODE != 0;
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  __shared__ __align__(16) unsigned s_key[N];
  __shared__ double s_val[NUM ? N : 1];
  __shared__ EscShare<W> s_share;
  static_assert(K == 8, "two 16-byte accesses per lane");
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const LaneLimits lim(lane);
  const int count = *R.count_of(bin);
  const int* items = R.bin_items + (int64_t)bin * R.bin_stride;
  for (int idx = blockIdx.x; idx < count; idx += gridDim.x) {
    const int fr = items[idx];
    const TileDev<T, RP> tile = R.tiles[R.blk_tile[fr >> 8]];
    const int64_t i = fr - tile.flat0;
    unsigned key[K];
    esc_expand<K, NUM>(tile, glob(tile.a_rp)[i], glob(tile.a_rp)[i + 1], w * kEscChunk, lane, key, s_val);
    esc_sort(key, lane, lim);
    // Merge: for each block size S = 1024 .. N, a mirror stage (position E against E ^ (S - 1)) and half-cleaners at
    // distances S / 4 .. 1. Distances of 512 or more cross wavefronts and go through LDS, where a lane's eight keys are two
    // 16-byte halves, each with neighbouring lanes side by side; shorter ones stay in registers and lanes.
    // One stage across wavefronts: against wavefront w ^ dw, mirrored or not; the lower wavefront keeps the minimum.
    auto cross = [&](int dw, auto mirror_tag, bool lower) {
      constexpr bool mirrored = decltype(mirror_tag)::value;
      u32x4* mine = reinterpret_cast<u32x4*>(s_key + w * kEscChunk);
      const u32x4* other = reinterpret_cast<const u32x4*>(s_key + (w ^ dw) * kEscChunk);
      mine[lane] = u32x4{key[0], key[1], key[2], key[3]};
      mine[64 + lane] = u32x4{key[4], key[5], key[6], key[7]};
      __syncthreads();
      const int l = mirrored ? 63 - lane : lane;
      const u32x4 p = other[l], q = other[64 + l];
      unsigned o[K];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        o[u] = mirrored ? q[3 - u] : p[u];
        o[4 + u] = mirrored ? p[3 - u] : q[u];
      }
#pragma unroll
      for (int u = 0; u < K; u++) key[u] = lower ? min(key[u], o[u]) : max(key[u], o[u]);
      __syncthreads();
    };
#pragma unroll 1
    for (int s = 2; s <= W; s <<= 1) {
      cross(s - 1, std::true_type{}, (w & (s >> 1)) == 0);
#pragma unroll 1
      for (int d = s >> 2; d > 0; d >>= 1) cross(d, std::false_type{}, (w & d) == 0);
      esc_half_clean(key, lim);
    }
    esc_compress<K, W, MODE>(R, tile, fr, key, w, lane, s_key, s_val, s_share, [] { __syncthreads(); });
  }
}

// ------------------------------------------------------------------------------------------------------------
// Heavy rows (more products than the sort-based bins take and more output entries than the hash tables are given),
// rank-slice accumulator: one workgroup per row, or per part of a split row, everything in LDS.
//   pass 1: LDS bitmap of the row's columns (one atomicOr per product) and prefix counts per group of kHRGroup
//           words, so every column's output rank is known and nnz(C_i) is exact;
//   pass 2 (numeric modes), per slice of hr_slice() ranks: the slice's columns are written from the bitmap, and the
//           products whose columns fall in its column range are added in float64 into an LDS array indexed by
//           rank - slice start (ds_add_f64), then written out with unit stride. Most rows fit one slice; larger
//           rows enumerate their products once per slice.
// Modes as in k_hash: 0 symbolic, 1 numeric at off[fr], 2 predicted (slot if nnz <= cap, else bump-allocate),
// 3 bump-allocate. Needs n <= 32 * kHRWords; wider tiles use k_heavy (global dense accumulator).
//
// A row with more products than heavy_part_size() is split by columns into parts of about that many: an R-MAT
// square at scale 16 has one row of 0.2 % of its products, and the workgroup that ran it alone took 1.6 times the
// average (19 M cycles of 10 M on average in a stage of 4 x 4 tiles at scale 21). Order of a pass:
//   k_order_heavy   picks the rows to split and orders the others by size
//   k_heavy_split   samples a split row's columns and cuts them into ranges with equal samples
//   k_heavy_rank<0> counts each part's entries (symbolic: and the whole rows')
//   k_heavy_place   sums a row's parts and, in modes 2 and 3, gives them their places in C
//   k_heavy_rank    the parts (largest pieces) first, then the whole rows, from one queue
// A part finds its share of each B row by binary search, and so does a slice of a row or part of several slices. B rows
// should be sorted, but nothing is lost where they are not: the counting pass checks each product's column against the
// part's range, and the numeric pass against the slice's. Shares tile every B row (or part of it), so if all columns are
// inside, nothing is missed. Otherwise the row runs whole, or its slices again over all of its products.
// R-MAT square at scale 16 (122 M products): symbolic 0.53 -> 0.20 ms, numeric 1.76 -> 0.62 ms with the parts, the
// product loop of enumerate_waves and a word of the bitmap per lane when the columns are written. Bound now by LDS latency and
// atomics with one workgroup of 16 wavefronts per CU.
// ------------------------------------------------------------------------------------------------------------

constexpr int kHRWords = 16384;  // bitmap words: tiles up to 2^19 columns
// Words per prefix group: a column's rank is its group's prefix plus the bits before it in the group, read as one
// 16-byte LDS load. Narrow groups cost prefix space (16 KB for 2^19 columns) but keep the per-product LDS reads at
// 20 bytes; 16-word groups (four loads) were measured 0.75 ms slower on the s22 stage despite larger slices.
constexpr int kHRGroup = 4;
// float64 accumulators per slice: what LDS holds beside the bitmap, the prefixes and the entry staging (64 KB or 56 KB)
template <typename T, typename RP>
constexpr int hr_slice() { return sizeof(T) == 4 && sizeof(RP) == 4 ? 8192 : 7168; }
// symbolic: 512 threads, two workgroups per CU; numeric: 1024 threads, one workgroup per CU (bitmap + slice)
template <int MODE>
constexpr int hr_block() { return MODE == 0 ? 512 : 1024; }

typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
static_assert(kHRGroup == 4, "hr_rank reads one 16-byte group");

// Output rank of column j: set bits before j. The group prefix counts the bits before j's group; the group (j's word
// and the words before it) is one 16-byte LDS load.
__device__ inline int hr_rank(const unsigned* bits, const int* gpre, int j) {
  const int w = j >> 5, g = w / kHRGroup, wi = w % kHRGroup;
  const u32x4_t x = *reinterpret_cast<const u32x4_t*>(bits + g * kHRGroup);
  const unsigned below = (1u << (j & 31)) - 1u;
  return gpre[g] + (wi > 0 ? __popc(x.x) : 0) + (wi > 1 ? __popc(x.y) : 0) + (wi > 2 ? __popc(x.z) : 0) +
         __popc((wi == 0 ? x.x : wi == 1 ? x.y : wi == 2 ? x.z : x.w) & below);
}

// Column of output rank r (0 <= r < number of set bits): the r-th set bit of groups [g0, g1). One thread.
__device__ inline int hr_select(const unsigned* bits, const int* gpre, int g0, int g1, int r) {
  int lo = g0, hi = g1;  // last group with gpre <= r
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (gpre[mid] <= r) lo = mid; else hi = mid;
  }
  int left = r - gpre[lo];
  int w = lo * kHRGroup;
  while (true) {
    const int c = __popc(bits[w]);
    if (left < c) break;
    left -= c;
    w++;
  }
  unsigned word = bits[w];
  for (int q = 0; q < left; q++) word &= word - 1;
  return w * 32 + (__ffs(word) - 1);
}

// First position in [lo0, len) of the B row at st whose column is >= c (binary search in global memory).
template <typename RP>
__device__ inline RP hr_lower_bound(const int* b_col, RP st, RP lo0, RP len, int c) {
  RP lo = lo0, hi = len;
  while (lo < hi) {
    const RP mid = (lo + hi) >> 1;
    if (b_col[st + mid] < c) lo = mid + 1; else hi = mid;
  }
  return lo;
}

// [lo, hi) of the B row at st of len entries whose columns are in [c_lo, c_hi) (binary searches in global memory, side by
// side).
template <typename RP>
__device__ inline void hr_column_range(const int* b_col, RP st, RP len, int c_lo, int c_hi, RP* lo, RP* hi) {
  RP l0 = 0, l1 = len, h0 = 0, h1 = len;
  while (l0 < l1 || h0 < h1) {
    const RP lm = (l0 + l1) >> 1, hm = (h0 + h1) >> 1;
    const int lc = l0 < l1 ? glob(b_col)[st + lm] : 0, hc = h0 < h1 ? glob(b_col)[st + hm] : 0;
    if (l0 < l1) {
      if (lc < c_lo) l0 = lm + 1; else l1 = lm;
    }
    if (h0 < h1) {
      if (hc < c_hi) h0 = hm + 1; else h1 = hm;
    }
  }
  *lo = l0;
  *hi = h0;
}

// The heavy bin before its rows run: decides which rows are split (BUILD; the numeric pass that follows a symbolic one
// keeps that pass's parts) and orders the others by decreasing products (classes of equal floor(log2 P)), so that the
// queue of k_heavy_rank starts the largest first and the small ones fill in behind them. One block.
template <bool BUILD, typename T, typename RP>
__global__ __launch_bounds__(1024) void k_order_heavy(RowsDev<T, RP> R) {
  constexpr int U = 8;
  __shared__ int s_hist[32], s_next[32];
  __shared__ int s_parts, s_split;
  __shared__ long long s_scan[17];
  const int tid = threadIdx.x;
  const int cnt = *R.count_of(kHeavyBin);
  int* items = R.bin_items + (int64_t)kHeavyBin * R.bin_stride;
  if (tid < 32) s_hist[tid] = 0;
  if (tid == 0) {
    s_parts = 0;
    s_split = 0;
    *R.heavy_queue = 0ull;
  }
  auto each = [&](auto&& f) {  // f(row, products), U rows in flight per thread
    for (int q0 = tid; q0 < cnt; q0 += U * 1024) {
      int fr[U];
      long long p[U];
#pragma unroll
      for (int u = 0; u < U; u++) fr[u] = q0 + u * 1024 < cnt ? items[q0 + u * 1024] : -1;
#pragma unroll
      for (int u = 0; u < U; u++) p[u] = fr[u] >= 0 ? R.prod[fr[u]] : 0;
#pragma unroll
      for (int u = 0; u < U; u++)
        if (fr[u] >= 0) f(fr[u], p[u]);
    }
  };
  auto cls = [&](long long p) {  // 31 - floor(log2 P), clamped to [0, 31]: larger rows first
    const int lg = 63 - __clzll((unsigned long long)(p > 1 ? p : 1));
    return 31 - (lg < 31 ? lg : 31);
  };
  long long size = LLONG_MAX;
  if (BUILD) {
    long long mine = 0;
    each([&](int, long long p) { mine += p; });
    size = heavy_part_size(block_sum<1024, long long>(mine, s_scan));
  }
  __syncthreads();
  each([&](int fr, long long p) {
    bool split = false;
    if (BUILD) {
      int first = -1;
      if (p > size) {
        const int n = R.tiles[R.blk_tile[fr >> 8]].n;
        const int k = (int)min(min((p + size - 1) / size, (long long)kMaxRowParts), (long long)(n / (32 * kHRGroup)));
        if (k > 1) {
          first = atomicAdd(&s_parts, k);
          R.heavy_parts[first].fr = fr;
          R.heavy_parts[first].parts = k;
          R.heavy_parts[first].bad = 0;
          R.heavy_parts[atomicAdd(&s_split, 1)].split_row = first;
          split = true;
        }
      }
      R.heavy_first[fr] = first;
    } else {
      const int first = R.heavy_first[fr];
      split = first >= 0 && !R.heavy_parts[first].bad;
    }
    if (!split) atomicAdd(&s_hist[cls(p)], 1);
  });
  __syncthreads();
  if (tid == 0) {
    int run = 0;
    for (int c = 0; c < 32; c++) {
      s_next[c] = run;
      run += s_hist[c];
    }
    R.heavy_head->ordered = run;
    R.heavy_head->rows = run;
    if (BUILD) {
      R.heavy_head->parts = s_parts;
      R.heavy_head->split_rows = s_split;
    }
  }
  __syncthreads();
  each([&](int fr, long long p) {
    const int first = R.heavy_first[fr];
    if (first < 0 || (!BUILD && R.heavy_parts[first].bad)) R.tmp_items[atomicAdd(&s_next[cls(p)], 1)] = fr;
  });
  __syncthreads();
  for (int q = tid; q < s_next[31]; q += 1024) items[q] = R.tmp_items[q];  // s_next[31] is now the end of the list
}

// Cuts the columns of each split row into ranges of about equal products: a histogram, by groups of kHRGroup words, of the columns
// of 8192 to 16384 products at equal distances in product order. One workgroup per row.
template <typename T, typename RP>
__global__ __launch_bounds__(1024) void k_heavy_split(RowsDev<T, RP> R) {
  constexpr int kSpan = 32 * kHRGroup;  // columns per group
  __shared__ int s_hist[kHRWords / kHRGroup];
  __shared__ RP s_delta[1024];
  __shared__ int s_pre[1024];
  __shared__ int s_scan[2][16];
  const int tid = threadIdx.x;
  const int nsplit = R.heavy_head->split_rows;
  for (int q = blockIdx.x; q < nsplit; q += gridDim.x) {
    const int first = R.heavy_parts[q].split_row;
    HeavyPart* parts = R.heavy_parts + first;
    const int fr = parts->fr, k = parts->parts;
    const TileDev<T, RP> tile = R.tiles[R.blk_tile[fr >> 8]];
    const RP a0 = tile.a_rp[fr - tile.flat0], a1 = tile.a_rp[fr - tile.flat0 + 1];
    const long long p = R.prod[fr], stride = p / 8192 > 1 ? p / 8192 : 1;
    const int groups = (tile.n + kSpan - 1) / kSpan;
    for (int g = tid; g < groups; g += 1024) s_hist[g] = 0;
    long long base = 0;  // products of the chunks before
    for (RP c0 = a0; c0 < a1; c0 += 1024) {
      const int ne = (int)((a1 - c0) < (RP)1024 ? (a1 - c0) : (RP)1024);
      RP st = 0;
      int len = 0;
      if (tid < ne) {
        const int kk = tile.a_col[c0 + tid];
        st = tile.b_rp[kk];
        len = (int)(tile.b_rp[kk + 1] - st);
      }
      int total;
      const int ex = block_scan_dpp<1024>(len, &total, s_scan[0]);
      if (tid < ne) {
        s_delta[tid] = st - (RP)ex;
        s_pre[tid] = ex;
      }
      __syncthreads();
      int top = 1;
      while (top < ne) top <<= 1;
      top >>= 1;
      for (long long smp = (base + stride - 1) / stride + tid; smp * stride < base + total; smp += 1024) {
        const int t = (int)(smp * stride - base);
        int e = 0;
        for (int step = top; step > 0; step >>= 1)
          if (e + step < ne && s_pre[e + step] <= t) e += step;
        atomicAdd(&s_hist[tile.b_col[s_delta[e] + (RP)t] / kSpan], 1);
      }
      base += total;
      __syncthreads();
    }
    // part x starts at the end of the group in which the running count passes x / k of the samples
    constexpr int kPer = kHRWords / kHRGroup / 1024;
    int mine = 0;
#pragma unroll
    for (int u = 0; u < kPer; u++) mine += tid * kPer + u < groups ? s_hist[tid * kPer + u] : 0;
    int ns;
    long long run = block_scan_dpp<1024>(mine, &ns, s_scan[1]);
    for (int u = 0; u < kPer; u++) {
      const int g = tid * kPer + u;
      if (g >= groups) break;
      const long long next = run + s_hist[g];
      for (long long x = run * k / ns + 1; x < k && x * ns <= next * k; x++) {
        parts[x].lo = (g + 1) * kSpan;
        parts[x - 1].hi = (g + 1) * kSpan;
      }
      run = next;
    }
    if (tid == 0) {
      parts[0].lo = 0;
      parts[k - 1].hi = groups * kSpan;
    }
    for (int x = tid; x < k; x += 1024) {
      parts[x].fr = fr;
      parts[x].nnz = 0;
    }
    __syncthreads();
  }
}

// After the parts are counted: a split row's entries are their sum; modes 2 and 3 also place it in C. Rows whose parts
// met unsorted B rows join the list of whole rows. One wavefront per row.
template <int MODE, typename T, typename RP>
__global__ __launch_bounds__(256) void k_heavy_place(RowsDev<T, RP> R) {
  const int lane = threadIdx.x & 63, nwaves = gridDim.x * 4;
  const int nsplit = R.heavy_head->split_rows;
  int* items = R.bin_items + (int64_t)kHeavyBin * R.bin_stride;
  if (blockIdx.x == 0 && threadIdx.x == 0) *R.heavy_queue = 0ull;
  for (int q = blockIdx.x * 4 + (threadIdx.x >> 6); q < nsplit; q += nwaves) {
    const int first = R.heavy_parts[q].split_row;
    HeavyPart* parts = R.heavy_parts + first;
    const int fr = parts->fr, k = parts->parts;
    const bool bad = parts->bad != 0;
    static_assert(kMaxRowParts == 4 * 64, "four parts per lane");
    int cnt[4], mine = 0;
#pragma unroll
    for (int u = 0; u < 4; u++) {
      cnt[u] = lane * 4 + u < k ? parts[lane * 4 + u].nnz : 0;
      mine += cnt[u];
    }
    const int inc = wave_scan_dpp(mine);
    const int total = __builtin_amdgcn_readlane(inc, 63);
    long long b = 0;
    if (lane == 0) {
      if (bad) {
        items[atomicAdd(&R.heavy_head->rows, 1)] = fr;
      } else {
        if (MODE != 0) {
          if (MODE == 2 && total <= R.cap[fr]) {
            b = R.off[fr];
          } else {
            b = (long long)atomicAdd(R.cursor, (unsigned long long)total);
            R.off[fr] = b;
          }
          if (b + total > R.out_limit) {  // refused, as a whole row is
            R.stats[3] = 1ull;
            b = -1;
            R.off[fr] = 0;
          }
        }
        R.nnz[fr] = b < 0 ? 0 : total;
        atomicAdd(&R.stats[1], 1ull);
      }
    }
    b = __shfl(b, 0, 64);
    long long off = b + inc - mine;
#pragma unroll
    for (int u = 0; u < 4; u++) {
      if (lane * 4 + u < k) parts[lane * 4 + u].off = b < 0 ? -1 : off;
      off += cnt[u];
    }
  }
}

// The product loop of a staged chunk of A entries, a run of consecutive products per wavefront. Entry e's products are
// t in [e_pre[e], e_pre[e + 1]) at B positions e_delta[e] + t (e_pre[0] = 0; the last entry ends at `total`). A wavefront keeps
// the entry of its next product and, for each 64 products, reads the starts of the 64 entries that follow:
// the few that lie inside are broadcast and counted per lane (a B row of a heavy row is mostly longer than 64), more than
// eight are searched. A binary search per product over the whole chunk took 5 to 10 dependent LDS reads
// and more instructions than everything else in the pass. U * 64 products are loaded at a time, ahead of the
// ones being added. f(column, a, b) per product.
template <int BLOCK, bool NUM, int U, typename T, typename RP, typename F>
__device__ inline void enumerate_waves(const TileDev<T, RP>& tile, int ne, int total, int tid, const RP* e_delta,
                                       const int* e_pre, const T* e_val, F&& f) {
  static_assert(BLOCK <= 1024, "the entry search takes two steps of 64 for at most 4096 entries");
  constexpr int NW = BLOCK / 64;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int seg = (total + NW * 64 - 1) / (NW * 64) * 64;
  const int t_beg = w * seg, t_end = min(total, t_beg + seg);
  if (t_beg >= t_end) return;
  int e;  // an entry that starts at or before the next product, with none but empty ones between them
  {
    const int step = (ne + 63) >> 6;
    e = (__popcll(__ballot(lane * step < ne && e_pre[lane * step < ne ? lane * step : 0] <= t_beg)) - 1) * step;
    const int x = e + lane;
    e += __popcll(__ballot(lane < step && x < ne && e_pre[x < ne ? x : 0] <= t_beg)) - 1;
  }
  struct Batch {
    int j[U];
    T a[U], b[U];
  };
  auto fetch = [&](int t0, Batch& r) {
    RP q[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int tu = t0 + 64 * u, t = tu + lane;
      q[u] = 0;
      if (tu < t_end) {  // uniform
        const int x = e + 1 + lane;
        const int start = x < ne ? e_pre[x] : INT_MAX;
        const int in = __popcll(__ballot(start <= tu + 63));
        int c = 0;
        if (in <= 8) {
          for (int i = 0; i < in; i++) c += __builtin_amdgcn_readlane(start, i) <= t ? 1 : 0;
        } else {
          for (int step = in < 64 ? 32 : 512; step > 0; step >>= 1)
            if (e + c + step < ne && e_pre[e + c + step] <= t) c += step;
        }
        const int et = e + c;
        q[u] = e_delta[et] + (RP)t;
        if (NUM) r.a[u] = e_val[et];
        e = in < 64 ? e + in : __builtin_amdgcn_readlane(et, 63);
      }
    }
#pragma unroll
    for (int u = 0; u < U; u++)
      if (t0 + 64 * u + lane < t_end) {
        r.j[u] = glob(tile.b_col)[q[u]];
        if (NUM) r.b[u] = glob(tile.b_val)[q[u]];
      }
  };
  auto use = [&](int t0, const Batch& r) {
#pragma unroll
    for (int u = 0; u < U; u++)
      if (t0 + 64 * u + lane < t_end) f(r.j[u], NUM ? r.a[u] : T(0), NUM ? r.b[u] : T(0));
  };
  Batch now, next;
  for (int t0 = t_beg - 64 * U; t0 < t_end; t0 += 64 * U) {
    if (t0 + 64 * U < t_end) fetch(t0 + 64 * U, next);
    if (t0 >= t_beg) use(t0, now);
    now = next;
  }
}

// A value that is the same in every lane, in scalar registers.
template <typename V>
__device__ inline V uniform(V v) {
  static_assert(sizeof(V) == 4 || sizeof(V) == 8, "one or two registers");
  int x[sizeof(V) / 4];
  __builtin_memcpy(x, &v, sizeof(V));
#pragma unroll
  for (unsigned u = 0; u < sizeof(V) / 4; u++) x[u] = __builtin_amdgcn_readfirstlane(x[u]);
  __builtin_memcpy(&v, x, sizeof(V));
  return v;
}

// what k_heavy_rank takes: parts and whole rows; parts only; the rows k_heavy_place appended
constexpr int kHeavyAll = 0, kHeavyParts = 1, kHeavyBad = 2;

template <int MODE, typename T, typename RP>
__global__ __launch_bounds__(hr_block<MODE>()) void k_heavy_rank(RowsDev<T, RP> R, int what) {
  constexpr int BLOCK = hr_block<MODE>();
  constexpr bool NUM = MODE != 0;
  constexpr int kHRSlice = hr_slice<T, RP>();
  __shared__ __align__(16) unsigned s_bits[kHRWords];
  __shared__ int s_gpre[NUM ? kHRWords / kHRGroup : 1];  // the symbolic pass needs only the total
  __shared__ __align__(16) double s_acc[NUM ? kHRSlice : 1];  // a slice's columns (as int), then its values
  __shared__ long long s_base;
  __shared__ int s_crange[2];
  __shared__ int s_outside;  // a product of a slice's share is not in the slice's columns
  __shared__ RP s_delta[BLOCK];
  // product prefixes of one staged chunk fit 32 bits: at most BLOCK entries, each a B row of at most 2^19 columns
  __shared__ int s_pre[BLOCK];
  __shared__ T s_val[NUM ? BLOCK : 1];
  __shared__ int s_scan[2][BLOCK / 64];
  const int tid = threadIdx.x;
  const HeavyHead head = *R.heavy_head;
  const int nparts = what == kHeavyBad ? 0 : head.parts;
  const int row0 = what == kHeavyBad ? head.ordered : 0;
  const int count = nparts + (what == kHeavyParts ? 0 : head.rows - row0);
  const int* items = R.bin_items + (int64_t)kHeavyBin * R.bin_stride + row0;
  int* s_colbuf = reinterpret_cast<int*>(s_acc);
  __shared__ int s_idx;
  // Parts and rows are taken from a queue (largest first), so one block's share is not fixed in advance. The next one is
  // fetched while the current one runs: its queue slot when the current one starts, then one dependent load per
  // barrier (bin item, tile, A row bounds, each entry's A column and value, its B-row range). A
  // row then starts with its staging in registers instead of behind a chain of global round trips.
  int nq = 0;        // thread 0: the next one's queue slot
  int pst = 0;       // fetch steps done for it (uniform)
  int n_idx = 0, n_fr = 0, n_tix = 0, n_kk = 0, n_cap = 0;  // n_cap, n_off: thread 0 only
  int n_lo = 0, n_hi = 0;  // its columns; n_hi 0: none (nothing to do)
  bool n_skip = false;
  long long n_off = 0;
  RP n_a0 = 0, n_a1 = 0, n_st = 0;
  int n_len = 0;
  T n_av = T(0);
  auto advance = [&](int upto) {  // all threads, uniform upto; a barrier separates steps 1 and 2
    if (pst < 1 && upto >= 1) {
      if (tid == 0) s_idx = nq;
      pst = 1;
      if (upto >= 2) __syncthreads();
    }
    if (pst < 2 && upto >= 2) {
      n_idx = __builtin_amdgcn_readfirstlane(s_idx);
      if (n_idx < count) n_fr = uniform(n_idx < nparts ? R.heavy_parts[n_idx].fr : items[n_idx - nparts]);
      pst = 2;
    }
    if (pst < 3 && upto >= 3) {
      n_skip = false;
      if (n_idx < count) {
        n_tix = uniform((int)R.blk_tile[n_fr >> 8]);
        if (n_idx < nparts) {
          const HeavyPart& x = R.heavy_parts[n_idx];
          n_lo = uniform(x.lo);
          n_hi = uniform(x.hi);
          n_skip = n_lo >= n_hi || (NUM && (x.nnz == 0 || x.off < 0));
        }
      }
      pst = 3;
    }
    if (pst < 4 && upto >= 4) {
      if (n_idx < count) {
        const TileDev<T, RP>& t = R.tiles[n_tix];
        const int64_t ni = n_fr - t.flat0;
        n_a0 = uniform(t.a_rp[ni]);
        n_a1 = uniform(t.a_rp[ni + 1]);
        if (n_idx < nparts) {
          if (NUM) {
            n_skip = n_skip || R.heavy_parts[R.heavy_first[n_fr]].bad;
            n_off = R.heavy_parts[n_idx].off;
            if (MODE == 1) {  // the row may hash now that its count is known, or not fit
              n_off += R.off[n_fr];
              n_skip = n_skip || bin_for(R.nnz[n_fr], R.prod[n_fr], R.tn, t.n, true) != kHeavyBin;
              if (!n_skip && R.off[n_fr] + R.nnz[n_fr] > R.out_limit) {
                if (tid == 0) R.stats[3] = 1ull;
                n_skip = true;
              }
            }
          }
        } else if (NUM && tid == 0) {  // only this block reads or rewrites the row's slot
          n_cap = R.cap[n_fr];
          n_off = R.off[n_fr];
        }
      }
      pst = 4;
    }
    if (pst < 5 && upto >= 5) {
      if (n_idx < count && n_a1 - n_a0 <= (RP)BLOCK && tid < (int)(n_a1 - n_a0)) {
        const TileDev<T, RP>& t = R.tiles[n_tix];
        n_kk = t.a_col[n_a0 + tid];
        if (NUM) n_av = t.a_val[n_a0 + tid];
      }
      pst = 5;
    }
    if (pst < 6 && upto >= 6) {
      if (n_idx < count && n_a1 - n_a0 <= (RP)BLOCK && tid < (int)(n_a1 - n_a0)) {
        const TileDev<T, RP>& t = R.tiles[n_tix];
        n_st = t.b_rp[n_kk];
        n_len = (int)(t.b_rp[n_kk + 1] - n_st);
      }
      pst = 6;
    }
  };
  if (tid == 0) nq = (int)atomicAdd(R.heavy_queue, 1ull);
  advance(6);  // the first one: the whole chain, unhidden
  for (;;) {
    if (n_idx >= count) break;
    const bool part = n_idx < nparts, skip = uniform((int)n_skip) != 0;
    const int idx = n_idx, fr = n_fr;
    TileDev<T, RP> tile = R.tiles[n_tix];
    tile.a_col = uniform(tile.a_col);
    tile.a_val = uniform(tile.a_val);
    tile.b_rp = uniform(tile.b_rp);
    tile.b_col = uniform(tile.b_col);
    tile.b_val = uniform(tile.b_val);
    tile.c_col = uniform(tile.c_col);
    tile.c_val = uniform(tile.c_val);
    tile.n = uniform(tile.n);
    const int W = (tile.n + 31) / 32;
    const int Wr = (W + kHRGroup - 1) / kHRGroup * kHRGroup;  // whole groups (the tail words stay zero)
    const int lo = part ? n_lo : 0, hi = part ? n_hi : INT_MAX;
    const int w0 = lo >> 5, w1 = part ? hi >> 5 : Wr;  // the words in use: a part's, whole groups, or all
    if (!skip)
      for (int w = w0 + tid; w < w1; w += BLOCK) s_bits[w] = 0u;
    const RP a0 = n_a0, a1 = n_a1;
    const int na = (int)(a1 - a0);
    const bool one_chunk = na <= BLOCK;  // one entry per thread, staged once and kept in registers
    RP my_st = n_st;
    int my_len = n_len;
    const T my_av = n_av;
    const int my_cap = n_cap;
    const long long my_off = n_off;
    if (tid == 0) nq = (int)atomicAdd(R.heavy_queue, 1ull);
    pst = 0;
    n_st = 0;
    n_len = 0;
    n_av = T(0);
    do {
      __syncthreads();
      if (skip) break;
      bool bad = false;  // MODE 0, parts: a product outside the part's columns
      // Stage (start, length, value) of the row's entries, one per thread and BLOCK at a time, and run the product loop.
      // One chunk: st and len are the caller's. More: each chunk is loaded, and cut to the columns [c_lo, c_hi)
      // of a part.
      auto run_row = [&](RP st, int len, int c_lo, int c_hi, auto&& f, auto num_tag) {
        constexpr bool kNum = decltype(num_tag)::value;
        for (RP c0 = a0; c0 < a1; c0 += BLOCK) {
          const int ne = (int)((a1 - c0) < (RP)BLOCK ? (a1 - c0) : (RP)BLOCK);
          T av = my_av;
          if (!one_chunk) {
            st = 0;
            len = 0;
            if (tid < ne) {
              const int kk = glob(tile.a_col)[c0 + tid];
              st = glob(tile.b_rp)[kk];
              const RP l = glob(tile.b_rp)[kk + 1] - st;
              len = (int)l;
              if (kNum) av = glob(tile.a_val)[c0 + tid];
              if (part) {
                RP x, y;
                hr_column_range(tile.b_col, st, l, c_lo, c_hi, &x, &y);
                bad = bad || y < x;
                st += x;
                len = y > x ? (int)(y - x) : 0;
              }
            }
          }
          int tot;
          const int ex = block_scan_dpp<BLOCK>(tid < ne ? len : 0, &tot, s_scan[0]);
          if (tid < ne) {
            s_delta[tid] = st - (RP)ex;
            s_pre[tid] = ex;
            if constexpr (kNum) s_val[tid] = av;
          }
          __syncthreads();
          enumerate_waves<BLOCK, kNum, sizeof(T) + sizeof(RP) == 8 ? 4 : 2>(tile, ne, tot, tid, s_delta, s_pre, s_val, f);
          __syncthreads();
        }
      };
      if (part && one_chunk && tid < na) {  // the entry's share of its B row
        RP x, y;
        hr_column_range(tile.b_col, my_st, (RP)my_len, lo, hi, &x, &y);
        bad = y < x;
        my_st += x;
        my_len = y > x ? (int)(y - x) : 0;
      }
      auto set_bit = [&](int j, T, T) {
        atomicOr(&s_bits[j >> 5], 1u << (j & 31));
        if (MODE == 0 && part) bad = bad || (unsigned)(j - lo) >= (unsigned)(hi - lo);
      };
      run_row(my_st, my_len, lo, hi, set_bit, std::false_type{});
      if (MODE == 0 && part && bad) R.heavy_parts[R.heavy_first[fr]].bad = 1;
      advance(1);
      __syncthreads();
      advance(2);
      // group prefixes, in order: thread t counts `per` groups from g0 + t * per
      const int g0 = w0 / kHRGroup, g1 = w1 / kHRGroup;
      const int per = (g1 - g0 + BLOCK - 1) / BLOCK;
      int c = 0;
      for (int g = g0 + tid * per; g < min(g1, g0 + (tid + 1) * per); g++) {
        const u32x4_t x = *reinterpret_cast<const u32x4_t*>(s_bits + g * kHRGroup);
        const int n1 = __popc(x.x) + __popc(x.y) + __popc(x.z) + __popc(x.w);
        if (NUM) s_gpre[g] = n1;
        c += n1;
      }
      int total;
      int run = block_scan_dpp<BLOCK>(c, &total, s_scan[1]);
      advance(3);
      if (MODE == 0) {
        if (tid == 0) {
          if (part) {
            R.heavy_parts[idx].nnz = total;
          } else {
            R.nnz[fr] = total;
            atomicAdd(&R.stats[1], 1ull);
          }
        }
        __syncthreads();
        break;
      }
      for (int g = g0 + tid * per; g < min(g1, g0 + (tid + 1) * per); g++) {
        const int n1 = s_gpre[g];
        s_gpre[g] = run;
        run += n1;
      }
      if (tid == 0) {
        long long b = my_off;
        if (!part) {
          if (!(MODE == 1 || (MODE == 2 && total <= my_cap))) {
            b = (long long)atomicAdd(R.cursor, (unsigned long long)total);
            R.off[fr] = b;
          }
          if (b + total > R.out_limit) {  // refused: nothing is written and, after this pass, the row holds 0 entries
            R.stats[3] = 1ull;
            b = -1;
            if (MODE != 1) R.off[fr] = 0;
          }
          R.nnz[fr] = (b < 0 && MODE != 1) ? 0 : total;
          atomicAdd(&R.stats[1], 1ull);
        }
        s_base = b;
        s_outside = 0;
      }
      __syncthreads();
      const long long base = uniform(s_base);
      advance(4);
      if (base < 0) {  // refused: nothing is written
        __syncthreads();
        break;
      }
      // one rank slice at a time: columns (staged in LDS by rank, then stored with unit stride), then values. A
      // slice's first column and each entry's first B position in it are where the previous slice ended.
      RP my_lo = 0;
      bool search = one_chunk || part;  // each slice finds its share of the B rows (uniform)
      for (int s0 = 0; s0 < total; s0 += kHRSlice) {
        const int len = total - s0 < kHRSlice ? total - s0 : kHRSlice;
        const bool whole = s0 == 0 && len == total;
        int c_lo = lo, c_hi = hi;
        if (!whole) {
          if (tid == 0) {  // column range of the slice
            s_crange[0] = s0 == 0 ? lo : s_crange[1];
            s_crange[1] = s0 + len >= total ? hi : hr_select(s_bits, s_gpre, g0, g1, s0 + len);
          }
          __syncthreads();
          c_lo = uniform(s_crange[0]);
          c_hi = uniform(s_crange[1]);
        }
        const int w_lo = c_lo >> 5, w_hi = c_hi == INT_MAX ? W - 1 : (c_hi - 1) >> 5;
        // a wavefront takes 64 consecutive words (whole groups) at a time: each word's rank base is its group prefix
        // plus the bits of the group's earlier words (a kHRGroup-lane scan of popcounts). A lane per word keeps
        // the lanes of a wavefront alike; 16 words per thread left one wavefront with all of a skewed row's dense words
        // (20700 of 130000 cycles per row of an R-MAT square at scale 16).
        for (int wb = (w_lo & ~63) + (tid & ~63); wb <= w_hi; wb += BLOCK) {
          const int lane = tid & 63, w = wb + lane;
          const unsigned full = w >= w0 && w < w1 && w < W ? s_bits[w] : 0u;
          const int pc = __popc(full);
          int inc = pc;
#pragma unroll
          for (int d = 1; d < kHRGroup; d <<= 1) {
            const int t = __shfl_up(inc, d, kHRGroup);
            if ((lane & (kHRGroup - 1)) >= d) inc += t;
          }
          unsigned m = (w >= w_lo && w <= w_hi) ? full : 0u;
          if (w == w_lo) m &= ~((1u << (c_lo & 31)) - 1u);
          if (c_hi != INT_MAX && w == (c_hi >> 5)) m &= (1u << (c_hi & 31)) - 1u;
          if (m) {
            int r = s_gpre[w / kHRGroup] + inc - pc - s0 + __popc(full & ((m & (0u - m)) - 1u));
            while (m) {
              s_colbuf[r++] = w * 32 + (__ffs(m) - 1);
              m &= m - 1;
            }
          }
        }
        __syncthreads();
        if (s0 == 0) advance(5);
        for (int t = tid; t < len; t += BLOCK) __builtin_nontemporal_store(s_colbuf[t], &glob(tile.c_col)[base + s0 + t]);
        __syncthreads();
        for (int t = tid; t < len; t += BLOCK) s_acc[t] = 0.0;
        if (s0 == 0) advance(6);
        auto add = [&](int j, T a, T b) {
          if (whole || (j >= c_lo && j < c_hi))
            atomicAdd(&s_acc[hr_rank(s_bits, s_gpre, j) - s0], (double)a * (double)b);
          else
            s_outside = 1;
        };
        RP st = my_st;
        int ln = my_len;
        if (search && one_chunk && !whole && tid < na) {  // the part of the entry's B row inside the slice's columns
          const RP x = my_lo;
          const RP y = s0 + len >= total ? (RP)my_len : hr_lower_bound(tile.b_col, my_st, x, (RP)my_len, c_hi);
          st = my_st + x;
          ln = (int)(y - x);
          my_lo = y;
        }
        run_row(st, ln, search ? c_lo : lo, search ? c_hi : hi, add, std::true_type{});
        for (int t = tid; t < len; t += BLOCK) __builtin_nontemporal_store((T)s_acc[t], &glob(tile.c_val)[base + s0 + t]);
        __syncthreads();
        if (!whole && search && s0 + len >= total && uniform(s_outside)) {  // an unsorted B row: all slices again
          search = false;
          s0 = -kHRSlice;
        }
      }
    } while (false);
    advance(6);  // rows that ended early (symbolic, refused, skipped) finish the next row's fetch here
  }
}

// ------------------------------------------------------------------------------------------------------------
// Heavy rows: one workgroup per row, a bitmap of the row's columns (LDS when it fits, else global) and a dense
// float64 accumulator of n entries in HBM (one zeroed slot per resident workgroup; emission re-zeroes it).
// The bitmap gives the sorted column order and the exact count without a sort.
//   MODE 0 symbolic -> nnz[fr]; MODE 1 numeric at off[fr];
//   MODE 2 predicted: write at off[fr] when count <= cap[fr], else bump-allocate; MODE 3 bump-allocate.
// ------------------------------------------------------------------------------------------------------------

// The dense accumulator (and the bitmap when it is in global memory) is private to one workgroup: every access is
// a workgroup-scope atomic (performed in L2) ordered by workgroup barriers, so no device-scope fence is needed.
template <bool LDS_BITMAP>
__device__ inline void heavy_bit_set(unsigned* bits, int j) {
  if (LDS_BITMAP) atomicOr(&bits[j >> 5], 1u << (j & 31));
  else __hip_atomic_fetch_or(&bits[j >> 5], 1u << (j & 31), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
template <bool LDS_BITMAP>
__device__ inline unsigned heavy_bit_word(unsigned* bits, int64_t w) {
  if (LDS_BITMAP) return bits[w];
  return __hip_atomic_load(&bits[w], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <int MODE, bool LDS_BITMAP, typename T, typename RP>
__global__ __launch_bounds__(kHeavyThreads) void k_heavy(RowsDev<T, RP> R, int bin, double* dense_slots,
                                                         int64_t slot_doubles, unsigned* gbits, int64_t words) {
  extern __shared__ unsigned s_dyn[];
  __shared__ long long s_scan[kHeavyThreads / 64 + 1];
  __shared__ long long s_base;
  constexpr bool NUM = MODE != 0;
  const int tid = threadIdx.x;
  double* dense = dense_slots + (int64_t)blockIdx.x * slot_doubles;
  unsigned* bits = LDS_BITMAP ? s_dyn : gbits + (int64_t)blockIdx.x * words;
  const int count = *R.count_of(bin);
  const int* items = R.bin_items + (int64_t)bin * R.bin_stride;
  for (int idx = blockIdx.x; idx < count; idx += gridDim.x) {
    const int fr = items[idx];
    const TileDev<T, RP> tile = R.tiles[R.blk_tile[fr >> 8]];
    const int64_t i = fr - tile.flat0;
    const int64_t W = ((int64_t)tile.n + 31) / 32;
    if (LDS_BITMAP)
      for (int64_t w = tid; w < W; w += kHeavyThreads) bits[w] = 0u;
    __syncthreads();
    const RP a0 = tile.a_rp[i], a1 = tile.a_rp[i + 1];
    const long long prod = R.prod[fr];
    const long long na = (long long)(a1 - a0);
    const long long avg = (prod + na - 1) / (na > 0 ? na : 1);
    int lg = 0;
    while ((1 << lg) < avg && (1 << lg) < kHeavyThreads) lg++;
    const int L = 1 << lg, S = kHeavyThreads >> lg;
    const int sub = tid >> lg, sl = tid & (L - 1);
    for (RP p = a0 + sub; p < a1; p += S) {
      const int kk = tile.a_col[p];
      const double av = NUM ? (double)tile.a_val[p] : 0.0;
      const RP b0 = tile.b_rp[kk], b1 = tile.b_rp[kk + 1];
      for (RP q = b0 + sl; q < b1; q += L) {
        const int j = tile.b_col[q];
        heavy_bit_set<LDS_BITMAP>(bits, j);
        if (NUM)
          __hip_atomic_fetch_add(&dense[j], av * (double)tile.b_val[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    }
    __syncthreads();
    const int64_t per = (W + kHeavyThreads - 1) / kHeavyThreads;
    const int64_t w0 = tid * per, w1 = (w0 + per < W) ? w0 + per : W;
    long long c = 0;
    for (int64_t w = w0; w < w1; w++) c += __popc(heavy_bit_word<LDS_BITMAP>(bits, w));
    long long total;
    const long long pre = block_excl_scan<kHeavyThreads, long long>(c, &total, s_scan);
    if (MODE == 0) {
      if (tid == 0) R.nnz[fr] = (int)total;
      if (!LDS_BITMAP)
        for (int64_t w = w0; w < w1; w++) __hip_atomic_store(&bits[w], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    } else {
      if (tid == 0) {
        long long b;
        if (MODE == 1) {
          b = R.off[fr];
        } else if (MODE == 2 && total <= (long long)R.cap[fr]) {
          b = R.off[fr];
        } else {
          b = (long long)atomicAdd(R.cursor, (unsigned long long)total);
          R.off[fr] = b;
        }
        if (b + total > R.out_limit) {  // refused: nothing is written and, after this pass, the row holds 0 entries
          R.stats[3] = 1ull;
          b = -1;
          if (MODE != 1) R.off[fr] = 0;
        }
        s_base = b;
        R.nnz[fr] = (b < 0 && MODE != 1) ? 0 : (int)total;
      }
      __syncthreads();
      const bool fits = s_base >= 0;
      long long pos = s_base + pre;
      for (int64_t w = w0; w < w1; w++) {
        unsigned word = heavy_bit_word<LDS_BITMAP>(bits, w);
        while (word) {  // read and re-zero the accumulator whether or not the row is written
          const int bit = __ffs(word) - 1;
          const int j = (int)(w * 32 + bit);
          const double v = __hip_atomic_exchange(&dense[j], 0.0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          if (fits) {
            __builtin_nontemporal_store(j, &tile.c_col[pos]);
            __builtin_nontemporal_store((T)v, &tile.c_val[pos]);
            pos++;
          }
          word &= word - 1;
        }
        if (!LDS_BITMAP) __hip_atomic_store(&bits[w], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    }
    if (tid == 0) atomicAdd(&R.stats[1], 1ull);
    __syncthreads();
  }
}

// ------------------------------------------------------------------------------------------------------------
// Scans over flat rows: off[r] = sum_{q < r} cnt[q] (int32 counts -> int64 offsets), off[n] = total.
// Three launches: per-block sums, scan of block sums (one block), per-block scan with base.
// ------------------------------------------------------------------------------------------------------------

constexpr int kScanBlock = 1024;
constexpr int kScanPer = 4;
constexpr int kScanTile = kScanBlock * kScanPer;

// kScanPer consecutive counts of a thread: one 16-byte load inside the array (cnt is 16-byte aligned), else scalars
__device__ inline void scan_load4(const int32_t* cnt, int64_t n, int64_t r0, long long* v) {
  static_assert(kScanPer == 4, "one int4 per thread");
  if (r0 + 3 < n) {
    const int4 x = *reinterpret_cast<const int4*>(cnt + r0);
    v[0] = x.x;
    v[1] = x.y;
    v[2] = x.z;
    v[3] = x.w;
  } else {
#pragma unroll
    for (int q = 0; q < kScanPer; q++) v[q] = r0 + q < n ? cnt[r0 + q] : 0;
  }
}

static __global__ __launch_bounds__(kScanBlock) void k_scan_reduce(const int32_t* cnt, int64_t n, long long* partial) {
  __shared__ long long sm[kScanBlock / 64 + 1];
  const int64_t r0 = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanPer;
  long long v[kScanPer];
  scan_load4(cnt, n, r0, v);
  long long s = v[0] + v[1] + v[2] + v[3];
  s = block_sum<kScanBlock, long long>(s, sm);
  if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

static __global__ __launch_bounds__(kScanBlock) void k_scan_top(long long* partial, int64_t nblocks, int64_t* total_out) {
  __shared__ long long sm[kScanBlock / 64 + 1];
  long long run = 0;
  for (int64_t base = 0; base < nblocks; base += kScanBlock) {
    const int64_t r = base + threadIdx.x;
    long long v = r < nblocks ? partial[r] : 0;
    long long tot;
    long long ex = block_excl_scan<kScanBlock, long long>(v, &tot, sm);
    if (r < nblocks) partial[r] = run + ex;
    run += tot;
  }
  if (threadIdx.x == 0 && total_out) *total_out = run;
}

static __global__ __launch_bounds__(kScanBlock) void k_scan_final(const int32_t* cnt, int64_t n, const long long* partial,
                                                           int64_t* off, int64_t off_add) {
  __shared__ long long sm[kScanBlock / 64 + 1];
  const int64_t base = (int64_t)blockIdx.x * kScanTile;
  // each thread owns kScanPer consecutive elements
  const int64_t r0 = base + (int64_t)threadIdx.x * kScanPer;
  long long v[kScanPer];
  scan_load4(cnt, n, r0, v);
  const long long s = v[0] + v[1] + v[2] + v[3];
  long long tot;
  long long ex = block_excl_scan<kScanBlock, long long>(s, &tot, sm);
  long long run = partial[blockIdx.x] + ex + off_add;
  if (r0 + 3 < n) {  // two 16-byte stores (off is 16-byte aligned and r0 a multiple of 4)
    typedef long long ll2 __attribute__((ext_vector_type(2)));
    ll2* o = reinterpret_cast<ll2*>(off + r0);
    o[0] = ll2{run, run + v[0]};
    o[1] = ll2{run + v[0] + v[1], run + v[0] + v[1] + v[2]};
    run += s;
  } else {
    for (int q = 0; q < kScanPer; q++) {
      if (r0 + q < n) off[r0 + q] = run;
      run += v[q];
    }
  }
  if (r0 + kScanPer >= n && r0 < n) off[n] = run;  // the thread holding the last element writes the total
}

// Compaction of the learned path: each row's entries move from the arena (at off[fr], nnz[fr] long) to the final
// CSR (at dst_off[fr]). Work is split by output entries, not rows, so a block of hub rows (tens of thousands of
// entries each) costs the same as any other: block c copies entries [c * kCompactChunk, (c + 1) * kCompactChunk).
constexpr int kCompactChunk = 8192;

// chunk_row[c] = the flat row holding output entry c * kCompactChunk.
static __global__ __launch_bounds__(kRowBlock) void k_chunk_rows(const int64_t* dst_off, int64_t nflat,
                                                                 long long max_out, int32_t* chunk_row) {
  const int64_t r = (int64_t)blockIdx.x * kRowBlock + threadIdx.x;
  if (r >= nflat) return;
  const long long a = dst_off[r], b = dst_off[r + 1] < max_out ? dst_off[r + 1] : max_out;
  for (long long c = (a + kCompactChunk - 1) / kCompactChunk; c * kCompactChunk < b; c++) chunk_row[c] = (int32_t)r;
}

// One block per chunk. The block walks windows of 256 row offsets (LDS) from the chunk's first row; each thread
// finds the row of its entry by binary search in the window and copies it. Loads and stores are unit-stride across
// the wavefront, four entries in flight per thread.
template <typename T, typename RP>
__global__ __launch_bounds__(kRowBlock) void k_compact(RowsDev<T, RP> R, const int64_t* dst_off, int64_t nflat,
                                                       const int32_t* chunk_row, long long max_out, int* dst_col,
                                                       T* dst_val, const int* src_col, const T* src_val) {
  __shared__ long long s_dst[kRowBlock + 1];
  __shared__ long long s_src[kRowBlock];
  const int tid = threadIdx.x;
  long long total = dst_off[nflat];
  if (total > max_out) {  // more entries than the output holds: refuse the excess and flag it
    if (blockIdx.x == 0 && tid == 0) R.stats[3] = 1ull;
    total = max_out;
  }
  const long long c0 = (long long)blockIdx.x * kCompactChunk;
  if (c0 >= total) return;
  const long long c1 = c0 + kCompactChunk < total ? c0 + kCompactChunk : total;
  int64_t r0 = chunk_row[blockIdx.x];
  long long e = c0;
  while (e < c1) {
    const int64_t r = r0 + tid;
    s_dst[tid] = dst_off[r < nflat ? r : nflat];
    s_src[tid] = r < nflat ? R.off[r] : 0;
    if (tid == 0) s_dst[kRowBlock] = dst_off[r0 + kRowBlock < nflat ? r0 + kRowBlock : nflat];
    __syncthreads();
    const long long we = s_dst[kRowBlock] < c1 ? s_dst[kRowBlock] : c1;
    for (long long x0 = e; x0 < we; x0 += 4LL * kRowBlock) {
      long long src[4];
      bool ok[4];
      int a[4];  // largest a with s_dst[a] <= x: four branchless searches in lockstep
#pragma unroll
      for (int q = 0; q < 4; q++) a[q] = 0;
#pragma unroll
      for (int step = kRowBlock / 2; step > 0; step >>= 1) {
#pragma unroll
        for (int q = 0; q < 4; q++)
          if (s_dst[a[q] + step] <= x0 + (long long)q * kRowBlock + tid) a[q] += step;
      }
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const long long x = x0 + (long long)q * kRowBlock + tid;
        ok[q] = x < we;
        src[q] = s_src[a[q]] + (x - s_dst[a[q]]);
      }
      int cv[4];
      T vv[4];
#pragma unroll
      for (int q = 0; q < 4; q++)
        if (ok[q]) {
          // the arena is read once: streaming loads, as the stores
          cv[q] = __builtin_nontemporal_load(&src_col[src[q]]);
          vv[q] = __builtin_nontemporal_load(&src_val[src[q]]);
        }
#pragma unroll
      for (int q = 0; q < 4; q++)
        if (ok[q]) {
          const long long x = x0 + (long long)q * kRowBlock + tid;
          __builtin_nontemporal_store(cv[q], &dst_col[x]);
          __builtin_nontemporal_store(vv[q], &dst_val[x]);
        }
    }
    e = we;
    r0 += kRowBlock;
    __syncthreads();
  }
}

// Scan of at most kScanOneMax counts by one workgroup: one launch instead of three. A wavefront takes 1024 neighbouring
// counts, 64 per instruction, scans them by DPP, and the block meets at one barrier: 16384 rows 8.3 us (9.4 with four counts
// per thread side by side, bound by the 8-byte stores of neighbouring lanes going to different lines; three launches
// 8.3 and two more gaps between them). report (may be null): the bin counts and the total go to pinned host
// memory, kNumBins + 1 values, as k_report writes them.
constexpr int kScanOnePer = 16;
constexpr int64_t kScanOneMax = 2 * 1024 * kScanOnePer;

// Inclusive scan of one 64-bit value per lane of a wavefront, by DPP.
__device__ inline long long wave_scan_dpp64(long long v) {
  auto step = [&](auto ctrl, auto rows) {
    const int lo = __builtin_amdgcn_update_dpp(0, (int)v, decltype(ctrl)::value, decltype(rows)::value, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(v >> 32), decltype(ctrl)::value, decltype(rows)::value, 0xF, false);
    v += (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
  };
  constexpr std::integral_constant<int, 0xF> all{};
  step(std::integral_constant<int, 0x111>{}, all);  // row_shr:1, 2, 4, 8
  step(std::integral_constant<int, 0x112>{}, all);
  step(std::integral_constant<int, 0x114>{}, all);
  step(std::integral_constant<int, 0x118>{}, all);
  step(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xA>{});  // row_bcast:15 into rows 1 and 3
  step(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xC>{});  // row_bcast:31 into rows 2 and 3
  return v;
}
__device__ inline long long read_lane64(long long v, int lane) {
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)v, lane);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(v >> 32), lane);
  return (long long)(((unsigned long long)hi << 32) | lo);
}

static __global__ __launch_bounds__(1024) void k_scan_one(const int32_t* cnt, int64_t n, int64_t* off, int64_t off_add,
                                                          int64_t* total_out, const int32_t* bin_count, int64_t* report) {
  __shared__ long long s_wave[2][16];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  if (report && threadIdx.x < kNumBins) report[threadIdx.x] = bin_count[threadIdx.x * kCountStride];
  long long base = off_add;
  int turn = 0;
  for (int64_t b = 0; b < n; b += 1024 * kScanOnePer, turn ^= 1) {
    const int64_t r0 = b + w * 64 * kScanOnePer + lane;
    int v[kScanOnePer];
#pragma unroll
    for (int q = 0; q < kScanOnePer; q++) v[q] = r0 + q * 64 < n ? cnt[r0 + q * 64] : 0;
    long long ex[kScanOnePer], mine = 0;  // exclusive in the wavefront; its total so far
#pragma unroll
    for (int q = 0; q < kScanOnePer; q++) {
      ex[q] = 0;
      if (r0 - lane + q * 64 < n) {  // uniform
        const long long inc = wave_scan_dpp64(v[q]);
        ex[q] = mine + inc - v[q];
        mine += read_lane64(inc, 63);
      }
    }
    if (lane == 0) s_wave[turn][w] = mine;
    __syncthreads();
    const long long waves = wave_scan_dpp64(lane < 16 ? s_wave[turn][lane] : 0ll);
    const long long run = base + (w > 0 ? read_lane64(waves, w - 1) : 0ll);
#pragma unroll
    for (int q = 0; q < kScanOnePer; q++)
      if (r0 + q * 64 < n) off[r0 + q * 64] = run + ex[q];
    base += read_lane64(waves, 15);
  }
  if (threadIdx.x == 0) {
    off[n] = base;
    if (total_out) *total_out = base - off_add;
    if (report) report[kNumBins] = base - off_add;
  }
}

// One launch before a product's passes: its tile, the (single) product of every row block, all counters cleared.
template <typename T, typename RP>
__global__ __launch_bounds__(256) void k_prepare_one(TileDev<T, RP> tile, RowsDev<T, RP> R, int64_t nblocks) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, step = (int64_t)gridDim.x * 256;
  if (i == 0) *const_cast<TileDev<T, RP>*>(R.tiles) = tile;
  for (int64_t b = i; b < nblocks; b += step) const_cast<uint16_t*>(R.blk_tile)[b] = 0;
  for (int64_t b = i; b < kNumBins * kCountStride; b += step) R.bin_count[b] = 0;
  if (i < 3) R.ovf_count[i] = 0;  // overflow, predicted and long rows
  if (i < 8) R.stats[i] = 0;
}

// The bin counts and the last scan's total, written to pinned host memory (kNumBins + 1 values): the host waits for the
// stream and reads them, with no copy in between.
template <typename T, typename RP>
__global__ void k_report(RowsDev<T, RP> R, const int64_t* total, int64_t* out) {
  if (threadIdx.x < kNumBins) out[threadIdx.x] = *R.count_of(threadIdx.x);
  if (threadIdx.x == kNumBins) out[kNumBins] = *total;
}

// One launch before the numeric pass: C's row_ptr (m < 0: not yet), and the arrays its entries go to.
template <typename OUT, typename T, typename RP>
__global__ void k_begin_numeric(RowsDev<T, RP> R, int64_t m, OUT* rp, int* c_col, T* c_val) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i <= m) rp[i] = (OUT)(R.off[i] - R.off[0]);
  if (i == 0) {
    TileDev<T, RP>* t = const_cast<TileDev<T, RP>*>(R.tiles);
    t->c_col = c_col;
    t->c_val = c_val;
  }
}

// Per-product row_ptr from flat offsets: rp[i] = off[flat0 + i] - off[flat0] (int32 or int64 out).
template <typename OUT>
__global__ void k_rowptr(const int64_t* off, int64_t flat0, int64_t m, OUT* rp) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i <= m) rp[i] = (OUT)(off[flat0 + i] - off[flat0]);
}

}  // namespace bclx
