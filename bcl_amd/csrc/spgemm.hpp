// SpGEMM host-side building blocks shared by the two-phase path and the batched stage pipeline.
#pragma once

#include <memory>
#include <vector>

#include "internal.hpp"
#include "spgemm_kernels.hpp"

namespace bclx {

void fill_i32(hipStream_t s, int32_t* p, int64_t n, int32_t v);
void fill_u64(hipStream_t s, unsigned long long* p, int64_t n, unsigned long long v);
int rows_per_block(int bin);
// off[0..n] = exclusive scan of cnt[0..n) (off[n] = total, also written to *total when non-null);
// partial needs scan_partials(n) entries.
int64_t scan_partials(int64_t n);
void scan_counts(hipStream_t s, const int32_t* cnt, int64_t n, int64_t* off, long long* partial, int64_t* total);
void check_pair(const bclx_csr* A, const bclx_csr* B);

template <typename T, typename RP>
TileDev<T, RP> make_tile(const bclx_csr* A, const bclx_csr* B);

// Device workspace over the flat-row space of one batch of products.
template <typename T, typename RP>
struct FlatRows {
  bclx_handle* h = nullptr;
  std::vector<TileDev<T, RP>> tiles;
  int ntiles = 0;
  int64_t nflat = 0, nblocks = 0, max_n = 1;
  Arena arena;
  RowsDev<T, RP> R{};
  long long* scan_partial = nullptr;
  int64_t* scan_total = nullptr;
  DevBuf gbits;  // per-workgroup column bitmaps of the wide-tile heavy kernel (kept zeroed between rows)

  void setup(bclx_handle* h, const std::vector<TileDev<T, RP>>& tiles, bool with_cap);
  // the same for one product, without any GPU work: prepare_one() writes its tables. pooled: the workspace may be the
  // handle's (then it is given back by the owner)
  bool setup_one(bclx_handle* h, const TileDev<T, RP>& tile, bool pooled);
  void prepare_one(hipStream_t s);
  void upload_tiles();
  void reset_counters(hipStream_t s);
  // pred_min >= 0 (learned path): also write cap = min(prod, n) and list the rows with more than pred_min products
  // with_stats: also count products (stats[0]) and rows bound for the heavy bin (stats[5])
  // cleared: the counters (the long-row count among them) are zero already
  void analyze(hipStream_t s, bool do_bin, long long pred_min = -1, bool with_stats = true, bool cleared = false);
  void bin(hipStream_t s, int src);
  // exclusive scan of cnt over all flat rows into off (nflat + 1 entries), plus off_add; total -> *scan_total
  // with_report: a one-launch scan also writes what report() waits for
  void scan(hipStream_t s, const int32_t* cnt, int64_t* off, int64_t off_add, bool with_report = false);
  // planned: plan_heavy() ran before (the heavy bin)
  void run_bin(hipStream_t s, int mode, int b, int64_t count_hint, bool planned = false);
  // The heavy bin's small kernels (order, split and, in modes 2 and 3, counting and placing the parts). Callers that run
  // bins side by side launch them first: behind the other bins' workgroups, which fill the GPU, splitting the rows of
  // a stage of 4 x 4 tiles at scale 21 took 1290 us instead of 25.
  void plan_heavy(hipStream_t s, int mode);
  // max_out >= dst_off[nflat]; chunk_row holds div_up(max_out, kCompactChunk) entries
  void compact(hipStream_t s, const int64_t* dst_off, int* dst_col, T* dst_val, const int* src_col, const T* src_val,
               int64_t max_out, int32_t* chunk_row);
  // heavy rows: allocate the zeroed accumulators of the heavy kernel (before any graph capture)
  void prepare_heavy();
  bool heavy_lds_bitmap() const;  // wide-tile heavy kernel: bitmap in LDS (else per-workgroup global bitmaps)
  int64_t read_stat(int q);
  void read_counts(hipStream_t s, int32_t* dst);  // kNumBins bin counts (synchronises s)
  int64_t report(hipStream_t s, int32_t* counts);  // the bin counts and the last scan's total (synchronises s)

 private:
  bool reported = false;  // the last scan wrote the report
  void layout(bool with_cap, bool pooled, bool* from_pool);
};

// The two-phase product C = A * B of one tile pair (symbolic, then numeric into caller-allocated C).
template <typename T, typename RP>
struct TwoPhase {
  bclx_handle* h;
  FlatRows<T, RP> F;
  int64_t nnz_c = -1;
  int64_t m = 0;
  // bins of the symbolic pass; when no row hashed, the numeric pass reuses them (sorted rows are binned by their
  // products alone)
  int32_t sym_counts[kNumBins] = {0};
  bool reuse_bins = false;
  bool from_pool = false;        // the workspace is the handle's
  unsigned stream_changes = 0;   // of the handle, when the workspace was taken
  // scratch / scratch_bytes: device memory the workspace is laid out in instead of being allocated. pooled: the handle's
  // workspace may be taken (by one product at a time)
  TwoPhase(bclx_handle* h_, const TileDev<T, RP>& tile, const BinTuning& tn, void* scratch = nullptr,
           size_t scratch_bytes = 0, bool pooled = false)
      : h(h_) {
    if (scratch) F.arena.use_external(scratch, scratch_bytes);
    from_pool = F.setup_one(h, tile, pooled);
    stream_changes = h->stream_changes;
    F.R.tn = tn;
    m = tile.m;
  }
  // The handle's workspace goes back once nothing uses it: the work of this product is on the handle's stream, or on an
  // earlier one where bclx_set_stream was called in between.
  ~TwoPhase() {
    if (!from_pool) return;
    if (stream_changes == h->stream_changes) (void)hipStreamSynchronize(h->stream);
    else (void)hipDeviceSynchronize();
    h->plan_ws_busy = false;
  }
  TwoPhase(const TwoPhase&) = delete;
  TwoPhase& operator=(const TwoPhase&) = delete;
  int64_t symbolic();
  // A's and B's arrays, where the caller's row_ptr may be one of them
  struct Range {
    const void* p = nullptr;
    size_t bytes = 0;
  } inputs[6];
  void reads(const bclx_csr* A, const bclx_csr* B) {
    int q = 0;
    for (const bclx_csr* x : {A, B}) {
      inputs[q++] = {x->row_ptr, (size_t)(x->m + 1) * sizeof(RP)};
      inputs[q++] = {x->col_idx, (size_t)x->nnz * sizeof(int)};
      inputs[q++] = {x->vals, (size_t)x->nnz * sizeof(T)};
    }
  }
  // writes col/val into c_col/c_val (capacity c_cap entries) and row_ptr (m+1 entries of 4 or 8 bytes)
  void numeric(int* c_col, T* c_val, int64_t c_cap, void* row_ptr, int ptr_width);
};


}  // namespace bclx
