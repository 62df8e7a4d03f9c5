// Internal runtime of the bclx library: handle, error reporting, device buffers.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <string>
#include <vector>

#include "../../include/bclx.h"

namespace bclx {

void set_error(const std::string& msg);

struct Error {
  bclx_status status;
  std::string msg;
};

#define BCLX_HIP(call)                                                                                    \
  do {                                                                                                     \
    hipError_t e_ = (call);                                                                                \
    if (e_ != hipSuccess) {                                                                                \
      throw ::bclx::Error{e_ == hipErrorOutOfMemory ? BCLX_ERR_ALLOC : BCLX_ERR_HIP,                      \
                          std::string(#call) + ": " + hipGetErrorString(e_) + " at " + __FILE__ + ":" +   \
                              std::to_string(__LINE__)};                                                   \
    }                                                                                                      \
  } while (0)

#define BCLX_REQUIRE(cond, status, msg)                       \
  do {                                                        \
    if (!(cond)) throw ::bclx::Error{(status), (msg)};        \
  } while (0)

// The device allocator of the calling thread's current handle (bclx_set_allocator; hipMalloc / hipFree when unset).
// Every entry point selects its handle's allocator through set_device() before it allocates.
struct AllocFns {
  bclx_alloc_fn alloc = nullptr;
  bclx_free_fn free = nullptr;
  void* user = nullptr;
};
extern thread_local AllocFns g_alloc;

// Device memory from the current allocator; freed with the allocator it came from.
void* dev_alloc(size_t bytes, const AllocFns& how);
void dev_free(void* p, const AllocFns& how);

// Device buffer owned by the library. Move-only; remembers the allocator that made it.
struct DevBuf {
  void* p = nullptr;
  size_t bytes = 0;
  AllocFns how;
  DevBuf() = default;
  explicit DevBuf(size_t n) { alloc(n); }
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  DevBuf(DevBuf&& o) noexcept : p(o.p), bytes(o.bytes), how(o.how) { o.p = nullptr; o.bytes = 0; }
  DevBuf& operator=(DevBuf&& o) noexcept {
    if (this != &o) { release(); p = o.p; bytes = o.bytes; how = o.how; o.p = nullptr; o.bytes = 0; }
    return *this;
  }
  ~DevBuf() { release(); }
  void alloc(size_t n) {
    release();
    if (n == 0) n = 256;
    how = g_alloc;
    p = dev_alloc(n, how);
    bytes = n;
  }
  // grow-only
  void reserve(size_t n) { if (n > bytes) alloc(n); }
  void release() {
    if (p) dev_free(p, how);
    p = nullptr;
    bytes = 0;
  }
  template <typename T> T* as() const { return static_cast<T*>(p); }
};

// Bump allocator over one device buffer: sub-buffers are 256-byte aligned. The buffer is the arena's own (allocated
// at commit), or caller memory given to use_external (nothing is allocated; commit fails when it is too small).
struct Arena {
  DevBuf buf;
  char* ext = nullptr;
  size_t ext_bytes = 0;
  size_t used = 0;
  size_t reserve(size_t bytes) {
    size_t off = (used + 255) & ~size_t(255);
    used = off + bytes;
    return off;
  }
  void use_external(void* p, size_t bytes) {
    ext = static_cast<char*>(p);
    ext_bytes = bytes;
  }
  void commit() {
    if (ext) {
      BCLX_REQUIRE(used <= ext_bytes, BCLX_ERR_OVERFLOW,
                   "workspace of " + std::to_string(used) + " bytes exceeds the " + std::to_string(ext_bytes) +
                       "-byte scratch");
    } else {
      buf.reserve(used);
    }
  }
  template <typename T> T* at(size_t off) const {
    return reinterpret_cast<T*>((ext ? ext : static_cast<char*>(buf.p)) + off);
  }
};

}  // namespace bclx

struct bclx_handle {
  int device = 0;
  bclx::AllocFns alloc;  // device allocator of this handle (bclx_set_allocator)
  hipStream_t stream = nullptr;
  int num_cus = 256;
  size_t lds_per_block = 65536;
  // operands and partial sums of dense products (grow-only; dense_scratch()). A product may still run when its call
  // returns: scratch_stream is where the last one was launched, and where the handle is on another stream by now,
  // scratch_left was recorded there when it moved on.
  bclx::DevBuf scratch;
  bool scratch_used = false;
  hipStream_t scratch_stream = nullptr;
  hipEvent_t scratch_left = nullptr;
  bclx::DevBuf call_ws;  // CallWorkspace; hipMalloc'd handles only
  bclx::DevBuf dense_slots;  // heavy-row dense accumulators, kept zeroed between uses
  size_t dense_slot_doubles = 0;
  int dense_nslots = 0;
  int64_t* h_pinned = nullptr;  // kPinnedCounts values in pinned host memory, written by k_report
  // workspace of the last spgemm plan, kept for the next one (at most kPlanKeep bytes; hipMalloc'd handles only)
  bclx::DevBuf plan_ws;
  bool plan_ws_busy = false;
  unsigned stream_changes = 0;  // bclx_set_stream calls that changed the stream
  ~bclx_handle() {
    if (h_pinned) (void)hipHostFree(h_pinned);
    if (scratch_left) (void)hipEventDestroy(scratch_left);
  }
};

namespace bclx {

constexpr size_t kPlanKeep = size_t(4) << 30;
constexpr int kPinnedCounts = 64;

// Wraps a C-ABI body: converts exceptions to status codes and records the message.
template <typename F>
bclx_status guarded(F&& f) {
  try {
    f();
    return BCLX_OK;
  } catch (const Error& e) {
    set_error(e.msg);
    return e.status;
  } catch (const std::bad_alloc&) {
    set_error("host allocation failed");
    return BCLX_ERR_ALLOC;
  } catch (const std::exception& e) {
    set_error(e.what());
    return BCLX_ERR_INVALID;
  }
}

inline void set_device(bclx_handle* h) {
  BCLX_HIP(hipSetDevice(h->device));
  g_alloc = h->alloc;
}

// Do two arrays (n bytes each; none where n is 0) have memory in common?
inline bool share_memory(const void* a, size_t na, const void* b, size_t nb) {
  const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
  return na > 0 && nb > 0 && x < y + nb && y < x + na;
}

inline unsigned div_up(int64_t a, int64_t b) { return (unsigned)((a + b - 1) / b); }

// Device memory of a call that waits for its stream before it returns, so nothing of the call still uses it then, on any
// stream. Kept by the handle for the next such call, up to kCallKeep bytes; a handle with a caller's allocator keeps
// nothing.
constexpr size_t kCallKeep = size_t(1) << 30;
struct CallWorkspace {
  bclx_handle* h;
  DevBuf own;
  CallWorkspace(bclx_handle* h_, Arena& ws) : h(h_) {
    DevBuf& b = h->alloc.alloc ? own : h->call_ws;
    b.reserve(ws.used);
    ws.use_external(b.p, b.bytes);
  }
  ~CallWorkspace() {
    if (!own.p && h->call_ws.bytes <= kCallKeep) return;
    (void)hipStreamSynchronize(h->stream);
    if (!own.p) h->call_ws.release();
  }
  CallWorkspace(const CallWorkspace&) = delete;
  CallWorkspace& operator=(const CallWorkspace&) = delete;
};

// The handle's scratch for a dense product on its stream: what an earlier product left running on another stream
// (bclx_set_stream in between) comes first.
char* dense_scratch(bclx_handle* h, size_t bytes);
// Waits for the dense products that still use the scratch.
void finish_dense(bclx_handle* h);
// The handle is about to leave its stream.
void leave_dense(bclx_handle* h);

// Looks up, once per device and with that device current, the address of the fixed scratch array that
// bclx_spgemm_noalloc works in.
void init_noalloc_scratch(int device);

// Zeroed heavy-row accumulators: nslots x ndoubles, grown on demand, zeroed once when (re)allocated.
void ensure_dense_slots(bclx_handle* h, int nslots, size_t ndoubles);

}  // namespace bclx
