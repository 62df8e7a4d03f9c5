// Handle lifecycle, error reporting and version of the bclx C ABI.
#include <memory>

#include "internal.hpp"

namespace bclx {
static thread_local std::string g_last_error;
void set_error(const std::string& msg) { g_last_error = msg; }

thread_local AllocFns g_alloc;

void* dev_alloc(size_t bytes, const AllocFns& how) {
  void* p = nullptr;
  if (how.alloc) {
    p = how.alloc(bytes, how.user);
    BCLX_REQUIRE(p != nullptr, BCLX_ERR_ALLOC,
                 "the handle's allocator returned NULL for " + std::to_string(bytes) + " bytes");
  } else {
    BCLX_HIP(hipMalloc(&p, bytes));
  }
  return p;
}

void dev_free(void* p, const AllocFns& how) {
  if (how.free) how.free(p, how.user);
  else (void)hipFree(p);
}

// hipSuccess: the stream is not being captured. hipErrorStreamCaptureImplicit: it is, or is the null stream beside one
// that is: it may not be waited for, nor events recorded on it. Others: not a stream any more.
static hipError_t stream_state(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  const hipError_t e = hipStreamIsCapturing(s, &st);
  if (e != hipSuccess) (void)hipGetLastError();
  return e == hipSuccess && st != hipStreamCaptureStatusNone ? hipErrorStreamCaptureImplicit : e;
}

void finish_dense(bclx_handle* h) {
  if (!h->scratch_used) return;
  if (h->scratch_stream == h->stream) (void)hipStreamSynchronize(h->stream);
  else (void)hipEventSynchronize(h->scratch_left);
}

void leave_dense(bclx_handle* h) {
  if (!h->scratch_used || h->scratch_stream != h->stream) return;
  const hipError_t e = stream_state(h->stream);
  if (e == hipSuccess && hipEventRecord(h->scratch_left, h->stream) == hipSuccess) return;
  if (e != hipErrorStreamCaptureImplicit) {  // destroyed before it was left
    (void)hipGetLastError();
    (void)hipSetDevice(h->device);
    (void)hipDeviceSynchronize();
  }
  h->scratch_used = false;
}

// Under capture nothing runs yet, so nothing is waited for: ordering a graph's launches is the caller's.
char* dense_scratch(bclx_handle* h, size_t bytes) {
  const bool runs = stream_state(h->stream) == hipSuccess;
  if (runs && h->scratch_used) {
    if (bytes > h->scratch.bytes) finish_dense(h);
    else if (h->scratch_stream != h->stream) BCLX_HIP(hipStreamWaitEvent(h->stream, h->scratch_left, 0));
  }
  h->scratch.reserve(bytes);
  if (runs) {
    h->scratch_used = true;
    h->scratch_stream = h->stream;
  }
  return h->scratch.as<char>();
}
}  // namespace bclx

using namespace bclx;

extern "C" {

const char* bclx_last_error(void) { return g_last_error.c_str(); }

const char* bclx_version(void) { return "bclx 0.1 (gfx950)"; }

bclx_status bclx_create(int device, void* stream, bclx_handle** out) {
  return guarded([&] {
    BCLX_REQUIRE(out != nullptr, BCLX_ERR_INVALID, "out is null");
    int ndev = 0;
    BCLX_HIP(hipGetDeviceCount(&ndev));
    BCLX_REQUIRE(device >= 0 && device < ndev, BCLX_ERR_INVALID,
                 "device " + std::to_string(device) + " not present (" + std::to_string(ndev) + " devices)");
    BCLX_HIP(hipSetDevice(device));
    std::unique_ptr<bclx_handle> h(new bclx_handle());
    h->device = device;
    h->stream = static_cast<hipStream_t>(stream);
    int cus = 0, lds = 0;
    BCLX_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
    BCLX_HIP(hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, device));
    h->num_cus = cus > 0 ? cus : 256;
    h->lds_per_block = lds > 0 ? (size_t)lds : 65536;
    init_noalloc_scratch(device);
    BCLX_HIP(hipHostMalloc(reinterpret_cast<void**>(&h->h_pinned), sizeof(int64_t) * kPinnedCounts, hipHostMallocDefault));
    BCLX_HIP(hipEventCreateWithFlags(&h->scratch_left, hipEventDisableTiming));
    *out = h.release();
  });
}

bclx_status bclx_destroy(bclx_handle* h) {
  return guarded([&] {
    if (!h) return;
    (void)hipSetDevice(h->device);
    (void)hipStreamSynchronize(h->stream);
    finish_dense(h);
    delete h;
  });
}

bclx_status bclx_set_allocator(bclx_handle* h, bclx_alloc_fn alloc, bclx_free_fn free_fn, void* user) {
  return guarded([&] {
    BCLX_REQUIRE(h != nullptr, BCLX_ERR_INVALID, "null handle");
    BCLX_REQUIRE((alloc == nullptr) == (free_fn == nullptr), BCLX_ERR_INVALID,
                 "give both allocator functions, or neither (hipMalloc / hipFree)");
    // what the handle keeps for later calls, and no call or plan uses now, goes back to the allocator it came from
    BCLX_HIP(hipSetDevice(h->device));
    h->call_ws.release();
    if (!h->plan_ws_busy) h->plan_ws.release();
    h->alloc = AllocFns{alloc, free_fn, user};
  });
}

bclx_status bclx_set_stream(bclx_handle* h, void* stream) {
  return guarded([&] {
    BCLX_REQUIRE(h != nullptr, BCLX_ERR_INVALID, "null handle");
    if (h->stream == static_cast<hipStream_t>(stream)) return;
    leave_dense(h);
    h->stream_changes++;
    h->stream = static_cast<hipStream_t>(stream);
  });
}

bclx_status bclx_synchronize(bclx_handle* h) {
  return guarded([&] {
    BCLX_REQUIRE(h != nullptr, BCLX_ERR_INVALID, "null handle");
    set_device(h);
    BCLX_HIP(hipStreamSynchronize(h->stream));
  });
}

}  // extern "C"
