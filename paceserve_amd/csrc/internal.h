// Shared declarations between the translation units of libpace_kv.so.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "pace_kv.h"

// Returns from the enclosing function with the status of `expr` if non-zero.
#define PACE_KV_TRY(expr)  \
  do {                     \
    int rc_ = (expr);      \
    if (rc_) return rc_;   \
  } while (0)

namespace pace_kv {

// Records `msg` (printf-style) as the calling thread's last error and returns
// `code`, so call sites read `return fail(PACE_KV_EINVAL, "...")`.
int fail(int code, const char* fmt, ...);

// Converts a HIP error into the ABI's status convention (positive hipError_t)
// and records its message; returns 0 for hipSuccess.
int hip_status(hipError_t err, const char* what);

// Division by a divisor known on the host, by the multiply-and-shift form
// (Granlund and Montgomery, "Division by invariant integers using
// multiplication", figure 4.1), exact for every 32-bit n and divisor >= 1.
struct FastDiv {
  uint32_t mul, shift1, shift2;
};

inline FastDiv fast_div(uint32_t divisor) {
  uint32_t log2_up = 0;
  while ((uint64_t(1) << log2_up) < divisor) ++log2_up;
  return FastDiv{static_cast<uint32_t>((((uint64_t(1) << log2_up) - divisor) << 32) / divisor + 1),
                 log2_up > 0 ? 1u : 0u, log2_up > 0 ? log2_up - 1 : 0u};
}

#ifdef __HIP__
__device__ __forceinline__ uint32_t over(const FastDiv& d, uint32_t n) {
  const uint32_t q = __umulhi(d.mul, n);
  return (q + ((n - q) >> d.shift1)) >> d.shift2;
}
#endif

// One side of a page copy: per-layer base pointers plus optional page ids, in
// a device array or (n_pages <= PACE_KV_INLINE_IDS) in a host array whose ids
// travel in the kernel arguments.  Without either, page j of layer l is at
// base[l] + j*page_bytes, which is how the contiguous transfer buffer is
// addressed.
struct Side {
  const char* const* layers;  // host array, num_layers entries
  const int32_t* ids;         // device array of n_pages ids, or nullptr
  int64_t pool_pages;         // ids must lie in [0, pool_pages)
  const int32_t* host_ids = nullptr;
};

// The page ids of one side of a call: a device array, or a host array of at
// most PACE_KV_INLINE_IDS entries that travel in the kernel arguments.
struct IdList {
  const int32_t* dev;
  const int32_t* host;
  bool null() const { return dev == nullptr && host == nullptr; }
};

// Store flavour of a copy: both write through the L2 at device scope; kStream
// also marks the stores nontemporal, while kPack (a pack into a transfer
// buffer that an unpack reads next) leaves them cacheable, so that the unpack
// finds them in the memory-side cache.  kLink is kStream across the host link
// (ids on both sides, in device memory), where short pages go one to a wave.
enum class StorePolicy { kStream, kPack, kLink };

// A second destination of a copy with ids on both sides: page j of layer l
// also goes to base + l * layer_stride + j * page_bytes.
struct Tee {
  char* base;
  int64_t layer_stride;
};

// Validates arguments and enqueues the copy dst[l][dst_id(j)] = src[l][src_id(j)]
// for l < num_layers, j < n_pages on `stream`, in launches of at most
// PACE_KV_MAX_LAYERS_PER_LAUNCH layers.  With a tee the pools and its buffer
// must not share memory.
int launch_page_copy(const Side& src, const Side& dst, int num_layers,
                     int64_t n_pages, int64_t page_bytes, int32_t* err_count,
                     hipStream_t stream, StorePolicy policy = StorePolicy::kStream, const Tee* tee = nullptr);

// src -> buffer -> dst in chunks of buffer_layers layers: the bytes of a pack
// into `buffer` and an unpack out of it, which stays filled.  One launch per
// chunk reads each page once and writes it to both, unless source, buffer and
// destination share memory.  Ids as in launch_page_copy; the caller has
// checked page_bytes, buffer_layers >= 1 and the buffer's stride.
int buffered_copy(const Side& src, const Side& dst, char* buffer, int64_t buffer_layer_stride, int buffer_layers,
                  int num_layers, int64_t n_pages, int64_t page_bytes, int32_t* err_count, hipStream_t stream);

// launch_page_copy between device pages (`pool`, with ids) and pinned memory
// that the device addresses (`host`: a pool with device ids, or, without ids,
// [num_layers][n_pages][page_bytes] in one piece), out to the host (to_host) or in
// from it, with few waves.  `done`, if given, is recorded behind a copy whose
// every launch succeeded.
int launch_host_leg(const Side& pool, const Side& host, bool to_host, int num_layers, int64_t n_pages,
                    int64_t page_bytes, int32_t* err_count, hipStream_t stream, hipEvent_t done = nullptr);

// The same with the host side laid out [num_layers][n_pages][page_bytes].
int launch_host_leg(const Side& pool, char* host, bool to_host, int num_layers, int64_t n_pages, int64_t page_bytes,
                    int32_t* err_count, hipStream_t stream, hipEvent_t done = nullptr);

// pace_kv_pack and pace_kv_unpack for ids of either kind.
int pack(const void* const* src_layers, int num_layers, int64_t pool_pages, const IdList& ids, int64_t n_pages,
         int64_t page_bytes, void* out, int64_t out_layer_stride, int32_t* err_count, hipStream_t stream);
int unpack(const void* buf, int64_t buf_layer_stride, void* const* dst_layers, int num_layers, int64_t pool_pages,
           const IdList& ids, int64_t n_pages, int64_t page_bytes, int32_t* err_count, hipStream_t stream);

// Builds the layer table of a contiguous buffer [num_layers][layer_stride].
void buffer_layers(const void* base, int64_t layer_stride, int num_layers,
                      const char** out);

}  // namespace pace_kv
