// Paged KV append (the producer of page contents): writes newly computed K/V
// rows of appended tokens into their page slots, in the layout the migration
// path moves.  Equivalent to the three FlashInfer calls the reference makes per
// layer (paceserve/model_executor/attention/flashinfer_attention_wrapper.py:
// 241-255): get_seq_lens, get_batch_indices_positions, append_paged_kv_cache.
//
//   seq_len[b]   = max(kv_indptr[b+1] - kv_indptr[b] - 1, 0) * P + kv_last_page_len[b]
//                  (computed by the caller: get_seq_lens)
//   token i of request b (append_indptr[b] <= i < append_indptr[b+1]) sits at
//   pos = seq_len[b] - (append_indptr[b+1] - append_indptr[b]) + (i - append_indptr[b])
//   cache[kv_indices[kv_indptr[b] + pos / P]][0 (K) | 1 (V)][pos % P] = key[i] | value[i]
//
// pace_kv_append takes b and pos per token (get_batch_indices_positions);
// pace_kv_append_indptr derives them in the same launch from append_indptr,
// kv_indptr and kv_last_page_len, so a layer's append is one launch.
//
// One wave64 workgroup carries 1 KiB of the key rows and the same 1 KiB of the
// value rows, one 16-byte vector of each per lane, stored with the page copy's
// device-scope write-through store.  A token's two rows go to the same slot of
// the two halves of a page, so they share one chain of index loads.  Rows of
// whole KiB give a wave one token, whose indices are scalar; other rows are
// taken end to end, vector after vector, so that every lane carries one and a
// wave holds several tokens (or the end of one and the start of the next).
//
// Bound by HBM from some 16 MiB up, and below by the launch and by the chain
// of two to four dependent index loads.  Measured on MI355X per launch in a
// graph of 32 on the same buffers (up to 64 MiB partly from the memory-side
// cache), fused form and the other, against one wave per K or V row (or 16 KiB):
//   256-byte rows, 16384 tokens               3.9, 3.4 us, before 10.7, 8.9
//   256-byte rows, 32768 tokens               5.3, 4.7 us, before 19.4, 16.0
//   384-byte rows, 8500 tokens                3.8, 3.3 us, before 6.7, 5.7
//   2 KiB rows, 8500 tokens                   10.9, 11.3 us, before 12.7, 11.5
//   2 KiB rows, 256 tokens of a decode step   1.96, 2.28 us, before 2.41, 2.34
//   8 KiB rows, 8190 tokens                   39.6, 39.3 us, before 40.5, 40.2
// Launches of up to 300 tokens with rows of less than a KiB, 2.1 to 2.3 us, are
// up to 0.06 us slower than that.
// Waves that end with a row (idle lanes, scalar indices) never measured
// faster than rows end to end, not in decode either, and up to 40% slower at
// 16384 tokens.  Every index is checked: a token whose request, page slot or
// page id is out of range is skipped and counted.
#include "internal.h"

namespace pace_kv {
namespace {

constexpr int kThreads = 64;
constexpr int kVecBytes = 16;
// Workgroups per launch: grid * 64 threads stays within the 32-bit limit; a
// longer batch uses more launches.
constexpr int64_t kMaxGroupsPerLaunch = int64_t(1) << 25;

// Appends of at most this many key bytes load their rows with plain loads,
// larger ones nontemporally.  Measured on MI355X, 2 KiB rows: 512 KiB of keys
// 2.4 us plain, 2.6 nontemporal; 1 MiB the same either way; 2 MiB 3.8 against
// 4.05 and 32 MiB 24.0 against 23.1.
constexpr int64_t kCachedLoadBytes = int64_t(1) << 20;
// Blocks of 64 append_indptr entries that one round of the search loads.
constexpr int kSearchBlocks = 4;
// Most entries that a wave of several requests hands round one by one.
constexpr uint32_t kHandRound = 8;

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

struct AppendParams {
  const char* key;
  const char* value;
  int64_t token_stride;      // bytes between tokens in key / value
  const int32_t* batch_indices;  // precomputed token -> request (or nullptr: derive from append_indptr)
  const int32_t* positions;
  const int32_t* append_indptr;  // batch_size + 1 entries (the fused form)
  const int32_t* kv_last_page_len;  // batch_size entries (the fused form)
  const int32_t* kv_indices;
  const int32_t* kv_indptr;  // batch_size + 1 entries
  int64_t num_indices;       // entries of kv_indices
  char* cache;               // [num_pages, 2, P, H, D]
  int32_t* err;
  int64_t row_bytes;         // H * D * elem: one token's K (or V) row
  uint32_t batch_size;
  uint32_t num_pages;
  uint32_t page_size;
  int32_t page_log2;         // log2(page_size), or -1 when it is no power of two
  uint32_t row_vecs;         // row_bytes / 16
  uint32_t row_div;          // waves (rows of whole KiB) or lanes per row
  FastDiv by_row;            // division by row_div
  uint32_t first_token;      // of this launch
  uint32_t total_items;      // lanes of this launch: its tokens * row_vecs
  uint32_t guess_own_request;  // fused form, nnz <= batch_size: try request i for token i first
};

// A store of more than 64 bits reads its data registers after it issues; the
// asm carries the wait states the compiler cannot add for it (s_nop 1).
__device__ __forceinline__ void store_row_vec(u32x4* d, const u32x4 v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" : : "v"(d), "v"(v) : "memory");
}

// The search for a token's request in the fused form, the largest
// b < batch_size with append_indptr[b] <= token: the whole wave searches at
// once, each lane loading one entry of each block of 64 (four blocks per round,
// loaded before any is tested, so up to 256 requests cost one load latency),
// and the entries that pass are counted.
__device__ __forceinline__ void search_load(const AppendParams& p, uint32_t base, int32_t* x) {
#pragma unroll
  for (int k = 0; k < kSearchBlocks; ++k) {
    x[k] = INT32_MAX;
    if (k > 0 && base + k * kThreads >= p.batch_size) continue;
    const uint32_t e = base + k * kThreads + threadIdx.x;
    if (e < p.batch_size) x[k] = p.append_indptr[e];
  }
}

// How many of the entries x, summed over the wave, are at most t.
__device__ __forceinline__ uint32_t search_count(const int32_t* x, int32_t t) {
  uint32_t n = 0;
#pragma unroll
  for (int k = 0; k < kSearchBlocks; ++k) n += __popcll(__ballot(x[k] <= t));
  return n;
}

// What the first round of index loads gives: the guessed request's offsets in
// the fused form, the token's request and position in the other.
struct FirstRound {
  int32_t a0, a1, k0, k1, len;
  int32_t b, pos;
  bool guessed;
  int32_t x[kSearchBlocks];  // the search's first round, where there is no guess
};

__device__ __forceinline__ void request_offsets(const AppendParams& p, uint32_t b, FirstRound* f) {
  f->a0 = p.append_indptr[b];
  f->a1 = p.append_indptr[b + 1];
  f->k0 = p.kv_indptr[b];
  f->k1 = p.kv_indptr[b + 1];
  f->len = p.kv_last_page_len[b];
}

template <bool FUSED, bool UNIFORM>
__device__ __forceinline__ FirstRound first_round(const AppendParams& p, uint32_t i) {
  FirstRound f = {};
  if (!FUSED) {
    f.b = p.batch_indices[i];
    f.pos = p.positions[i];
  } else if (p.guess_own_request) {  // i < nnz <= batch_size
    // A decode batch (no more tokens than requests) usually appends one
    // token per request: guess that token i is request i's and load every
    // index that places it in one round.
    f.guessed = true;
    request_offsets(p, i, &f);
  } else if (UNIFORM) {
    search_load(p, 0, f.x);
  }
  return f;
}

// Page and slot of the lane's token, or false when any index is out of range.
template <bool FUSED, bool UNIFORM>
__device__ __forceinline__ bool locate(const AppendParams& p, FirstRound f, uint32_t first_i, uint32_t last_i,
                                       uint32_t i, uint32_t* page, uint32_t* slot) {
  int32_t pos;
  int64_t first, last;
  if (FUSED) {
    const int32_t t = static_cast<int32_t>(i);
    // The guess holds exactly when append_indptr[i] <= i < append_indptr[i+1],
    // which is when the search finds request i.
    const bool found = f.guessed && f.a0 <= t && t < f.a1;
    if (UNIFORM ? !found : __ballot(!found) != 0) {
      const int32_t t0 = static_cast<int32_t>(first_i), t1 = static_cast<int32_t>(last_i);
      if (!UNIFORM || f.guessed) search_load(p, 0, f.x);
      uint32_t lo = search_count(f.x, t0), hi = UNIFORM ? 0 : search_count(f.x, t1);
      for (uint32_t base = kSearchBlocks * kThreads; base < p.batch_size; base += kSearchBlocks * kThreads) {
        search_load(p, base, f.x);
        lo += search_count(f.x, t0);
        if (!UNIFORM) hi += search_count(f.x, t1);
      }
      if (UNIFORM) hi = lo;
      // A wave of several requests: the entries between its first and its last
      // token's.  A few that the wave still holds are handed round, which spares
      // a small launch a round of loads (MI355X, 256 tokens of 16 requests, rows
      // of 160 B 2.56 -> 2.25 us; 1000 of 200, rows of 384 B 2.70 -> 2.40; the
      // same to 2% from 4096 tokens on); else they are loaded once more and
      // counted for each token.  (Counting all that are held for each token
      // measured the same or 1% slower than that.)
      uint32_t count = lo;
      const bool held = hi - lo <= kHandRound && p.batch_size <= kSearchBlocks * kThreads;
      for (uint32_t e = lo; held && e < hi; ++e) {
        const uint32_t block = e / kThreads;
        const int32_t x = block == 0 ? f.x[0] : block == 1 ? f.x[1] : block == 2 ? f.x[2] : f.x[3];
        if (__builtin_amdgcn_readlane(x, e % kThreads) <= t) ++count;
      }
      for (uint32_t base = lo; !held && base < hi; base += kThreads) {
        const uint32_t e = base + threadIdx.x;
        const int32_t x = e < hi ? p.append_indptr[e] : INT32_MAX;
        for (int32_t k = t0 + 1; k <= t1; ++k) {
          const uint32_t n = __popcll(__ballot(x <= k));
          if (t == k) count += n;
        }
      }
      if (!found) {
        if (count == 0) return false;
        // Request count - 1 < batch_size: its offsets are loaded in one round,
        // before the range check; by scalar loads where the wave has one
        // request.
        if (lo == hi) request_offsets(p, __builtin_amdgcn_readfirstlane(lo) - 1, &f);
        else request_offsets(p, count - 1, &f);
        if (t >= f.a1) return false;
      }
    }
    const int32_t pages = f.k1 - f.k0;
    const int32_t seq_len = (pages > 1 ? pages - 1 : 0) * static_cast<int32_t>(p.page_size) + f.len;
    pos = seq_len - (f.a1 - f.a0) + (t - f.a0);
    first = f.k0;
    last = f.k1;
  } else {
    pos = f.pos;
    if (f.b < 0 || static_cast<uint32_t>(f.b) >= p.batch_size) return false;
    first = p.kv_indptr[f.b];
    last = p.kv_indptr[f.b + 1];
  }
  if (pos < 0) return false;
  const uint32_t upos = static_cast<uint32_t>(pos);
  const uint32_t nth = p.page_log2 >= 0 ? upos >> p.page_log2 : upos / p.page_size;
  const int64_t it = first + nth;
  if (first < 0 || it >= last || it >= p.num_indices) return false;
  *page = static_cast<uint32_t>(p.kv_indices[it]);
  if (*page >= p.num_pages) return false;
  *slot = upos - nth * p.page_size;
  return true;
}

template <bool NT>
__device__ __forceinline__ u32x4 load_vec(const u32x4* s) {
  return NT ? __builtin_nontemporal_load(s) : *s;
}

// UNIFORM: rows of whole KiB, so that a wave holds one token and its index
// loads are scalar.
template <bool FUSED, bool UNIFORM, bool NT>
__global__ __launch_bounds__(kThreads) void append_kernel(const AppendParams p) {
  uint32_t i, vec, first_i, last_i;
  bool live = true;
  if (UNIFORM) {
    const uint32_t t = over(p.by_row, blockIdx.x);
    vec = (blockIdx.x - t * p.row_div) * kThreads + threadIdx.x;
    i = first_i = last_i = p.first_token + t;
  } else {
    uint32_t g = blockIdx.x * kThreads + threadIdx.x;
    live = g < p.total_items;
    if (!live) g = p.total_items - 1;  // the lane stays for the wave's search
    const uint32_t t = over(p.by_row, g);
    vec = g - t * p.row_div;
    i = p.first_token + t;
    first_i = __builtin_amdgcn_readlane(i, 0);
    last_i = __builtin_amdgcn_readlane(i, kThreads - 1);
  }
  FirstRound f;
  if (!UNIFORM) {
    // Per-lane index loads share the row loads' counter, which counts in
    // order: the first round goes ahead of them.
    f = first_round<FUSED, false>(p, i);
    __builtin_amdgcn_sched_barrier(0);
  }
  // The rows' loads depend on the token alone (always in range): they are
  // issued before the index loads that place it, so their latencies overlap.
  const int64_t at = static_cast<int64_t>(i) * p.token_stride;
  const u32x4 k = load_vec<NT>(reinterpret_cast<const u32x4*>(p.key + at) + vec);
  const u32x4 v = load_vec<NT>(reinterpret_cast<const u32x4*>(p.value + at) + vec);
  // Without this barrier the compiler sinks the row loads below the index
  // loads (into the block that stores the row), and the two latencies add up
  // again (measured: 1 us of a 20.8 us prefill launch).
  __builtin_amdgcn_sched_barrier(0);
  if (UNIFORM) f = first_round<FUSED, true>(p, i);
  uint32_t page = 0, slot = 0;
  if (!locate<FUSED, UNIFORM>(p, f, first_i, last_i, i, &page, &slot)) {
    if (live && vec == 0 && p.err != nullptr) atomicAdd(p.err, 1);
    return;
  }
  if (!live) return;
  const int64_t half = static_cast<int64_t>(p.page_size) * p.row_bytes;
  char* row = p.cache + 2 * half * page + static_cast<int64_t>(slot) * p.row_bytes;
  store_row_vec(reinterpret_cast<u32x4*>(row) + vec, k);
  store_row_vec(reinterpret_cast<u32x4*>(row + half) + vec, v);
}

// Sequence length of each request, in 32-bit arithmetic that wraps as torch's
// does.  Bound by its launch: one instead of the five elementwise ones that
// tensor arithmetic takes (MI355X: FlashInfer's form of a prefill of 2 x 4095
// tokens, 4 layers, 194.6 -> 184.4 us).
__global__ __launch_bounds__(256) void seq_lens_kernel(const int32_t* __restrict__ kv_indptr,
                                                       const int32_t* __restrict__ last_page_len, uint32_t batch_size,
                                                       uint32_t page_size, int32_t* __restrict__ out) {
  const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= batch_size) return;
  const int32_t before_last = static_cast<int32_t>(static_cast<uint32_t>(kv_indptr[b + 1]) -
                                                   static_cast<uint32_t>(kv_indptr[b]) - 1u);
  const uint32_t full = before_last > 0 ? static_cast<uint32_t>(before_last) : 0u;
  out[b] = static_cast<int32_t>(full * page_size + static_cast<uint32_t>(last_page_len[b]));
}

// One thread per appended token: finds its request by binary search over
// append_indptr and derives its position from the request's sequence length.
__global__ __launch_bounds__(256) void positions_kernel(const int32_t* __restrict__ append_indptr,
                                                        const int32_t* __restrict__ seq_lens,
                                                        uint32_t batch_size, uint32_t nnz,
                                                        int32_t* __restrict__ batch_indices,
                                                        int32_t* __restrict__ positions) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nnz) return;
  // largest b in [0, batch_size) with append_indptr[b] <= i
  uint32_t lo = 0, hi = batch_size;
  while (hi - lo > 1) {
    const uint32_t mid = lo + (hi - lo) / 2;
    if (append_indptr[mid] <= static_cast<int32_t>(i)) lo = mid; else hi = mid;
  }
  const int32_t a0 = append_indptr[lo], a1 = append_indptr[lo + 1];
  if (static_cast<int32_t>(i) < a0 || static_cast<int32_t>(i) >= a1) {
    batch_indices[i] = -1;   // not covered by any request: the append skips it
    positions[i] = -1;
    return;
  }
  batch_indices[i] = static_cast<int32_t>(lo);
  positions[i] = seq_lens[lo] - (a1 - a0) + (static_cast<int32_t>(i) - a0);
}

}  // namespace
}  // namespace pace_kv

namespace pace_kv {
namespace {

int32_t exact_log2(int64_t n) {
  return (n & (n - 1)) == 0 ? static_cast<int32_t>(__builtin_ctzll(static_cast<uint64_t>(n))) : -1;
}

template <bool FUSED, bool UNIFORM>
const void* kernel_of(bool nt) {
  return nt ? reinterpret_cast<const void*>(&append_kernel<FUSED, UNIFORM, true>)
            : reinterpret_cast<const void*>(&append_kernel<FUSED, UNIFORM, false>);
}

template <bool FUSED>
const void* pick_kernel(bool uniform, bool nt) {
  return uniform ? kernel_of<FUSED, true>(nt) : kernel_of<FUSED, false>(nt);
}

// Checks the arguments both forms share, sizes the grid and launches.
int launch_append(AppendParams& p, int64_t nnz, int batch_size, int64_t num_pages, int64_t num_indices,
                  int page_size, int64_t token_stride_bytes, int64_t row_bytes, bool fused, hipStream_t stream) {
  if (nnz < 0 || batch_size < 0 || num_pages < 0 || num_indices < 0)
    return fail(PACE_KV_EINVAL, "append: negative size");
  if (nnz == 0) return PACE_KV_OK;
  if (!p.key || !p.value || !p.cache || !p.kv_indices || !p.kv_indptr)
    return fail(PACE_KV_EINVAL, "append: NULL argument");
  if (page_size <= 0) return fail(PACE_KV_EINVAL, "append: page_size must be >= 1");
  if (row_bytes <= 0 || row_bytes % kVecBytes != 0)
    return fail(PACE_KV_EINVAL, "append: row bytes (H*D*elem) must be a positive multiple of 16");
  if (token_stride_bytes < row_bytes || token_stride_bytes % kVecBytes != 0)
    return fail(PACE_KV_EINVAL, "append: token stride must be >= row bytes and a multiple of 16");
  if ((reinterpret_cast<uintptr_t>(p.key) | reinterpret_cast<uintptr_t>(p.value) |
       reinterpret_cast<uintptr_t>(p.cache)) & 15u)
    return fail(PACE_KV_EINVAL, "append: keys, values and cache must be 16-byte aligned");
  if (num_pages > INT32_MAX) return fail(PACE_KV_ERANGE, "append: too many pages");
  const int64_t row_vecs = row_bytes / kVecBytes;
  // The most one call takes, whatever its launches could: fewer than 2^24 rows
  // per side, a row longer than 16 KiB counting once per 16 KiB.
  const int64_t pieces = (row_bytes + (16 << 10) - 1) / (16 << 10);
  if (nnz > INT32_MAX || nnz * 2 * pieces >= (int64_t(1) << 25))
    return fail(PACE_KV_ERANGE, "append: too many tokens for one call (%lld)", (long long)nnz);
  p.token_stride = token_stride_bytes;
  p.num_indices = num_indices;
  p.row_bytes = row_bytes;
  p.batch_size = static_cast<uint32_t>(batch_size);
  p.num_pages = static_cast<uint32_t>(num_pages);
  p.page_size = static_cast<uint32_t>(page_size);
  p.page_log2 = exact_log2(page_size);
  p.row_vecs = static_cast<uint32_t>(row_vecs);
  p.guess_own_request = fused && nnz <= batch_size ? 1u : 0u;
  const bool uniform = row_vecs % kThreads == 0;
  const bool nt = nnz * row_bytes > kCachedLoadBytes;
  const int64_t waves_per_row = (row_vecs + kThreads - 1) / kThreads;
  p.row_div = static_cast<uint32_t>(uniform ? waves_per_row : row_vecs);
  p.by_row = fast_div(p.row_div);
  const void* fn = fused ? pick_kernel<true>(uniform, nt) : pick_kernel<false>(uniform, nt);
  const int64_t max_tokens = kMaxGroupsPerLaunch / waves_per_row;
  if (max_tokens < 1) return fail(PACE_KV_ERANGE, "append: row bytes too large (%lld)", (long long)row_bytes);
  for (int64_t t0 = 0; t0 < nnz; t0 += max_tokens) {
    const int64_t n = nnz - t0 < max_tokens ? nnz - t0 : max_tokens;
    const int64_t groups = (n * row_vecs + kThreads - 1) / kThreads;
    p.first_token = static_cast<uint32_t>(t0);
    p.total_items = static_cast<uint32_t>(n * row_vecs);
    void* args[] = {&p};
    PACE_KV_TRY(hip_status(hipLaunchKernel(fn, dim3(static_cast<uint32_t>(groups)),
                                           dim3(kThreads), args, 0, stream), "append launch"));
  }
  return PACE_KV_OK;
}

}  // namespace
}  // namespace pace_kv

using pace_kv::fail;
using pace_kv::hip_status;

extern "C" {

int pace_kv_append(const void* keys, const void* values, int64_t token_stride_bytes, int64_t nnz,
                   const int32_t* batch_indices, const int32_t* positions, int batch_size,
                   void* cache, int64_t num_pages, const int32_t* kv_indices, int64_t num_indices,
                   const int32_t* kv_indptr, int page_size, int64_t row_bytes, int32_t* err_count,
                   void* stream) {
  if (nnz > 0 && (!batch_indices || !positions)) return fail(PACE_KV_EINVAL, "append: NULL argument");
  pace_kv::AppendParams p = {};
  p.key = static_cast<const char*>(keys);
  p.value = static_cast<const char*>(values);
  p.batch_indices = batch_indices;
  p.positions = positions;
  p.kv_indices = kv_indices;
  p.kv_indptr = kv_indptr;
  p.cache = static_cast<char*>(cache);
  p.err = err_count;
  return pace_kv::launch_append(p, nnz, batch_size, num_pages, num_indices, page_size, token_stride_bytes,
                                row_bytes, false, static_cast<hipStream_t>(stream));
}

int pace_kv_append_indptr(const void* keys, const void* values, int64_t token_stride_bytes, int64_t nnz,
                          const int32_t* append_indptr, int batch_size, void* cache, int64_t num_pages,
                          const int32_t* kv_indices, int64_t num_indices, const int32_t* kv_indptr,
                          const int32_t* kv_last_page_len, int page_size, int64_t row_bytes,
                          int32_t* err_count, void* stream) {
  if (nnz > 0 && batch_size == 0) return fail(PACE_KV_EINVAL, "append: tokens without requests");
  if (nnz > 0 && (!append_indptr || !kv_last_page_len)) return fail(PACE_KV_EINVAL, "append: NULL argument");
  pace_kv::AppendParams p = {};
  p.key = static_cast<const char*>(keys);
  p.value = static_cast<const char*>(values);
  p.append_indptr = append_indptr;
  p.kv_last_page_len = kv_last_page_len;
  p.kv_indices = kv_indices;
  p.kv_indptr = kv_indptr;
  p.cache = static_cast<char*>(cache);
  p.err = err_count;
  return pace_kv::launch_append(p, nnz, batch_size, num_pages, num_indices, page_size, token_stride_bytes,
                                row_bytes, true, static_cast<hipStream_t>(stream));
}

int pace_kv_seq_lens(const int32_t* kv_indptr, const int32_t* kv_last_page_len, int batch_size, int page_size,
                     int32_t* seq_lens, void* stream) {
  if (batch_size < 0) return fail(PACE_KV_EINVAL, "seq_lens: negative size");
  if (batch_size == 0) return PACE_KV_OK;
  if (!kv_indptr || !kv_last_page_len || !seq_lens) return fail(PACE_KV_EINVAL, "seq_lens: NULL argument");
  uint32_t bs = static_cast<uint32_t>(batch_size), ps = static_cast<uint32_t>(page_size);
  void* args[] = {&kv_indptr, &kv_last_page_len, &bs, &ps, &seq_lens};
  return hip_status(hipLaunchKernel(reinterpret_cast<const void*>(&pace_kv::seq_lens_kernel), dim3((bs + 255) / 256),
                                    dim3(256), args, 0, static_cast<hipStream_t>(stream)),
                    "seq_lens launch");
}

int pace_kv_batch_indices_positions(const int32_t* append_indptr, const int32_t* seq_lens,
                                    int batch_size, int64_t nnz, int32_t* batch_indices,
                                    int32_t* positions, void* stream) {
  if (nnz < 0 || batch_size < 0) return fail(PACE_KV_EINVAL, "positions: negative size");
  if (nnz == 0) return PACE_KV_OK;
  if (batch_size == 0) return fail(PACE_KV_EINVAL, "positions: tokens without requests");
  if (!append_indptr || !seq_lens || !batch_indices || !positions)
    return fail(PACE_KV_EINVAL, "positions: NULL argument");
  if (nnz > INT32_MAX) return fail(PACE_KV_ERANGE, "positions: too many tokens");
  uint32_t n = static_cast<uint32_t>(nnz);
  uint32_t bs = static_cast<uint32_t>(batch_size);
  const uint32_t blocks = (n + 255) / 256;
  void* args[] = {const_cast<int32_t**>(&append_indptr), const_cast<int32_t**>(&seq_lens), &bs, &n,
                  &batch_indices, &positions};
  return hip_status(hipLaunchKernel(reinterpret_cast<const void*>(&pace_kv::positions_kernel), dim3(blocks),
                                    dim3(256), args, 0, static_cast<hipStream_t>(stream)),
                    "positions launch");
}

}  // extern "C"
