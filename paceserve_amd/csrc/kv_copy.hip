// Paged KV-cache page copies for MI355X (gfx950): pack (gather), unpack
// (scatter) and move (fused gather+scatter), and their C ABI.
//
// Data movement only: no arithmetic, no MFMA.  The kernels are bound by HBM
// bandwidth, so the design goals are (1) every byte read and written exactly
// once, in full 16-byte vectors, fully coalesced per wavefront; (2) no per-page
// host work: one launch covers every (layer, page) pair of a batch of
// requests, with each page id read from the device block table once per
// wavefront (a uniform load, served from L2 after the first wavefront of the
// page); (3) a compact set of in-flight addresses.
//
// Work decomposition.  A page of one layer is `page_bytes` contiguous bytes
// (K half then V half).  It is split into 1 KiB rows; one workgroup of one
// wave64 copies one row, each lane moving one 16-byte vector with a
// nontemporal load and a write-through store, and then retires.  The grid is
// (rows x pages) x layers: blockIdx.x walks the rows of a layer's pages, row
// fastest, and blockIdx.y is the layer, so workgroups dispatched together read
// (unpack) or write (pack) adjacent rows of the transfer buffer and adjacent
// rows of each pool page.  A wave splits blockIdx.x into page and row with a
// shift when a page has a power-of-two number of rows (every common KV page),
// else with one division; pages that are no whole number of rows are taken end
// to end (enum Shape).  An unpack wave issues its buffer load before its
// destination page id arrives.  Measured on MI355X, this fine grain keeps
// the chip's in-flight accesses within a narrow address window and copies at
// ~6.6 TB/s, against ~5.6-5.9 TB/s for 8-32 KiB per workgroup, persistent
// grid-stride loops or ids staged in LDS (a persistent loop serialises each
// trip's loads behind the previous trip's stores on the shared vmcnt counter).
#include <hip/hip_ext.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "internal.h"

namespace pace_kv {

namespace {

constexpr int kThreads = 64;              // one wave64 per workgroup
constexpr int kVecBytes = 16;
constexpr int kRowBytes = kThreads * kVecBytes;  // 1 KiB per workgroup
constexpr int kMaxLayers = PACE_KV_MAX_LAYERS_PER_LAUNCH;
// Workgroups per launch stay below 2^25 so that grid * 64 threads fits the
// 32-bit launch limit with room to spare; larger batches use more launches.
constexpr int64_t kMaxItemsPerLaunch = int64_t(1) << 25;

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

thread_local char g_last_error[512] = "";

struct CopyParams {
  const char* src[kMaxLayers];
  char* dst[kMaxLayers];
  const int32_t* src_ids;  // nullptr: identity (page j)
  const int32_t* dst_ids;  // nullptr: identity (page j)
  int32_t* err;            // optional skipped-tile counter
  int64_t page_bytes;
  uint32_t src_pool_pages;
  uint32_t dst_pool_pages;
  uint32_t page_vecs;      // page_bytes / 16
  uint32_t n_pages;        // of this launch, per layer
  FastDiv by_page;         // pages end to end: division by page_vecs
  uint32_t total_vecs;     // n_pages * page_vecs
  uint32_t rows_per_page;  // page_bytes / kRowBytes (pages of whole rows)
  uint32_t rows_log2;      // log2(rows_per_page) when that is a power of two
  char* tee;               // Kind::kTee: page j of layer l also goes to tee + l * tee_stride + j * page_bytes
  int64_t tee_stride;
};

// What a launch copies: kStream (unpack, move, swap), kPack (into a transfer
// buffer that an unpack reads next), kTee (a move that also leaves the pages
// in a transfer buffer).
enum Kind { kStream = 0, kPack = 1, kTee = 2 };

// How a launch splits a layer's pages over its waves.  Pages of a power-of-two
// number of 1 KiB rows (kPow2) or of another whole number (kRows): one row per
// wave.  Other pages are taken end to end, vector after vector, so that every
// lane carries a vector and a wave may hold several pages, or the end of one
// and the start of the next: each lane loads its own page's ids (kLaneFlat), or
// the wave loads the at most kSpan ids per side that its lanes choose from by
// scalar loads (kSpanFlat: pages of at least kSpanVecs vectors, 336 bytes, with
// ids on both sides, or packs of up to kSpanPackBytes a launch).
// Measured on MI355X, 32 layers, 150 MiB, against waves that end with a page:
//   move    160 B 210 -> 103 us, 256 B 132 -> 52, 512 B 67.4 -> 50.3, 1280 B
//           57 -> 50, 1536 B 53.7 -> 49.8, the same from 2560 B on
//   pack    160 B 210 -> 60, 512 B 67 -> 46, 1280 B 54.5 -> 46.3, 1536 B and
//           more the same or up to 2% faster
//   unpack  160 B 210 -> 85, 512 B 67.5 -> 48.9, 1280 B 56.4 -> 48.8
// and on 6 MiB in a graph, 512 B: move 4.3 -> 3.2 us, pack 4.3 -> 3.3, unpack
// 4.3 -> 3.2.  Below 2.5 MiB, where a launch takes 1.9 to 2.6 us, moves and packs
// are from 13% faster to 4% slower, unpacks from 15% faster to 5% slower.
// A move by lanes' own ids is 3-4% slower than by scalar ids (its id loads go
// ahead of the page's in one chain).  A pack by lanes' own ids is slower up to
// 64 MiB (kSpanPackBytes; 1.75 MiB of 1536 B 2.46 against 2.24 us, 2.24 by waves
// that end with a page; 48 MiB 3 to 17% and 64 MiB 0 to 10%) and 1 to 5% faster from 96 MiB
// on; an unpack by scalar ids, its eight waits as below, was 4-8% slower at 150 MiB.
// Across the host link what counts is the number of pieces in which pages
// travel: pages of up to kLinkPageBytes go one to a wave (kOnePage).
// Measured on MI355X, swaps of 8 MiB against waves end to end: 160 B out 167
// against 176 us, in 250 against 304; 400 B 159 against 167 and 192 against 234.
enum Shape { kPow2 = 0, kRows = 1, kSpanFlat = 2, kLaneFlat = 3, kOnePage = 4 };
constexpr int kLinkPageBytes = 512;
constexpr int64_t kSpanPackBytes = 64 << 20;
constexpr int kSpan = 4;
constexpr int kSpanVecs = kThreads / (kSpan - 1);

// Page ids carried in the kernel arguments (small promotions): no device id
// array, so no upload has to precede the launch.
struct CopyParamsInline {
  CopyParams base;
  int32_t src_ids[PACE_KV_INLINE_IDS];
  int32_t dst_ids[PACE_KV_INLINE_IDS];
};

// Stores carry the device-scope bit (sc1): an XCD's L2 is not coherent with
// the other XCDs', so such a store writes through it to the memory side, and
// the launch leaves no dirty L2 lines to write back when it ends.  A pack
// (PACK) stores with sc1 alone, so the rows also stay in the memory-side cache
// for the unpack that reads them next; every other copy adds nt (streaming).
// Measured on MI355X against plain (launches <= 1 GiB) or nontemporal pack
// stores and nontemporal unpack stores, pack+unpack runs 0.8% (16 GiB of
// 256 KiB pages) to 5.9% (64 MiB) faster, and a fused move 0.5% to 4.2%.
// A store of more than 64 bits reads its data registers after it issues, so
// the next instructions must not overwrite them; the compiler inserts those
// wait states for the stores it emits itself but cannot for one written as
// asm, so the asm carries them (s_nop 1: two wait states).  Without them a
// variant that computed its next address into the stored registers wrote
// wrong data.
template <bool CACHED>
__device__ __forceinline__ void store_vec(const u32x4 v, u32x4* d) {
  if (CACHED) asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" : : "v"(d), "v"(v) : "memory");
  else asm volatile("global_store_dwordx4 %0, %1, off nt sc1\n\ts_nop 1" : : "v"(d), "v"(v) : "memory");
}

// The tee's copy of one vector: pool page sp to page j of the transfer buffer
// and to pool page dp, from one read.  The same bytes and the same counts as a
// pack followed by an unpack, including a source id outside its pool, where
// the pack leaves the buffer's page as it was and the unpack copies that.
//
// Bound by HBM, and by its writes: 3 bytes of traffic per payload byte, two of
// them written, against the 4 of a pack and an unpack.  Measured on MI355X
// against those two launches: 512 MiB of 64 KiB pages 259 us (6.2 TB/s) against
// 300-310; 2.8 GB of 8 KiB pages, 80 layers, 1.47 ms against 1.79.  Of the
// shapes and policies tried, one wave per 1 KiB row with streaming stores and
// plain loads is the fastest: cacheable buffer stores cost 0.5%, cacheable
// stores on both sides 4-7%, nontemporal loads 0.5-1%, the destination store
// first 0.2-1%; 128 threads are 0.5% faster on 512 MiB and 2% slower on 2.8 GB,
// 256 and 512 threads slower on both.
__device__ __forceinline__ void tee_row(const CopyParams& p, uint32_t j, uint32_t layer, uint32_t vec,
                                        uint32_t sp, uint32_t dp) {
  u32x4* buf = reinterpret_cast<u32x4*>(p.tee + layer * p.tee_stride + static_cast<int64_t>(j) * p.page_bytes) + vec;
  const bool src_ok = sp < p.src_pool_pages, dst_ok = dp < p.dst_pool_pages;
  if (!(src_ok && dst_ok) && vec == 0 && p.err != nullptr)
    atomicAdd(p.err, static_cast<int>(!src_ok) + static_cast<int>(!dst_ok));
  const u32x4* s = src_ok ? reinterpret_cast<const u32x4*>(p.src[layer] + static_cast<int64_t>(sp) * p.page_bytes) + vec
                          : buf;
  const u32x4 v = *s;
  if (src_ok) store_vec<false>(v, buf);
  if (dst_ok)
    store_vec<false>(v, reinterpret_cast<u32x4*>(p.dst[layer] + static_cast<int64_t>(dp) * p.page_bytes) + vec);
}

// The copy of one 1 KiB row: item blockIdx.x of layer blockIdx.y.  For pages
// of whole rows (kPow2, kRows) that is row r of page j, the grid is exactly
// (rows x pages) x layers and every index is scalar; else it is the next
// 64 vectors of the layer's pages.  sids / dids are the
// sides' page ids (device or kernel-argument arrays), nullptr for a contiguous
// side.  Loads are nontemporal but in a tee; KIND selects the store policy
// (store_vec) and the tee.
template <Shape SHAPE, Kind KIND>
__device__ __forceinline__ void copy_row(const CopyParams& p, const int32_t* sids,
                                         const int32_t* dids) {
  const uint32_t x = blockIdx.x;
  const uint32_t layer = blockIdx.y;
  uint32_t j, vec, sp, dp;
  bool inside = true;
  if (SHAPE == kSpanFlat) {
    // The arguments are all loaded behind one wait, and then the ids behind
    // another: left to itself the compiler loads each where it is first used,
    // eight waits in a row, which small launches showed (a move of 256 KiB of
    // 512-byte pages 2.06 us, now 1.88).  In kLaneFlat the same was up to 4%
    // faster below 512 KiB and up to 10% slower at 1 MiB.
    uint32_t g0 = x * kThreads;
    if (KIND == kTee) asm("" : "+s"(g0) : "s"(p.tee), "s"(p.tee_stride));
    asm("" : "+s"(g0) : "s"(p.src[layer]), "s"(p.dst[layer]), "s"(p.err), "s"(p.page_bytes), "s"(p.src_pool_pages),
                        "s"(p.dst_pool_pages), "s"(p.page_vecs), "s"(p.by_page.mul), "s"(p.by_page.shift1),
                        "s"(p.by_page.shift2), "s"(p.n_pages), "s"(p.total_vecs));
    inside = g0 + threadIdx.x < p.total_vecs;
    const uint32_t j0 = over(p.by_page, g0), last = p.n_pages - 1;
    const uint32_t j1 = min(j0 + 1, last), j2 = min(j0 + 2, last), j3 = min(j0 + 3, last);
    int32_t s0 = sids[j0], s1 = sids[j1], s2 = sids[j2], s3 = sids[j3];
    int32_t d0 = 0, d1 = 0, d2 = 0, d3 = 0;
    if (KIND == kPack) {
      asm("" : "+s"(s0), "+s"(s1), "+s"(s2), "+s"(s3));
    } else {
      d0 = dids[j0], d1 = dids[j1], d2 = dids[j2], d3 = dids[j3];
      asm("" : "+s"(s0), "+s"(s1), "+s"(s2), "+s"(s3), "+s"(d0), "+s"(d1), "+s"(d2), "+s"(d3));
    }
    vec = g0 - j0 * p.page_vecs + threadIdx.x;
    const bool past1 = vec >= p.page_vecs, past2 = vec >= 2 * p.page_vecs, past3 = vec >= 3 * p.page_vecs;
    j = j0 + past1 + past2 + past3;
    vec -= past3 ? 3 * p.page_vecs : past2 ? 2 * p.page_vecs : past1 ? p.page_vecs : 0;
    sp = static_cast<uint32_t>(past3 ? s3 : past2 ? s2 : past1 ? s1 : s0);
    dp = KIND == kPack ? j : static_cast<uint32_t>(past3 ? d3 : past2 ? d2 : past1 ? d1 : d0);
  } else if (SHAPE == kLaneFlat) {
    const uint32_t g = x * kThreads + threadIdx.x;
    if (g >= p.total_vecs) return;
    j = over(p.by_page, g);
    vec = g - j * p.page_vecs;
  } else if (SHAPE == kOnePage) {
    j = x;
    vec = threadIdx.x;
    if (vec >= p.page_vecs) return;
  } else {
    j = SHAPE == kPow2 ? x >> p.rows_log2 : x / p.rows_per_page;
    const uint32_t row = SHAPE == kPow2 ? x & (p.rows_per_page - 1) : x - j * p.rows_per_page;
    vec = row * kThreads + threadIdx.x;
  }
  if (!inside) return;
  if (SHAPE != kSpanFlat && sids == nullptr) {
    // Contiguous source (unpack): page j of the buffer is always in bounds,
    // so the load is issued before the destination id is known.
    const u32x4 v = __builtin_nontemporal_load(
        reinterpret_cast<const u32x4*>(p.src[layer] + static_cast<int64_t>(j) * p.page_bytes) + vec);
    dp = dids ? static_cast<uint32_t>(dids[j]) : j;
    if (dp >= p.dst_pool_pages) {
      if (vec == 0 && p.err != nullptr) atomicAdd(p.err, 1);
      return;
    }
    store_vec<KIND == kPack>(v, reinterpret_cast<u32x4*>(p.dst[layer] + static_cast<int64_t>(dp) * p.page_bytes) + vec);
    return;
  }
  if (SHAPE != kSpanFlat) {
    sp = static_cast<uint32_t>(sids[j]);
    dp = dids ? static_cast<uint32_t>(dids[j]) : j;
  }
  if (KIND == kTee) {
    tee_row(p, j, layer, vec, sp, dp);
    return;
  }
  // Negative ids wrap to large unsigned values and fail the same test.
  if (sp >= p.src_pool_pages || dp >= p.dst_pool_pages) {
    if (vec == 0 && p.err != nullptr) atomicAdd(p.err, 1);
    return;
  }
  const u32x4 v = __builtin_nontemporal_load(
      reinterpret_cast<const u32x4*>(p.src[layer] + static_cast<int64_t>(sp) * p.page_bytes) + vec);
  store_vec<KIND == kPack>(v, reinterpret_cast<u32x4*>(p.dst[layer] + static_cast<int64_t>(dp) * p.page_bytes) + vec);
}

template <Shape SHAPE, Kind KIND>
__global__ __launch_bounds__(kThreads) void page_copy_kernel(const CopyParams p) {
  copy_row<SHAPE, KIND>(p, p.src_ids, p.dst_ids);
}

// Same copy with the ids in the kernel arguments.  A side whose ids are not
// inline (the contiguous buffer of a pack or unpack) indexes pages by
// position.
template <Shape SHAPE, Kind KIND, bool SRC_INLINE, bool DST_INLINE>
__global__ __launch_bounds__(kThreads) void page_copy_inline_kernel(const CopyParamsInline p) {
  copy_row<SHAPE, KIND>(p.base, SRC_INLINE ? p.src_ids : nullptr, DST_INLINE ? p.dst_ids : nullptr);
}

// Inline ids on both sides (move), the source only (pack) or the destination
// only (unpack).
enum InlineSides { kBothInline = 0, kSrcInline = 1, kDstInline = 2 };

template <Shape SHAPE>
const void* kernel_of(Kind kind) {
  switch (kind) {
    case kPack: return reinterpret_cast<const void*>(&page_copy_kernel<SHAPE, kPack>);
    case kTee: return reinterpret_cast<const void*>(&page_copy_kernel<SHAPE, kTee>);
    default: return reinterpret_cast<const void*>(&page_copy_kernel<SHAPE, kStream>);
  }
}

template <Shape SHAPE, Kind KIND>
const void* inline_kernel_of(InlineSides sides) {
  switch (sides) {
    case kSrcInline: return reinterpret_cast<const void*>(&page_copy_inline_kernel<SHAPE, KIND, true, false>);
    case kDstInline: return reinterpret_cast<const void*>(&page_copy_inline_kernel<SHAPE, KIND, false, true>);
    default: return reinterpret_cast<const void*>(&page_copy_inline_kernel<SHAPE, KIND, true, true>);
  }
}

template <Shape SHAPE>
const void* inline_kernel_of(Kind kind, InlineSides sides) {
  switch (kind) {
    case kPack: return inline_kernel_of<SHAPE, kPack>(sides);
    // a tee has ids on both sides
    case kTee: return reinterpret_cast<const void*>(&page_copy_inline_kernel<SHAPE, kTee, true, true>);
    default: return inline_kernel_of<SHAPE, kStream>(sides);
  }
}

// Pages between a pool and pinned host memory, without a device buffer between
// them.
//
// Bound by the link (56-57 GB/s per direction), so what counts is to keep
// enough of it in flight with few waves: the rest of the chip's CUs stay free
// for other streams, and more waves slow the other direction's traffic.  Each
// lane keeps UNROLL vectors in flight and loads the next round's ids behind
// them.  Measured on MI355X at 14 and 56 MiB, by workgroups of 256:
//   out, 16 vectors   4: 54.5 and 56.2 GB/s, 6 to 12 within 2% either way
//                     (short pages 4: 16 MiB of 160 B 341 us, of 400 B 326;
//                     8: 310 and 309)
//   in, 8 vectors     8: 33, 16: 55.4 and 56.8, 24 to 64: 54 to 56.5;
//                     16 vectors the same or slower
// Beside host-to-device DMA copies 4 workgroups out keep 48.6 GB/s per
// direction, 32 workgroups 44; a read stream by waves beside a write stream
// falls to 28, so only short copies read the host this way.
// What other streams run meanwhile is slowed by more than those CUs: 1 GiB HBM
// copies for 6.05 ms, or bf16 matrix products for 11.3 ms, take 6.9 and 12.7 ms
// beside two legs out of 56 MiB (the same beside a pack and a copy kernel), 7.6
// and 12.7 beside two legs in (6.1 and 11.4 beside two DMA copies in, which take
// 1.065 ms each against 1.035), and 7.4 to 7.7 and 12.7 beside two swaps (8.1
// and 13.1 to 13.3 by the page copy).
constexpr int kHostThreads = 256;
constexpr int kOutGroups = 4, kOutUnroll = 16;
constexpr int kInGroups = 16, kInUnroll = 8;
// Between two paged pools (swaps) both sides' ids take registers: 8 vectors
// either way, out from 32 workgroups (12 to 16 are 1-4% slower).  Measured
// against the page copy's one wave per row, 63 pages of 64 KiB, 32 layers: out
// 2379 -> 2328 us, in 2412 -> 2326; 7 pages out 270 -> 264, in 290 -> 265; 500
// pages of 8 KiB out 2362 -> 2307, in 2384 -> 2306; 777 of 1536 B out 689 -> 680,
// in 696 -> 679.  Short pages and small swaps are the page copy's (swap_copy).
constexpr int kPagedOutGroups = 32;

struct HostLegParams {
  char* layers[kMaxLayers];
  char* host[kMaxLayers];  // the host side: pages in order, or chosen by host_ids (PAGED)
  const int32_t* ids;      // device arrays; unused by the inline kernel
  const int32_t* host_ids;
  int32_t* err;
  int64_t page_bytes;
  uint32_t pool_pages;     // at least 1, on both sides
  uint32_t host_pages;
  uint32_t page_vecs;
  uint32_t n_pages;
  uint32_t total_vecs;
  FastDiv by_page;         // division by page_vecs
  FastDiv by_count;        // division by n_pages
};

struct HostLegParamsInline {
  HostLegParams base;
  int32_t ids[PACE_KV_INLINE_IDS];
};

// What a lane needs to know of the UNROLL vectors of one round.
template <int UNROLL>
struct HostRound {
  uint32_t vec[UNROLL], id[UNROLL], host_id[UNROLL];
  char* base[UNROLL];
  char* host[UNROLL];
};

template <int UNROLL, bool PAGED>
__device__ __forceinline__ void next_round(const HostLegParams& p, const int32_t* ids, uint32_t i, uint32_t stride,
                                           HostRound<UNROLL>* r) {
#pragma unroll
  for (int u = 0; u < UNROLL; ++u) {
    const uint32_t k = min(i + u * stride, p.total_vecs - 1);
    const uint32_t at = over(p.by_page, k);
    r->vec[u] = k - at * p.page_vecs;
    const uint32_t layer = over(p.by_count, at);
    const uint32_t j = at - layer * p.n_pages;
    r->base[u] = p.layers[layer];
    r->id[u] = static_cast<uint32_t>(ids[j]);
    r->host[u] = PAGED ? p.host[layer] : p.host[0];
    r->host_id[u] = PAGED ? static_cast<uint32_t>(p.host_ids[j]) : at;
  }
}

// The loads of a round are free of branches, so that all of a lane's are in
// flight together: a vector past the end repeats the last one's and a page id
// out of range reads page 0, and neither is stored.  The next round's ids are
// loaded behind this round's vectors.
template <bool TO_HOST, int UNROLL, bool PAGED>
__device__ __forceinline__ void host_leg(const HostLegParams& p, const int32_t* ids) {
  const uint32_t stride = gridDim.x * kHostThreads;
  uint32_t i = blockIdx.x * kHostThreads + threadIdx.x;
  HostRound<UNROLL> r;
  next_round<UNROLL, PAGED>(p, ids, i, stride, &r);
  for (; i < p.total_vecs; i += UNROLL * stride) {
    u32x4* to[UNROLL];
    u32x4 v[UNROLL];
    bool ok[UNROLL], first[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const bool id_ok = r.id[u] < p.pool_pages, host_ok = !PAGED || r.host_id[u] < p.host_pages;
      u32x4* const pool =
          reinterpret_cast<u32x4*>(r.base[u] + static_cast<int64_t>(id_ok ? r.id[u] : 0) * p.page_bytes) + r.vec[u];
      u32x4* const host =
          reinterpret_cast<u32x4*>(r.host[u] + static_cast<int64_t>(host_ok ? r.host_id[u] : 0) * p.page_bytes) +
          r.vec[u];
      v[u] = __builtin_nontemporal_load(TO_HOST ? pool : host);
      to[u] = TO_HOST ? host : pool;
      ok[u] = id_ok && host_ok;
      first[u] = r.vec[u] == 0;
    }
    __builtin_amdgcn_sched_barrier(0);
    next_round<UNROLL, PAGED>(p, ids, i + UNROLL * stride, stride, &r);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      if (i + u * stride >= p.total_vecs) continue;
      if (ok[u]) store_vec<false>(v[u], to[u]);
      else if (first[u] && p.err != nullptr) atomicAdd(p.err, 1);
    }
  }
}

template <bool TO_HOST, bool PAGED>
__global__ __launch_bounds__(kHostThreads) void host_leg_kernel(const HostLegParams p) {
  host_leg<TO_HOST, TO_HOST && !PAGED ? kOutUnroll : kInUnroll, PAGED>(p, p.ids);
}

template <bool TO_HOST>
__global__ __launch_bounds__(kHostThreads) void host_leg_inline_kernel(const HostLegParamsInline p) {
  host_leg<TO_HOST, TO_HOST ? kOutUnroll : kInUnroll, false>(p.base, p.ids);
}

const void* pick_kernel(Shape shape, Kind kind) {
  switch (shape) {
    case kOnePage: return reinterpret_cast<const void*>(&page_copy_kernel<kOnePage, kStream>);
    case kPow2: return kernel_of<kPow2>(kind);
    case kRows: return kernel_of<kRows>(kind);
    case kSpanFlat: return kernel_of<kSpanFlat>(kind);  // a move, a tee or a small pack
    default: return kernel_of<kLaneFlat>(kind);
  }
}

const void* pick_inline_kernel(Shape shape, Kind kind, InlineSides sides) {
  switch (shape) {
    case kPow2: return inline_kernel_of<kPow2>(kind, sides);
    case kRows: return inline_kernel_of<kRows>(kind, sides);
    case kSpanFlat:
      switch (kind) {
        case kPack: return reinterpret_cast<const void*>(&page_copy_inline_kernel<kSpanFlat, kPack, true, false>);
        case kTee: return reinterpret_cast<const void*>(&page_copy_inline_kernel<kSpanFlat, kTee, true, true>);
        default: return reinterpret_cast<const void*>(&page_copy_inline_kernel<kSpanFlat, kStream, true, true>);
      }
    default: return inline_kernel_of<kLaneFlat>(kind, sides);
  }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int check_layers(const char* const* layers, int num_layers, const char* what) {
  if (num_layers > 0 && layers == nullptr) return fail(PACE_KV_EINVAL, "%s: layer table is NULL", what);
  for (int l = 0; l < num_layers; ++l) {
    if (layers[l] == nullptr) return fail(PACE_KV_EINVAL, "%s: layer %d pointer is NULL", what, l);
    if (!aligned16(layers[l]))
      return fail(PACE_KV_EINVAL, "%s: layer %d pointer is not 16-byte aligned", what, l);
  }
  return PACE_KV_OK;
}

}  // namespace

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_last_error, sizeof(g_last_error), fmt, ap);
  va_end(ap);
  return code;
}

int hip_status(hipError_t err, const char* what) {
  if (err == hipSuccess) return PACE_KV_OK;
  return fail(static_cast<int>(err), "%s: %s (hipError %d)", what, hipGetErrorString(err),
              static_cast<int>(err));
}

void buffer_layers(const void* base, int64_t layer_stride, int num_layers, const char** out) {
  for (int l = 0; l < num_layers; ++l)
    out[l] = static_cast<const char*>(base) + static_cast<int64_t>(l) * layer_stride;
}

int launch_page_copy(const Side& src, const Side& dst, int num_layers, int64_t n_pages,
                     int64_t page_bytes, int32_t* err_count, hipStream_t stream, StorePolicy policy,
                     const Tee* tee) {
  const int32_t *const host_src_ids = src.host_ids, *const host_dst_ids = dst.host_ids;
  if (num_layers < 0) return fail(PACE_KV_EINVAL, "num_layers must be >= 0 (got %d)", num_layers);
  if (n_pages < 0) return fail(PACE_KV_EINVAL, "n_pages must be >= 0 (got %lld)", (long long)n_pages);
  if (page_bytes <= 0 || page_bytes % kVecBytes != 0)
    return fail(PACE_KV_EINVAL, "page_bytes must be a positive multiple of 16 (got %lld)",
                (long long)page_bytes);
  if (page_bytes / kVecBytes > INT32_MAX)
    return fail(PACE_KV_ERANGE, "page_bytes too large (%lld)", (long long)page_bytes);
  if (n_pages > INT32_MAX) return fail(PACE_KV_ERANGE, "n_pages exceeds int32 range");
  if (src.pool_pages < 0 || dst.pool_pages < 0) return fail(PACE_KV_EINVAL, "pool_pages must be >= 0");
  if (num_layers == 0 || n_pages == 0) return PACE_KV_OK;
  const bool src_indexed = src.ids != nullptr || host_src_ids != nullptr;
  const bool dst_indexed = dst.ids != nullptr || host_dst_ids != nullptr;
  if ((!src_indexed && src.pool_pages < n_pages) || (!dst_indexed && dst.pool_pages < n_pages))
    return fail(PACE_KV_ERANGE, "contiguous buffer holds fewer pages than n_pages");
  int rc = check_layers(src.layers, num_layers, "source");
  if (rc) return rc;
  rc = check_layers(dst.layers, num_layers, "destination");
  if (rc) return rc;
  if (tee != nullptr && (!src_indexed || !dst_indexed || !aligned16(tee->base) || tee->layer_stride % kVecBytes != 0))
    return fail(PACE_KV_EINVAL, "tee: needs page ids on both sides and a 16-byte aligned buffer");
  const bool inline_ids = host_src_ids != nullptr || host_dst_ids != nullptr;
  // The inline kernels index a side without inline ids by position.
  if (inline_ids && ((host_src_ids == nullptr && src.ids != nullptr) ||
                     (host_dst_ids == nullptr && dst.ids != nullptr)))
    return fail(PACE_KV_EINVAL, "a launch cannot mix device and kernel-argument page ids");
  if (inline_ids && n_pages > PACE_KV_INLINE_IDS)
    return fail(PACE_KV_ERANGE, "more than %d pages cannot travel in the kernel arguments",
                PACE_KV_INLINE_IDS);
  if (src.ids != nullptr && (reinterpret_cast<uintptr_t>(src.ids) & 3u))
    return fail(PACE_KV_EINVAL, "source page ids are not 4-byte aligned");
  if (dst.ids != nullptr && (reinterpret_cast<uintptr_t>(dst.ids) & 3u))
    return fail(PACE_KV_EINVAL, "destination page ids are not 4-byte aligned");

  const int64_t rows_per_page = (page_bytes + kRowBytes - 1) / kRowBytes;

  const auto clamp_pool = [](int64_t pages) -> uint32_t {
    return pages > INT32_MAX ? static_cast<uint32_t>(INT32_MAX) : static_cast<uint32_t>(pages);
  };

  uint32_t rows_log2 = 0;
  while ((int64_t(1) << rows_log2) < rows_per_page) ++rows_log2;
  const bool whole_rows = page_bytes % kRowBytes == 0;
  const bool small_pack = policy == StorePolicy::kPack && src_indexed && !dst_indexed &&
                          n_pages <= kSpanPackBytes / page_bytes / std::min(num_layers, kMaxLayers);
  const bool span = page_bytes >= kSpanVecs * kVecBytes &&
                    ((src_indexed && dst_indexed && policy != StorePolicy::kPack) || small_pack);
  const bool one_page =
      policy == StorePolicy::kLink && page_bytes <= kLinkPageBytes && !inline_ids && tee == nullptr;
  const Shape shape = whole_rows ? ((int64_t(1) << rows_log2) == rows_per_page ? kPow2 : kRows)
                      : one_page ? kOnePage
                      : span     ? kSpanFlat
                                 : kLaneFlat;

  for (int l0 = 0; l0 < num_layers; l0 += kMaxLayers) {
    const int nl = num_layers - l0 < kMaxLayers ? num_layers - l0 : kMaxLayers;
    const int64_t max_pages = kMaxItemsPerLaunch / (int64_t(nl) * rows_per_page);
    if (max_pages < 1)
      return fail(PACE_KV_ERANGE, "page_bytes too large for one launch (%lld)", (long long)page_bytes);
    for (int64_t j0 = 0; j0 < n_pages; j0 += max_pages) {
      const int64_t nj = n_pages - j0 < max_pages ? n_pages - j0 : max_pages;
      CopyParams p;
      memset(&p, 0, sizeof(p));
      for (int l = 0; l < nl; ++l) {
        p.src[l] = src.layers[l0 + l] + (src_indexed ? 0 : j0 * page_bytes);
        p.dst[l] = const_cast<char*>(dst.layers[l0 + l]) + (dst_indexed ? 0 : j0 * page_bytes);
      }
      p.src_ids = src.ids ? src.ids + j0 : nullptr;
      p.dst_ids = dst.ids ? dst.ids + j0 : nullptr;
      p.err = err_count;
      p.page_bytes = page_bytes;
      p.src_pool_pages = src_indexed ? clamp_pool(src.pool_pages) : static_cast<uint32_t>(nj);
      p.dst_pool_pages = dst_indexed ? clamp_pool(dst.pool_pages) : static_cast<uint32_t>(nj);
      p.page_vecs = static_cast<uint32_t>(page_bytes / kVecBytes);
      p.rows_per_page = static_cast<uint32_t>(rows_per_page);
      p.rows_log2 = rows_log2;
      p.by_page = fast_div(p.page_vecs);
      p.n_pages = static_cast<uint32_t>(nj);
      p.total_vecs = static_cast<uint32_t>(nj * p.page_vecs);  // < 2^25 * 64: see max_pages
      if (tee != nullptr) {
        p.tee = tee->base + l0 * tee->layer_stride + j0 * page_bytes;
        p.tee_stride = tee->layer_stride;
      }
      const int64_t groups =
          whole_rows || one_page ? rows_per_page * nj : (nj * p.page_vecs + kThreads - 1) / kThreads;
      const dim3 grid(static_cast<uint32_t>(groups), static_cast<uint32_t>(nl));
      const Kind kind = tee != nullptr ? kTee : (policy == StorePolicy::kPack ? kPack : kStream);
      if (inline_ids) {
        CopyParamsInline q;
        q.base = p;
        if (host_src_ids) memcpy(q.src_ids, host_src_ids + j0, nj * sizeof(int32_t));
        if (host_dst_ids) memcpy(q.dst_ids, host_dst_ids + j0, nj * sizeof(int32_t));
        const InlineSides sides =
            host_src_ids && host_dst_ids ? kBothInline : (host_src_ids ? kSrcInline : kDstInline);
        void* args[] = {&q};
        rc = hip_status(hipLaunchKernel(pick_inline_kernel(shape, kind, sides), grid, dim3(kThreads), args, 0, stream),
                        "page copy launch");
      } else {
        void* args[] = {&p};
        rc = hip_status(hipLaunchKernel(pick_kernel(shape, kind), grid, dim3(kThreads), args, 0, stream),
                        "page copy launch");
      }
      if (rc) return rc;
    }
  }
  return PACE_KV_OK;
}

namespace {

// Whether no byte of any [a[i], a[i] + a_bytes) lies in any [b[k], b[k] + b_bytes).
bool disjoint(const char* const* a, int64_t a_bytes, const char* const* b, int64_t b_bytes, int n) {
  const auto hull = [n](const char* const* t) { return std::minmax_element(t, t + n); };
  const auto ha = hull(a), hb = hull(b);
  // Pools allocated one after the other, the usual case: all of one side
  // lies below all of the other.
  if (*ha.second + a_bytes <= *hb.first || *hb.second + b_bytes <= *ha.first) return true;
  std::vector<const char*> sa(a, a + n), sb(b, b + n);
  std::sort(sa.begin(), sa.end());
  std::sort(sb.begin(), sb.end());
  for (int i = 0, k = 0; i < n && k < n;) {
    if (sa[i] + a_bytes <= sb[k]) ++i;
    else if (sb[k] + b_bytes <= sa[i]) ++k;
    else return false;
  }
  return true;
}

}  // namespace

int launch_host_leg(const Side& pool, const Side& host, bool to_host, int num_layers, int64_t n_pages,
                    int64_t page_bytes, int32_t* err_count, hipStream_t stream, hipEvent_t done) {
  constexpr int64_t kMaxVecs = int64_t(1) << 31;  // of one launch: 32-bit indexes, with room for a round past the end
  const bool paged = host.ids != nullptr;
  const int64_t page_vecs = page_bytes / kVecBytes;
  // The page copy would take a side without ids for a contiguous buffer.
  if (num_layers > 0 && n_pages > 0 && pool.ids == nullptr && pool.host_ids == nullptr)
    return fail(PACE_KV_EINVAL, "host leg: NULL page ids");
  // Other refusals, empty pools (no page to read in a bad id's place) and
  // layers of 32 GiB and more are the page copy's.
  if (num_layers <= 0 || n_pages <= 0 || page_vecs <= 0 || page_bytes % kVecBytes != 0 || pool.pool_pages < 1 ||
      host.pool_pages < (paged ? 1 : n_pages) || n_pages > kMaxVecs / page_vecs ||
      host.host_ids != nullptr ||
      (paged && pool.host_ids != nullptr) || (reinterpret_cast<uintptr_t>(pool.ids) & 3u) != 0 ||
      (reinterpret_cast<uintptr_t>(host.ids) & 3u) != 0 || (pool.host_ids != nullptr && n_pages > PACE_KV_INLINE_IDS)) {
    PACE_KV_TRY(launch_page_copy(to_host ? pool : host, to_host ? host : pool, num_layers, n_pages, page_bytes,
                                 err_count, stream));
    return done != nullptr ? hip_status(hipEventRecord(done, stream), "host leg record") : PACE_KV_OK;
  }
  PACE_KV_TRY(check_layers((to_host ? pool : host).layers, num_layers, "source"));
  PACE_KV_TRY(check_layers((to_host ? host : pool).layers, num_layers, "destination"));
  const int64_t fit = kMaxVecs / (n_pages * page_vecs);
  const int step = static_cast<int>(std::min<int64_t>({fit, kMaxLayers, num_layers}));
  for (int l0 = 0; l0 < num_layers; l0 += step) {
    const int nl = std::min(step, num_layers - l0);
    HostLegParamsInline q;
    memset(&q.base, 0, sizeof(q.base));
    HostLegParams& p = q.base;
    for (int l = 0; l < nl; ++l) {
      p.layers[l] = const_cast<char*>(pool.layers[l0 + l]);
      p.host[l] = const_cast<char*>(host.layers[l0 + l]);
    }
    p.ids = pool.ids;
    p.host_ids = host.ids;
    p.err = err_count;
    p.page_bytes = page_bytes;
    p.pool_pages = static_cast<uint32_t>(std::min<int64_t>(pool.pool_pages, INT32_MAX));
    p.host_pages = static_cast<uint32_t>(std::min<int64_t>(host.pool_pages, INT32_MAX));
    p.page_vecs = static_cast<uint32_t>(page_vecs);
    p.n_pages = static_cast<uint32_t>(n_pages);
    p.total_vecs = static_cast<uint32_t>(nl * n_pages * page_vecs);
    p.by_page = fast_div(p.page_vecs);
    p.by_count = fast_div(p.n_pages);
    const int64_t most = (int64_t(p.total_vecs) + kHostThreads - 1) / kHostThreads;
    const int groups = !to_host ? kInGroups
                       : paged  ? kPagedOutGroups
                                : (page_bytes < kLinkPageBytes ? 2 : 1) * kOutGroups;
    const dim3 grid(static_cast<uint32_t>(std::min<int64_t>(groups, most)));
    const void* fn;
    void* args[] = {&p};
    if (paged) {
      fn = to_host ? reinterpret_cast<const void*>(&host_leg_kernel<true, true>)
                   : reinterpret_cast<const void*>(&host_leg_kernel<false, true>);
    } else if (pool.host_ids == nullptr) {
      fn = to_host ? reinterpret_cast<const void*>(&host_leg_kernel<true, false>)
                   : reinterpret_cast<const void*>(&host_leg_kernel<false, false>);
    } else {
      memcpy(q.ids, pool.host_ids, n_pages * sizeof(int32_t));
      args[0] = &q;
      fn = to_host ? reinterpret_cast<const void*>(&host_leg_inline_kernel<true>)
                   : reinterpret_cast<const void*>(&host_leg_inline_kernel<false>);
    }
    // The launch records the event itself: a record behind it would be a packet
    // of its own, with a wait around it.  Measured on MI355X, a pair of legs
    // that each end with a record of the caller's: 4 us longer with the event
    // here, 9 with a record.
    if (done != nullptr && l0 + nl == num_layers)
      PACE_KV_TRY(hip_status(hipExtLaunchKernel(fn, grid, dim3(kHostThreads), args, 0, stream, nullptr, done, 0),
                             "host leg launch"));
    else
      PACE_KV_TRY(hip_status(hipLaunchKernel(fn, grid, dim3(kHostThreads), args, 0, stream), "host leg launch"));
  }
  return PACE_KV_OK;
}

int launch_host_leg(const Side& pool, char* host, bool to_host, int num_layers, int64_t n_pages, int64_t page_bytes,
                    int32_t* err_count, hipStream_t stream, hipEvent_t done) {
  std::vector<const char*> buf(std::max(num_layers, 0));
  buffer_layers(host, n_pages * page_bytes, num_layers, buf.data());
  return launch_host_leg(pool, Side{buf.data(), nullptr, n_pages}, to_host, num_layers, n_pages, page_bytes, err_count,
                         stream, done);
}

int buffered_copy(const Side& src, const Side& dst, char* buffer, int64_t buffer_layer_stride, int buffer_layers,
                  int num_layers, int64_t n_pages, int64_t page_bytes, int32_t* err_count, hipStream_t stream) {
  if (num_layers == 0 || n_pages == 0) return PACE_KV_OK;
  PACE_KV_TRY(check_layers(src.layers, num_layers, "source"));
  PACE_KV_TRY(check_layers(dst.layers, num_layers, "destination"));
  const int nb = buffer_layers < num_layers ? buffer_layers : num_layers;
  // A pack reads every source page before the unpack writes the first
  // destination page, so the two steps also serve pools that share memory (and
  // a buffer inside a pool); the tee does not, and needs all three apart.
  bool tee = page_bytes > 0 && src.pool_pages >= 0 && dst.pool_pages >= 0 &&
             src.pool_pages <= INT64_MAX / 4 / page_bytes && dst.pool_pages <= INT64_MAX / 4 / page_bytes;
  if (tee) {
    const int64_t sb = src.pool_pages * page_bytes, db = dst.pool_pages * page_bytes;
    const char* const lo = buffer;
    const char* const hi = buffer + (nb - 1) * buffer_layer_stride + n_pages * page_bytes;
    tee = disjoint(src.layers, sb, dst.layers, db, num_layers);
    for (int l = 0; l < num_layers && tee; ++l)
      tee = (src.layers[l] + sb <= lo || hi <= src.layers[l]) && (dst.layers[l] + db <= lo || hi <= dst.layers[l]);
  }
  std::vector<const char*> buf;
  if (!tee) {
    buf.resize(nb);
    pace_kv::buffer_layers(buffer, buffer_layer_stride, nb, buf.data());
  }
  for (int l0 = 0; l0 < num_layers; l0 += nb) {
    const int nl = num_layers - l0 < nb ? num_layers - l0 : nb;
    const Side s{src.layers + l0, src.ids, src.pool_pages, src.host_ids};
    const Side d{dst.layers + l0, dst.ids, dst.pool_pages, dst.host_ids};
    if (tee) {
      const Tee t{buffer, buffer_layer_stride};
      PACE_KV_TRY(launch_page_copy(s, d, nl, n_pages, page_bytes, err_count, stream, StorePolicy::kStream, &t));
      continue;
    }
    const Side b{buf.data(), nullptr, n_pages};
    PACE_KV_TRY(launch_page_copy(s, b, nl, n_pages, page_bytes, err_count, stream, StorePolicy::kPack));
    PACE_KV_TRY(launch_page_copy(b, d, nl, n_pages, page_bytes, err_count, stream));
  }
  return PACE_KV_OK;
}

int pack(const void* const* src_layers, int num_layers, int64_t pool_pages, const IdList& ids, int64_t n_pages,
         int64_t page_bytes, void* out, int64_t out_layer_stride, int32_t* err_count, hipStream_t stream) {
  if (num_layers < 0) return fail(PACE_KV_EINVAL, "num_layers must be >= 0");
  if (num_layers == 0 || n_pages == 0) return PACE_KV_OK;
  if (ids.null() || out == nullptr) return fail(PACE_KV_EINVAL, "pack: NULL page_ids or out");
  if (n_pages > 0 && page_bytes > 0 &&
      (n_pages > INT64_MAX / page_bytes || out_layer_stride < n_pages * page_bytes))
    return fail(PACE_KV_ERANGE, "pack: out_layer_stride %lld < n_pages*page_bytes",
                (long long)out_layer_stride);
  if (out_layer_stride % 16 != 0) return fail(PACE_KV_EINVAL, "pack: out_layer_stride not a multiple of 16");
  std::vector<const char*> buf(num_layers);
  buffer_layers(out, out_layer_stride, num_layers, buf.data());
  const Side src{reinterpret_cast<const char* const*>(src_layers), ids.dev, pool_pages, ids.host};
  const Side dst{buf.data(), nullptr, n_pages};
  return launch_page_copy(src, dst, num_layers, n_pages, page_bytes, err_count, stream, StorePolicy::kPack);
}

int unpack(const void* buf, int64_t buf_layer_stride, void* const* dst_layers, int num_layers, int64_t pool_pages,
           const IdList& ids, int64_t n_pages, int64_t page_bytes, int32_t* err_count, hipStream_t stream) {
  if (num_layers < 0) return fail(PACE_KV_EINVAL, "num_layers must be >= 0");
  if (num_layers == 0 || n_pages == 0) return PACE_KV_OK;
  if (ids.null() || buf == nullptr) return fail(PACE_KV_EINVAL, "unpack: NULL page_ids or buf");
  if (n_pages > 0 && page_bytes > 0 &&
      (n_pages > INT64_MAX / page_bytes || buf_layer_stride < n_pages * page_bytes))
    return fail(PACE_KV_ERANGE, "unpack: buf_layer_stride %lld < n_pages*page_bytes",
                (long long)buf_layer_stride);
  if (buf_layer_stride % 16 != 0) return fail(PACE_KV_EINVAL, "unpack: buf_layer_stride not a multiple of 16");
  std::vector<const char*> src_tab(num_layers);
  buffer_layers(buf, buf_layer_stride, num_layers, src_tab.data());
  const Side src{src_tab.data(), nullptr, n_pages};
  const Side dst{reinterpret_cast<const char* const*>(dst_layers), ids.dev, pool_pages, ids.host};
  return launch_page_copy(src, dst, num_layers, n_pages, page_bytes, err_count, stream);
}

// Resolves num_layers host or device layer pointers to the addresses the
// kernel uses, after checking that each lies in a registered allocation of
// the expected kind (pinned host memory mapped for the device, or device
// memory of the current device) that holds pool_bytes from the pointer on.
// Unregistered (pageable) host memory is rejected: the kernel would fault.
int resolve_layers(const void* const* layers, int num_layers, int64_t pool_bytes, bool host,
                   std::vector<const char*>& out, const char* what) {
  if (num_layers > 0 && layers == nullptr) return fail(PACE_KV_EINVAL, "%s: layer table is NULL", what);
  int dev = -1;
  PACE_KV_TRY(hip_status(hipGetDevice(&dev), "hipGetDevice"));
  out.resize(num_layers);
  for (int l = 0; l < num_layers; ++l) {
    const void* p = layers[l];
    hipPointerAttribute_t attr;
    memset(&attr, 0, sizeof(attr));
    hipError_t e = hipPointerGetAttributes(&attr, p);
    const hipMemoryType want = host ? hipMemoryTypeHost : hipMemoryTypeDevice;
    if (e != hipSuccess || attr.type != want || attr.devicePointer == nullptr) {
      (void)hipGetLastError();
      return fail(PACE_KV_EINVAL, "%s: layer %d is not %s memory", what, l,
                  host ? "pinned host (hipHostMalloc)" : "device");
    }
    if (!host && attr.device != dev)
      return fail(PACE_KV_EINVAL, "%s: layer %d lives on device %d, current device is %d", what, l,
                  attr.device, dev);
    // The allocation's range comes from hipMemGetAddressRange: on ROCm 7.2,
    // hipPointerGetAttribute(HIP_POINTER_ATTRIBUTE_RANGE_SIZE) reports the
    // size modulo 2^32 (a 4 GiB allocation reads 0), which would reject a
    // valid pool carved out of a large allocation or accept a short one.
    hipDeviceptr_t start = nullptr;
    size_t size = 0;
    e = hipMemGetAddressRange(&start, &size, const_cast<void*>(p));
    if (e != hipSuccess) {
      (void)hipGetLastError();
      return fail(PACE_KV_EINVAL, "%s: layer %d allocation range unknown", what, l);
    }
    const uintptr_t begin = reinterpret_cast<uintptr_t>(p);
    const uintptr_t lo = reinterpret_cast<uintptr_t>(start);
    if (begin < lo || begin - lo + static_cast<uint64_t>(pool_bytes) > size)
      return fail(PACE_KV_ERANGE, "%s: layer %d allocation holds %zu bytes from its start, "
                  "the pool needs %lld from offset %llu", what, l, size, (long long)pool_bytes,
                  (unsigned long long)(begin - lo));
    out[l] = static_cast<const char*>(attr.devicePointer);
  }
  return PACE_KV_OK;
}

int swap_copy(const void* const* src_layers, int64_t src_pool_pages, const int32_t* src_ids,
              bool src_host, const void* const* dst_layers, int64_t dst_pool_pages,
              const int32_t* dst_ids, bool dst_host, int num_layers, int64_t n_pages,
              int64_t page_bytes, int32_t* err_count, hipStream_t stream, const char* what) {
  if (num_layers < 0 || n_pages < 0) return fail(PACE_KV_EINVAL, "%s: negative size", what);
  if (num_layers == 0 || n_pages == 0) return PACE_KV_OK;
  if (src_ids == nullptr || dst_ids == nullptr) return fail(PACE_KV_EINVAL, "%s: NULL page ids", what);
  if (page_bytes <= 0 || page_bytes % kVecBytes != 0)
    return fail(PACE_KV_EINVAL, "%s: page_bytes must be a positive multiple of 16", what);
  if (src_pool_pages < 0 || dst_pool_pages < 0 || src_pool_pages > INT64_MAX / page_bytes ||
      dst_pool_pages > INT64_MAX / page_bytes)
    return fail(PACE_KV_EINVAL, "%s: bad pool size", what);
  std::vector<const char*> s, d;
  PACE_KV_TRY(resolve_layers(src_layers, num_layers, src_pool_pages * page_bytes, src_host, s, what));
  PACE_KV_TRY(resolve_layers(dst_layers, num_layers, dst_pool_pages * page_bytes, dst_host, d, what));
  const Side src{s.data(), src_ids, src_pool_pages}, dst{d.data(), dst_ids, dst_pool_pages};
  // The page copy is the faster one for short pages (see enum Shape; 512 B, 8
  // MiB: out 154 against 156 us by the host leg, in 162 against 158) and for
  // small swaps, where its waves carry one vector each: measured on MI355X,
  // pages of 8 KiB, alone, 64 KiB in 19.5 against 20.5 us, 256 KiB out 29.0
  // against 29.8 and in 30.8 against 30.6, 512 KiB in 37.1 against 35.6, 1 MiB
  // out 43.7 against 44.4 and in 49.6 against 46.4, 2 MiB out 63.1 against 62.4.
  const int64_t small_bytes = dst_host ? 2 << 20 : 512 << 10;
  if (page_bytes < kLinkPageBytes + (dst_host ? 1 : 0) || n_pages <= (small_bytes - 1) / page_bytes / num_layers)
    return launch_page_copy(src, dst, num_layers, n_pages, page_bytes, err_count, stream, StorePolicy::kLink);
  return launch_host_leg(dst_host ? src : dst, dst_host ? dst : src, dst_host, num_layers, n_pages, page_bytes,
                         err_count, stream);
}

}  // namespace pace_kv

using pace_kv::fail;
using pace_kv::Side;

extern "C" {

int pace_kv_abi_version(void) { return PACE_KV_ABI_VERSION; }

const char* pace_kv_last_error(void) { return pace_kv::g_last_error; }

int pace_kv_pack(const void* const* src_layers, int num_layers, int64_t pool_pages,
                 const int32_t* page_ids, int64_t n_pages, int64_t page_bytes, void* out,
                 int64_t out_layer_stride, int32_t* err_count, void* stream) {
  return pace_kv::pack(src_layers, num_layers, pool_pages, {page_ids, nullptr}, n_pages, page_bytes, out,
                       out_layer_stride, err_count, static_cast<hipStream_t>(stream));
}

int pace_kv_pack_inline(const void* const* src_layers, int num_layers, int64_t pool_pages,
                        const int32_t* host_page_ids, int64_t n_pages, int64_t page_bytes, void* out,
                        int64_t out_layer_stride, int32_t* err_count, void* stream) {
  return pace_kv::pack(src_layers, num_layers, pool_pages, {nullptr, host_page_ids}, n_pages, page_bytes, out,
                       out_layer_stride, err_count, static_cast<hipStream_t>(stream));
}

int pace_kv_unpack(const void* buf, int64_t buf_layer_stride, void* const* dst_layers,
                   int num_layers, int64_t pool_pages, const int32_t* page_ids, int64_t n_pages,
                   int64_t page_bytes, int32_t* err_count, void* stream) {
  return pace_kv::unpack(buf, buf_layer_stride, dst_layers, num_layers, pool_pages, {page_ids, nullptr}, n_pages,
                         page_bytes, err_count, static_cast<hipStream_t>(stream));
}

int pace_kv_unpack_inline(const void* buf, int64_t buf_layer_stride, void* const* dst_layers, int num_layers,
                          int64_t pool_pages, const int32_t* host_page_ids, int64_t n_pages, int64_t page_bytes,
                          int32_t* err_count, void* stream) {
  return pace_kv::unpack(buf, buf_layer_stride, dst_layers, num_layers, pool_pages, {nullptr, host_page_ids}, n_pages,
                         page_bytes, err_count, static_cast<hipStream_t>(stream));
}

int pace_kv_swap_out(const void* const* dev_layers, int64_t dev_pool_pages, const int32_t* dev_ids,
                     void* const* host_layers, int64_t host_pool_pages, const int32_t* host_ids,
                     int num_layers, int64_t n_pages, int64_t page_bytes, int32_t* err_count,
                     void* stream) {
  return pace_kv::swap_copy(dev_layers, dev_pool_pages, dev_ids, false,
                            reinterpret_cast<const void* const*>(host_layers), host_pool_pages,
                            host_ids, true, num_layers, n_pages, page_bytes, err_count,
                            static_cast<hipStream_t>(stream), "swap_out");
}

int pace_kv_swap_in(const void* const* host_layers, int64_t host_pool_pages, const int32_t* host_ids,
                    void* const* dev_layers, int64_t dev_pool_pages, const int32_t* dev_ids,
                    int num_layers, int64_t n_pages, int64_t page_bytes, int32_t* err_count,
                    void* stream) {
  return pace_kv::swap_copy(host_layers, host_pool_pages, host_ids, true,
                            reinterpret_cast<const void* const*>(dev_layers), dev_pool_pages,
                            dev_ids, false, num_layers, n_pages, page_bytes, err_count,
                            static_cast<hipStream_t>(stream), "swap_in");
}

int pace_kv_move(const void* const* src_layers, int64_t src_pool_pages, const int32_t* src_ids,
                 void* const* dst_layers, int64_t dst_pool_pages, const int32_t* dst_ids,
                 int num_layers, int64_t n_pages, int64_t page_bytes, int32_t* err_count,
                 void* stream) {
  if (num_layers < 0) return fail(PACE_KV_EINVAL, "num_layers must be >= 0");
  if (num_layers == 0 || n_pages == 0) return PACE_KV_OK;
  if (src_ids == nullptr || dst_ids == nullptr) return fail(PACE_KV_EINVAL, "move: NULL page ids");
  Side src{reinterpret_cast<const char* const*>(src_layers), src_ids, src_pool_pages};
  Side dst{reinterpret_cast<const char* const*>(dst_layers), dst_ids, dst_pool_pages};
  return pace_kv::launch_page_copy(src, dst, num_layers, n_pages, page_bytes, err_count,
                                   static_cast<hipStream_t>(stream));
}

int pace_kv_move_buffered(const void* const* src_layers, int64_t src_pool_pages, const int32_t* src_ids,
                          void* buffer, int64_t buffer_layer_stride, int buffer_layers,
                          void* const* dst_layers, int64_t dst_pool_pages, const int32_t* dst_ids,
                          int num_layers, int64_t n_pages, int64_t page_bytes, int32_t* err_count,
                          void* stream) {
  if (num_layers < 0 || n_pages < 0) return fail(PACE_KV_EINVAL, "move_buffered: negative size");
  if (num_layers == 0 || n_pages == 0) return PACE_KV_OK;
  if (src_ids == nullptr || dst_ids == nullptr || buffer == nullptr)
    return fail(PACE_KV_EINVAL, "move_buffered: NULL page ids or buffer");
  if (buffer_layers <= 0) return fail(PACE_KV_EINVAL, "move_buffered: buffer_layers must be >= 1");
  if (page_bytes <= 0 || page_bytes % 16 != 0)
    return fail(PACE_KV_EINVAL, "page_bytes must be a positive multiple of 16 (got %lld)", (long long)page_bytes);
  if (n_pages > INT64_MAX / page_bytes || buffer_layer_stride < n_pages * page_bytes || buffer_layer_stride % 16 != 0)
    return fail(PACE_KV_ERANGE, "move_buffered: buffer_layer_stride must be >= n_pages*page_bytes and a multiple of 16");
  Side src{reinterpret_cast<const char* const*>(src_layers), src_ids, src_pool_pages};
  Side dst{reinterpret_cast<const char* const*>(dst_layers), dst_ids, dst_pool_pages};
  return pace_kv::buffered_copy(src, dst, static_cast<char*>(buffer), buffer_layer_stride, buffer_layers, num_layers,
                                n_pages, page_bytes, err_count, static_cast<hipStream_t>(stream));
}

}  // extern "C"
