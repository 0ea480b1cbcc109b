// libaegkv: KV-cache block movement for MI355X (gfx950).
//
// Three operations, all pure byte movement (no arithmetic on the payload):
//   * swap-out  : device K/V tiles -> composite pages of a pinned host pool
//   * swap-in   : composite host pages -> device K/V tiles
//   * copy_blocks: device block -> device block, every backing tensor
//
// One "tile mover" kernel family does all of it. A work item is one chunk of
// one tile (a segment's bytes of one entry or pair): WG lanes move WG * 16 * U
// bytes with all U loads issued before the first store. Swaps are link-bound:
// a few persistent workgroups of 256 lanes stride over items in entry order,
// so that consecutive ones walk one composite host page in address order (good
// for PCIe write combining and host DRAM pages). Copies are HBM-bound: one
// workgroup of 64 or 256 lanes (1024 for whole tiles on masked streams) per
// item, segment by segment (copy_walk.h).
//
// Two host-transfer designs share the kernel:
//   DIRECT: the "host side" pointer is the pinned host pool itself (mapped
//           into the GPU address space by hipHostMalloc); the kernel's
//           loads/stores cross PCIe.
//   STAGED: the "host side" pointer is a contiguous device staging buffer
//           laid out like the host pages; hipMemcpyAsync moves merged runs
//           between staging and the host pool (the runtime runs each copy
//           as a blit kernel or on an SDMA engine).
//
// Entry-point contracts are in include/aegkv.h.

#include <hip/hip_runtime.h>
#include "aegkv.h"
#include "copy_walk.h"
#include "errors.h"
#include "staged_runs.h"

#include <algorithm>
#include <cstdarg>
#include <cstddef>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <mutex>
#include <vector>

// ---------------------------------------------------------------- errors --

namespace {
thread_local char g_err[512] = "";
}  // namespace

int aegkv_set_error(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

void aegkv_clear_error() { g_err[0] = '\0'; }

namespace {

#define fail aegkv_set_error

// Report a failed HIP call and clear the runtime's last-error state, which
// would otherwise make a later launch check report this failure again.
int hip_fail(hipError_t e, const char* what) {
  (void)hipGetLastError();
  return fail(static_cast<int>(e), "%s failed: %s (%d)", what, hipGetErrorString(e),
              static_cast<int>(e));
}

#define AEGKV_HIP(call)                          \
  do {                                           \
    hipError_t e_ = (call);                      \
    if (e_ != hipSuccess) return hip_fail(e_, #call); \
  } while (0)

// --------------------------------------------------------------- tunables --

struct Tunables {
  // Swap kernels: persistent workgroups in total, per direction, each lane
  // with swap_unroll 16 B loads in flight. The swaps are link-bound: about
  // 1 MiB in flight per direction saturates PCIe, and the few workgroups
  // leave the other CUs to concurrent copies. Two loads per lane with twice
  // the workgroups keep the same bytes in flight and share the link better
  // when both directions run at once (model switch 105 -> 103 ms), at the
  // same rate for one direction alone (57.1 / 57.5 GB/s).
  int64_t swap_out_workgroups = 64;
  int64_t swap_in_workgroups = 128;
  // Swap-out into an uncached pool: alone 64-224 workgroups all reach the
  // link rate, and beside a swap-in 112 leave the swap-in more of the link
  // (with 4 loads per lane: 32 -> 56 workgroups, 108.5 -> 105 ms). Into a
  // cached pool 64 stay best alone (56.6 GB/s; 55.8 at 112) and equal
  // beside a swap-in.
  int64_t swap_out_workgroups_uncached = 112;
  int64_t staging_bytes = int64_t(512) << 20;
  int64_t auto_d2h = AEGKV_MODE_DIRECT;
  int64_t auto_h2d = AEGKV_MODE_DIRECT;
  int64_t nt_stores = 1;
  int64_t copy_wgs_per_cu = 0;   // copy_blocks: 0 = one workgroup per work item
  int64_t copy_unroll = 0;       // copy_blocks: 0 = shape from the page size
  int64_t copy_lanes = 0;        // copy_blocks with copy_unroll: 256 or 1024 lanes (0 = 1024)
  int64_t swap_shape_auto = 0;   // swap kernels: 1 = page-sized shape as copy_blocks
  int64_t swap_unroll = 2;       // swap kernels: 16 B loads per lane (256-lane shape)
  int64_t staged_workgroups = 0; // STAGED gather/scatter grid: 0 = one workgroup per item
  int64_t staged_dma_streams = 2; // STAGED copies: library streams (<= 1: caller stream)
  // STAGED over library streams: two staging chunks in flight (bit 0
  // swap-out, bit 1 swap-in), so the gather or scatter of one chunk runs
  // while another chunk's copies use the link. Qwen3-4B, 1024 blocks (GB/s
  // out / in): one call at a time 43.4 / 50.9 -> 54.3 / 55.4; swap-out and
  // swap-in at once 174 -> 121 ms for a model switch; beside a GEMM the
  // swaps end at 52 / 56 ms instead of 74 / 105. Where the host enqueues
  // far ahead with block copies between the swaps, the runtime moved the
  // swap-out's copies to SDMA and it fell to 29 GB/s (35 one chunk at a
  // time); set bit 0 off for that pattern.
  int64_t staged_overlap = 3;
  int64_t staged_short_runs = 1;  // STAGED calls of short runs go DIRECT (runs_are_short)
  // copy_blocks, 1024-lane shapes with items of >= 32 KiB (a fixed unroll):
  // LDS reserved per workgroup so that one workgroup holds a CU (HBM copy
  // rate +1-5 % on 32-160 KiB tiles).
  int64_t copy_lds_bytes = int64_t(96) << 10;
  // copy_blocks: the order in which pairs reach the kernel (0: the caller's,
  // 1: by target id, 2: by source id; the checks make the result
  // order-free). The kernel's walk (CopyWalk) relies on target order to
  // write near by; see there for the rates.
  int64_t copy_order = 1;
};
Tunables g_tune;
std::mutex g_tune_mu;
constexpr int64_t kMaxLdsPerWorkgroup = int64_t(160) << 10;  // gfx950: 160 KiB per CU

// Environment overrides, read once per process: AEGKV_AUTO_D2H and
// AEGKV_AUTO_H2D ("direct" or "staged") choose what mode AUTO resolves to,
// AEGKV_STAGING_BYTES (>= 1 MiB) the STAGED chunk. An invalid value makes
// every entry point that moves data fail with AEGKV_EINVAL naming it.
std::once_flag g_env_once;
char g_env_err[256] = "";

void read_env() {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  auto mode = [](const char* name, int64_t* slot) {
    const char* v = std::getenv(name);
    if (!v || !*v) return;
    if (!std::strcmp(v, "direct")) *slot = AEGKV_MODE_DIRECT;
    else if (!std::strcmp(v, "staged")) *slot = AEGKV_MODE_STAGED;
    else std::snprintf(g_env_err, sizeof(g_env_err), "%s=%s: expected direct or staged", name, v);
  };
  mode("AEGKV_AUTO_D2H", &g_tune.auto_d2h);
  mode("AEGKV_AUTO_H2D", &g_tune.auto_h2d);
  const char* v = std::getenv("AEGKV_STAGING_BYTES");
  if (v && *v) {
    char* end = nullptr;
    const long long x = std::strtoll(v, &end, 10);
    if (*end != '\0' || x < (1ll << 20))
      std::snprintf(g_env_err, sizeof(g_env_err),
                    "AEGKV_STAGING_BYTES=%s: expected an integer >= 1048576", v);
    else
      g_tune.staging_bytes = x;
  }
}

int env_status() {
  std::call_once(g_env_once, read_env);
  return g_env_err[0] ? fail(AEGKV_EINVAL, "%s", g_env_err) : 0;
}

Tunables tunables() {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  return g_tune;
}

// ------------------------------------------------------ device descriptors --

struct SegDesc {            // one backing tensor
  char* base;
  int64_t page_bytes;
  int64_t host_offset;
  uint64_t owner_mask;
};
static_assert(sizeof(SegDesc) == 32, "SegDesc layout");

struct EntDesc {            // one swap entry, already resolved to sides
  int64_t dev_block;        // block id in every backing tensor
  int64_t host_slot;        // host block id (DIRECT) or staging slot (STAGED)
  int32_t group;
  int32_t first;            // first kernel block of the extent
  int32_t valid;            // kernel blocks in the extent
  int32_t pad;
};
static_assert(sizeof(EntDesc) == 32, "EntDesc layout");

struct PairDesc {
  int64_t src;
  int64_t dst;
};

struct CopySeg {            // one backing tensor of a block copy
  const char* src;          // source cache's tensor
  char* dst;                // target cache's tensor (== src within one cache)
  int64_t page_bytes;
  int64_t pad;
};
static_assert(sizeof(CopySeg) == 32, "CopySeg layout");
static_assert(sizeof(PairDesc) == 16, "PairDesc layout (descriptors are whole 16-byte words)");

typedef unsigned int v4u __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) v4u gv4u;  // global (VM) address space
typedef v4u v4u_any __attribute__((aligned(1)));     // 16 bytes at any address
typedef __attribute__((address_space(1))) v4u_any gv4u_any;
typedef __attribute__((address_space(1))) char gchar;

// A kernel "shape": WG lanes per workgroup, U 16-byte loads in flight per
// lane, so one work item (chunk) is WG * 16 * U bytes.
template <int WG, int U>
struct Shape {
  static constexpr int kLanes = WG;
  static constexpr int kLoads = U;
  static constexpr int64_t kChunk = int64_t(WG) * 16 * U;
};

// Where the 16-byte words of one chunk go and how they are stored; `dst` and
// `nbytes` are the same for the whole workgroup.
//   kPlain:     targets in the host pool
//   kStreaming: non-temporal, targets in HBM
//   kThrough:   also at device scope, so that the L2 writes whole lines through
//               as they come instead of keeping them for a later write-back.
//               Only buffer stores can be told so.
// Copies of random blocks, streaming -> through (TB/s, read plus written): 16
// KiB pages 5.88 -> 5.99, 20 KiB 5.90 -> 5.98, 32 KiB 6.04 -> 6.12, 64 KiB 6.27
// -> 6.42, 160 KiB 6.40 -> 6.57; plain stores 5.1-5.6. The scope bits of the
// loads change nothing. Tiles that
// do not begin and end on 128-byte lines write lines in parts, and lose by it
// (16,388-byte pages 5.7 -> 5.2, 16,400 5.5 -> 5.4), as do shapes with several
// loads per lane on few CUs (8 of 32 per XCD: 3.14 -> 3.04): these stay
// streaming.
enum StoreKind { kPlain, kStreaming, kThrough };
constexpr int kBufferNt = 2, kBufferDeviceScope = 16;  // cache bits of a buffer store
constexpr int kRawBufferWord3 = 0x00027000;            // untyped 32-bit data, no swizzle

template <StoreKind K>
struct Words {
  gv4u* d;
  __device__ __forceinline__ Words(char* dst, uint32_t, bool) : d((gv4u*)dst) {}
  __device__ __forceinline__ void put(uint32_t i, v4u x) const {
    if (K == kStreaming)
      __builtin_nontemporal_store(x, d + i);
    else
      d[i] = x;
  }
};

template <>
struct Words<kThrough> {
  __amdgpu_buffer_rsrc_t r;
  bool lines;  // the tile is made of whole 128-byte lines
  __device__ __forceinline__ Words(char* dst, uint32_t nbytes, bool whole_lines)
      : r(__builtin_amdgcn_make_buffer_rsrc(dst, 0, static_cast<int>(nbytes), kRawBufferWord3)),
        lines(whole_lines) {}
  __device__ __forceinline__ void put(uint32_t i, v4u x) const {
    const int at = static_cast<int>(i * 16u);
    if (lines)
      __builtin_amdgcn_raw_buffer_store_b128(x, r, at, 0, kBufferNt | kBufferDeviceScope);
    else
      __builtin_amdgcn_raw_buffer_store_b128(x, r, at, 0, kBufferNt);
  }
};

__device__ __forceinline__ bool whole_lines(const char* tile, int64_t bytes) {
  return ((reinterpret_cast<uintptr_t>(tile) | static_cast<uintptr_t>(bytes)) & 127u) == 0;
}

// The stores of a shape: through the L2 with one load per lane.
template <int WG, int U, bool NT_STORE>
using ShapeWords = Words<!NT_STORE ? kPlain : U == 1 && WG <= 256 ? kThrough : kStreaming>;

// The guarded U loads of a tail chunk, all issued before the first store.
// Recursion keeps every value in registers of its own: an array of U values
// filled under conditions became one wide value that was copied whole at each
// (252 VGPRs for U = 8, and with 1024 lanes scratch memory: 128 KiB tiles
// copied at 1.3 TB/s).
//
// Load and store stand under conditions of their own, so the compiler takes a
// tail's load for possibly unfinished behind them, and the loops over items of
// swaps and weight loads wait for all of an item's memory operations, its
// stores among them, where they next use the register: before the next item's
// loads. That wait is wanted. Without it (the store nested under
// its load's condition) the same grid keeps twice the requests to the host in
// the memory queues, and what else uses HBM or the link waits behind them: a
// copy beside a swap-out of 24 / 32 workgroups runs at 6.0 / 5.8 TB/s, 4.5 / 2.1
// without; beside a swap-in of 48 at 5.9, 2.2 without; beside both at 24 / 24 at
// 5.9, 3.6 without. Both directions at 16 / 16 reach 92-95 GB/s (88-92), a switch
// at the default grids 11.6 ms (11.7), with a weight load beside it 22.4 (23.2).
// It costs swaps both ways at 20 to 48 workgroups of two loads, or 12 to 16 of
// four, with nothing beside them (24 / 24 14.9 ms a switch, 12.9 without; 32 / 32
// 13.6, 12.4), and one direction over 4 to 8 workgroups (4: 32 GB/s, 40 without).
// Asked for in the source right before the loads, behind the addresses, it made
// both ways at 12 to 32 workgroups another 4-9 % slower.
template <int WG, int U, typename Out>
__device__ __forceinline__ void move_tail16(const gv4u* s, const Out& d, uint32_t i,
                                            uint32_t n16) {
  v4u x;
  if (i < n16) x = __builtin_nontemporal_load(s + i);
  if constexpr (U > 1) move_tail16<WG, U - 1>(s, d, i + WG, n16);
  if (i < n16) d.put(i, x);
}

// Move nbytes (multiple of 16, at most one chunk) with 16 B per lane. A full
// chunk issues all U loads back to back before the first store; only a tail
// chunk pays for per-load guards.
template <int WG, int U, bool NT_STORE>
__device__ __forceinline__ void move_chunk16(const char* src, char* dst, uint32_t nbytes,
                                             bool lines = false) {
  const gv4u* s = (const gv4u*)src;  // generic -> global address space
  const ShapeWords<WG, U, NT_STORE> d(dst, nbytes, lines);
  const uint32_t tid = threadIdx.x;
  if (nbytes != static_cast<uint32_t>(Shape<WG, U>::kChunk)) {
    move_tail16<WG, U>(s, d, tid, nbytes >> 4);
    return;
  }
  v4u r[U];
#pragma unroll
  for (int u = 0; u < U; ++u) r[u] = __builtin_nontemporal_load(s + tid + u * WG);
#pragma unroll
  for (int u = 0; u < U; ++u) d.put(tid + u * WG, r[u]);
}

// A move guard is a word a stream's fence waits set when they give up or
// see a failed source (aegkv_fence_wait). Kernels over full grids
// (migrations, STAGED gathers and scatters) move nothing when the word that
// their descriptor's staging kernel left is set: that kernel reads the guard
// once per launch, at system scope (it may live in pinned host memory), into
// a device word behind the descriptor. DIRECT swaps, over a few persistent
// workgroups, read the guard themselves (guard_set_at_source).
//
// Read by every wave of the moving kernel instead, a guard in pinned host
// memory costs 83-88 ns per wave, one after another whatever the grid: a
// 12,288-workgroup migration (1.6 GB) took 17.3 ms instead of 0.28, a STAGED
// gather of 57,600 workgroups 19.1 ms instead of 0.15.
__device__ __forceinline__ bool guard_set(const uint64_t* __restrict__ seen) {
  return seen != nullptr && *seen != 0;
}

// Bring a call's descriptor from the pinned ring to the device (16 B per
// lane; one launch costs the host the 3 us a small runtime copy does) and
// take the guard's value along.
constexpr uint32_t kStageLanes = 256;

__global__ __launch_bounds__(kStageLanes) void desc_stage_kernel(const v4u* __restrict__ host,
                                                                 v4u* __restrict__ dev,
                                                                 uint32_t words,
                                                                 const uint64_t* guard,
                                                                 uint64_t* seen) {
  const uint32_t i = blockIdx.x * kStageLanes + threadIdx.x;
  if (i < words) dev[i] = host[i];
  if (i == 0 && guard != nullptr)
    *seen = __hip_atomic_load(guard, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Move nbytes from any address to any other: 16 B per lane, loads at the
// source's own alignment (the hardware takes any) and stores on the target's
// 16-byte words, with single bytes at both ends. 16,388-byte pages, one byte
// per lane -> this: block copy 1.7 -> 5.7 TB/s (read plus written), swap-out
// 34.9 (uncached pool 13.8) -> 51.2 GB/s, swap-in 24.6 -> 52.1, a weight load
// at odd addresses 24.7 -> 55.4.
template <int WG, int U, bool NT_STORE>
__device__ __forceinline__ void move_any(const char* src, char* dst, uint32_t nbytes) {
  const uint32_t tid = threadIdx.x;
  uint32_t head = static_cast<uint32_t>(-reinterpret_cast<uintptr_t>(dst)) & 15u;
  if (head > nbytes) head = nbytes;
  const uint32_t n16 = (nbytes - head) >> 4;
  // lanes 0-15 carry the bytes before the first whole word, lanes 16-31
  // those behind the last one
  const uint32_t at = tid < 16 ? tid : head + n16 * 16 + (tid - 16);
  const bool edge = tid < 16 ? tid < head : tid < 32 && at < nbytes;
  char b = 0;
  if (edge) b = ((const gchar*)src)[at];
  const gchar* s = (const gchar*)src + head;
  const Words<NT_STORE ? kStreaming : kPlain> d(dst + head, n16 * 16u, false);
  uint32_t i = tid;
  for (; i + (U - 1) * WG < n16; i += U * WG) {
    v4u r[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      r[u] = __builtin_nontemporal_load((const gv4u_any*)(s + (i + u * WG) * 16u));
#pragma unroll
    for (int u = 0; u < U; ++u) d.put(i + u * WG, r[u]);
  }
  for (; i < n16; i += WG)
    d.put(i, __builtin_nontemporal_load((const gv4u_any*)(s + i * 16u)));
  if (edge) ((gchar*)dst)[at] = b;
}

// A guard in the caller's own place, pinned host memory perhaps: one lane of
// each workgroup reads it (83 ns a read, one after another: for grids of a
// few workgroups). Every lane of the workgroup gets the same answer.
__device__ __forceinline__ bool guard_set_at_source(const uint64_t* guard) {
  if (guard == nullptr) return false;
  __shared__ uint32_t set;
  if (threadIdx.x == 0)
    set = __hip_atomic_load(guard, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) != 0;
  __syncthreads();
  return set != 0;
}

// What a swap kernel needs beside its tables.
struct SwapWalk {
  char* host_base;
  int64_t host_stride, host_rank_offset;
  uint32_t num_segs, num_items, chunks_per_tile;
};

// Swap tile mover. Item w -> (entry e, segment s, chunk c), entry-major.
// TO_HOST: device tile -> host side; otherwise host side -> device tile.
// The host keeps num_items + gridDim.x below 2^32 (launch_items), so the
// 32-bit grid-stride loop never wraps.
template <int WG, int U, bool TO_HOST, bool VEC, bool NT_STORE, typename Segs, typename Ents,
          typename Kpp>
__device__ __forceinline__ void swap_items(Segs segs, Ents ents, Kpp kpp, const SwapWalk& k) {
  constexpr int64_t kChunk = Shape<WG, U>::kChunk;
  for (uint32_t w = blockIdx.x; w < k.num_items; w += gridDim.x) {
    const uint32_t tile = w / k.chunks_per_tile;
    const uint32_t c = w - tile * k.chunks_per_tile;
    const uint32_t e = tile / k.num_segs;
    const uint32_t s = tile - e * k.num_segs;
    const int32_t group = ents[e].group;
    const int64_t page = segs[s].page_bytes;
    if (!((segs[s].owner_mask >> group) & 1ull)) continue;
    const int64_t unit = page / kpp[group];
    const int64_t off = unit * ents[e].first;
    const int64_t len = unit * ents[e].valid;
    char* dev = segs[s].base + ents[e].dev_block * page + off;
    char* host = k.host_base + ents[e].host_slot * k.host_stride + k.host_rank_offset +
                 segs[s].host_offset + off;
    const char* src = TO_HOST ? dev : host;
    char* dst = TO_HOST ? host : dev;
    if (VEC) {
      const int64_t begin = static_cast<int64_t>(c) * kChunk;
      if (begin >= len) continue;
      const uint32_t nbytes =
          static_cast<uint32_t>((len - begin < kChunk) ? (len - begin) : kChunk);
      move_chunk16<WG, U, NT_STORE>(src + begin, dst + begin, nbytes);
    } else {
      const Extent x = any_chunk<kChunk>(dst, len, c, k.chunks_per_tile - 1);
      if (x.nbytes) move_any<WG, U, NT_STORE>(src + x.begin, dst + x.begin, x.nbytes);
    }
  }
}

// `seen`: the guard's value as the descriptor's staging kernel found it (a
// STAGED gather or scatter, over a full grid); `guard`: the guard itself (a
// DIRECT swap, over a few persistent workgroups). Either may be null.
template <int WG, int U, bool TO_HOST, bool VEC, bool NT_STORE>
__global__ __launch_bounds__(WG) void swap_tiles_kernel(
    const SegDesc* __restrict__ segs, const EntDesc* __restrict__ ents,
    const int64_t* __restrict__ kpp, SwapWalk walk, const uint64_t* seen,
    const uint64_t* guard) {
  if (guard_set(seen) || guard_set_at_source(guard)) return;
  swap_items<WG, U, TO_HOST, VEC, NT_STORE>(segs, ents, kpp, walk);
}

// A short DIRECT swap's whole descriptor in the kernel's own arguments, as
// InlineCopy below: one launch. 72 segments and 45 entries.
//
// While the link is full, whatever the GPU fetches from host memory waits
// behind the transfers (100-200 us a time), a launch's packet and a staged
// descriptor among them, so a launch less counts double there.
constexpr uint32_t kInlineSwapBytes = 3776;
typedef __attribute__((address_space(4))) const char kernarg_char;
struct alignas(16) InlineSwap {
  SwapWalk walk;
  uint32_t kpp_offset, ent_offset;
  uint32_t pad;
  const uint64_t* guard;
  unsigned char data[kInlineSwapBytes];
};
static_assert(offsetof(InlineSwap, data) % 16 == 0 && sizeof(InlineSwap) <= 3840,
              "InlineSwap layout: 4 KiB of arguments, 256 bytes of them hidden ones");

template <bool TO_HOST, bool VEC, bool NT_STORE>
__global__ __launch_bounds__(256) void swap_inline_kernel(InlineSwap a) {
  typedef __attribute__((address_space(4))) const SegDesc kernarg_seg_desc;
  typedef __attribute__((address_space(4))) const EntDesc kernarg_ent;
  typedef __attribute__((address_space(4))) const int64_t kernarg_i64;
  if (guard_set_at_source(a.guard)) return;
  kernarg_char* data =
      (kernarg_char*)__builtin_amdgcn_kernarg_segment_ptr() + offsetof(InlineSwap, data);
  swap_items<256, 2, TO_HOST, VEC, NT_STORE>((kernarg_seg_desc*)data,
                                             (kernarg_ent*)(data + a.ent_offset),
                                             (kernarg_i64*)(data + a.kpp_offset), a.walk);
}

// The classes of a walk behind the first, a kernel's last argument: none
// (OneClass), or CopyClasses, read where the launch put them (indexed as a
// parameter they would be copied to scratch memory). Kernels for caches with
// one page size are built without them: looking for the class, and with 224
// bytes more the arguments and the grid's size in several lines of 64 bytes,
// took 0.1-0.5 % of a copy and 2-4 % of a probe.
struct CopyArgs {
  const CopySeg* segs;
  const PairDesc* pairs;
  CopyWalk walk;
  const uint64_t* guard;  // a probe's sink and magic
  CopyClasses classes;
};
static_assert(offsetof(CopyArgs, classes) == 64, "CopyArgs layout");
typedef __attribute__((address_space(4))) const CopyClass kernarg_class;

template <typename Classes>
__device__ __forceinline__ auto argument_classes() {
  if constexpr (sizeof(Classes) == sizeof(CopyClasses))
    return (kernarg_class*)((kernarg_char*)__builtin_amdgcn_kernarg_segment_ptr() +
                            offsetof(CopyArgs, classes));
  else
    return OneClass{};
}

// copy_blocks: one item is one chunk of one (segment, pair) tile. The host
// keeps num_items + gridDim.x below 2^32 (launch_items).
template <int WG, int U, bool VEC, bool NT_STORE, typename Segs, typename Pairs,
          typename Classes>
__device__ __forceinline__ void copy_items(Segs segs, Pairs pairs, const CopyWalk& walk,
                                           Classes classes) {
  constexpr int64_t kChunk = Shape<WG, U>::kChunk;
  for (uint32_t w = blockIdx.x; w < walk.num_items; w += gridDim.x) {
    const CopyItem it = copy_item(walk, classes, w);
    const int64_t src_block = pairs[it.pair].src, dst_block = pairs[it.pair].dst;
    const int64_t page = segs[it.segment].page_bytes;
    const char* src = segs[it.segment].src + src_block * page;
    char* dst = segs[it.segment].dst + dst_block * page;
    // both descriptor entries are wanted at once, not the addresses only
    // behind a branch on the page's size (two trips through the scalar cache)
    asm("" : "+s"(src), "+s"(dst));
    if (VEC) {
      const int64_t begin = static_cast<int64_t>(it.chunk) * kChunk;
      if (begin >= page) continue;
      const uint32_t nbytes =
          static_cast<uint32_t>((page - begin < kChunk) ? (page - begin) : kChunk);
      move_chunk16<WG, U, NT_STORE>(src + begin, dst + begin, nbytes, whole_lines(dst, page));
    } else {
      const Extent x = any_chunk<kChunk>(dst, page, it.chunk, it.last);
      if (x.nbytes) move_any<WG, U, NT_STORE>(src + x.begin, dst + x.begin, x.nbytes);
    }
  }
}

template <int WG, int U, bool VEC, bool NT_STORE, typename Classes>
__global__ __launch_bounds__(WG) void copy_blocks_kernel(const CopySeg* __restrict__ segs,
                                                         const PairDesc* __restrict__ pairs,
                                                         CopyWalk walk,
                                                         const uint64_t* __restrict__ guard,
                                                         Classes) {
  if (guard_set(guard)) return;
  copy_items<WG, U, VEC, NT_STORE>(segs, pairs, walk, argument_classes<Classes>());
}

// A short copy's whole descriptor (segment table, classes of the walk behind
// the first, pair table) in the kernel's own arguments, which the runtime copies when the launch is
// enqueued (a graph that captures it keeps its own copy) and every workgroup
// reads through the scalar cache: the call is one launch, with no upload in
// front of it, no ring region and no event behind it.
// Copying one block of 72 segments takes the host 8 us through the library
// instead of 14 and the caller 19 instead of 22 until it is done; 63 blocks of
// 72 x 32 KiB take 54 us a pass instead of 61.
// kInlineBytes keeps all arguments, hidden ones among them, within 4 KiB: 72
// segments and 94 pairs.
constexpr uint32_t kInlineBytes = 3808;
struct alignas(32) InlineCopy {
  CopyWalk walk;
  uint32_t class_offset, pair_offset;  // from data
  unsigned char data[kInlineBytes];
};
static_assert(offsetof(InlineCopy, data) % alignof(CopyClass) == 0 && sizeof(InlineCopy) <= 3840,
              "InlineCopy layout: 4 KiB of arguments, 256 bytes of them hidden ones");
typedef __attribute__((address_space(4))) const CopySeg kernarg_seg;
typedef __attribute__((address_space(4))) const PairDesc kernarg_pair;

template <int WG, bool VEC, bool NT_STORE, typename Classes>
__global__ __launch_bounds__(WG) void copy_blocks_inline_kernel(InlineCopy a) {
  // the tables are indexed where the launch put them: `a` is the kernel's
  // only argument and starts its argument segment
  kernarg_char* data =
      (kernarg_char*)__builtin_amdgcn_kernarg_segment_ptr() + offsetof(InlineCopy, data);
  kernarg_seg* segs = (kernarg_seg*)data;
  kernarg_pair* pairs = (kernarg_pair*)(data + a.pair_offset);
  if constexpr (sizeof(Classes) == sizeof(CopyClasses))
    copy_items<WG, 1, VEC, NT_STORE>(segs, pairs, a.walk, (kernarg_class*)(data + a.class_offset));
  else
    copy_items<WG, 1, VEC, NT_STORE>(segs, pairs, a.walk, OneClass{});
}

// Measurement twins of copy_blocks_kernel (aegkv_copy_probe): the same
// item walk over the same tiles and the same grid, either reading the
// source tiles only (PROBE_READ; the loads are XOR-folded and the fold is
// stored only if it equals `magic`, so no load can be dropped and nearly
// nothing is written) or writing a fixed pattern to the target tiles only
// (PROBE_WRITE). Their rates bound what a copy of that tile pattern can
// reach on the memory system at hand.
constexpr int PROBE_READ = 1;
constexpr int PROBE_WRITE = 2;

template <int WG, int U, int KIND, bool NT_STORE, typename Classes>
__global__ __launch_bounds__(WG) void copy_probe_kernel(const CopySeg* __restrict__ segs,
                                                        const PairDesc* __restrict__ pairs,
                                                        CopyWalk walk, uint32_t* sink,
                                                        uint32_t magic, Classes) {
  constexpr int64_t kChunk = Shape<WG, U>::kChunk;
  const uint32_t tid = threadIdx.x;
  v4u acc = {0u, 0u, 0u, 0u};
  const v4u pattern = {tid, blockIdx.x, 0x5a5a5a5au, magic};
  for (uint32_t w = blockIdx.x; w < walk.num_items; w += gridDim.x) {
    const CopyItem it = copy_item(walk, argument_classes<Classes>(), w);
    const PairDesc pr = pairs[it.pair];
    const CopySeg seg = segs[it.segment];
    const int64_t begin = static_cast<int64_t>(it.chunk) * kChunk;
    if (begin >= seg.page_bytes) continue;
    const uint32_t n16 = static_cast<uint32_t>(
        ((seg.page_bytes - begin < kChunk) ? (seg.page_bytes - begin) : kChunk) >> 4);
    if (KIND == PROBE_READ) {
      const gv4u* src = (const gv4u*)(seg.src + pr.src * seg.page_bytes + begin);
      v4u r[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t i = tid + u * WG;
        r[u] = i < n16 ? __builtin_nontemporal_load(src + i) : v4u{0u, 0u, 0u, 0u};
      }
#pragma unroll
      for (int u = 0; u < U; ++u) acc ^= r[u];
    } else {
      char* tile = seg.dst + pr.dst * seg.page_bytes;
      const ShapeWords<WG, U, NT_STORE> dst(tile + begin, n16 * 16u,
                                            whole_lines(tile, seg.page_bytes));
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t i = tid + u * WG;
        if (i < n16) dst.put(i, pattern);
      }
    }
  }
  if (KIND == PROBE_READ) {
    const uint32_t x = acc.x ^ acc.y ^ acc.z ^ acc.w;
    if (x == magic) sink[0] = x;
  }
}

// One contiguous slice of a weight load: `bytes` bytes from src to dst; its
// work items start at first_item.
struct SliceDesc {
  char* dst;
  const char* src;
  int64_t bytes;
  int64_t first_item;
};
static_assert(sizeof(SliceDesc) == 32, "SliceDesc layout");

// Contiguous slices, host to device (weight loads): item w -> the slice
// that holds it (the last one whose first_item <= w, found by a binary
// search over the uniform descriptor) and its chunk in that slice. Empty
// slices are dropped on the host, so every slice has at least one item.
template <int WG, int U, bool VEC, bool NT_STORE>
__global__ __launch_bounds__(WG) void slices_kernel(const SliceDesc* __restrict__ slices,
                                                    uint32_t num_slices, uint32_t num_items) {
  constexpr int64_t kChunk = Shape<WG, U>::kChunk;
  for (uint32_t w = blockIdx.x; w < num_items; w += gridDim.x) {
    uint32_t lo = 0, hi = num_slices - 1;
    while (lo < hi) {
      const uint32_t mid = (lo + hi + 1) >> 1;
      if (slices[mid].first_item <= static_cast<int64_t>(w))
        lo = mid;
      else
        hi = mid - 1;
    }
    const SliceDesc sl = slices[lo];
    const uint32_t c = static_cast<uint32_t>(static_cast<int64_t>(w) - sl.first_item);
    if (VEC) {
      const int64_t begin = static_cast<int64_t>(c) * kChunk;
      const uint32_t nbytes =
          static_cast<uint32_t>((sl.bytes - begin < kChunk) ? (sl.bytes - begin) : kChunk);
      move_chunk16<WG, U, NT_STORE>(sl.src + begin, sl.dst + begin, nbytes);
    } else {
      const uint32_t last = static_cast<uint32_t>((sl.bytes - 1) / kChunk);
      const Extent x = any_chunk<kChunk>(sl.dst, sl.bytes, c, last);
      if (x.nbytes) move_any<WG, U, NT_STORE>(sl.src + x.begin, sl.dst + x.begin, x.nbytes);
    }
  }
}

// A part of an allocation-free copy's descriptor in one launch's kernel
// arguments, packed, and unpacked into the tables by the launch: 16 bytes a
// segment (address and page), then 8 bytes a pair (32-bit ids; 16 bytes where
// a cache has more blocks than those name). The runtime copies a launch's
// arguments when the launch is enqueued, and a graph that captures the launch
// keeps its own copy, so the host buffer they came from is free as soon as the
// launch call returns.
//
// One such launch takes 4.9 us on the stream whatever it carries, so they
// carry all that 4 KiB of arguments hold (hidden ones among them): 72
// segments and 600 pairs go out in two launches, where 2 KiB of finished
// table entries a launch took six.
constexpr uint32_t kFillBytes = 3776;
constexpr uint32_t kFillLanes = 512;
struct FillSeg {
  char* base;
  int64_t page_bytes;
};
struct FillPair {
  uint32_t src, dst;
};
struct alignas(16) FillArgs {
  CopySeg* segs;
  PairDesc* pairs;
  uint32_t num_segs;
  uint32_t num_pairs;
  uint32_t wide;  // pairs are PairDesc
  uint32_t pad;
  unsigned char data[kFillBytes];
};
static_assert(kFillBytes / sizeof(FillPair) <= kFillLanes &&
              offsetof(FillArgs, data) % 16 == 0 && kFillBytes % 16 == 0, "FillArgs layout");

__global__ __launch_bounds__(kFillLanes) void desc_fill_kernel(FillArgs a) {
  const uint32_t i = threadIdx.x;
  if (i < a.num_segs) {
    const FillSeg s = reinterpret_cast<const FillSeg*>(a.data)[i];
    a.segs[i] = CopySeg{s.base, s.base, s.page_bytes, 0};
  }
  const unsigned char* pairs = a.data + a.num_segs * sizeof(FillSeg);
  if (i < a.num_pairs) {
    if (a.wide) {
      a.pairs[i] = reinterpret_cast<const PairDesc*>(pairs)[i];
    } else {
      const FillPair p = reinterpret_cast<const FillPair*>(pairs)[i];
      a.pairs[i] = PairDesc{p.src, p.dst};
    }
  }
}

// Shapes that move a whole tile per workgroup (swaps asked for them, copies
// of more chunks than one launch holds). 1024-lane shapes move 16 KiB rows; a
// tile that is a multiple of 16 KiB gets the largest U dividing its row
// count, so one workgroup moves a whole tile (up to 160 KiB) with no tail
// chunk. Smaller tiles use 256-lane (4 KiB) rows.
struct ShapeSel {
  int wg;
  int u;
  int64_t chunk() const { return int64_t(wg) * 16 * u; }
};

ShapeSel auto_shape(int64_t page) {
  static const int kBigU[] = {10, 8, 6, 5, 4, 3, 2, 1};
  const int64_t row = 1024 * 16;
  if (page >= row && page % row == 0) {
    const int64_t rows = page / row;
    for (int u : kBigU)
      if (rows % u == 0) return {1024, u};
  }
  if (page >= row) return {1024, 4};
  const int64_t small_rows = (page + 4095) / 4096;
  return {256, small_rows <= 1 ? 1 : (small_rows <= 2 ? 2 : 4)};
}

// Shape of copy_blocks: one load per lane, so an item is 4 KiB, or 1 KiB (one
// wave) where pages are no multiple of 4 KiB and 4 KiB items would leave
// lanes idle in the last one. In the order of copy_item, few bytes per item
// keep what the chip writes at any moment close together: 160 KiB tiles run
// at 6.45 TB/s (streaming stores) with 4 KiB items, 6.18 with 8 or 16 KiB,
// 6.03 with one item a tile; 12.5 KiB tiles at 5.69 with 4 KiB items and 6.02
// with 1 KiB, 1 KiB tiles at 3.84 and 6.19. On multiples of 4 KiB the two are
// within 1 %.
//
// One load per lane keeps 32 KiB in flight on a CU, which fills the chip's
// memory system only with all CUs. A stream masked to some of them
// (aegkv_stream_create_masked) gets more bytes per CU: whole-tile items from
// 64 KiB, else two loads per lane. On 24 / 16 / 8 of each XCD's 32 CUs, TB/s:
// 160 KiB tiles 6.07 / 4.52 / 2.40 with one load, 6.09 / 5.34 / 3.09 whole;
// 64 KiB 5.88 / 4.48 / 2.40, 6.15 / 4.97 / 2.75 whole; 32 KiB 5.47 / 4.33 /
// 2.38, 5.58 / 5.07 / 2.99 with two.
ShapeSel copy_shape(int64_t page, bool all_cus) {
  if (all_cus || page <= 4096) return ShapeSel{page % 4096 == 0 ? 256 : 64, 1};
  const int64_t row = 1024 * 16;
  return page >= 4 * row && page % row == 0 ? auto_shape(page) : ShapeSel{256, 2};
}

// Whether work on `stream` may use every one of the device's CUs (0.3 us).
bool stream_has_all_cus(hipStream_t stream, int num_cus) {
  uint32_t mask[32] = {};
  if (hipExtStreamGetCUMask(stream, 32, mask) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  int n = 0;
  for (uint32_t m : mask) n += __builtin_popcount(m);
  return n >= num_cus;
}

bool valid_copy_unroll(int64_t u) {
  return u == 1 || u == 2 || u == 3 || u == 4 || u == 5 || u == 6 || u == 8 || u == 10;
}

// ------------------------------------------------------- per-device state --

// Stream-ordered pinned->device upload ring for call descriptors. A region
// is reused only after the event recorded behind the call that read it has
// completed, whatever stream that call ran on. Every event remembers the
// stream it was last recorded on, so that a stream about to be destroyed
// can take its events with it (forget_stream): an event is never queried,
// waited on or re-recorded after the stream that recorded it is gone. A
// region whose event was dropped that way (ev == nullptr) has completed.
struct Ring {
  char* host = nullptr;
  char* host_dev = nullptr;  // the device's address of `host`
  char* dev = nullptr;
  size_t cap = 0;
  size_t head = 0;
  struct Region {
    size_t begin, end;
    hipEvent_t ev;
    hipStream_t stream;
  };
  struct Spare {
    hipEvent_t ev;
    hipStream_t last;  // stream it was last recorded on
  };
  std::deque<Region> inflight;
  std::vector<Spare> spare;
};

constexpr int kMaxDmaStreams = 4;

struct DeviceCtx {
  int device = -1;
  int num_cus = 0;
  std::mutex mu;
  Ring ring;
  // STAGED mode: library-owned streams the per-run copies fan out over,
  // forked from and joined back into the caller's stream with events, one
  // set per direction (dma[0] swap-out, dma[1] swap-in) so a swap-out and
  // a swap-in at once do not queue their copies behind each other (with
  // one shared set, a swap-in beside a swap-out finished at 88-120 ms
  // instead of 56 ms).
  // A staged call holds the set's mutex from its first fork to its last
  // join, so its events are not re-recorded by another call in between.
  // fork_ev and kernel_ev are recorded on callers' streams; fork_on and
  // kernel_on name the stream of their last record (forget_stream).
  struct DmaSet {
    std::mutex mu;
    int streams = 0;
    hipStream_t st[kMaxDmaStreams] = {};
    hipEvent_t fork_ev = nullptr;
    hipEvent_t join_ev[2][kMaxDmaStreams] = {};  // copies done, per staging buffer
    hipEvent_t kernel_ev[2] = {};                // gather / scatter done, per staging buffer
    hipStream_t fork_on = nullptr;
    hipStream_t kernel_on[2] = {};
  } dma[2];
};

std::mutex g_ctx_mu;
std::map<int, DeviceCtx*> g_ctx;

std::mutex g_host_mu;
std::map<uintptr_t, size_t> g_host_allocs;  // live pools: start -> bytes asked for
// Uncached host memory is never returned to the runtime. Every uncached
// block hipHostMalloc gave stays mapped until the process ends, and live
// uncached pools are carved out of those blocks: a freed pool's range goes
// back to a free list (coalesced with its free neighbours in the same
// block), and a later uncached pool takes the smallest free range that fits
// before any new block is allocated. A process whose pools come and go in
// different sizes thus pins no more than its largest set of live pools,
// which keeps it under the host's cap on pinned memory.
constexpr size_t kHostPage = 4096;
std::map<uintptr_t, size_t> g_uncached_blocks;  // block base -> bytes
std::map<uintptr_t, size_t> g_uncached_pools;   // live pool start -> bytes carved
std::map<uintptr_t, size_t> g_uncached_free;    // free range start -> bytes

int get_ctx(DeviceCtx** out) {
  int dev = -1;
  AEGKV_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(g_ctx_mu);
  auto it = g_ctx.find(dev);
  if (it != g_ctx.end()) {
    *out = it->second;
    return 0;
  }
  auto* ctx = new DeviceCtx();
  ctx->device = dev;
  AEGKV_HIP(hipDeviceGetAttribute(&ctx->num_cus, hipDeviceAttributeMultiprocessorCount, dev));
  if (ctx->num_cus <= 0) ctx->num_cus = 1;
  // Keep stream-ordered staging memory cached in the pool between calls.
  hipMemPool_t pool = nullptr;
  if (hipDeviceGetDefaultMemPool(&pool, dev) == hipSuccess && pool) {
    uint64_t threshold = UINT64_MAX;
    (void)hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &threshold);
  }
  (void)hipGetLastError();
  g_ctx[dev] = ctx;
  *out = ctx;
  return 0;
}

// Entry points that upload their descriptors through the host ring cannot
// be captured into a graph: a replay would copy the descriptor from the
// ring slot as a later call left it. They refuse a capturing stream before
// anything is enqueued (aegkv_copy_blocks_noalloc is the capturable copy).
int refuse_capture(hipStream_t stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  const hipError_t e = hipStreamIsCapturing(stream, &status);
  if (e != hipSuccess) return hip_fail(e, "hipStreamIsCapturing");
  if (status != hipStreamCaptureStatusNone)
    return fail(AEGKV_EINVAL, "the stream is being captured: this call uploads its descriptor "
                "through a host ring that later calls reuse, so a graph replay would read "
                "another call's descriptor (aegkv_copy_blocks_noalloc can be captured)");
  return 0;
}

// Hand a completed region's event back to the spare list (caller holds
// ctx->mu; the region is popped by the caller).
void ring_retire(Ring& r, const Ring::Region& reg) {
  if (reg.ev) r.spare.push_back({reg.ev, reg.stream});
}

// True once the oldest region's reader has finished (never blocks).
bool ring_front_done(Ring& r) {
  const Ring::Region& f = r.inflight.front();
  return f.ev == nullptr || hipEventQuery(f.ev) == hipSuccess;
}

// Wait for the oldest region's reader, then retire it.
int ring_wait_front(Ring& r) {
  const Ring::Region f = r.inflight.front();
  if (f.ev) AEGKV_HIP(hipEventSynchronize(f.ev));
  ring_retire(r, f);
  r.inflight.pop_front();
  return 0;
}

int ring_grow(Ring& r, size_t need) {
  // Retire everything, then replace the buffers.
  while (!r.inflight.empty()) {
    int rc = ring_wait_front(r);
    if (rc) return rc;
  }
  if (r.host) AEGKV_HIP(hipHostFree(r.host));
  if (r.dev) AEGKV_HIP(hipFree(r.dev));
  r.host = nullptr;
  r.dev = nullptr;
  r.cap = 0;
  size_t cap = size_t(4) << 20;
  while (cap < need) cap <<= 1;
  AEGKV_HIP(hipHostMalloc(reinterpret_cast<void**>(&r.host), cap, hipHostMallocDefault));
  void* mapped = nullptr;
  AEGKV_HIP(hipHostGetDevicePointer(&mapped, r.host, 0));
  r.host_dev = static_cast<char*>(mapped);
  AEGKV_HIP(hipMalloc(reinterpret_cast<void**>(&r.dev), cap));
  r.cap = cap;
  r.head = 0;
  return 0;
}

// Reserve `bytes` of the ring (caller holds ctx->mu). Returns offset.
int ring_reserve(Ring& r, size_t bytes, size_t* offset) {
  bytes = (bytes + 255) & ~size_t(255);
  if (bytes == 0) bytes = 256;
  if (bytes > r.cap) {
    int rc = ring_grow(r, bytes);
    if (rc) return rc;
  }
  // Retire completed regions without blocking.
  while (!r.inflight.empty() && ring_front_done(r)) {
    ring_retire(r, r.inflight.front());
    r.inflight.pop_front();
  }
  size_t start = r.head;
  if (start + bytes > r.cap) start = 0;
  const size_t end = start + bytes;
  auto overlaps = [&](const Ring::Region& g) { return g.begin < end && start < g.end; };
  for (;;) {
    bool any = false;
    for (auto& g : r.inflight)
      if (overlaps(g)) {
        any = true;
        break;
      }
    if (!any) break;
    int rc = ring_wait_front(r);
    if (rc) return rc;
  }
  r.head = end;
  *offset = start;
  return 0;
}

int ring_commit(Ring& r, size_t offset, size_t bytes, hipStream_t stream) {
  bytes = (bytes + 255) & ~size_t(255);
  if (bytes == 0) bytes = 256;
  Ring::Spare sp{nullptr, nullptr};
  if (!r.spare.empty()) {
    sp = r.spare.back();
    r.spare.pop_back();
  } else {
    AEGKV_HIP(hipEventCreateWithFlags(&sp.ev, hipEventDisableTiming));
  }
  hipError_t e = hipEventRecord(sp.ev, stream);
  if (e != hipSuccess) {
    r.spare.push_back(sp);
    return hip_fail(e, "hipEventRecord");
  }
  r.inflight.push_back({offset, offset + bytes, sp.ev, stream});
  return 0;
}

// A descriptor region in the ring: `bytes` of descriptor (a multiple of 16)
// and, behind it, the device word that holds the guard's value.
struct Desc {
  size_t off = 0;
  size_t bytes = 0;
  size_t total() const { return bytes + 16; }
};

int desc_reserve(Ring& r, size_t bytes, Desc* d) {
  d->bytes = (bytes + 15) & ~size_t(15);
  return ring_reserve(r, d->total(), &d->off);
}

// Enqueue the descriptor's way to the device. *seen: the word the moving
// kernel tests for `guard`, or null without one.
int desc_stage(Ring& r, const Desc& d, const uint64_t* guard, const uint64_t** seen,
               hipStream_t stream) {
  char* dev = r.dev + d.off;
  uint64_t* word = guard ? reinterpret_cast<uint64_t*>(dev + d.bytes) : nullptr;
  const uint32_t words = static_cast<uint32_t>(d.bytes / 16);
  (void)hipGetLastError();  // clear a stale error: the check below is for this launch
  hipLaunchKernelGGL(desc_stage_kernel, dim3((words + kStageLanes - 1) / kStageLanes),
                     dim3(kStageLanes), 0, stream,
                     reinterpret_cast<const v4u*>(r.host_dev + d.off),
                     reinterpret_cast<v4u*>(dev), words, guard, word);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(e, "desc_stage_kernel launch");
  *seen = word;
  return 0;
}

// Drop every event this library last recorded on `stream`, which the caller
// has synchronized and is about to destroy: ring regions it read are
// complete (their events are destroyed and the regions count as done),
// spare events recorded there are destroyed, and the DMA sets' fork and
// kernel events are replaced by fresh ones.
int forget_stream(hipStream_t stream) {
  std::vector<DeviceCtx*> ctxs;
  {
    std::lock_guard<std::mutex> lk(g_ctx_mu);
    for (auto& kv : g_ctx) ctxs.push_back(kv.second);
  }
  for (DeviceCtx* ctx : ctxs) {
    {
      std::lock_guard<std::mutex> lk(ctx->mu);
      Ring& r = ctx->ring;
      for (Ring::Region& g : r.inflight)
        if (g.ev && g.stream == stream) {
          (void)hipEventDestroy(g.ev);
          g.ev = nullptr;
        }
      auto keep = r.spare.begin();
      for (auto it = r.spare.begin(); it != r.spare.end(); ++it) {
        if (it->last == stream)
          (void)hipEventDestroy(it->ev);
        else
          *keep++ = *it;
      }
      r.spare.erase(keep, r.spare.end());
    }
    for (DeviceCtx::DmaSet& d : ctx->dma) {
      std::lock_guard<std::mutex> lk(d.mu);
      auto renew = [&](hipEvent_t* ev, hipStream_t* on) -> int {
        if (*ev == nullptr || *on != stream) return 0;
        (void)hipEventDestroy(*ev);
        *ev = nullptr;
        *on = nullptr;
        AEGKV_HIP(hipEventCreateWithFlags(ev, hipEventDisableTiming));
        return 0;
      };
      int rc = renew(&d.fork_ev, &d.fork_on);
      for (int b = 0; b < 2 && !rc; ++b) rc = renew(&d.kernel_ev[b], &d.kernel_on[b]);
      if (rc) return rc;
    }
  }
  (void)hipGetLastError();
  return 0;
}

// ------------------------------------------------------------- validation --

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Checks [ptr, ptr + bytes) lies inside one HIP device allocation.
int check_device_range(const void* ptr, int64_t bytes, const char* what) {
  if (bytes == 0) return 0;
  void* base = nullptr;
  size_t size = 0;
  hipError_t e = hipMemGetAddressRange(&base, &size, const_cast<void*>(ptr));
  if (e != hipSuccess || base == nullptr) {
    (void)hipGetLastError();
    return fail(AEGKV_EINVAL, "%s (%p) is not HIP device memory", what, ptr);
  }
  const uintptr_t b = reinterpret_cast<uintptr_t>(base);
  const uintptr_t p = reinterpret_cast<uintptr_t>(ptr);
  if (p < b || p + static_cast<uint64_t>(bytes) > b + size)
    return fail(AEGKV_ERANGE, "%s: %lld bytes at %p exceed its allocation (%zu bytes at %p)",
                what, static_cast<long long>(bytes), ptr, size, base);
  return 0;
}

// Checks a host pool is pinned and device-visible; kernels dereference it
// directly in DIRECT mode.
int check_host_range(const void* ptr, int64_t bytes, const char* what) {
  if (bytes == 0) return 0;
  {
    std::lock_guard<std::mutex> lk(g_host_mu);
    auto it = g_host_allocs.upper_bound(reinterpret_cast<uintptr_t>(ptr));
    if (it != g_host_allocs.begin()) {
      --it;
      const uintptr_t b = it->first;
      const uintptr_t p = reinterpret_cast<uintptr_t>(ptr);
      if (p >= b && p < b + it->second) {
        if (p + static_cast<uint64_t>(bytes) > b + it->second)
          return fail(AEGKV_ERANGE, "%s: %lld bytes at %p exceed its pinned pool", what,
                      static_cast<long long>(bytes), ptr);
        return 0;
      }
    }
  }
  hipPointerAttribute_t attr;
  std::memset(&attr, 0, sizeof(attr));
  hipError_t e = hipPointerGetAttributes(&attr, ptr);
  if (e != hipSuccess || attr.type != hipMemoryTypeHost) {
    (void)hipGetLastError();
    return fail(AEGKV_EINVAL, "%s (%p) is not pinned host memory (use aegkv_host_alloc)",
                what, ptr);
  }
  return 0;
}

// True when p lies in a pool from aegkv_host_alloc_flags(AEGKV_HOST_UNCACHED).
bool in_uncached_pool(const void* p) {
  std::lock_guard<std::mutex> lk(g_host_mu);
  const uintptr_t a = reinterpret_cast<uintptr_t>(p);
  auto it = g_uncached_pools.upper_bound(a);
  if (it == g_uncached_pools.begin()) return false;
  --it;
  return a < it->first + it->second;
}

// ----------------------------------------------------------- launching --

// Workgroups to launch for `items` work items: at most `limit` when limit > 0
// (the kernels' grid-stride loops cover the rest), else one per item. An HSA
// dispatch counts work-items in 32 bits, so the grid is also capped at
// (2^32 - 1) / lanes, for narrow workgroups at that of 256 lanes
// (kMaxLaunchItems), and to whole turns of the 8 XCDs.
int64_t launch_grid(int64_t limit, int64_t items, int lanes) {
  const int64_t cap = static_cast<int64_t>(UINT32_MAX) / std::max(lanes, 256) / 8 * 8;
  int64_t g = items;
  if (limit > 0) g = std::min<int64_t>(g, limit);
  return std::max<int64_t>(1, std::min<int64_t>(g, cap));
}

int too_many_items(int64_t a, int64_t b, int64_t c, const char* what) {
  return fail(AEGKV_EINVAL, "%lld %s x %lld segments x %lld chunks exceed the %lld work items "
              "of one launch; split the call", static_cast<long long>(a), what,
              static_cast<long long>(b), static_cast<long long>(c),
              static_cast<long long>(kMaxLaunchItems));
}

struct SwapArgs {
  const SegDesc* segs;
  const EntDesc* ents;
  const int64_t* kpp;
  SwapWalk walk;
  const uint64_t* seen;   // the staged guard value, or null
  const uint64_t* guard;  // the guard itself, or null
};

template <int WG, int U, bool TO_HOST, bool VEC, bool NT>
hipError_t launch_swap_t(int64_t grid, hipStream_t st, const SwapArgs& a) {
  (void)hipGetLastError();  // clear a stale error: the check below is for this launch
  hipLaunchKernelGGL((swap_tiles_kernel<WG, U, TO_HOST, VEC, NT>),
                     dim3(static_cast<uint32_t>(grid)), dim3(WG), 0, st, a.segs, a.ents, a.kpp,
                     a.walk, a.seen, a.guard);
  return hipGetLastError();
}

template <bool TO_HOST, bool VEC, bool NT>
hipError_t launch_inline_swap_t(int64_t grid, hipStream_t st, const InlineSwap& a) {
  (void)hipGetLastError();  // clear a stale error: the check below is for this launch
  hipLaunchKernelGGL((swap_inline_kernel<TO_HOST, VEC, NT>), dim3(static_cast<uint32_t>(grid)),
                     dim3(256), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_inline_swap(bool to_host, bool vec, bool nt, int64_t grid, hipStream_t st,
                              const InlineSwap& a) {
  if (to_host)  // never with non-temporal stores: the target is the host pool
    return vec ? launch_inline_swap_t<true, true, false>(grid, st, a)
               : launch_inline_swap_t<true, false, false>(grid, st, a);
  if (nt)
    return vec ? launch_inline_swap_t<false, true, true>(grid, st, a)
               : launch_inline_swap_t<false, false, true>(grid, st, a);
  return vec ? launch_inline_swap_t<false, true, false>(grid, st, a)
             : launch_inline_swap_t<false, false, false>(grid, st, a);
}

template <int WG, int U>
hipError_t launch_swap_shape(bool to_host, bool nt, int64_t grid, hipStream_t st,
                             const SwapArgs& a) {
  if (to_host)
    return nt ? launch_swap_t<WG, U, true, true, true>(grid, st, a)
              : launch_swap_t<WG, U, true, true, false>(grid, st, a);
  return nt ? launch_swap_t<WG, U, false, true, true>(grid, st, a)
            : launch_swap_t<WG, U, false, true, false>(grid, st, a);
}

hipError_t launch_swap(ShapeSel sh, bool to_host, bool vec, bool nt, int64_t grid,
                       hipStream_t st, const SwapArgs& a) {
  if (!vec) {
    if (to_host)
      return nt ? launch_swap_t<256, 2, true, false, true>(grid, st, a)
                : launch_swap_t<256, 2, true, false, false>(grid, st, a);
    return nt ? launch_swap_t<256, 2, false, false, true>(grid, st, a)
              : launch_swap_t<256, 2, false, false, false>(grid, st, a);
  }
#define AEGKV_SW(W, UU) \
  if (sh.wg == W && sh.u == UU) return launch_swap_shape<W, UU>(to_host, nt, grid, st, a);
  AEGKV_SW(256, 1) AEGKV_SW(256, 2) AEGKV_SW(256, 4)
  AEGKV_SW(1024, 1) AEGKV_SW(1024, 2) AEGKV_SW(1024, 3) AEGKV_SW(1024, 4)
  AEGKV_SW(1024, 5) AEGKV_SW(1024, 6) AEGKV_SW(1024, 8) AEGKV_SW(1024, 10)
#undef AEGKV_SW
  return hipErrorInvalidValue;
}

// `lds`: dynamic LDS reserved per workgroup. The kernel does not use it; it
// caps how many workgroups share a CU.
template <int WG, int U, bool VEC, bool NT>
hipError_t launch_copy_t(int64_t grid, unsigned lds, hipStream_t st, const CopySeg* s,
                         const PairDesc* p, const CopyLayout& l, const uint64_t* guard) {
  (void)hipGetLastError();  // clear a stale error: the check below is for this launch
  const dim3 g(static_cast<uint32_t>(grid));
  if (l.num_classes)
    hipLaunchKernelGGL((copy_blocks_kernel<WG, U, VEC, NT, CopyClasses>), g, dim3(WG), lds, st, s,
                       p, l.walk, guard, l.classes);
  else
    hipLaunchKernelGGL((copy_blocks_kernel<WG, U, VEC, NT, OneClass>), g, dim3(WG), lds, st, s, p,
                       l.walk, guard, OneClass{});
  return hipGetLastError();
}

hipError_t launch_copy(ShapeSel sh, bool vec, bool nt, int64_t grid, unsigned lds,
                       hipStream_t st, const CopySeg* s, const PairDesc* p, const CopyLayout& l,
                       const uint64_t* guard) {
  if (!vec) {
    if (sh.wg == 64)
      return nt ? launch_copy_t<64, 1, false, true>(grid, 0, st, s, p, l, guard)
                : launch_copy_t<64, 1, false, false>(grid, 0, st, s, p, l, guard);
    return nt ? launch_copy_t<256, 1, false, true>(grid, 0, st, s, p, l, guard)
              : launch_copy_t<256, 1, false, false>(grid, 0, st, s, p, l, guard);
  }
#define AEGKV_CP(W, UU)                                                               \
  if (sh.wg == W && sh.u == UU)                                                       \
    return nt ? launch_copy_t<W, UU, true, true>(grid, lds, st, s, p, l, guard)       \
              : launch_copy_t<W, UU, true, false>(grid, lds, st, s, p, l, guard);
  AEGKV_CP(64, 1) AEGKV_CP(256, 1) AEGKV_CP(256, 2) AEGKV_CP(256, 4) AEGKV_CP(256, 8)
  AEGKV_CP(1024, 1) AEGKV_CP(1024, 2) AEGKV_CP(1024, 3) AEGKV_CP(1024, 4)
  AEGKV_CP(1024, 5) AEGKV_CP(1024, 6) AEGKV_CP(1024, 8) AEGKV_CP(1024, 10)
#undef AEGKV_CP
  return hipErrorInvalidValue;
}

template <int WG, bool VEC, bool NT>
hipError_t launch_inline_t(bool one_class, int64_t grid, hipStream_t st, const InlineCopy& a) {
  (void)hipGetLastError();  // clear a stale error: the check below is for this launch
  const dim3 g(static_cast<uint32_t>(grid));
  if (one_class)
    hipLaunchKernelGGL((copy_blocks_inline_kernel<WG, VEC, NT, OneClass>), g, dim3(WG), 0, st, a);
  else
    hipLaunchKernelGGL((copy_blocks_inline_kernel<WG, VEC, NT, CopyClasses>), g, dim3(WG), 0, st,
                       a);
  return hipGetLastError();
}

hipError_t launch_inline(int lanes, bool vec, bool nt, bool one, int64_t grid,
                         hipStream_t st, const InlineCopy& a) {
  if (!vec)
    return nt ? launch_inline_t<64, false, true>(one, grid, st, a)
              : launch_inline_t<64, false, false>(one, grid, st, a);
  if (lanes == 64)
    return nt ? launch_inline_t<64, true, true>(one, grid, st, a)
              : launch_inline_t<64, true, false>(one, grid, st, a);
  return nt ? launch_inline_t<256, true, true>(one, grid, st, a)
            : launch_inline_t<256, true, false>(one, grid, st, a);
}

template <int WG, int U, int KIND, bool NT>
hipError_t launch_probe_t(int64_t grid, unsigned lds, hipStream_t st, const CopySeg* s,
                          const PairDesc* p, const CopyLayout& l, uint32_t* sink,
                          uint32_t magic) {
  (void)hipGetLastError();  // clear a stale error: the check below is for this launch
  const dim3 g(static_cast<uint32_t>(grid));
  if (l.num_classes)
    hipLaunchKernelGGL((copy_probe_kernel<WG, U, KIND, NT, CopyClasses>), g, dim3(WG), lds, st, s,
                       p, l.walk, sink, magic, l.classes);
  else
    hipLaunchKernelGGL((copy_probe_kernel<WG, U, KIND, NT, OneClass>), g, dim3(WG), lds, st, s, p,
                       l.walk, sink, magic, OneClass{});
  return hipGetLastError();
}

hipError_t launch_probe(ShapeSel sh, int kind, bool nt, int64_t grid, unsigned lds,
                        hipStream_t st, const CopySeg* s, const PairDesc* p,
                        const CopyLayout& l, uint32_t* sink, uint32_t magic) {
#define AEGKV_PR(W, UU)                                                                        \
  if (sh.wg == W && sh.u == UU) {                                                              \
    if (kind == PROBE_READ)                                                                    \
      return launch_probe_t<W, UU, PROBE_READ, false>(grid, lds, st, s, p, l, sink, magic); \
    return nt ? launch_probe_t<W, UU, PROBE_WRITE, true>(grid, lds, st, s, p, l, sink,      \
                                                         magic)                                \
              : launch_probe_t<W, UU, PROBE_WRITE, false>(grid, lds, st, s, p, l, sink,     \
                                                          magic);                              \
  }
  AEGKV_PR(64, 1) AEGKV_PR(256, 1) AEGKV_PR(256, 2) AEGKV_PR(256, 4) AEGKV_PR(256, 8)
  AEGKV_PR(1024, 1) AEGKV_PR(1024, 2) AEGKV_PR(1024, 3) AEGKV_PR(1024, 4)
  AEGKV_PR(1024, 5) AEGKV_PR(1024, 6) AEGKV_PR(1024, 8) AEGKV_PR(1024, 10)
#undef AEGKV_PR
  return hipErrorInvalidValue;
}

hipError_t launch_slices(bool vec, bool nt, int64_t grid, hipStream_t st,
                         const SliceDesc* slices, uint32_t num_slices, uint32_t items) {
  (void)hipGetLastError();  // clear a stale error: the check below is for this launch
  const dim3 g(static_cast<uint32_t>(grid));
  if (!vec && nt)
    hipLaunchKernelGGL((slices_kernel<256, 2, false, true>), g, dim3(256), 0, st, slices,
                       num_slices, items);
  else if (!vec)
    hipLaunchKernelGGL((slices_kernel<256, 2, false, false>), g, dim3(256), 0, st, slices,
                       num_slices, items);
  else if (nt)
    hipLaunchKernelGGL((slices_kernel<256, 2, true, true>), g, dim3(256), 0, st, slices,
                       num_slices, items);
  else
    hipLaunchKernelGGL((slices_kernel<256, 2, true, false>), g, dim3(256), 0, st, slices,
                       num_slices, items);
  return hipGetLastError();
}

// ------------------------------------------------------------ swap core --

bool mul_fits(int64_t a, int64_t b) { return a >= 0 && b >= 0 && (b == 0 || a <= INT64_MAX / b); }

// Argument checks that need no HIP call (run first, so a bad argument costs
// nothing on the device side). dev_vec: every device tile extent is 16 B
// aligned; host_vec: so is every host-pool extent. The 16 B kernel path needs
// both sides aligned.
int validate_layout(const SwapLayout& L, int64_t* composite_bytes, bool* dev_vec,
                    bool* host_vec) {
  if (L.num_segments <= 0) return fail(AEGKV_EINVAL, "num_segments must be positive");
  if (!L.bases || !L.page_bytes || !L.host_offsets || !L.owner_masks)
    return fail(AEGKV_EINVAL, "segment arrays must not be null");
  if (L.device_num_blocks <= 0) return fail(AEGKV_EINVAL, "device_num_blocks must be positive");
  if (L.num_groups <= 0 || L.num_groups > 64)
    return fail(AEGKV_EINVAL, "num_groups must be in [1, 64], got %d", L.num_groups);
  if (!L.kpp) return fail(AEGKV_EINVAL, "group_kernel_blocks_per_page must not be null");
  if (!L.host_pool) return fail(AEGKV_EINVAL, "host_pool must not be null");
  if (L.host_num_blocks <= 0 || L.host_page_bytes <= 0)
    return fail(AEGKV_EINVAL, "host pool geometry must be positive");
  if (!mul_fits(L.host_num_blocks, L.host_page_bytes))
    return fail(AEGKV_ERANGE, "host pool of %lld x %lld bytes overflows",
                static_cast<long long>(L.host_num_blocks),
                static_cast<long long>(L.host_page_bytes));
  if (L.host_rank_offset < 0 || L.host_rank_offset >= L.host_page_bytes)
    return fail(AEGKV_EINVAL, "host_rank_offset must be in [0, host_page_bytes)");
  for (int32_t g = 0; g < L.num_groups; ++g)
    if (L.kpp[g] <= 0 || L.kpp[g] > INT32_MAX)
      return fail(AEGKV_EINVAL, "kernel_blocks_per_page[%d]=%lld must be in [1, 2^31)", g,
                  static_cast<long long>(L.kpp[g]));
  bool v = true;
  int64_t composite = 0;
  for (int32_t s = 0; s < L.num_segments; ++s) {
    const int64_t pb = L.page_bytes[s];
    const int64_t ho = L.host_offsets[s];
    if (!L.bases[s]) return fail(AEGKV_EINVAL, "segment %d base is null", s);
    if (pb <= 0) return fail(AEGKV_EINVAL, "segment %d page_bytes must be positive", s);
    if (ho < 0) return fail(AEGKV_EINVAL, "segment %d host offset must be >= 0", s);
    if (!mul_fits(L.device_num_blocks, pb))
      return fail(AEGKV_ERANGE, "segment %d of %lld x %lld bytes overflows", s,
                  static_cast<long long>(L.device_num_blocks), static_cast<long long>(pb));
    // rank offset + host offset + page must stay inside one host page
    if (ho > L.host_page_bytes || pb > L.host_page_bytes - ho ||
        L.host_rank_offset > L.host_page_bytes - ho - pb)
      return fail(AEGKV_ERANGE,
                  "segment %d [%lld, +%lld) at rank offset %lld overruns the %lld-byte host page",
                  s, static_cast<long long>(ho), static_cast<long long>(pb),
                  static_cast<long long>(L.host_rank_offset),
                  static_cast<long long>(L.host_page_bytes));
    if (L.owner_masks[s] == 0) return fail(AEGKV_EINVAL, "segment %d has no owning group", s);
    for (int32_t g = 0; g < L.num_groups; ++g)
      if (((L.owner_masks[s] >> g) & 1ull) && pb % L.kpp[g] != 0)
        return fail(AEGKV_EEXTENT,
                    "segment %d page of %lld bytes does not split into %lld equal kernel blocks", s,
                    static_cast<long long>(pb), static_cast<long long>(L.kpp[g]));
    if (L.num_groups < 64 && (L.owner_masks[s] >> L.num_groups) != 0)
      return fail(AEGKV_ERANGE, "segment %d owner mask names a group >= %d", s, L.num_groups);
    v = v && aligned16(L.bases[s]) && pb % 16 == 0 && ho % 16 == 0;
    for (int32_t g = 0; g < L.num_groups && v; ++g)
      if ((L.owner_masks[s] >> g) & 1ull) v = (pb / L.kpp[g]) % 16 == 0;
    composite = std::max(composite, ho + pb);
  }
  *composite_bytes = composite;
  *dev_vec = v;
  *host_vec = aligned16(L.host_pool) && L.host_page_bytes % 16 == 0 &&
              L.host_rank_offset % 16 == 0;
  return 0;
}

// Pointer checks through the HIP runtime: every segment lies inside one
// device allocation, and the host pool is pinned and mapped in both modes
// (DIRECT kernels dereference it; STAGED copies of a pageable pool would be
// staged again by the runtime, so they are refused too).
int check_layout_pointers(const SwapLayout& L) {
  for (int32_t s = 0; s < L.num_segments; ++s) {
    int rc = check_device_range(L.bases[s], L.device_num_blocks * L.page_bytes[s],
                                "segment base");
    if (rc) return rc;
  }
  return check_host_range(L.host_pool, L.host_num_blocks * L.host_page_bytes, "host_pool");
}

int validate_list(const SwapLayout& L, const SwapList& E, bool is_swap_in) {
  if (E.n < 0) return fail(AEGKV_EINVAL, "num_entries must be >= 0");
  if (E.n == 0) return 0;
  if (!E.src || !E.dst) return fail(AEGKV_EINVAL, "block id arrays must not be null");
  const int64_t src_lim = is_swap_in ? L.host_num_blocks : L.device_num_blocks;
  const int64_t dst_lim = is_swap_in ? L.device_num_blocks : L.host_num_blocks;
  std::vector<uint8_t> seen(static_cast<size_t>(dst_lim), 0);
  for (int64_t i = 0; i < E.n; ++i) {
    if (E.src[i] < 0 || E.src[i] >= src_lim)
      return fail(AEGKV_ERANGE, "source block id %lld at %lld outside [0, %lld)",
                  static_cast<long long>(E.src[i]), static_cast<long long>(i),
                  static_cast<long long>(src_lim));
    if (E.dst[i] < 0 || E.dst[i] >= dst_lim)
      return fail(AEGKV_ERANGE, "target block id %lld at %lld outside [0, %lld)",
                  static_cast<long long>(E.dst[i]), static_cast<long long>(i),
                  static_cast<long long>(dst_lim));
    if (seen[static_cast<size_t>(E.dst[i])])
      return fail(AEGKV_EDUP, "target block id %lld appears twice",
                  static_cast<long long>(E.dst[i]));
    seen[static_cast<size_t>(E.dst[i])] = 1;
    const int32_t g = E.group ? E.group[i] : 0;
    if (g < 0 || g >= L.num_groups)
      return fail(AEGKV_ERANGE, "group id %d at %lld outside [0, %d)", g,
                  static_cast<long long>(i), L.num_groups);
    const int64_t k = L.kpp[g];
    const int64_t first = E.first ? E.first[i] : 0;
    const int64_t valid = E.valid ? E.valid[i] : k;
    if (first < 0 || valid < 0 || first > k || valid > k - first)
      return fail(AEGKV_EEXTENT, "kernel blocks [%lld, %lld) of entry %lld run past a page of %lld",
                  static_cast<long long>(first), static_cast<long long>(first + valid),
                  static_cast<long long>(i), static_cast<long long>(k));
  }
  return 0;
}

// Launch shape of the swap kernels: 256 lanes with the tuned loads per
// lane, or (tuning key 8) a whole-tile shape; two loads where addresses or
// lengths are no multiples of 16.
ShapeSel swap_shape(const Tunables& t, bool vec, int64_t max_page) {
  if (!vec) return ShapeSel{256, 2};
  return t.swap_shape_auto ? auto_shape(max_page)
                           : ShapeSel{256, static_cast<int>(t.swap_unroll)};
}

// The tables of a swap of entries order[lo, hi), at h: segments, then kernel
// blocks per page, then entries resolved to the given host side.
void pack_swap_desc(char* h, size_t kpp_off, size_t ent_off, const SwapLayout& L,
                    const SwapList& E, const std::vector<int64_t>& order, size_t lo, size_t hi,
                    bool is_swap_in, bool staged) {
  SegDesc* hs = reinterpret_cast<SegDesc*>(h);
  for (int32_t s = 0; s < L.num_segments; ++s)
    hs[s] = SegDesc{static_cast<char*>(L.bases[s]), L.page_bytes[s], L.host_offsets[s],
                    L.owner_masks[s]};
  std::memcpy(h + kpp_off, L.kpp, sizeof(int64_t) * L.num_groups);
  EntDesc* he = reinterpret_cast<EntDesc*>(h + ent_off);
  for (size_t j = 0; j < hi - lo; ++j) {
    const int64_t i = order[lo + j];
    const int32_t g = E.group ? E.group[i] : 0;
    EntDesc d;
    d.dev_block = is_swap_in ? E.dst[i] : E.src[i];
    const int64_t host_id = is_swap_in ? E.src[i] : E.dst[i];
    d.host_slot = staged ? static_cast<int64_t>(j) : host_id;
    d.group = g;
    d.first = static_cast<int32_t>(E.first ? E.first[i] : 0);
    d.valid = static_cast<int32_t>(E.valid ? E.valid[i] : L.kpp[g]);
    d.pad = 0;
    he[j] = d;
  }
}

// Enqueue the descriptor and the kernel for entries order[lo, hi) resolved to
// the given host side. Caller holds ctx->mu.
//
// A DIRECT swap's descriptor reaches the device inside the launch where it is
// short, else by a runtime copy: those of a swap-out and a swap-in enqueued
// together are both done (5.5 us each) before either fills the link. A
// staging kernel read the second one from the host while the first swap had
// the link, for 500-890 us (a model switch in a process with other swappers:
// 12.4 ms, 11.9 so). A swap-out of one block of 72 x 32 KiB takes 68 us a
// pass in one launch, 77 in two. STAGED kernels keep the staging kernel,
// which reads the guard once for their full grids.
int enqueue_swap_kernel(DeviceCtx* ctx, const SwapLayout& L, const SwapList& E,
                        const std::vector<int64_t>& order, size_t lo, size_t hi,
                        bool is_swap_in, bool staged, char* host_side, int64_t host_stride,
                        int64_t host_rank_off, bool vec, int64_t wgs, hipStream_t stream) {
  const int32_t S = L.num_segments;
  const int64_t n = static_cast<int64_t>(hi - lo);
  if (n == 0) return 0;
  const Tunables t = tunables();
  int64_t max_page = 0;
  for (int32_t s = 0; s < S; ++s) max_page = std::max(max_page, L.page_bytes[s]);
  const ShapeSel sh = swap_shape(t, vec, max_page);
  const int64_t cpt = (max_page + sh.chunk() - 1) / sh.chunk();
  const int64_t items = launch_items(n, S, cpt);
  if (items < 0) return too_many_items(n, S, cpt, "entries");
  const int64_t grid = launch_grid(wgs, items, sh.wg);
  const SwapWalk walk{host_side, host_stride, host_rank_off, static_cast<uint32_t>(S),
                      static_cast<uint32_t>(items), static_cast<uint32_t>(cpt)};
  // Non-temporal stores only where the destination is HBM: plain stores to
  // the host pool measured faster (no L2 residency to avoid there).
  const bool nt = t.nt_stores != 0 && !(!is_swap_in && !staged);
  const size_t seg_bytes = sizeof(SegDesc) * S;
  const size_t kpp_bytes = sizeof(int64_t) * L.num_groups;
  const size_t ent_bytes = sizeof(EntDesc) * n;

  const size_t short_ent_off = (seg_bytes + kpp_bytes + 15) & ~size_t(15);
  if (!staged && sh.wg == 256 && sh.u == 2 && short_ent_off + ent_bytes <= kInlineSwapBytes) {
    InlineSwap a;
    a.walk = walk;
    a.kpp_offset = static_cast<uint32_t>(seg_bytes);
    a.ent_offset = static_cast<uint32_t>(short_ent_off);
    a.pad = 0;
    a.guard = E.guard;
    pack_swap_desc(reinterpret_cast<char*>(a.data), seg_bytes, short_ent_off, L, E, order, lo, hi,
                   is_swap_in, false);
    const hipError_t e = launch_inline_swap(!is_swap_in, vec, nt, grid, stream, a);
    return e == hipSuccess ? 0 : hip_fail(e, "swap_inline_kernel launch");
  }

  const size_t kpp_off = (seg_bytes + 255) & ~size_t(255);
  const size_t ent_off = (kpp_off + kpp_bytes + 255) & ~size_t(255);
  Desc desc;
  int rc = desc_reserve(ctx->ring, ent_off + ent_bytes, &desc);
  if (rc) return rc;
  pack_swap_desc(ctx->ring.host + desc.off, kpp_off, ent_off, L, E, order, lo, hi, is_swap_in,
                 staged);
  char* dv = ctx->ring.dev + desc.off;
  const uint64_t* seen = nullptr;
  if (staged) {
    rc = desc_stage(ctx->ring, desc, E.guard, &seen, stream);
    if (rc) return rc;
  } else {
    AEGKV_HIP(hipMemcpyAsync(dv, ctx->ring.host + desc.off, desc.bytes, hipMemcpyHostToDevice,
                             stream));
  }
  SwapArgs a{reinterpret_cast<const SegDesc*>(dv), reinterpret_cast<const EntDesc*>(dv + ent_off),
             reinterpret_cast<const int64_t*>(dv + kpp_off), walk, seen,
             staged ? nullptr : E.guard};
  const hipError_t e = launch_swap(sh, !is_swap_in, vec, nt, grid, stream, a);
  if (e != hipSuccess) {
    // the descriptor's way to the device is already enqueued: retire its
    // region in order
    (void)hipGetLastError();
    (void)ring_commit(ctx->ring, desc.off, desc.total(), stream);
    return hip_fail(e, "swap_tiles_kernel launch");
  }
  return ring_commit(ctx->ring, desc.off, desc.total(), stream);
}

// A staged chunk with more host runs than this counts as scattered.
constexpr size_t kManyRuns = 16;

// A stream on a hardware queue of its own: a stream created with a CU mask
// gets a dedicated queue (here the mask enables every CU), while plain
// streams share the process's GPU_MAX_HW_QUEUES queues, and two copies whose
// streams share a queue run one after the other.
hipError_t dedicated_stream(hipStream_t* out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  int cus = 0;
  e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (e != hipSuccess) return e;
  std::vector<uint32_t> mask(static_cast<size_t>((cus + 31) / 32), 0xFFFFFFFFu);
  return hipExtStreamCreateWithCUMask(out, static_cast<uint32_t>(mask.size()), mask.data());
}

// Create the DMA streams and events once (caller holds the set's mutex).
int ensure_dma(DeviceCtx::DmaSet& d, int k) {
  if (!d.fork_ev) {
    AEGKV_HIP(hipEventCreateWithFlags(&d.kernel_ev[0], hipEventDisableTiming));
    AEGKV_HIP(hipEventCreateWithFlags(&d.kernel_ev[1], hipEventDisableTiming));
    AEGKV_HIP(hipEventCreateWithFlags(&d.fork_ev, hipEventDisableTiming));
  }
  while (d.streams < k) {
    const int i = d.streams;
    AEGKV_HIP(hipStreamCreateWithFlags(&d.st[i], hipStreamNonBlocking));
    AEGKV_HIP(hipEventCreateWithFlags(&d.join_ev[0][i], hipEventDisableTiming));
    AEGKV_HIP(hipEventCreateWithFlags(&d.join_ev[1][i], hipEventDisableTiming));
    ++d.streams;
  }
  return 0;
}

hipError_t copy_run(const Run& r, bool to_device, char* staging, char* host, hipStream_t st) {
  char* s_ptr = staging + r.stage_off;
  char* h_ptr = host + r.host_off;
  const size_t len = static_cast<size_t>(r.len);
  return to_device ? hipMemcpyAsync(s_ptr, h_ptr, len, hipMemcpyHostToDevice, st)
                   : hipMemcpyAsync(h_ptr, s_ptr, len, hipMemcpyDeviceToHost, st);
}

// Copy the staged runs of one chunk between staging and the host pool over
// the k DMA streams, balanced by bytes, and record join[i] behind stream i's
// share (caller holds the set's mutex).
int runs_on_dma(DeviceCtx::DmaSet& d, int k, const std::vector<Run>& runs, bool to_device,
                char* staging, char* host, hipEvent_t* join) {
  int64_t load[kMaxDmaStreams] = {};
  for (const Run& r : runs) {
    const int i = static_cast<int>(std::min_element(load, load + k) - load);
    load[i] += r.len;
    hipError_t e = copy_run(r, to_device, staging, host, d.st[i]);
    if (e != hipSuccess) return hip_fail(e, "hipMemcpyAsync(staged run)");
  }
  for (int i = 0; i < k; ++i) AEGKV_HIP(hipEventRecord(join[i], d.st[i]));
  return 0;
}

// The gather (swap-out) or scatter (swap-in) kernel of staged chunk
// order[lo, hi) whose host side is `staging` (one composite page per entry).
// It moves HBM to HBM, so it gets a full grid, except a swap-out whose chunk
// leaves many host runs (scattered host ids, one page-sized copy each):
// there the copies measured faster beside the slower persistent grid
// (41.9 -> 50.1 GB/s), while a few large runs gain from the full grid
// (51.1 -> 55.3 GB/s).
int staged_kernel(DeviceCtx* ctx, const SwapLayout& L, const SwapList& E,
                  const std::vector<int64_t>& order, size_t lo, size_t hi, bool is_swap_in,
                  char* staging, int64_t composite, bool vec_stage, size_t num_runs,
                  const Tunables& t, hipStream_t stream) {
  const int64_t wgs = !is_swap_in && num_runs > kManyRuns ? t.swap_out_workgroups
                                                          : t.staged_workgroups;
  std::lock_guard<std::mutex> lk(ctx->mu);
  return enqueue_swap_kernel(ctx, L, E, order, lo, hi, is_swap_in, true, staging, composite, 0,
                             vec_stage, wgs, stream);
}

// Copy one chunk's runs between staging and the host pool and return the
// caller's stream to after them: on the caller's stream itself (k <= 1), or
// forked over the k DMA streams (after everything the caller's stream
// holds) and joined back, which overlaps the runtime's per-copy gaps.
int chunk_copies(DeviceCtx* ctx, int k, const std::vector<Run>& runs, bool to_device,
                 char* staging, char* host, hipStream_t stream) {
  const int dir = to_device ? 1 : 0;
  if (k <= 1) {
    for (const Run& r : runs) {
      hipError_t e = copy_run(r, to_device, staging, host, stream);
      if (e != hipSuccess) return hip_fail(e, "hipMemcpyAsync(staged run)");
    }
    return 0;
  }
  DeviceCtx::DmaSet& d = ctx->dma[dir];
  std::lock_guard<std::mutex> lk(d.mu);
  int rc = ensure_dma(d, k);
  if (rc) return rc;
  d.fork_on = stream;
  AEGKV_HIP(hipEventRecord(d.fork_ev, stream));
  for (int j = 0; j < k; ++j) AEGKV_HIP(hipStreamWaitEvent(d.st[j], d.fork_ev, 0));
  rc = runs_on_dma(d, k, runs, to_device, staging, host, d.join_ev[0]);
  // join whatever was enqueued, also after a failed copy
  for (int j = 0; j < k; ++j) {
    if (rc && hipEventRecord(d.join_ev[0][j], d.st[j]) != hipSuccess) continue;
    hipError_t e = hipStreamWaitEvent(stream, d.join_ev[0][j], 0);
    if (e != hipSuccess && !rc) rc = hip_fail(e, "hipStreamWaitEvent(staged copies)");
  }
  return rc;
}

// STAGED one chunk after another, each through its own stream-ordered
// staging allocation: swap-out gathers a chunk and then copies it to the
// host, swap-in copies a chunk from the host and then scatters it. `runs`
// arrives with those of the first chunk.
int staged_serial(DeviceCtx* ctx, const SwapLayout& L, const SwapList& E,
                  const std::vector<int64_t>& order, bool is_swap_in, int64_t composite,
                  size_t step, std::vector<Run>& runs, bool vec_stage, const Tunables& t, int k,
                  hipStream_t stream) {
  for (size_t lo = 0; lo < order.size(); lo += step) {
    const size_t hi = std::min(order.size(), lo + step);
    if (lo > 0) chunk_runs(L, E, order, lo, hi, is_swap_in, composite, runs);
    void* p = nullptr;
    AEGKV_HIP(hipMallocAsync(&p, (hi - lo) * static_cast<size_t>(composite), stream));
    char* buf = static_cast<char*>(p);
    int rc = 0;
    if (is_swap_in) rc = chunk_copies(ctx, k, runs, true, buf, L.host_pool, stream);
    if (!rc)
      rc = staged_kernel(ctx, L, E, order, lo, hi, is_swap_in, buf, composite, vec_stage,
                         runs.size(), t, stream);
    if (!rc && !is_swap_in) rc = chunk_copies(ctx, k, runs, false, buf, L.host_pool, stream);
    if (rc) {
      (void)hipFreeAsync(buf, stream);
      return rc;
    }
    AEGKV_HIP(hipFreeAsync(buf, stream));
  }
  return 0;
}

// STAGED with the copies on the library's k DMA streams and two staging
// buffers, so the gather (swap-out) or scatter (swap-in) of one chunk runs
// while another chunk's copies use the link. Chunk c uses buffer b = c % 2:
//   swap-out: the caller's stream waits the copies of chunk c-2 and gathers
//             chunk c into buffer b; the DMA streams wait that gather, copy
//             the chunk to the host and record join_ev[b];
//   swap-in:  the DMA streams wait the scatter of chunk c-2, copy chunk c
//             from the host into buffer b and record join_ev[b]; the
//             caller's stream waits those and scatters the chunk.
// The DMA streams start after everything the caller's stream holds, the
// staging allocations included; the caller's stream ends after every copy
// and frees the buffers there.
int staged_overlapped(DeviceCtx* ctx, const SwapLayout& L, const SwapList& E,
                      const std::vector<int64_t>& order, bool is_swap_in, int64_t composite,
                      size_t step, std::vector<Run>& runs, bool vec_stage, const Tunables& t,
                      int k, hipStream_t stream) {
  DeviceCtx::DmaSet& d = ctx->dma[is_swap_in ? 1 : 0];
  std::lock_guard<std::mutex> lk(d.mu);
  int rc = ensure_dma(d, k);
  if (rc) return rc;
  const size_t n = order.size();
  const size_t chunks = (n + step - 1) / step;
  const int nbuf = chunks > 1 ? 2 : 1;
  const size_t buf_bytes = std::min(step, n) * static_cast<size_t>(composite);
  char* buf[2] = {nullptr, nullptr};
  for (int b = 0; b < nbuf; ++b) {
    void* p = nullptr;
    hipError_t e = hipMallocAsync(&p, buf_bytes, stream);
    if (e != hipSuccess) {
      if (b) (void)hipFreeAsync(buf[0], stream);
      return hip_fail(e, "hipMallocAsync(staging)");
    }
    buf[b] = static_cast<char*>(p);
  }
  // On a failure after work was enqueued: join every DMA stream back into
  // the caller's stream and free the buffers behind it.
  auto unwind = [&](int status) {
    for (int j = 0; j < k; ++j)
      if (hipEventRecord(d.join_ev[0][j], d.st[j]) == hipSuccess)
        (void)hipStreamWaitEvent(stream, d.join_ev[0][j], 0);
    for (int b = 0; b < nbuf; ++b) (void)hipFreeAsync(buf[b], stream);
    (void)hipGetLastError();
    return status;
  };
  // every DMA stream waits `ev`, recorded on `on` (which *ev_on notes)
  auto fan_in = [&](hipEvent_t ev, hipStream_t* ev_on, hipStream_t on) {
    *ev_on = on;
    hipError_t e = hipEventRecord(ev, on);
    for (int j = 0; j < k && e == hipSuccess; ++j) e = hipStreamWaitEvent(d.st[j], ev, 0);
    return e;
  };
  // the caller's stream waits the copies that recorded join_ev[b]
  auto join = [&](int b) {
    hipError_t e = hipSuccess;
    for (int j = 0; j < k && e == hipSuccess; ++j) e = hipStreamWaitEvent(stream, d.join_ev[b][j], 0);
    return e;
  };
  hipError_t e = fan_in(d.fork_ev, &d.fork_on, stream);
  if (e != hipSuccess) return unwind(hip_fail(e, "staged fork"));
  for (size_t c = 0; c < chunks; ++c) {
    const size_t lo = c * step, hi = std::min(n, lo + step);
    const int b = static_cast<int>(c & 1);
    if (c > 0) chunk_runs(L, E, order, lo, hi, is_swap_in, composite, runs);
    if (!is_swap_in) {
      if (c >= 2 && (e = join(b)) != hipSuccess)
        return unwind(hip_fail(e, "hipStreamWaitEvent(staged copies)"));
      rc = staged_kernel(ctx, L, E, order, lo, hi, false, buf[b], composite, vec_stage,
                         runs.size(), t, stream);
      if (rc) return unwind(rc);
      if ((e = fan_in(d.kernel_ev[b], &d.kernel_on[b], stream)) != hipSuccess)
        return unwind(hip_fail(e, "staged gather event"));
      rc = runs_on_dma(d, k, runs, false, buf[b], L.host_pool, d.join_ev[b]);
      if (rc) return unwind(rc);
    } else {
      for (int j = 0; c >= 2 && j < k && e == hipSuccess; ++j)
        e = hipStreamWaitEvent(d.st[j], d.kernel_ev[b], 0);
      if (e != hipSuccess) return unwind(hip_fail(e, "hipStreamWaitEvent(staged scatter)"));
      rc = runs_on_dma(d, k, runs, true, buf[b], L.host_pool, d.join_ev[b]);
      if (rc) return unwind(rc);
      if ((e = join(b)) != hipSuccess)
        return unwind(hip_fail(e, "hipStreamWaitEvent(staged copies)"));
      rc = staged_kernel(ctx, L, E, order, lo, hi, true, buf[b], composite, vec_stage,
                         runs.size(), t, stream);
      if (rc) return unwind(rc);
      d.kernel_on[b] = stream;
      if ((e = hipEventRecord(d.kernel_ev[b], stream)) != hipSuccess)
        return unwind(hip_fail(e, "staged scatter event"));
    }
  }
  // swap-out: each DMA stream's last join follows all of its earlier copies
  if (!is_swap_in && (e = join(static_cast<int>((chunks - 1) & 1))) != hipSuccess)
    return unwind(hip_fail(e, "hipStreamWaitEvent(staged copies)"));
  for (int b = 0; b < nbuf; ++b) AEGKV_HIP(hipFreeAsync(buf[b], stream));
  return 0;
}

int swap_core(const SwapLayout& L, const SwapList& E, bool is_swap_in, int mode,
              hipStream_t stream) {
  if (mode < AEGKV_MODE_AUTO || mode > AEGKV_MODE_STAGED)
    return fail(AEGKV_EINVAL, "unknown transfer mode %d", mode);
  const Tunables t = tunables();
  if (mode == AEGKV_MODE_AUTO)
    mode = static_cast<int>(is_swap_in ? t.auto_h2d : t.auto_d2h);
  const bool staged = mode == AEGKV_MODE_STAGED;
  int64_t composite = 0;
  bool dev_vec = false, host_vec = false;
  int rc = validate_layout(L, &composite, &dev_vec, &host_vec);
  if (rc) return rc;
  rc = validate_list(L, E, is_swap_in);
  if (rc) return rc;
  if (E.n == 0) return 0;
  int64_t max_page = 0;
  for (int32_t s = 0; s < L.num_segments; ++s) max_page = std::max(max_page, L.page_bytes[s]);
  auto chunks = [&](bool vec) {
    const int64_t chunk = swap_shape(t, vec, max_page).chunk();
    return (max_page + chunk - 1) / chunk;
  };
  // the whole list in one launch (a staged chunk holds fewer entries)
  const int64_t cpt = chunks(dev_vec && (staged ? composite % 16 == 0 : host_vec));
  if (launch_items(E.n, L.num_segments, cpt) < 0)
    return too_many_items(E.n, L.num_segments, cpt, "entries");
  const bool direct_fits = launch_items(E.n, L.num_segments, chunks(dev_vec && host_vec)) >= 0;
  rc = check_layout_pointers(L);
  if (rc) return rc;
  rc = refuse_capture(stream);
  if (rc) return rc;
  DeviceCtx* ctx = nullptr;
  rc = get_ctx(&ctx);
  if (rc) return rc;

  std::vector<int64_t> order(static_cast<size_t>(E.n));
  for (int64_t i = 0; i < E.n; ++i) order[static_cast<size_t>(i)] = i;

  auto direct = [&] {
    std::lock_guard<std::mutex> lk(ctx->mu);
    // link-bound: a few persistent workgroups
    const int64_t wgs = is_swap_in                        ? t.swap_in_workgroups
                        : in_uncached_pool(L.host_pool) ? t.swap_out_workgroups_uncached
                                                        : t.swap_out_workgroups;
    return enqueue_swap_kernel(ctx, L, E, order, 0, order.size(), is_swap_in, false,
                               L.host_pool, L.host_page_bytes, L.host_rank_offset,
                               dev_vec && host_vec, wgs, stream);
  };
  if (!staged) return direct();

  // STAGED: host-id order lets consecutive host pages merge into one DMA.
  const int64_t* host_ids = is_swap_in ? E.src : E.dst;
  std::stable_sort(order.begin(), order.end(),
                   [&](int64_t a, int64_t b) { return host_ids[a] < host_ids[b]; });
  const size_t step = static_cast<size_t>(
      std::max<int64_t>(1, std::min<int64_t>(E.n, t.staging_bytes / composite)));
  std::vector<Run> runs;
  chunk_runs(L, E, order, 0, step, is_swap_in, composite, runs);
  if (t.staged_short_runs && direct_fits &&
      cheap_as_direct(order.size() <= step ? run_totals(runs)
                                           : call_runs(L, E, order, is_swap_in, composite, step)))
    return direct();
  // Staging comes from hipMallocAsync (256 B aligned) with a composite stride.
  const bool vec_stage = dev_vec && composite % 16 == 0;
  int k = static_cast<int>(std::min<int64_t>(t.staged_dma_streams, kMaxDmaStreams));
  if (order.size() <= step && static_cast<int64_t>(runs.size()) <= kFewRuns) k = 0;
  const bool overlap = (t.staged_overlap >> (is_swap_in ? 1 : 0)) & 1;
  if (k <= 1 || !overlap)
    return staged_serial(ctx, L, E, order, is_swap_in, composite, step, runs, vec_stage, t, k,
                         stream);
  return staged_overlapped(ctx, L, E, order, is_swap_in, composite, step, runs, vec_stage, t,
                           k, stream);
}

// Whole-block copies from a source cache to a target cache (the same cache
// for copy_blocks), in steps shared by the allocating and the
// allocation-free entry points: layout checks, id checks, device-range
// checks, the launch shape, then descriptor upload and launch.

// Checks that need no HIP call and no memory: segment geometry and the
// 16 B path. *max_page receives the largest page.
int copy_check_layout(int32_t num_segments, void* const* src_bases, void* const* dst_bases,
                      const int64_t* page_bytes, int64_t src_num_blocks,
                      int64_t dst_num_blocks, int64_t num_pairs, const int64_t* src_ids,
                      const int64_t* dst_ids, bool same_cache, bool* vec, int64_t* max_page) {
  if (num_segments <= 0) return fail(AEGKV_EINVAL, "num_segments must be positive");
  if (!src_bases || !dst_bases || !page_bytes)
    return fail(AEGKV_EINVAL, "segment arrays must not be null");
  if (src_num_blocks <= 0 || dst_num_blocks <= 0)
    return fail(AEGKV_EINVAL, "device_num_blocks must be positive");
  if (num_pairs < 0) return fail(AEGKV_EINVAL, "num_pairs must be >= 0");
  if (num_pairs > 0 && (!src_ids || !dst_ids))
    return fail(AEGKV_EINVAL, "block id arrays must not be null");
  bool v = true;
  int64_t mp = 0;
  for (int32_t s = 0; s < num_segments; ++s) {
    if (!src_bases[s] || !dst_bases[s]) return fail(AEGKV_EINVAL, "segment %d base is null", s);
    if (page_bytes[s] <= 0)
      return fail(AEGKV_EINVAL, "segment %d page_bytes must be positive", s);
    if (!mul_fits(src_num_blocks, page_bytes[s]) || !mul_fits(dst_num_blocks, page_bytes[s]))
      return fail(AEGKV_ERANGE, "segment %d of %lld x %lld bytes overflows", s,
                  static_cast<long long>(std::max(src_num_blocks, dst_num_blocks)),
                  static_cast<long long>(page_bytes[s]));
    if (!same_cache) {
      const uintptr_t a0 = reinterpret_cast<uintptr_t>(src_bases[s]);
      const uintptr_t b0 = reinterpret_cast<uintptr_t>(dst_bases[s]);
      const uintptr_t a1 = a0 + static_cast<uint64_t>(src_num_blocks * page_bytes[s]);
      const uintptr_t b1 = b0 + static_cast<uint64_t>(dst_num_blocks * page_bytes[s]);
      if (a0 < b1 && b0 < a1)
        return fail(AEGKV_EOVERLAP,
                    "segment %d: source and target caches overlap (copy within one cache "
                    "with aegkv_copy_blocks)", s);
    }
    v = v && aligned16(src_bases[s]) && aligned16(dst_bases[s]) && page_bytes[s] % 16 == 0;
    mp = std::max(mp, page_bytes[s]);
  }
  *vec = v;
  *max_page = mp;
  return 0;
}

// Every id inside its cache (first offending pair in pair order).
int copy_check_ranges(int64_t src_num_blocks, int64_t dst_num_blocks, int64_t num_pairs,
                      const int64_t* src_ids, const int64_t* dst_ids) {
  for (int64_t i = 0; i < num_pairs; ++i) {
    const int64_t s = src_ids[i], d = dst_ids[i];
    if (s < 0 || s >= src_num_blocks || d < 0 || d >= dst_num_blocks)
      return fail(AEGKV_ERANGE, "pair %lld (%lld -> %lld) outside [0, %lld) -> [0, %lld)",
                  static_cast<long long>(i), static_cast<long long>(s),
                  static_cast<long long>(d), static_cast<long long>(src_num_blocks),
                  static_cast<long long>(dst_num_blocks));
  }
  return 0;
}

int dup_target(int64_t id) {
  return fail(AEGKV_EDUP, "target block id %lld appears twice", static_cast<long long>(id));
}

int source_is_target(int64_t id) {
  return fail(AEGKV_EOVERLAP, "block %lld is both a source and a target",
              static_cast<long long>(id));
}

// Distinct targets, and (within one cache) no source that is also a
// target, with a block-indexed map. Ids are in range.
int copy_check_ids_map(int64_t dst_num_blocks, int64_t num_pairs, const int64_t* src_ids,
                       const int64_t* dst_ids, bool same_cache) {
  std::vector<uint8_t> target(static_cast<size_t>(dst_num_blocks), 0);
  for (int64_t i = 0; i < num_pairs; ++i) {
    uint8_t& t = target[static_cast<size_t>(dst_ids[i])];
    if (t) return dup_target(dst_ids[i]);
    t = 1;
  }
  if (same_cache)
    for (int64_t i = 0; i < num_pairs; ++i)
      if (target[static_cast<size_t>(src_ids[i])]) return source_is_target(src_ids[i]);
  return 0;
}

// The same checks without memory of the block count's size: sorted copies
// of the ids in the caller's work arrays (num_pairs entries each).
int copy_check_ids_sorted(int64_t num_pairs, const int64_t* src_ids, const int64_t* dst_ids,
                          bool same_cache, int64_t* work_src, int64_t* work_dst) {
  std::copy(dst_ids, dst_ids + num_pairs, work_dst);
  std::sort(work_dst, work_dst + num_pairs);
  for (int64_t i = 1; i < num_pairs; ++i)
    if (work_dst[i] == work_dst[i - 1]) return dup_target(work_dst[i]);
  if (!same_cache) return 0;
  std::copy(src_ids, src_ids + num_pairs, work_src);
  std::sort(work_src, work_src + num_pairs);
  for (int64_t i = 0, j = 0; i < num_pairs && j < num_pairs;) {
    if (work_src[i] == work_dst[j]) return source_is_target(work_src[i]);
    if (work_src[i] < work_dst[j]) ++i;
    else ++j;
  }
  return 0;
}

int copy_check_device(int32_t num_segments, void* const* src_bases, void* const* dst_bases,
                      const int64_t* page_bytes, int64_t src_num_blocks,
                      int64_t dst_num_blocks, bool same_cache) {
  for (int32_t s = 0; s < num_segments; ++s) {
    int rc = check_device_range(src_bases[s], src_num_blocks * page_bytes[s], "segment base");
    if (rc) return rc;
    if (!same_cache) {
      rc = check_device_range(dst_bases[s], dst_num_blocks * page_bytes[s], "target segment base");
      if (rc) return rc;
    }
  }
  return 0;
}

struct CopyPlan {
  ShapeSel sh;
  bool vec;
  CopyLayout lay;
};

int copy_plan(const Tunables& t, bool vec, const int64_t* page_bytes, int64_t max_page,
              bool all_cus, int32_t num_segments, int64_t num_pairs, CopyPlan* out) {
  out->vec = vec;
  auto lay = [&](ShapeSel sh) {
    out->sh = sh;
    return lay_walk(page_bytes, num_segments, num_pairs, sh.chunk(), vec, &out->lay);
  };
  ShapeSel sh = copy_shape(max_page, all_cus);
  if (t.copy_unroll > 0)
    sh = ShapeSel{t.copy_lanes == 256 ? 256 : 1024, static_cast<int>(t.copy_unroll)};
  if (lay(vec ? sh : ShapeSel{64, 1})) return 0;
  if (!vec || t.copy_unroll == 0) {
    // more small items than one launch holds
    if (lay(vec ? auto_shape(max_page) : ShapeSel{256, 1})) return 0;
  }
  return too_many_items(num_pairs, num_segments, tile_chunks(max_page, out->sh.chunk(), vec),
                        "pairs");
}

// Byte offset of the pair table after num_segments CopySeg entries.
size_t copy_pair_offset(int32_t num_segments) {
  return (sizeof(CopySeg) * static_cast<size_t>(num_segments) + 255) & ~size_t(255);
}

// Pairs in order of their target ids (by_dst) or source ids, by a stable
// least-significant-byte-first counting sort: one pass over the pairs per
// byte of the largest id, with `tmp` (num_pairs entries) as the other
// buffer. Pairs already in order are left alone.
void sort_pairs(PairDesc* a, int64_t n, bool by_dst, PairDesc* tmp) {
  auto key = [by_dst](const PairDesc& x) { return by_dst ? x.dst : x.src; };
  int64_t top = 0;
  bool sorted = true;
  for (int64_t i = 0; i < n; ++i) {
    top = std::max(top, key(a[i]));
    if (i > 0 && key(a[i]) < key(a[i - 1])) sorted = false;
  }
  if (sorted) return;
  PairDesc* from = a;
  PairDesc* to = tmp;
  for (int shift = 0; shift < 64 && (top >> shift) != 0; shift += 8) {
    int64_t start[257] = {};
    for (int64_t i = 0; i < n; ++i) ++start[((key(from[i]) >> shift) & 255) + 1];
    for (int d = 0; d < 256; ++d) start[d + 1] += start[d];
    for (int64_t i = 0; i < n; ++i) to[start[(key(from[i]) >> shift) & 255]++] = from[i];
    std::swap(from, to);
  }
  if (from != a) std::copy(from, from + n, a);
}

// The tables of a copy at h: segments, class by class as the walk takes them,
// then pairs.
void pack_copy_desc(char* h, size_t pair_offset, const CopyPlan& plan, int32_t num_segments,
                    void* const* src_bases, void* const* dst_bases, const int64_t* page_bytes,
                    int64_t num_pairs, const int64_t* src_ids, const int64_t* dst_ids,
                    int64_t order, PairDesc* tmp) {
  const CopyLayout& l = plan.lay;
  CopySeg* hs = reinterpret_cast<CopySeg*>(h);
  for (int k = 0; k <= static_cast<int>(l.num_classes); ++k)
    for (int32_t s = 0; s < num_segments; ++s)
      if (l.num_classes == 0 ||
          l.class_of(tile_chunks(page_bytes[s], plan.sh.chunk(), plan.vec)) == k)
        *hs++ = CopySeg{static_cast<const char*>(src_bases[s]), static_cast<char*>(dst_bases[s]),
                        page_bytes[s], 0};
  PairDesc* hp = reinterpret_cast<PairDesc*>(h + pair_offset);
  for (int64_t i = 0; i < num_pairs; ++i) hp[i] = PairDesc{src_ids[i], dst_ids[i]};
  // Targets are distinct and never sources, so any order gives the same
  // result. Copies of small tiles run faster with their targets in order:
  // the workgroups running together then write near one another.
  if (order == 1 || order == 2) sort_pairs(hp, num_pairs, order == 1, tmp);
}

// What a copy call launches: the copy itself (guarded by `guard` when it is
// not null), or one of its measurement twins (aegkv_copy_probe) with the
// sink word and magic they take.
struct CopyKind {
  int probe = 0;            // 0 = copy, PROBE_READ or PROBE_WRITE
  uint32_t* sink = nullptr;
  uint32_t magic = 0;
  const uint64_t* guard = nullptr;
};

// Launch the copy kernel (or a probe twin) over descriptors already on the
// device at `dv`, with the copy's grid and LDS policy.
hipError_t copy_launch(const CopyPlan& p, const Tunables& t, int num_cus, int32_t num_segments,
                       const char* dv, hipStream_t stream, const CopyKind& kind = CopyKind()) {
  const int64_t grid = launch_grid(t.copy_wgs_per_cu * num_cus, p.lay.walk.num_items, p.sh.wg);
  const unsigned lds = p.sh.wg == 1024 && p.sh.chunk() >= (int64_t(32) << 10)
                           ? static_cast<unsigned>(t.copy_lds_bytes) : 0u;
  const CopySeg* segs = reinterpret_cast<const CopySeg*>(dv);
  const PairDesc* pairs = reinterpret_cast<const PairDesc*>(dv + copy_pair_offset(num_segments));
  if (kind.probe)
    return launch_probe(p.sh, kind.probe, t.nt_stores != 0, grid, lds, stream, segs, pairs,
                        p.lay, kind.sink, kind.magic);
  return launch_copy(p.sh, p.vec, t.nt_stores != 0, grid, lds, stream, segs, pairs, p.lay,
                     kind.guard);
}

// A copy whose descriptor fits a launch's arguments goes out as that one
// launch, in the shapes of the whole chip (one load per lane). *launched:
// whether it did.
int copy_inline(const CopyPlan& p, const Tunables& t, int num_cus, int32_t num_segments,
                void* const* src_bases, void* const* dst_bases, const int64_t* page_bytes,
                int64_t num_pairs, const int64_t* src_ids, const int64_t* dst_ids,
                hipStream_t stream, bool* launched) {
  const size_t class_offset = sizeof(CopySeg) * static_cast<size_t>(num_segments);
  const size_t pair_offset = class_offset + sizeof(CopyClass) * p.lay.num_classes;
  *launched = false;
  if (p.sh.u != 1 || p.sh.wg > 256 || (!p.vec && p.sh.wg != 64) ||
      pair_offset >= kInlineBytes ||
      num_pairs > static_cast<int64_t>((kInlineBytes - pair_offset) / sizeof(PairDesc)))
    return 0;
  InlineCopy a;
  a.walk = p.lay.walk;
  a.class_offset = static_cast<uint32_t>(class_offset);
  a.pair_offset = static_cast<uint32_t>(pair_offset);
  PairDesc tmp[kInlineBytes / sizeof(PairDesc)];
  pack_copy_desc(reinterpret_cast<char*>(a.data), pair_offset, p, num_segments, src_bases,
                 dst_bases, page_bytes, num_pairs, src_ids, dst_ids, t.copy_order, tmp);
  std::memcpy(a.data + class_offset, p.lay.classes.at, sizeof(CopyClass) * p.lay.num_classes);
  const int64_t grid = launch_grid(t.copy_wgs_per_cu * num_cus, p.lay.walk.num_items, p.sh.wg);
  const hipError_t e = launch_inline(p.sh.wg, p.vec, t.nt_stores != 0,
                                     p.lay.num_classes == 0, grid, stream, a);
  if (e != hipSuccess) return hip_fail(e, "copy_blocks_inline_kernel launch");
  *launched = true;
  return 0;
}

int copy_core(int32_t num_segments, void* const* src_bases, void* const* dst_bases,
              const int64_t* page_bytes, int64_t src_num_blocks, int64_t dst_num_blocks,
              int64_t num_pairs, const int64_t* src_ids, const int64_t* dst_ids, bool same_cache,
              hipStream_t stream, const CopyKind& kind = CopyKind()) {
  bool vec = false;
  int64_t max_page = 0;
  int rc = copy_check_layout(num_segments, src_bases, dst_bases, page_bytes, src_num_blocks,
                             dst_num_blocks, num_pairs, src_ids, dst_ids, same_cache, &vec,
                             &max_page);
  if (!rc) rc = copy_check_ranges(src_num_blocks, dst_num_blocks, num_pairs, src_ids, dst_ids);
  if (!rc) rc = copy_check_ids_map(dst_num_blocks, num_pairs, src_ids, dst_ids, same_cache);
  if (rc || num_pairs == 0) return rc;
  if (kind.probe && !vec)
    return fail(AEGKV_EINVAL, "the probes move 16 B per lane: bases and pages must be "
                "16 B multiples");
  const Tunables t = tunables();
  CopyPlan plan;
  rc = copy_plan(t, vec, page_bytes, max_page, true, num_segments, num_pairs, &plan);
  if (rc) return rc;
  rc = copy_check_device(num_segments, src_bases, dst_bases, page_bytes, src_num_blocks,
                         dst_num_blocks, same_cache);
  if (rc) return rc;
  rc = refuse_capture(stream);
  if (rc) return rc;
  DeviceCtx* ctx = nullptr;
  rc = get_ctx(&ctx);
  if (rc) return rc;
  if (!stream_has_all_cus(stream, ctx->num_cus))
    rc = copy_plan(t, vec, page_bytes, max_page, false, num_segments, num_pairs, &plan);
  if (rc) return rc;
  if (!kind.probe && !kind.guard) {
    bool launched = false;
    rc = copy_inline(plan, t, ctx->num_cus, num_segments, src_bases, dst_bases, page_bytes,
                     num_pairs, src_ids, dst_ids, stream, &launched);
    if (rc || launched) return rc;
  }
  std::lock_guard<std::mutex> lk(ctx->mu);
  Desc desc;
  rc = desc_reserve(ctx->ring, copy_pair_offset(num_segments) + sizeof(PairDesc) * num_pairs,
                    &desc);
  if (rc) return rc;
  char* h = ctx->ring.host + desc.off;
  std::vector<PairDesc> tmp(t.copy_order != 0 ? static_cast<size_t>(num_pairs) : 0);
  pack_copy_desc(h, copy_pair_offset(num_segments), plan, num_segments, src_bases, dst_bases,
                 page_bytes, num_pairs, src_ids, dst_ids, t.copy_order, tmp.data());
  CopyKind launch = kind;
  rc = desc_stage(ctx->ring, desc, kind.guard, &launch.guard, stream);
  if (rc) return rc;
  const hipError_t e = copy_launch(plan, t, ctx->num_cus, num_segments, ctx->ring.dev + desc.off,
                                   stream, launch);
  if (e != hipSuccess) {
    // the descriptor's staging is already enqueued: retire its region in order
    (void)hipGetLastError();
    (void)ring_commit(ctx->ring, desc.off, desc.total(), stream);
    return hip_fail(e, kind.probe ? "copy_probe_kernel launch" : "copy_blocks_kernel launch");
  }
  return ring_commit(ctx->ring, desc.off, desc.total(), stream);
}

// ------------------------------------------------ allocation-free copies --
//
// aegkv_copy_blocks_noalloc: aegkv_copy_blocks for callers that cannot
// allocate. The descriptor (segment table + pair table) goes to `scratch`,
// a fixed device array every GPU holds for the life of the process, instead
// of the library's upload ring; it travels in the kernel arguments of small
// fill launches, or of the copy itself where it is short (copy_inline), so a
// graph that captures the call replays its own descriptor. The ids are checked
// with fixed host arrays instead of a block-indexed map. Nothing is allocated
// on the host or the device. Every call on a device shares that device's array,
// so calls that overlap on one device (different streams, or threads, or a
// graph replayed beside other calls) race; calls on one stream are ordered.

constexpr int32_t kNoAllocMaxSegments = 1024;
constexpr int64_t kNoAllocMaxPairs = 65536;
constexpr size_t kNoAllocBytes =
    sizeof(CopySeg) * kNoAllocMaxSegments + sizeof(PairDesc) * kNoAllocMaxPairs;  // 1.03 MiB
constexpr int kNoAllocMaxDevices = 64;

static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

std::mutex g_noalloc_mu;                        // guards everything below
char* g_scratch_ptr[kNoAllocMaxDevices] = {};   // device address of `scratch`, per device
int g_noalloc_cus[kNoAllocMaxDevices] = {};
alignas(256) unsigned char g_noalloc_host[kNoAllocBytes];  // descriptor packing (pageable)
int64_t g_noalloc_work[2][kNoAllocMaxPairs];    // sorted id copies for the checks
PairDesc g_noalloc_order[kNoAllocMaxPairs];     // the other buffer of the pair sort

// Looks up this device's `scratch` address and CU count, once per device,
// with that device current (caller holds g_noalloc_mu). aegkv_init does it
// for every device at set-up.
int noalloc_resolve(int dev) {
  if (dev < 0 || dev >= kNoAllocMaxDevices)
    return fail(AEGKV_EINVAL, "device %d is outside the %d devices the allocation-free "
                "copy supports", dev, kNoAllocMaxDevices);
  if (g_scratch_ptr[dev]) return 0;
  void* p = nullptr;
  AEGKV_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  int cus = 0;
  AEGKV_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  g_noalloc_cus[dev] = cus > 0 ? cus : 1;
  g_scratch_ptr[dev] = static_cast<char*>(p);
  return 0;
}

// Device address of the current device's `scratch` (caller holds
// g_noalloc_mu). Without aegkv_init, the first call on a device looks it
// up, unless that call's stream is being captured: the lookup may load the
// library's code object, which must not happen inside a capture.
int noalloc_scratch(int dev, hipStream_t stream, char** out, int* num_cus) {
  if (dev < 0 || dev >= kNoAllocMaxDevices || !g_scratch_ptr[dev]) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    const hipError_t e = hipStreamIsCapturing(stream, &status);
    if (e != hipSuccess) return hip_fail(e, "hipStreamIsCapturing");
    if (status != hipStreamCaptureStatusNone)
      return fail(AEGKV_EINVAL, "the allocation-free copy's first call on device %d is being "
                  "captured; call aegkv_init() before capturing", dev);
    int rc = noalloc_resolve(dev);
    if (rc) return rc;
  }
  *out = g_scratch_ptr[dev];
  *num_cus = g_noalloc_cus[dev];
  return 0;
}

// The tables packed at g_noalloc_host to their places in `scratch`, kFillBytes
// of packed entries a launch of desc_fill_kernel.
hipError_t noalloc_fill(char* dst, const unsigned char* src, int32_t num_segments,
                        int64_t num_pairs, int64_t num_blocks, hipStream_t stream) {
  const size_t pair_offset = copy_pair_offset(num_segments);
  const CopySeg* segs = reinterpret_cast<const CopySeg*>(src);
  const PairDesc* pairs = reinterpret_cast<const PairDesc*>(src + pair_offset);
  FillArgs a;
  a.wide = num_blocks > (int64_t(1) << 32);
  a.pad = 0;
  const size_t pair_bytes = a.wide ? sizeof(PairDesc) : sizeof(FillPair);
  int64_t s = 0, p = 0;
  while (s < num_segments || p < num_pairs) {
    a.segs = reinterpret_cast<CopySeg*>(dst) + s;
    a.pairs = reinterpret_cast<PairDesc*>(dst + pair_offset) + p;
    a.num_segs = static_cast<uint32_t>(
        std::min<int64_t>(num_segments - s, kFillBytes / sizeof(FillSeg)));
    const size_t used = a.num_segs * sizeof(FillSeg);
    a.num_pairs = static_cast<uint32_t>(
        std::min<int64_t>(num_pairs - p, static_cast<int64_t>((kFillBytes - used) / pair_bytes)));
    FillSeg* fs = reinterpret_cast<FillSeg*>(a.data);
    for (uint32_t i = 0; i < a.num_segs; ++i)
      fs[i] = FillSeg{segs[s + i].dst, segs[s + i].page_bytes};
    if (a.wide) {
      std::memcpy(a.data + used, pairs + p, a.num_pairs * pair_bytes);
    } else {
      FillPair* fp = reinterpret_cast<FillPair*>(a.data + used);
      for (uint32_t i = 0; i < a.num_pairs; ++i)
        fp[i] = FillPair{static_cast<uint32_t>(pairs[p + i].src),
                         static_cast<uint32_t>(pairs[p + i].dst)};
    }
    s += a.num_segs;
    p += a.num_pairs;
    (void)hipGetLastError();  // clear a stale error: the check below is for this launch
    hipLaunchKernelGGL(desc_fill_kernel, dim3(1), dim3(kFillLanes), 0, stream, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

int copy_noalloc(int32_t num_segments, void* const* bases, const int64_t* page_bytes,
                 int64_t num_blocks, int64_t num_pairs, const int64_t* src_ids,
                 const int64_t* dst_ids, hipStream_t stream) {
  if (num_segments > kNoAllocMaxSegments)
    return fail(AEGKV_ENOMEM, "%d segments exceed the allocation-free copy's maximum of %d "
                "(use aegkv_copy_blocks)", num_segments, kNoAllocMaxSegments);
  if (num_pairs > kNoAllocMaxPairs)
    return fail(AEGKV_ENOMEM, "%lld pairs exceed the allocation-free copy's maximum of %lld "
                "(use aegkv_copy_blocks)", static_cast<long long>(num_pairs),
                static_cast<long long>(kNoAllocMaxPairs));
  bool vec = false;
  int64_t max_page = 0;
  int rc = copy_check_layout(num_segments, bases, bases, page_bytes, num_blocks, num_blocks,
                             num_pairs, src_ids, dst_ids, true, &vec, &max_page);
  if (!rc) rc = copy_check_ranges(num_blocks, num_blocks, num_pairs, src_ids, dst_ids);
  if (rc) return rc;
  std::lock_guard<std::mutex> lk(g_noalloc_mu);
  rc = copy_check_ids_sorted(num_pairs, src_ids, dst_ids, true, g_noalloc_work[0],
                             g_noalloc_work[1]);
  if (rc || num_pairs == 0) return rc;
  const Tunables t = tunables();
  CopyPlan plan;
  rc = copy_plan(t, vec, page_bytes, max_page, true, num_segments, num_pairs, &plan);
  if (rc) return rc;
  rc = copy_check_device(num_segments, bases, bases, page_bytes, num_blocks, num_blocks, true);
  if (rc) return rc;
  int dev = -1;
  AEGKV_HIP(hipGetDevice(&dev));
  char* dv = nullptr;
  int num_cus = 0;
  rc = noalloc_scratch(dev, stream, &dv, &num_cus);
  if (rc) return rc;
  if (!stream_has_all_cus(stream, num_cus))
    rc = copy_plan(t, vec, page_bytes, max_page, false, num_segments, num_pairs, &plan);
  if (rc) return rc;
  bool launched = false;
  rc = copy_inline(plan, t, num_cus, num_segments, bases, bases, page_bytes, num_pairs, src_ids,
                   dst_ids, stream, &launched);
  if (rc || launched) return rc;
  pack_copy_desc(reinterpret_cast<char*>(g_noalloc_host), copy_pair_offset(num_segments), plan,
                 num_segments, bases, bases, page_bytes, num_pairs, src_ids, dst_ids,
                 t.copy_order, g_noalloc_order);
  // The descriptor reaches `scratch` through kernel arguments, not a copy
  // from the packing area: a copy node captured into a graph would read the
  // packing area again at every replay, after later calls rewrote it.
  hipError_t e = noalloc_fill(dv, g_noalloc_host, num_segments, num_pairs, num_blocks, stream);
  if (e != hipSuccess) return hip_fail(e, "desc_fill_kernel launch");
  e = copy_launch(plan, t, num_cus, num_segments, dv, stream);
  if (e != hipSuccess) return hip_fail(e, "copy_blocks_kernel launch");
  return 0;
}

// Weight slices host -> device in one call (aegkv_load_slices).
int slices_core(int64_t n, void* const* dst, const void* const* src, const int64_t* bytes,
                int mode, hipStream_t stream) {
  if (n < 0) return fail(AEGKV_EINVAL, "num_slices must be >= 0");
  if (n > 0 && (!dst || !src || !bytes)) return fail(AEGKV_EINVAL, "slice arrays must not be null");
  if (mode < AEGKV_MODE_AUTO || mode > AEGKV_MODE_STAGED)
    return fail(AEGKV_EINVAL, "unknown transfer mode %d", mode);
  const Tunables t = tunables();
  if (mode == AEGKV_MODE_AUTO) mode = static_cast<int>(t.auto_h2d);
  // non-empty slices, checked; distinct targets
  std::vector<int64_t> keep;
  keep.reserve(static_cast<size_t>(n));
  bool vec = true;
  for (int64_t i = 0; i < n; ++i) {
    if (bytes[i] < 0)
      return fail(AEGKV_EINVAL, "slice %lld has %lld bytes", static_cast<long long>(i),
                  static_cast<long long>(bytes[i]));
    if (bytes[i] == 0) continue;
    if (!dst[i] || !src[i])
      return fail(AEGKV_EINVAL, "slice %lld has a null pointer", static_cast<long long>(i));
    keep.push_back(i);
    vec = vec && aligned16(dst[i]) && aligned16(src[i]) && bytes[i] % 16 == 0;
  }
  std::vector<int64_t> by_dst(keep);
  std::sort(by_dst.begin(), by_dst.end(), [&](int64_t a, int64_t b) {
    return reinterpret_cast<uintptr_t>(dst[a]) < reinterpret_cast<uintptr_t>(dst[b]);
  });
  for (size_t k = 1; k < by_dst.size(); ++k) {
    const int64_t a = by_dst[k - 1], b = by_dst[k];
    if (reinterpret_cast<uintptr_t>(dst[a]) + static_cast<uint64_t>(bytes[a]) >
        reinterpret_cast<uintptr_t>(dst[b]))
      return fail(AEGKV_EOVERLAP, "target slices %lld and %lld overlap",
                  static_cast<long long>(a), static_cast<long long>(b));
  }
  if (keep.empty()) return 0;
  const int64_t chunk = int64_t(256) * 16 * 2;
  int64_t items = 0;
  for (int64_t i : keep) {
    items += (bytes[i] + chunk - 1) / chunk;
    if (items > kMaxLaunchItems)
      return fail(AEGKV_EINVAL, "the slices need more than the %lld work items of one launch; "
                  "split the call", static_cast<long long>(kMaxLaunchItems));
  }
  for (int64_t i : keep) {
    int rc = check_device_range(dst[i], bytes[i], "target slice");
    if (!rc) rc = check_host_range(src[i], bytes[i], "source slice");
    if (rc) return rc;
  }
  if (mode == AEGKV_MODE_STAGED) {
    // the runtime's DMA copy per slice, as the reference's copy_ per slice
    for (int64_t i : keep)
      AEGKV_HIP(hipMemcpyAsync(dst[i], src[i], static_cast<size_t>(bytes[i]),
                               hipMemcpyHostToDevice, stream));
    return 0;
  }
  int rc = refuse_capture(stream);
  if (rc) return rc;
  DeviceCtx* ctx = nullptr;
  rc = get_ctx(&ctx);
  if (rc) return rc;
  std::lock_guard<std::mutex> lk(ctx->mu);
  Desc desc;
  rc = desc_reserve(ctx->ring, sizeof(SliceDesc) * keep.size(), &desc);
  if (rc) return rc;
  SliceDesc* h = reinterpret_cast<SliceDesc*>(ctx->ring.host + desc.off);
  int64_t first = 0;
  for (size_t k = 0; k < keep.size(); ++k) {
    const int64_t i = keep[k];
    h[k] = SliceDesc{static_cast<char*>(dst[i]), static_cast<const char*>(src[i]), bytes[i],
                     first};
    first += (bytes[i] + chunk - 1) / chunk;
  }
  const uint64_t* guard = nullptr;
  rc = desc_stage(ctx->ring, desc, nullptr, &guard, stream);
  if (rc) return rc;
  const hipError_t e =
      launch_slices(vec, t.nt_stores != 0, launch_grid(t.swap_in_workgroups, items, 256), stream,
                    reinterpret_cast<const SliceDesc*>(ctx->ring.dev + desc.off),
                    static_cast<uint32_t>(keep.size()), static_cast<uint32_t>(items));
  if (e != hipSuccess) {
    (void)hipGetLastError();
    (void)ring_commit(ctx->ring, desc.off, desc.total(), stream);
    return hip_fail(e, "slices_kernel launch");
  }
  return ring_commit(ctx->ring, desc.off, desc.total(), stream);
}

}  // namespace

// =============================================================== C ABI ==

extern "C" {

int aegkv_abi_version(void) { return AEGKV_ABI_VERSION; }

const char* aegkv_last_error(void) { return g_err; }

int64_t aegkv_tune(int key, int64_t value) {
  (void)env_status();  // environment overrides apply before the first change
  std::lock_guard<std::mutex> lk(g_tune_mu);
  int64_t* slot = nullptr;
  switch (key) {
    case AEGKV_TUNE_SWAP_OUT_WORKGROUPS: slot = &g_tune.swap_out_workgroups; break;
    case AEGKV_TUNE_SWAP_IN_WORKGROUPS: slot = &g_tune.swap_in_workgroups; break;
    case AEGKV_TUNE_STAGING_BYTES: slot = &g_tune.staging_bytes; break;
    case AEGKV_TUNE_AUTO_D2H: slot = &g_tune.auto_d2h; break;
    case AEGKV_TUNE_AUTO_H2D: slot = &g_tune.auto_h2d; break;
    case AEGKV_TUNE_NT_STORES: slot = &g_tune.nt_stores; break;
    case AEGKV_TUNE_COPY_WGS_PER_CU: slot = &g_tune.copy_wgs_per_cu; break;
    case AEGKV_TUNE_COPY_UNROLL: slot = &g_tune.copy_unroll; break;
    case AEGKV_TUNE_COPY_LANES: slot = &g_tune.copy_lanes; break;
    case AEGKV_TUNE_SWAP_SHAPE_AUTO: slot = &g_tune.swap_shape_auto; break;
    case AEGKV_TUNE_SWAP_UNROLL: slot = &g_tune.swap_unroll; break;
    case AEGKV_TUNE_STAGED_WORKGROUPS: slot = &g_tune.staged_workgroups; break;
    case AEGKV_TUNE_STAGED_DMA_STREAMS: slot = &g_tune.staged_dma_streams; break;
    case AEGKV_TUNE_COPY_LDS_BYTES: slot = &g_tune.copy_lds_bytes; break;
    case AEGKV_TUNE_STAGED_OVERLAP: slot = &g_tune.staged_overlap; break;
    case AEGKV_TUNE_SWAP_OUT_WORKGROUPS_UNCACHED: slot = &g_tune.swap_out_workgroups_uncached; break;
    case AEGKV_TUNE_COPY_ORDER: slot = &g_tune.copy_order; break;
    case AEGKV_TUNE_STAGED_SHORT_RUNS: slot = &g_tune.staged_short_runs; break;
    default: return fail(AEGKV_EINVAL, "unknown tuning key %d", key);
  }
  const int64_t prev = *slot;
  if (value >= 0) {
    if ((key == AEGKV_TUNE_AUTO_D2H || key == AEGKV_TUNE_AUTO_H2D) &&
        value != AEGKV_MODE_DIRECT && value != AEGKV_MODE_STAGED)
      return fail(AEGKV_EINVAL, "AUTO must resolve to DIRECT or STAGED");
    if ((key == AEGKV_TUNE_SWAP_OUT_WORKGROUPS || key == AEGKV_TUNE_SWAP_IN_WORKGROUPS ||
         key == AEGKV_TUNE_SWAP_OUT_WORKGROUPS_UNCACHED) &&
        (value < 1 || value > 65536))
      return fail(AEGKV_EINVAL, "swap workgroups must be in [1, 65536]");
    if (key == AEGKV_TUNE_STAGING_BYTES && value < (int64_t(1) << 20))
      return fail(AEGKV_EINVAL, "staging must be at least 1 MiB");
    if (key == AEGKV_TUNE_COPY_WGS_PER_CU && value > 64)
      return fail(AEGKV_EINVAL, "copy workgroups per CU must be in [0, 64]");
    if (key == AEGKV_TUNE_STAGED_WORKGROUPS && value > (int64_t(1) << 24))
      return fail(AEGKV_EINVAL, "staged workgroups must be in [0, 2^24]");
    if (key == AEGKV_TUNE_SWAP_UNROLL && value != 1 && value != 2 && value != 4)
      return fail(AEGKV_EINVAL, "swap unroll must be 1, 2 or 4");
    if (key == AEGKV_TUNE_COPY_LANES && value != 0 && value != 256 && value != 1024)
      return fail(AEGKV_EINVAL, "copy lanes must be 0, 256 or 1024");
    if (key == AEGKV_TUNE_COPY_UNROLL && value != 0 && g_tune.copy_lanes == 256 &&
        value != 1 && value != 2 && value != 4 && value != 8)
      return fail(AEGKV_EINVAL, "with 256 copy lanes the unroll must be 0, 1, 2, 4 or 8");
    if (key == AEGKV_TUNE_COPY_LANES && value == 256 && g_tune.copy_unroll != 0 &&
        g_tune.copy_unroll != 1 && g_tune.copy_unroll != 2 && g_tune.copy_unroll != 4 &&
        g_tune.copy_unroll != 8)
      return fail(AEGKV_EINVAL, "256 copy lanes take an unroll of 1, 2, 4 or 8");
    if (key == AEGKV_TUNE_COPY_UNROLL && value != 0 && !valid_copy_unroll(value))
      return fail(AEGKV_EINVAL, "copy unroll must be 0 (auto) or one of 1,2,3,4,5,6,8,10");
    if (key == AEGKV_TUNE_COPY_ORDER && value > 2)
      return fail(AEGKV_EINVAL, "copy order must be 0 (as given), 1 (by target) or 2 (by source)");
    if (key == AEGKV_TUNE_STAGED_DMA_STREAMS && value > kMaxDmaStreams)
      return fail(AEGKV_EINVAL, "staged DMA streams must be in [0, %d]", kMaxDmaStreams);
    if (key == AEGKV_TUNE_COPY_LDS_BYTES && value > kMaxLdsPerWorkgroup)
      return fail(AEGKV_EINVAL, "copy LDS reservation must be in [0, %lld]",
                  static_cast<long long>(kMaxLdsPerWorkgroup));
    if (key == AEGKV_TUNE_STAGED_SHORT_RUNS && value > 1)
      return fail(AEGKV_EINVAL, "tuning key %d takes 0 or 1", key);
    if (key == AEGKV_TUNE_SWAP_SHAPE_AUTO && value > 1)
      return fail(AEGKV_EINVAL, "swap shape selector is 0 or 1");
    if (key == AEGKV_TUNE_STAGED_OVERLAP && value > 3)
      return fail(AEGKV_EINVAL, "staged overlap is a 2-bit mask (0-3)");
    *slot = value;
  }
  return prev;
}

int aegkv_swap(const int64_t* source_block_ids, const int64_t* target_block_ids,
               int64_t num_ids, int is_swap_in, void* kv_cache, int64_t cache_num_blocks,
               void* kv_swap, int64_t swap_num_blocks, int64_t block_bytes, int mode,
               hipStream_t stream) {
  g_err[0] = '\0';
  if (int rc = env_status()) return rc;
  if (block_bytes <= 0) return fail(AEGKV_EINVAL, "block_bytes must be positive");
  void* bases[1] = {kv_cache};
  const int64_t page[1] = {block_bytes};
  const int64_t hoff[1] = {0};
  const uint64_t owner[1] = {1};
  const int64_t kpp[1] = {1};
  SwapLayout L{1, bases, page, hoff, owner, cache_num_blocks, 1, kpp,
               static_cast<char*>(kv_swap), swap_num_blocks, block_bytes, 0};
  SwapList E{num_ids, source_block_ids, target_block_ids, nullptr, nullptr, nullptr, nullptr};
  return swap_core(L, E, is_swap_in != 0, mode, stream);
}

int aegkv_swap_blocks(int32_t num_segments, void* const* segment_bases,
                      const int64_t* segment_page_bytes, const int64_t* segment_host_offsets,
                      const uint64_t* segment_owner_masks, int64_t device_num_blocks,
                      int32_t num_groups, const int64_t* group_kernel_blocks_per_page,
                      void* host_pool, int64_t host_num_blocks, int64_t host_page_bytes,
                      int64_t host_rank_offset, int64_t num_entries,
                      const int64_t* source_block_ids, const int64_t* target_block_ids,
                      const int32_t* group_ids, const int64_t* first_kernel_blocks,
                      const int64_t* valid_kernel_blocks, int is_swap_in, int mode,
                      const uint64_t* guard, hipStream_t stream) {
  g_err[0] = '\0';
  if (int rc = env_status()) return rc;
  if (num_entries > 0 && (!group_ids || !first_kernel_blocks || !valid_kernel_blocks))
    return fail(AEGKV_EINVAL, "entry metadata arrays must not be null");
  if (guard && (reinterpret_cast<uintptr_t>(guard) & 7u))
    return fail(AEGKV_EINVAL, "the move guard must be an 8-byte aligned word");
  SwapLayout L{num_segments, segment_bases, segment_page_bytes, segment_host_offsets,
               segment_owner_masks, device_num_blocks, num_groups,
               group_kernel_blocks_per_page, static_cast<char*>(host_pool), host_num_blocks,
               host_page_bytes, host_rank_offset};
  SwapList E{num_entries, source_block_ids, target_block_ids, group_ids, first_kernel_blocks,
             valid_kernel_blocks, guard};
  return swap_core(L, E, is_swap_in != 0, mode, stream);
}

int aegkv_copy_blocks(int32_t num_segments, void* const* segment_bases,
                      const int64_t* segment_page_bytes, int64_t device_num_blocks,
                      int64_t num_pairs, const int64_t* src_block_ids,
                      const int64_t* dst_block_ids, hipStream_t stream) {
  g_err[0] = '\0';
  if (int rc = env_status()) return rc;
  return copy_core(num_segments, segment_bases, segment_bases, segment_page_bytes,
                   device_num_blocks, device_num_blocks, num_pairs, src_block_ids,
                   dst_block_ids, true, stream);
}

int aegkv_copy_blocks_noalloc(int32_t num_segments, void* const* segment_bases,
                              const int64_t* segment_page_bytes, int64_t device_num_blocks,
                              int64_t num_pairs, const int64_t* src_block_ids,
                              const int64_t* dst_block_ids, hipStream_t stream) {
  g_err[0] = '\0';
  if (int rc = env_status()) return rc;
  return copy_noalloc(num_segments, segment_bases, segment_page_bytes, device_num_blocks,
                      num_pairs, src_block_ids, dst_block_ids, stream);
}

int aegkv_copy_probe(int kind, int32_t num_segments, void* const* segment_bases,
                     const int64_t* segment_page_bytes, int64_t device_num_blocks,
                     int64_t num_pairs, const int64_t* src_block_ids,
                     const int64_t* dst_block_ids, uint32_t* sink, uint32_t magic,
                     hipStream_t stream) {
  g_err[0] = '\0';
  if (int rc = env_status()) return rc;
  if (kind != AEGKV_PROBE_READ && kind != AEGKV_PROBE_WRITE)
    return fail(AEGKV_EINVAL, "probe kind %d is neither AEGKV_PROBE_READ nor AEGKV_PROBE_WRITE",
                kind);
  if (!sink || (reinterpret_cast<uintptr_t>(sink) & 3u))
    return fail(AEGKV_EINVAL, "the probe's sink must be a 4-byte aligned device word");
  CopyKind k;
  k.probe = kind == AEGKV_PROBE_READ ? PROBE_READ : PROBE_WRITE;
  k.sink = sink;
  k.magic = magic;
  return copy_core(num_segments, segment_bases, segment_bases, segment_page_bytes,
                   device_num_blocks, device_num_blocks, num_pairs, src_block_ids,
                   dst_block_ids, true, stream, k);
}

int aegkv_migrate_blocks(int32_t num_segments, void* const* src_segment_bases,
                         void* const* dst_segment_bases, const int64_t* segment_page_bytes,
                         int64_t src_num_blocks, int64_t dst_num_blocks, int64_t num_pairs,
                         const int64_t* src_block_ids, const int64_t* dst_block_ids,
                         const uint64_t* guard, hipStream_t stream) {
  g_err[0] = '\0';
  if (int rc = env_status()) return rc;
  if (!src_segment_bases || !dst_segment_bases)
    return fail(AEGKV_EINVAL, "segment arrays must not be null");
  if (guard && (reinterpret_cast<uintptr_t>(guard) & 7u))
    return fail(AEGKV_EINVAL, "the move guard must be an 8-byte aligned word");
  CopyKind k;
  k.guard = guard;
  return copy_core(num_segments, src_segment_bases, dst_segment_bases, segment_page_bytes,
                   src_num_blocks, dst_num_blocks, num_pairs, src_block_ids, dst_block_ids,
                   false, stream, k);
}

int aegkv_load_slices(int64_t num_slices, void* const* dst, const void* const* src,
                      const int64_t* bytes, int mode, hipStream_t stream) {
  g_err[0] = '\0';
  if (int rc = env_status()) return rc;
  return slices_core(num_slices, dst, src, bytes, mode, stream);
}

int aegkv_stream_create(hipStream_t* stream) {
  g_err[0] = '\0';
  if (!stream) return fail(AEGKV_EINVAL, "stream pointer must not be null");
  AEGKV_HIP(dedicated_stream(stream));
  return 0;
}

int aegkv_stream_create_masked(hipStream_t* stream, const uint32_t* cu_mask,
                               int32_t mask_words) {
  g_err[0] = '\0';
  if (!stream) return fail(AEGKV_EINVAL, "stream pointer must not be null");
  if (!cu_mask || mask_words <= 0) return fail(AEGKV_EINVAL, "CU mask must not be empty");
  int dev = -1, cus = 0;
  AEGKV_HIP(hipGetDevice(&dev));
  AEGKV_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  int64_t set = 0;
  for (int32_t w = 0; w < mask_words; ++w)
    for (int b = 0; b < 32; ++b)
      if ((cu_mask[w] >> b) & 1u) {
        if (int64_t(w) * 32 + b >= cus)
          return fail(AEGKV_ERANGE, "CU mask names CU %d; the device has %d", w * 32 + b, cus);
        ++set;
      }
  if (set == 0) return fail(AEGKV_EINVAL, "CU mask enables no CU");
  hipError_t e = hipExtStreamCreateWithCUMask(stream, static_cast<uint32_t>(mask_words), cu_mask);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return fail(static_cast<int>(e),
                "hipExtStreamCreateWithCUMask refused the mask (%s); the runtime takes runs "
                "of 8 or more consecutive CUs starting at a multiple of 8",
                hipGetErrorString(e));
  }
  return 0;
}

int aegkv_stream_release(hipStream_t stream) {
  g_err[0] = '\0';
  if (!stream) return fail(AEGKV_EINVAL, "stream must not be null");
  AEGKV_HIP(hipStreamSynchronize(stream));
  return forget_stream(stream);
}

int aegkv_stream_destroy(hipStream_t stream) {
  // the stream's queued work finishes first, whatever the caller dropped,
  // and no library event stays recorded on it
  if (int rc = aegkv_stream_release(stream)) return rc;
  AEGKV_HIP(hipStreamDestroy(stream));
  return 0;
}

int aegkv_init(void) {
  g_err[0] = '\0';
  int count = 0;
  if (hipGetDeviceCount(&count) != hipSuccess || count <= 0) {
    (void)hipGetLastError();
    return 0;  // no device: nothing to set up
  }
  int current = -1;
  AEGKV_HIP(hipGetDevice(&current));
  std::lock_guard<std::mutex> lk(g_noalloc_mu);
  // the current device first, with no device switch (a process with one
  // device never switches)
  int rc = current < kNoAllocMaxDevices ? noalloc_resolve(current) : 0;
  bool switched = false;
  for (int d = 0; d < count && d < kNoAllocMaxDevices && !rc; ++d) {
    if (d == current || g_scratch_ptr[d]) continue;
    const hipError_t e = hipSetDevice(d);
    switched = true;
    rc = e != hipSuccess ? hip_fail(e, "hipSetDevice") : noalloc_resolve(d);
  }
  if (switched) {
    const hipError_t e = hipSetDevice(current);
    if (!rc && e != hipSuccess) rc = hip_fail(e, "hipSetDevice");
  }
  return rc;
}

int aegkv_host_alloc(void** ptr, int64_t bytes) { return aegkv_host_alloc_flags(ptr, bytes, 0); }

int aegkv_host_alloc_flags(void** ptr, int64_t bytes, int flags) {
  g_err[0] = '\0';
  if (!ptr || bytes <= 0) return fail(AEGKV_EINVAL, "host_alloc needs a pointer and bytes > 0");
  if (flags & ~(AEGKV_HOST_UNCACHED | AEGKV_HOST_COHERENT))
    return fail(AEGKV_EINVAL, "unknown host_alloc flags 0x%x", flags);
  // hipHostMalloc refuses the pair; uncached memory bypasses every cache
  // already, and COHERENT is meant for cached pools
  if ((flags & AEGKV_HOST_UNCACHED) && (flags & AEGKV_HOST_COHERENT))
    return fail(AEGKV_EINVAL, "AEGKV_HOST_UNCACHED and AEGKV_HOST_COHERENT do not combine "
                "(uncached memory is coherent already)");
  const size_t n = static_cast<size_t>(bytes);
  const bool uncached = (flags & AEGKV_HOST_UNCACHED) != 0;
  unsigned hf = hipHostMallocMapped | hipHostMallocPortable;
  if (uncached) hf |= hipHostMallocUncached;
  if (flags & AEGKV_HOST_COHERENT) hf |= hipHostMallocCoherent;
  if (!uncached) {
    void* p = nullptr;
    AEGKV_HIP(hipHostMalloc(&p, n, hf));
    std::lock_guard<std::mutex> lk(g_host_mu);
    g_host_allocs[reinterpret_cast<uintptr_t>(p)] = n;
    *ptr = p;
    return 0;
  }
  const size_t want = (n + kHostPage - 1) / kHostPage * kHostPage;
  {
    // the smallest free range that fits
    std::lock_guard<std::mutex> lk(g_host_mu);
    auto best = g_uncached_free.end();
    for (auto it = g_uncached_free.begin(); it != g_uncached_free.end(); ++it)
      if (it->second >= want && (best == g_uncached_free.end() || it->second < best->second))
        best = it;
    if (best != g_uncached_free.end()) {
      const uintptr_t start = best->first;
      const size_t len = best->second;
      g_uncached_free.erase(best);
      if (len > want) g_uncached_free[start + want] = len - want;
      g_uncached_pools[start] = want;
      g_host_allocs[start] = n;
      *ptr = reinterpret_cast<void*>(start);
      return 0;
    }
  }
  void* p = nullptr;
  AEGKV_HIP(hipHostMalloc(&p, want, hf));
  std::lock_guard<std::mutex> lk(g_host_mu);
  const uintptr_t b = reinterpret_cast<uintptr_t>(p);
  g_uncached_blocks[b] = want;
  g_uncached_pools[b] = want;
  g_host_allocs[b] = n;
  *ptr = p;
  return 0;
}

int aegkv_host_usage(int64_t* pinned_bytes, int64_t* uncached_free_bytes) {
  g_err[0] = '\0';
  std::lock_guard<std::mutex> lk(g_host_mu);
  int64_t pinned = 0, free_bytes = 0;
  for (const auto& kv : g_host_allocs)
    if (!g_uncached_pools.count(kv.first)) pinned += static_cast<int64_t>(kv.second);
  for (const auto& kv : g_uncached_blocks) pinned += static_cast<int64_t>(kv.second);
  for (const auto& kv : g_uncached_free) free_bytes += static_cast<int64_t>(kv.second);
  if (pinned_bytes) *pinned_bytes = pinned;
  if (uncached_free_bytes) *uncached_free_bytes = free_bytes;
  return 0;
}

int aegkv_host_free(void* ptr) {
  g_err[0] = '\0';
  if (!ptr) return 0;
  {
    std::lock_guard<std::mutex> lk(g_host_mu);
    const uintptr_t b = reinterpret_cast<uintptr_t>(ptr);
    if (g_host_allocs.erase(b) == 0)
      return fail(AEGKV_EINVAL, "%p is not a live pool from aegkv_host_alloc", ptr);
    auto u = g_uncached_pools.find(b);
    if (u != g_uncached_pools.end()) {
      // back to the free list, merged with free neighbours of the same block
      uintptr_t start = b;
      size_t len = u->second;
      g_uncached_pools.erase(u);
      auto blk = g_uncached_blocks.upper_bound(start);
      --blk;  // the block holding the pool (every pool lies in one)
      const uintptr_t block_begin = blk->first, block_end = blk->first + blk->second;
      auto next = g_uncached_free.find(start + len);
      if (next != g_uncached_free.end() && start + len < block_end) {
        len += next->second;
        g_uncached_free.erase(next);
      }
      auto prev = g_uncached_free.lower_bound(start);
      if (prev != g_uncached_free.begin()) {
        --prev;
        if (prev->first >= block_begin && prev->first + prev->second == start) {
          prev->second += len;
          return 0;
        }
      }
      g_uncached_free[start] = len;
      return 0;
    }
  }
  AEGKV_HIP(hipHostFree(ptr));
  return 0;
}

}  // extern "C"
