// The runs of host bytes that a STAGED swap leaves to the runtime's copies, and
// whether a call is cheaper moved as DIRECT. Host code only; a CPU test drives
// it.
#pragma once

#include <cstddef>
#include <cstdint>
#include <vector>

struct SwapLayout {
  int32_t num_segments;
  void* const* bases;
  const int64_t* page_bytes;
  const int64_t* host_offsets;
  const uint64_t* owner_masks;
  int64_t device_num_blocks;
  int32_t num_groups;
  const int64_t* kpp;
  char* host_pool;
  int64_t host_num_blocks;
  int64_t host_page_bytes;
  int64_t host_rank_offset;
};

struct SwapList {
  int64_t n;
  const int64_t* src;
  const int64_t* dst;
  const int32_t* group;     // may be null: all group 0
  const int64_t* first;     // may be null: all 0
  const int64_t* valid;     // may be null: all kpp[group]
  const uint64_t* guard;    // may be null: the kernels move nothing once *guard != 0
};

struct Run {
  int64_t host_off;   // byte offset inside the host pool
  int64_t stage_off;  // byte offset inside staging
  int64_t len;
  // Takes r in if it follows on both sides.
  bool join(const Run& r) {
    if (host_off + len != r.host_off || stage_off + len != r.stage_off) return false;
    len += r.len;
    return true;
  }
};

// The host extents of one staged entry in order, add(Run) for each.
template <typename Add>
void entry_extents(const SwapLayout& L, const SwapList& E, int64_t i, bool is_swap_in,
                   int64_t slot, int64_t composite, Add add) {
  const int32_t g = E.group ? E.group[i] : 0;
  const int64_t k = L.kpp[g];
  const int64_t first = E.first ? E.first[i] : 0;
  const int64_t valid = E.valid ? E.valid[i] : k;
  const int64_t host_id = is_swap_in ? E.src[i] : E.dst[i];
  const int64_t host_page = host_id * L.host_page_bytes + L.host_rank_offset;
  const int64_t stage_page = slot * composite;
  for (int32_t s = 0; s < L.num_segments; ++s) {
    if (!((L.owner_masks[s] >> g) & 1ull)) continue;
    const int64_t unit = L.page_bytes[s] / k;
    const int64_t off = unit * first, len = unit * valid;
    if (len != 0)
      add(Run{host_page + L.host_offsets[s] + off, stage_page + L.host_offsets[s] + off, len});
  }
}

// The runs of a staged chunk, order[lo, hi), in staging slots of their own:
// its extents, joined where they are contiguous.
inline void chunk_runs(const SwapLayout& L, const SwapList& E,
                       const std::vector<int64_t>& order, size_t lo, size_t hi, bool is_swap_in,
                       int64_t composite, std::vector<Run>& runs) {
  runs.clear();
  for (size_t j = lo; j < hi; ++j)
    entry_extents(L, E, order[j], is_swap_in, static_cast<int64_t>(j - lo), composite,
                  [&](const Run& r) {
                    if (runs.empty() || !runs.back().join(r)) runs.push_back(r);
                  });
}

// The runs of all chunks of a STAGED call, `step` entries each.
struct RunTotals {
  int64_t runs = 0, bytes = 0;
};

inline RunTotals call_runs(const SwapLayout& L, const SwapList& E,
                           const std::vector<int64_t>& order, bool is_swap_in,
                           int64_t composite, size_t step) {
  RunTotals t;
  Run last{};
  for (size_t j = 0; j < order.size(); ++j) {
    if (j % step == 0) last = Run{-1, -1, 0};
    entry_extents(L, E, order[j], is_swap_in, static_cast<int64_t>(j % step), composite,
                  [&](const Run& r) {
                    t.bytes += r.len;
                    if (last.join(r)) return;
                    last = r;
                    ++t.runs;
                  });
  }
  return t;
}

inline RunTotals run_totals(const std::vector<Run>& runs) {
  RunTotals t;
  t.runs = static_cast<int64_t>(runs.size());
  for (const Run& r : runs) t.bytes += r.len;
  return t;
}

// Up to four runs in one chunk leave nothing to overlap, so their copies go
// on the caller's stream, without the events that fork to the library's
// streams and back. One stream -> two (us a swap-out): five runs of 160 KiB 74
// -> 106, of 512 KiB 105 -> 127, of 2.3 MiB 268 -> 285; six 86 -> 108, 124 ->
// 136, 318 -> 327; eight 109 -> 118, 159 -> 160, 420 -> 410; twelve 153 -> 138,
// 231 -> 208, 622 -> 600; twenty 250 -> 194, 385 -> 337. With several callers in
// turn, where the runtime moves some copies at 29 GB/s, one run of 472 MB took
// 10.4 ms over two streams and takes 9.15.
constexpr int64_t kFewRuns = 4;

// Whether a STAGED call goes out as the DIRECT kernel: its runs are short, and
// the kernel takes no more from work beside it than the copies would.
//
// The runtime takes 3-7 us a copy, over two streams, so runs below 128 KiB on
// average stay at a third of the link rate or less, where the kernel has all
// of it: 60 runs of 32 KiB take 335 us staged and 38 direct, of 128 KiB 453
// and 141.
//
// STAGED is there to leave the CUs to other work, though. A bf16 8192^3 GEMM
// beside swaps one after another lost, us a swap (out / in, direct against
// staged, uncached pool): 60 runs of 32 KiB 4 / 7 against 8 / 5, 48 KiB 11 / 9
// against 11 / 10, 64 KiB 17 / 15 against 13 / 10, 128 KiB 45 / 46 against 18 /
// 12; 20 runs of 64 KiB 7 / 8 against 8 / 6, 128 KiB 10 / 11 against 13 / 12; 8 of
// 128 KiB 8 / 9 against 11 / 11; 400 of 24 KiB 63 / 66 against 59 / 41, 64 KiB 232 /
// 201 against 96 / 54. The kernel costs what it moves beyond a megabyte or
// two, the copies about the same at any length, so the line runs along 2 MiB
// and 16 KiB a run more.
constexpr int64_t kShortRun = int64_t(128) << 10;
constexpr int64_t kDirectBytes = int64_t(2) << 20;
constexpr int64_t kDirectBytesPerRun = int64_t(16) << 10;

inline bool cheap_as_direct(const RunTotals& t) {
  return t.runs > kFewRuns && t.bytes < kShortRun * t.runs &&
         t.bytes <= kDirectBytes + kDirectBytesPerRun * t.runs;
}
