// The work items of a block copy: how many there are, in which order they are
// taken and which bytes each moves. The host lays the walk out (lay_walk),
// the kernels follow it (copy_item), and a CPU test enumerates it.
//
// The walk goes segment by segment, the pairs of one segment in the order of
// the descriptor, the chunks of one tile in address order. Workgroups are
// handed to the 8 XCDs in turn, so the items of a class below remap_end are
// renumbered to give every XCD whole runs of 2^run_shift consecutive items:
// with pairs in target order each XCD then writes one stretch of one segment
// at a time.
//
// HBM bounds the copy, and this order is what it answers best. Random halves
// of a cache, against pairs-first items over the whole chip (TB/s, read plus
// written, 4 KiB items): 160 KiB tiles 5.24 -> 6.45, 64 KiB 5.87 -> 6.19,
// 32 KiB 5.44 -> 5.88, 20 KiB 5.36 -> 6.01, 16 KiB 5.43 -> 5.99, 4 KiB
// 5.60 -> 6.15. Segment order alone gives 0-6 % of that, runs alone 2-4 %.
// (Measured with streaming stores; Words has what storing through adds.)
//
// Segments are grouped by the chunks their pages take, a class each, largest
// first, and every class is walked by itself.
#pragma once

#include <cstdint>

#ifdef __HIP__
#define AEGKV_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define AEGKV_HOST_DEVICE inline
#endif

// Work items one launch may hold. The kernels walk items with a 32-bit
// grid-stride loop (w += gridDim.x) over at most (2^32 - 1) / 256 workgroups,
// so with at most this many items, w + gridDim.x stays below 2^32 and the
// loop never wraps.
constexpr int64_t kMaxLaunchItems =
    static_cast<int64_t>(UINT32_MAX) - static_cast<int64_t>(UINT32_MAX) / 256;

// a * b * c work items, or -1 when that exceeds kMaxLaunchItems (or overflows).
inline int64_t launch_items(int64_t a, int64_t b, int64_t c) {
  if (a < 0 || b < 0 || c < 0) return -1;
  if (a == 0 || b == 0 || c == 0) return 0;
  if (a > kMaxLaunchItems / b) return -1;
  const int64_t ab = a * b;
  if (ab > kMaxLaunchItems / c) return -1;
  return ab * c;
}

// Tiles whose addresses or lengths are no multiples of 16 (a cache whose
// pages end in a scale, a pool that starts anywhere) are cut into chunks
// where their *target* crosses 16-byte boundaries: only the first chunk of a
// tile starts and only its last one ends inside a 16-byte word.
struct Extent {
  int64_t begin;
  uint32_t nbytes;
};

// Chunk `c` of a `len`-byte tile; the chunk numbered `last` takes the rest.
template <int64_t kChunk>
AEGKV_HOST_DEVICE Extent any_chunk(const char* dst_tile, int64_t len, uint32_t c, uint32_t last) {
  const int64_t head = static_cast<int64_t>(-reinterpret_cast<uintptr_t>(dst_tile) & 15u);
  const int64_t begin = c ? head + static_cast<int64_t>(c) * kChunk : 0;
  const int64_t next = head + (static_cast<int64_t>(c) + 1) * kChunk;
  const int64_t end = (c == last || next > len) ? len : next;
  return {begin, begin < end ? static_cast<uint32_t>(end - begin) : 0u};
}

// Chunks of a page's tiles. Unaligned tiles: the last chunk takes up to half
// a chunk more, so that a few bytes over do not cost a wave of their own.
inline int64_t tile_chunks(int64_t page, int64_t chunk, bool vec) {
  if (vec) return (page + chunk - 1) / chunk;
  const int64_t n = (page + chunk / 2) / chunk;
  return n > 0 ? n : 1;
}

// Consecutive segments whose tiles are cut into equally many chunks. A cache
// with one page size is one class, held in CopyWalk itself; further ones
// follow in a table. With the chunks of the largest page for every tile, the
// others' workgroups were empty: beside 63 tensors of 16 KiB pages one of 160
// KiB left 88 % of them so, and 1500 pairs took 2.29 ms where they now take
// 0.58 (6.2 TB/s, read plus written); 160 KiB, 16 KiB and 512 bytes in equal
// number 2.66 -> 1.69 ms, 41,984 and 8,448 bytes 0.96 -> 0.79.
struct alignas(32) CopyClass {
  uint32_t first_item, end;
  uint32_t first_segment, chunks_per_tile;
  uint32_t remap_end;  // counted from first_item, as the renumbering is
  uint32_t run_shift;
};
static_assert(sizeof(CopyClass) == 32, "CopyClass layout");

constexpr int kCopyClasses = 8;  // further sizes share the next larger one's

struct CopyWalk {
  uint32_t num_pairs;
  uint32_t num_items;
  uint32_t chunks_per_tile, remap_end, run_shift;  // the first class
  uint32_t first_end;                              // its items
};

struct CopyClasses {  // the others
  CopyClass at[kCopyClasses - 1];
};

struct OneClass {};  // in their place where there are none

struct CopyItem {
  uint32_t pair, segment, chunk, last;
};

// Item w of a class, counted from its first.
AEGKV_HOST_DEVICE CopyItem class_item(uint32_t num_pairs, uint32_t first_segment, uint32_t chunks,
                                      uint32_t remap_end, uint32_t shift, uint32_t w) {
  if (w < remap_end) {
    const uint32_t r = w & ((8u << shift) - 1u);
    w = w - r + ((r & 7u) << shift) + (r >> 3);
  }
  const uint32_t tile = w / chunks;
  const uint32_t s = tile / num_pairs;
  return {tile - s * num_pairs, first_segment + s, w - tile * chunks, chunks - 1};
}

// Item w (below num_items). `classes`: those behind the first one.
AEGKV_HOST_DEVICE CopyItem copy_item(const CopyWalk& k, OneClass, uint32_t w) {
  return class_item(k.num_pairs, 0, k.chunks_per_tile, k.remap_end, k.run_shift, w);
}

template <typename Classes>
AEGKV_HOST_DEVICE CopyItem copy_item(const CopyWalk& k, Classes classes, uint32_t w) {
  if (w < k.first_end) return copy_item(k, OneClass{}, w);
  uint32_t i = 0;
  while (w >= classes[i].end) ++i;
  return class_item(k.num_pairs, classes[i].first_segment, classes[i].chunks_per_tile,
                    classes[i].remap_end, classes[i].run_shift, w - classes[i].first_item);
}

// A walk as the host lays it out. The descriptor holds the segments class by
// class.
struct CopyLayout {
  CopyWalk walk;
  CopyClasses classes;
  uint32_t num_classes;               // behind the first one
  int64_t chunks[kCopyClasses];       // of every class, largest first
  // the class of a page of n chunks
  int class_of(int64_t n) const {
    int i = 0;
    while (i < static_cast<int>(num_classes) && n <= chunks[i + 1]) ++i;
    return i;
  }
};

// The walk over num_pairs pairs of the given pages (above 0) in items of
// `chunk` bytes, false where they are more than one launch holds. Needs no
// memory: callers that cannot allocate use it.
//
// A class's runs hold about 32 tiles: from 8 to 512 the rate moves by 2 %
// (least at 8 and 512 on 4-20 KiB tiles).
inline bool lay_walk(const int64_t* page_bytes, int32_t num_segments, int64_t num_pairs,
                     int64_t chunk, bool vec, CopyLayout* out) {
  // the different chunk counts, largest first; two that lie close become one
  // where there are more than the table holds
  constexpr int kSizes = 32;
  int64_t count[kSizes + 1] = {}, segments[kSizes + 1] = {};
  int n = 0;
  auto merge = [&] {
    int best = 1;
    for (int i = 2; i < n; ++i)
      if ((count[i - 1] - count[i]) * segments[i] <
          (count[best - 1] - count[best]) * segments[best])
        best = i;
    segments[best - 1] += segments[best];
    for (int i = best; i + 1 < n; ++i) {
      count[i] = count[i + 1];
      segments[i] = segments[i + 1];
    }
    --n;
  };
  int at = -1;  // the last segment's count
  for (int32_t s = 0; s < num_segments; ++s) {
    if (at >= 0 && page_bytes[s] == page_bytes[s - 1]) {
      ++segments[at];
      continue;
    }
    const int64_t c = tile_chunks(page_bytes[s], chunk, vec);
    if (launch_items(num_pairs, 1, c) < 0) return false;
    at = 0;
    while (at < n && count[at] > c) ++at;
    if (at == n || count[at] != c) {
      for (int j = n; j > at; --j) {
        count[j] = count[j - 1];
        segments[j] = segments[j - 1];
      }
      count[at] = c;
      segments[at] = 0;
      ++n;
    }
    ++segments[at];
    if (n > kSizes) {
      merge();
      at = -1;
    }
  }
  while (n > kCopyClasses) merge();
  out->num_classes = static_cast<uint32_t>(n - 1);
  for (int i = 0; i < n; ++i) out->chunks[i] = count[i];
  if (n > 1) {  // a joined size may have come again
    for (int i = 0; i < n; ++i) segments[i] = 0;
    for (int32_t s = 0; s < num_segments; ++s)
      ++segments[out->class_of(tile_chunks(page_bytes[s], chunk, vec))];
  }
  int64_t items = 0, segment = 0;
  for (int i = 0; i < n; ++i) {
    const int64_t mine = launch_items(num_pairs, segments[i], count[i]);
    if (mine < 0 || mine > kMaxLaunchItems - items) return false;
    uint32_t shift = 5;
    while (shift < 20 && (int64_t(1) << shift) < 32 * count[i]) ++shift;
    const int64_t span = int64_t(8) << shift;
    const CopyClass k{static_cast<uint32_t>(items),   static_cast<uint32_t>(items + mine),
                      static_cast<uint32_t>(segment), static_cast<uint32_t>(count[i]),
                      static_cast<uint32_t>(mine / span * span), shift};
    if (i == 0)
      out->walk = CopyWalk{static_cast<uint32_t>(num_pairs), 0, k.chunks_per_tile, k.remap_end,
                           k.run_shift, k.end};
    else
      out->classes.at[i - 1] = k;
    items += mine;
    segment += segments[i];
  }
  out->walk.num_items = static_cast<uint32_t>(items);
  return true;
}
