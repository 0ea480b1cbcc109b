// Enumerates the walk of a block copy (aegaeon_amd/csrc/copy_walk.h) on the
// CPU, built with sanitizers by tests/test_native_sanitized.py: every byte of
// every tile belongs to exactly one item, items without any bytes are few,
// and launch limits are refused. Prints "clean".

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "copy_walk.h"

#define CHECK(c)                                                           \
  do {                                                                     \
    if (!(c)) {                                                            \
      std::fprintf(stderr, "check failed at line %d: %s\n", __LINE__, #c); \
      std::exit(1);                                                        \
    }                                                                      \
  } while (0)

// Share of items without bytes of one walk in chunks of kChunk bytes; tiles
// start `shift` bytes behind a 16-byte boundary (0 where they are aligned).
template <int64_t kChunk>
double walk(const std::vector<int64_t>& pages, int64_t pairs, bool vec, int shift) {
  const int32_t S = static_cast<int32_t>(pages.size());
  CopyLayout l;
  CHECK(lay_walk(pages.data(), S, pairs, kChunk, vec, &l));
  CHECK(l.num_classes < static_cast<uint32_t>(kCopyClasses));
  // the segments as the descriptor holds them
  std::vector<int64_t> held;
  for (int k = 0; k <= static_cast<int>(l.num_classes); ++k)
    for (int64_t p : pages)
      if (l.class_of(tile_chunks(p, kChunk, vec)) == k) held.push_back(p);
  CHECK(held.size() == pages.size());
  // per tile, its extents
  std::vector<std::vector<std::pair<int64_t, int64_t>>> got(static_cast<size_t>(S * pairs));
  int64_t empty = 0;
  for (uint32_t w = 0; w < l.walk.num_items; ++w) {
    const CopyItem it = l.num_classes ? copy_item(l.walk, l.classes.at, w)
                                      : copy_item(l.walk, OneClass{}, w);
    CHECK(it.segment < static_cast<uint32_t>(S) && it.pair < pairs && it.chunk <= it.last);
    const int64_t page = held[it.segment];
    int64_t begin = static_cast<int64_t>(it.chunk) * kChunk;
    int64_t n = std::max<int64_t>(0, std::min<int64_t>(page - begin, kChunk));
    if (!vec) {
      const char* at = reinterpret_cast<const char*>(uintptr_t(4096 + shift));
      const Extent x = any_chunk<kChunk>(at, page, it.chunk, it.last);
      begin = x.begin;
      n = x.nbytes;
      CHECK(n <= kChunk + kChunk / 2 + 15);
    }
    if (n == 0)
      ++empty;
    else
      got[it.segment * pairs + it.pair].push_back({begin, n});
  }
  for (int32_t s = 0; s < S; ++s)
    for (int64_t p = 0; p < pairs; ++p) {
      auto& x = got[s * pairs + p];
      std::sort(x.begin(), x.end());
      int64_t at = 0;
      for (auto& e : x) {
        CHECK(e.first == at);
        at += e.second;
      }
      CHECK(at == held[s]);
    }
  return static_cast<double>(empty) / l.walk.num_items;
}

double walk_any(int64_t chunk, const std::vector<int64_t>& pages, int64_t pairs, bool vec,
                int shift = 0) {
  switch (chunk) {
    case 1024: return walk<1024>(pages, pairs, vec, shift);
    case 4096: return walk<4096>(pages, pairs, vec, shift);
    case 8192: return walk<8192>(pages, pairs, vec, shift);
    default: return walk<163840>(pages, pairs, vec, shift);
  }
}

std::vector<int64_t> times(int n, std::vector<int64_t> of) {
  std::vector<int64_t> out;
  for (int i = 0; i < n; ++i) out.insert(out.end(), of.begin(), of.end());
  return out;
}

int main() {
  const int64_t K = 1024;
  // caches of several page sizes leave no item empty
  std::vector<int64_t> one_large(64, 16 * K), state(8, 16 * K);
  one_large[5] = 160 * K;
  state[0] = 2048 * K;
  for (int64_t pairs : {1, 3, 24, 67}) {
    for (int64_t chunk : {1024, 4096}) {
      CHECK(walk_any(chunk, times(40, {160 * K}), pairs, true) == 0);
      CHECK(walk_any(chunk, times(20, {64 * K, 8 * K}), pairs, true) == 0);
      CHECK(walk_any(chunk, times(4, {160 * K, 16 * K, 512}), pairs, true) == 0);
      CHECK(walk_any(chunk, times(16, {41984, 8448}), pairs, true) == 0);
      CHECK(walk_any(chunk, one_large, pairs, true) == 0);
      CHECK(walk_any(chunk, state, pairs, true) == 0);
    }
    CHECK(walk_any(163840, one_large, pairs, true) == 0);
    for (int shift : {0, 1, 15})
      CHECK(walk_any(1024, times(5, {20484, 1028, 33, 1}), pairs, false, shift) == 0);
  }
  // more sizes than classes, and more than are told apart: few empty ones
  std::vector<int64_t> ten, many;
  for (int64_t k = 1; k <= 10; ++k) ten.push_back(16 * K * k);
  for (int64_t k = 1; k <= 70; ++k) many.push_back(K * ((k * 37) % 71));
  CHECK(walk_any(4096, times(3, ten), 9, true) < 0.08);
  // (70 evenly spread sizes in 8 classes as even as can be: 4 of 39.5 chunks a
  // tile, 10 %; the sizes are joined as they come)
  CHECK(walk_any(1024, many, 9, true) < 0.2);
  CHECK(walk_any(1024, times(2, many), 2, false, 7) < 0.2);
  // random mixtures
  std::mt19937_64 rng(7);
  auto rnd = [&](int64_t lo, int64_t hi) {  // inclusive
    return std::uniform_int_distribution<int64_t>(lo, hi)(rng);
  };
  for (int it = 0; it < 300; ++it) {
    std::vector<int64_t> sizes, pages;
    const bool vec = rnd(0, 1);
    for (int64_t i = rnd(1, 12); i > 0; --i)
      sizes.push_back(vec ? 16 * rnd(1, 4000) : rnd(1, 40000));
    for (int64_t i = rnd(1, 50); i > 0; --i) pages.push_back(sizes[rnd(0, sizes.size() - 1)]);
    const int64_t chunks[] = {1024, 4096, 8192, 163840};
    walk_any(chunks[rnd(0, 3)], pages, rnd(1, 40), vec, static_cast<int>(rnd(0, 15)));
  }
  // what one launch holds
  const int64_t huge[] = {4096, 1024};
  CopyLayout l;
  CHECK(lay_walk(huge, 1, kMaxLaunchItems, 4096, true, &l) &&
        l.walk.num_items == kMaxLaunchItems);
  CHECK(!lay_walk(huge, 1, kMaxLaunchItems + 1, 4096, true, &l));
  CHECK(!lay_walk(huge, 2, kMaxLaunchItems / 2 + 1, 4096, true, &l));
  CHECK(!lay_walk(huge, 2, kMaxLaunchItems / 4, 1024, true, &l));   // 4 + 1 chunks a pair
  CHECK(lay_walk(huge, 2, kMaxLaunchItems / 5, 1024, true, &l) &&
        l.walk.first_end == kMaxLaunchItems / 5 * 4);
  std::printf("clean\n");
  return 0;
}
