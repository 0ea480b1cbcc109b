// Drives the run counting of STAGED swaps (aegaeon_amd/csrc/staged_runs.h) on
// the CPU, built with sanitizers by tests/test_native_sanitized.py: the totals
// of a call are those of its chunks, and whether it goes DIRECT is decided by
// all of its runs, not by those of its first chunk. Prints "clean".

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <numeric>
#include <random>
#include <vector>

#include "staged_runs.h"

#define CHECK(c)                                                           \
  do {                                                                     \
    if (!(c)) {                                                            \
      std::fprintf(stderr, "check failed at line %d: %s\n", __LINE__, #c); \
      std::exit(1);                                                        \
    }                                                                      \
  } while (0)

constexpr int64_t K = 1024;

// One tensor of `page` bytes; entries in host-id order at the given host ids.
struct OneTensor {
  int64_t page[1], offset[1] = {0}, kpp[1] = {1};
  uint64_t owner[1] = {1};
  std::vector<int64_t> host, order;
  SwapLayout L{};
  SwapList E{};
  OneTensor(int64_t bytes, std::vector<int64_t> ids) : page{bytes}, host(std::move(ids)) {
    std::sort(host.begin(), host.end());
    order.resize(host.size());
    std::iota(order.begin(), order.end(), 0);
    L.num_segments = 1;
    L.page_bytes = page;
    L.host_offsets = offset;
    L.owner_masks = owner;
    L.num_groups = 1;
    L.kpp = kpp;
    L.host_page_bytes = bytes;
    E.n = static_cast<int64_t>(host.size());
    E.src = E.dst = host.data();
  }
  RunTotals first_chunk(size_t step) const {
    std::vector<Run> runs;
    chunk_runs(L, E, order, 0, std::min(step, order.size()), false, page[0], runs);
    return run_totals(runs);
  }
  RunTotals all(size_t step) const { return call_runs(L, E, order, false, page[0], step); }
};

std::vector<int64_t> ids(int64_t first, int64_t n, int64_t stride) {
  std::vector<int64_t> v;
  for (int64_t i = 0; i < n; ++i) v.push_back(first + i * stride);
  return v;
}

std::vector<int64_t> both(std::vector<int64_t> a, const std::vector<int64_t>& b) {
  a.insert(a.end(), b.begin(), b.end());
  return a;
}

int main() {
  // the line: short runs, up to 2 MiB and 16 KiB a run more, more than four
  CHECK(!cheap_as_direct({4, 4 * K}) && cheap_as_direct({5, 5 * K}));
  CHECK(cheap_as_direct({480, 480 * 9 * K}) && cheap_as_direct({60, 60 * 40 * K}));
  CHECK(cheap_as_direct({128, 128 * 32 * K}) && !cheap_as_direct({128, 128 * 32 * K + 1}));
  CHECK(!cheap_as_direct({400, 400 * 64 * K}) && !cheap_as_direct({60, 60 * 96 * K}));
  CHECK(!cheap_as_direct({5, 5 * 128 * K}) && cheap_as_direct({5, 5 * 128 * K - 1}));
  CHECK(!cheap_as_direct({0, 0}));

  // scattered pages first, long runs behind them: not DIRECT for the first
  // chunk's sake
  OneTensor long_behind(64 * K, both(ids(0, 8, 2), ids(100, 200, 1)));
  CHECK(cheap_as_direct(long_behind.first_chunk(8)));
  CHECK(!cheap_as_direct(long_behind.all(8)));
  CHECK(long_behind.all(8).runs == 8 + 25 && long_behind.all(8).bytes == 208 * 64 * K);
  // one long run first, scattered pages behind it: DIRECT in spite of it
  OneTensor short_behind(16 * K, both(ids(0, 8, 1), ids(100, 100, 3)));
  CHECK(!cheap_as_direct(short_behind.first_chunk(8)));
  CHECK(cheap_as_direct(short_behind.all(8)));

  // random layouts: the totals are those of the chunks
  std::mt19937_64 rng(11);
  auto rnd = [&](int64_t lo, int64_t hi) {  // inclusive
    return std::uniform_int_distribution<int64_t>(lo, hi)(rng);
  };
  for (int it = 0; it < 2000; ++it) {
    const int32_t S = static_cast<int32_t>(rnd(1, 6)), G = static_cast<int32_t>(rnd(1, 3));
    std::vector<int64_t> page(S), offset(S), kpp(G);
    std::vector<uint64_t> owner(S);
    for (auto& k : kpp) k = rnd(1, 2) * 2;
    int64_t composite = 0;
    for (int s = 0; s < S; ++s) {
      page[s] = 4 * rnd(1, 50);
      offset[s] = composite;
      composite += page[s];
      owner[s] = static_cast<uint64_t>(rnd(1, (1 << G) - 1));
    }
    const int64_t n = rnd(1, 40);
    std::vector<int64_t> host(60), first(n), valid(n), order(n);
    std::vector<int32_t> group(n);
    std::iota(host.begin(), host.end(), 0);
    std::shuffle(host.begin(), host.end(), rng);
    host.resize(n);
    if (rnd(0, 1)) std::sort(host.begin(), host.end());
    int64_t bytes = 0;
    for (int64_t i = 0; i < n; ++i) {
      group[i] = static_cast<int32_t>(rnd(0, G - 1));
      first[i] = rnd(0, kpp[group[i]]);
      valid[i] = rnd(0, kpp[group[i]] - first[i]);
      order[i] = i;
      for (int s = 0; s < S; ++s)
        if ((owner[s] >> group[i]) & 1) bytes += page[s] / kpp[group[i]] * valid[i];
    }
    std::sort(order.begin(), order.end(), [&](int64_t a, int64_t b) { return host[a] < host[b]; });
    const SwapLayout L{S, nullptr, page.data(), offset.data(), owner.data(), 60, G, kpp.data(),
                       nullptr, 60, composite + rnd(0, 1) * 8, 0};
    const SwapList E{n, host.data(), host.data(), group.data(), first.data(), valid.data(),
                     nullptr};
    for (bool in : {false, true}) {
      const size_t step = static_cast<size_t>(rnd(1, n));
      RunTotals sum;
      std::vector<Run> runs;
      for (size_t lo = 0; lo < order.size(); lo += step) {
        chunk_runs(L, E, order, lo, std::min(order.size(), lo + step), in, composite, runs);
        const RunTotals t = run_totals(runs);
        sum.runs += t.runs;
        sum.bytes += t.bytes;
        for (size_t r = 1; r < runs.size(); ++r)
          CHECK(runs[r].stage_off >= runs[r - 1].stage_off + runs[r - 1].len);
      }
      const RunTotals t = call_runs(L, E, order, in, composite, step);
      CHECK(t.runs == sum.runs && t.bytes == sum.bytes && t.bytes == bytes);
    }
  }
  std::printf("clean\n");
  return 0;
}
