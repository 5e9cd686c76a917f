// Checks graph_item (halloc_amd/csrc/ha_workload.h) against the sequence spelled
// out: builds in chunk order, each job's frees behind the build `lag` chunks
// after its last.
#include <cstdio>
#include <random>
#include <vector>

#include "../../halloc_amd/csrc/ha_workload.h"

using ha::u32;
using ha::u64;

int main() {
  std::mt19937 rng(7);
  for (u32 trial = 0; trial < 4000; ++trial) {
    const u32 njobs = 1 + rng() % (trial % 3 ? 9 : 70), most = 1 + rng() % (trial % 2 ? 3 : 40);
    std::vector<u32> offs(1, 0);
    for (u32 j = 0; j < njobs; ++j) offs.push_back(offs.back() + 1 + rng() % most);
    const u32 n = offs.back();
    const u64 lags[] = {1, 2, 3, n, n + 1ull, 2ull * n, 1ull << 33, 1 + rng() % (n + 1)};
    for (u64 lag : lags) {
      std::vector<u64> want, got(2 * (size_t)n, ~0ull);
      std::vector<bool> freed(njobs, false);
      auto frees = [&](u32 j) {
        for (u32 c = 0; c < offs[j + 1] - offs[j]; ++c) want.push_back(ha::GRAPH_FREE_ITEM | (u64)j << 32 | c);
        freed[j] = true;
      };
      for (u32 j = 0, b = 0; j < njobs; ++j)
        for (; b < offs[j + 1]; ++b) {
          want.push_back((u64)j << 32 | (b - offs[j]));
          for (u32 i = 0; i < njobs; ++i)
            if (offs[i + 1] - 1 + lag == b) frees(i);
        }
      for (u32 i = 0; i < njobs; ++i)
        if (!freed[i]) frees(i);
      for (u32 b = 0; b < n; ++b) {
        const ha::GraphItem g = ha::graph_item(offs.data(), njobs, lag, b);
        if (g.build_at >= got.size() || g.free_at >= got.size()) {
          std::printf("trial %u: place out of range\n", trial);
          return 1;
        }
        got[g.build_at] = g.item;
        got[g.free_at] = g.item | ha::GRAPH_FREE_ITEM;
      }
      if (got != want) {
        std::printf("trial %u: %u jobs, %u chunks, lag %llu\n", trial, njobs, n, (unsigned long long)lag);
        return 1;
      }
    }
  }
  std::printf("ok\n");
  return 0;
}
