// ha_workload.h -- workload arithmetic shared by the device drivers and the
// host tests: the Poisson(8) inversion table of the random-graph degrees, and
// the order in which the batched graph form builds and frees.
#pragma once

#include <cstdint>

#include "ha_bits.h"

namespace ha {

constexpr uint32_t POISSON8_N = 40;  // P(X >= 40) < 1e-14 for X ~ Poisson(8)

// t[k] = floor(2^24 * P(X <= k)), X ~ Poisson(8); a degree is the number of
// t[k] at or below a uniform 24-bit integer
struct PoissonCdf {
  uint32_t t[POISSON8_N];
};
constexpr PoissonCdf poisson8_cdf() {
  PoissonCdf c{};
  double p = 3.3546262790251185e-4;  // P(X = 0) = exp(-8)
  double cum = 0.0;
  for (uint32_t k = 0; k < POISSON8_N; ++k) {
    cum += p;
    c.t[k] = cum >= 1.0 ? 0x1000000u : (uint32_t)(cum * 16777216.0);
    p = p * 8.0 / (double)(k + 1);
  }
  return c;
}
constexpr PoissonCdf kPoisson8 = poisson8_cdf();

// The batched graph form's item sequence.  Chunks are numbered over all jobs,
// job j's are offs[j] .. offs[j + 1] - 1, every job has at least one.  Builds
// come in chunk order, and each job's frees directly behind the build that
// comes `lag` chunks after the job's last (behind the last build if there is
// none).  So the build of chunk b has before it the builds 0 .. b - 1 and the
// frees of the jobs that end at or before chunk b - lag, which are the chunks
// below the start of the job that holds chunk b - lag; and the free of job j's
// chunk c has before it the builds up to its place, and the frees of the
// jobs before j and of j's chunks before c.

// the job that holds x: offs[lo] <= x < offs[lo + 1] (offs[0] = 0)
template <class T>
HA_HD inline u32 job_at(const T* offs, u32 njobs, u64 x) {
  u32 lo = 0, hi = njobs;
  while (hi - lo > 1) {
    const u32 mid = (lo + hi) / 2;
    if ((u64)offs[mid] <= x) lo = mid;
    else hi = mid;
  }
  return lo;
}
constexpr u64 GRAPH_FREE_ITEM = 1ull << 63;  // else a build; job << 32 | chunk of the job
struct GraphItem {
  u64 item;            // the chunk's build; its free is this | GRAPH_FREE_ITEM
  u64 build_at, free_at;  // their places in the sequence of 2 * offs[njobs] items
};
HA_HD inline GraphItem graph_item(const u32* offs, u32 njobs, u64 lag, u32 b) {
  const u32 j = job_at(offs, njobs, b), n = offs[njobs];
  const u64 behind = (u64)offs[j + 1] + lag;
  GraphItem g;
  g.item = (u64)j << 32 | (b - offs[j]);
  g.build_at = b + (b >= lag ? (u64)offs[job_at(offs, njobs, b - lag)] : 0);
  g.free_at = (behind < n ? behind : n) + b;
  return g;
}

}  // namespace ha
