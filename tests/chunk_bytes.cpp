// Cuts lists of square-root jobs into chunks and adds up what each chunk holds on
// the device: prints "<kind> <shape> <share> <jobs> <bytes held> <budget> <packed>"
// per chunk; share 1: the budget is what a served group of the jobs is admitted with.
#include <cstdio>
#include <vector>

#include "cac_ks.h"

using namespace cac;

namespace {

size_t admitted(const std::vector<SqrtJob>& jobs) {
  size_t b = 0;
  for (const SqrtJob& j : jobs) b += job_sample_bytes(j) + job_ks_bytes(j);
  return b;
}

void run(const char* kind, int shape, const std::vector<SqrtJob>& jobs) {
  for (size_t share = 1; share <= 3; ++share) {
    const size_t budget = admitted(jobs) / share;
    for (size_t first = 0; first < jobs.size();) {
      const SqrtChunk c = sqrt_chunk(jobs, first, budget, false, CAC_SAMPLE_LC);
      if (c.jobs == 0 || first + c.jobs > jobs.size()) {
        std::printf("%s %d %zu 0 1 0 0\n", kind, shape, share);
        return;
      }
      // the sampling scratch, the packed graphs, and the levels at the entry size
      // that the graph's weight gives
      size_t held = c.sample + c.pack;
      for (size_t i = first; i < first + c.jobs; ++i)
        held += ks_live_bytes_per_root(jobs[i].t, jobs[i].total < (1ull << 31));
      std::printf("%s %d %zu %zu %zu %zu %zu\n", kind, shape, share, c.jobs, held, budget, c.pack);
      first += c.jobs;
    }
  }
}

// Trials of `graphs` graphs of n vertices and m edges that weigh `total` each.
void add(std::vector<SqrtJob>& jobs, uint32_t graphs, uint32_t trials, uint32_t n, uint64_t m, uint64_t total) {
  static cac_edge edges[1 << 10];
  for (uint32_t g = 0; g < graphs; ++g)
    for (uint32_t i = 0; i < trials; ++i)
      jobs.push_back({edges + g, m, n, sqrt_intermediate_size(n, m), i, (uint32_t)jobs.size(), 0u, total});
}

}  // namespace

int main() {
  const uint64_t light = (1ull << 31) - 1, heavy = 1ull << 31;
  const struct {
    uint32_t graphs, trials, n;
    uint64_t m;
  } shapes[] = {{1, 2, 3000, 20000}, {5, 3, 500, 4000},     {3, 2, 60000, 900000}, {1, 3, 1000, 499500},
                {6, 7, 200, 19900},  {4, 2, 70000, 600000}, {2, 40, 90, 100000},   {1, 1, 90, 100000}};
  for (int k = 0; k < (int)(sizeof shapes / sizeof shapes[0]); ++k) {
    const auto& s = shapes[k];
    for (const uint64_t total : {light, heavy, kTotalUnknown}) {
      std::vector<SqrtJob> jobs;
      add(jobs, s.graphs, s.trials, s.n, s.m, total);
      run(total == light ? "light" : total == heavy ? "heavy" : "unknown", k, jobs);
    }
    // heavy trials, and trials of graphs too large to pack, beside light ones
    std::vector<SqrtJob> mixed;
    add(mixed, 1, 3, 70001, 50000, heavy);
    add(mixed, 2, 2, 3001, 30000, heavy);
    add(mixed, s.graphs, s.trials, s.n, s.m, light);
    run("mixed", k, mixed);
  }
  return 0;
}
