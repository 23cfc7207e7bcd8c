// Splits job sizes into chunks the way large square-root trials run: prints
// "<jobs> <kind> <room> <chunks> <largest chunk> <chunks at the full room>
// <all / chunks> <largest job>" per list and room.
#include <cstdio>
#include <vector>

#include "cac_ks.h"

namespace {

// Chunks of at most `room` bytes (one job always runs), and the largest one.
size_t split(const std::vector<size_t>& jobs, size_t room, size_t* largest) {
  size_t chunks = 0;
  *largest = 0;
  for (size_t i = 0; i < jobs.size(); ++chunks) {
    size_t held = jobs[i++];
    while (i < jobs.size() && held + jobs[i] <= room) held += jobs[i++];
    if (held > *largest) *largest = held;
  }
  return chunks;
}

}  // namespace

int main() {
  for (const size_t count : {1, 2, 3, 7, 15, 16, 17, 31, 156}) {
    for (int kind = 0; kind < 3; ++kind) {
      std::vector<size_t> jobs;
      size_t all = 0, most = 0;
      for (size_t i = 0; i < count; ++i) {
        const size_t b = kind == 0 ? 1000 : kind == 1 ? 100 + (i * 7919) % 901 : (i == 0 ? 5000 : 10);
        jobs.push_back(b);
        all += b;
        most = b > most ? b : most;
      }
      for (const size_t room : {(size_t)0, (size_t)1, (size_t)999, (size_t)1000, (size_t)1001, (size_t)3500, (size_t)14000,
                                (size_t)50000, (size_t)1 << 40}) {
        size_t largest = 0, greedy_largest = 0;
        const size_t share = cac::even_share(all, most, room);
        const size_t n = split(jobs, share, &largest), greedy = split(jobs, room, &greedy_largest);
        std::printf("%zu %d %zu %zu %zu %zu %zu %zu\n", count, kind, room, n, largest, greedy, all / n, most);
      }
    }
  }
  return 0;
}
