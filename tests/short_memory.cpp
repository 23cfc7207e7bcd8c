// Finds the least device memory with which the approximate cut of a path succeeds:
// hipMalloc is interposed and refuses what would pass a cap on the bytes held, from
// the host, as a full device would.  Prints "<least bytes> <approx> <trials>".
#include <dlfcn.h>

#include <cstdint>
#include <cstdio>
#include <map>
#include <mutex>
#include <vector>

#include "cac.h"

namespace {
std::mutex mu;
std::map<void*, size_t> held;
size_t live = 0, cap = ~size_t(0);
}  // namespace

extern "C" int hipMalloc(void** p, size_t bytes) {
  static auto real = (int (*)(void**, size_t))dlsym(RTLD_NEXT, "hipMalloc");
  std::lock_guard<std::mutex> lock(mu);
  if (live + bytes > cap) return 2;  // hipErrorOutOfMemory
  const int e = real(p, bytes);
  if (e == 0) {
    held[*p] = bytes;
    live += bytes;
  }
  return e;
}

extern "C" int hipFree(void* p) {
  static auto real = (int (*)(void*))dlsym(RTLD_NEXT, "hipFree");
  std::lock_guard<std::mutex> lock(mu);
  auto it = held.find(p);
  if (it != held.end()) {
    live -= it->second;
    held.erase(it);
  }
  return real(p);
}

namespace {

int bad(const char* what, int rc) {
  std::printf("%s: %d\n", what, rc);
  return 1;
}

// The least cap, to a hundredth, on the bytes beyond those held now, with which a
// fresh context's call succeeds; any other error than CAC_ENOMEM ends the search.
template <class Call>
int least(Call call, size_t high, size_t* out) {
  size_t low = 0;
  while (high - low > high / 100) {
    const size_t mid = low + (high - low) / 2;
    cac_ctx* ctx = nullptr;
    int rc = cac_ctx_create(0, &ctx);
    if (rc) return bad("context", rc);
    cap = live + mid;
    rc = call(ctx);
    cap = ~size_t(0);
    cac_ctx_destroy(ctx);
    if (rc != CAC_OK && rc != CAC_ENOMEM) return bad("call", rc);
    if (rc == CAC_OK) high = mid;
    else low = mid;
  }
  *out = high;
  return 0;
}

}  // namespace

int main() {
  const uint32_t n = 100000;  // a path of equal weights
  std::vector<cac_edge> e;
  for (uint32_t v = 0; v + 1 < n; ++v) e.push_back({v, v + 1, 64});
  uint64_t approx = 0;
  uint32_t trials = 0;
  size_t need = 0;
  if (least([&](cac_ctx* c) { return cac_approx_cut(c, e.data(), e.size(), n, 0.95, 7, &approx, &trials); },
            (size_t)1 << 26, &need))
    return 1;
  std::printf("%zu %llu %u\n", need, (unsigned long long)approx, trials);
  return 0;
}
