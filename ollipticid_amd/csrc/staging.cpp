// See staging.hpp.
#include "staging.hpp"

#include <cstring>
#include <mutex>
#include <new>
#include <thread>

namespace oll {

namespace {
constexpr int kKeep = 16;
constexpr int kCopyThreads = 4;
constexpr size_t kThreadBytes = size_t(256) << 10;  // least share of a thread

std::mutex g_mu;
Staging *g_idle[kKeep];
int g_nidle = 0;
int g_handles = 0;

void destroy(Staging *s) {
  if (!s) return;
  for (char *p : s->half)
    if (p) (void)hipHostFree(p);
  delete s;
}
}  // namespace

hipError_t (*staging_malloc)(void **, size_t, unsigned) = hipHostMalloc;

Staging *staging_take(int halves) {
  Staging *s = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_mu);
    if (g_nidle > 0) s = g_idle[--g_nidle];
  }
  if (!s && !(s = new (std::nothrow) Staging())) return nullptr;
  for (int i = 0; i < halves; ++i) {
    char *&p = s->half[i];
    if (!p && staging_malloc(reinterpret_cast<void **>(&p), Staging::kBytes, hipHostMallocPortable) != hipSuccess) {
      (void)hipGetLastError();  // no later check reports it
      p = nullptr;
      destroy(s);
      return nullptr;
    }
  }
  return s;
}

void staging_give(Staging *s) {
  if (!s) return;
  {
    std::lock_guard<std::mutex> lock(g_mu);
    if (g_nidle < kKeep && g_nidle < g_handles) {
      g_idle[g_nidle++] = s;
      return;
    }
  }
  destroy(s);
}

void staging_retain() {
  std::lock_guard<std::mutex> lock(g_mu);
  ++g_handles;
}

void staging_release() {
  Staging *drop[kKeep];
  int n = 0;
  {
    std::lock_guard<std::mutex> lock(g_mu);
    --g_handles;
    while (g_nidle > g_handles) drop[n++] = g_idle[--g_nidle];
  }
  while (n > 0) destroy(drop[--n]);
}

void host_copy(void *dst, const void *src, size_t bytes) {
  char *d = static_cast<char *>(dst);
  const char *s = static_cast<const char *>(src);
  std::thread th[kCopyThreads - 1];
  size_t begin = 0;
  int started = 0;
  const size_t share = bytes / kCopyThreads / 4096 * 4096;
  if (share >= kThreadBytes) {
    try {
      for (; started < kCopyThreads - 1; ++started) {
        const size_t b = begin;
        th[started] = std::thread([d, s, b, share] { std::memcpy(d + b, s + b, share); });
        begin += share;
      }
    } catch (...) {  // no thread or no memory for one: the rest here
    }
  }
  std::memcpy(d + begin, s + begin, bytes - begin);
  for (int t = 0; t < started; ++t) th[t].join();
}

}  // namespace oll
