// Host check of ollipticid_amd/csrc/staging.cpp with the HIP calls replaced:
// copies that cannot start their threads.  Prints "ok" and exits 0, or what
// fails and exits 1.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <vector>

#include "../ollipticid_amd/csrc/staging.cpp"

static bool g_no_memory = false;
void *operator new(std::size_t n) {
  void *p = g_no_memory ? nullptr : std::malloc(n);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }

static int g_held = 0, g_mallocs = 0;  // buffers not freed, allocations so far
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  *p = std::malloc(n);
  ++g_held;
  ++g_mallocs;
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipHostFree(void *p) {
  std::free(p);
  --g_held;
  return hipSuccess;
}

namespace {

// sizes on both sides of the first that is shared among threads, whole and
// odd; with memory for the threads' states and without
int check_copy() {
  for (size_t bytes : {size_t(0), size_t(1), (size_t(1) << 20) - 1, size_t(1) << 20, (size_t(3) << 20) + 12345}) {
    std::vector<char> src(bytes + 1), dst(bytes + 1);
    for (size_t i = 0; i <= bytes; ++i) src[i] = char(i * 131 + (i >> 9));
    for (bool no_memory : {false, true}) {
      for (char &c : dst) c = char(0x55);
      g_no_memory = no_memory;
      oll::host_copy(dst.data(), src.data(), bytes);
      g_no_memory = false;
      for (size_t i = 0; i < bytes; ++i)
        if (dst[i] != src[i]) return std::printf("copy of %zu differs at %zu\n", bytes, i), 1;
      if (dst[bytes] != char(0x55)) return std::printf("copy of %zu runs over\n", bytes), 1;
    }
  }
  return 0;
}

// `callers` calls at once over `handles` handles: the second round allocates
// only what the bound (16, and one a handle) keeps from staying, and no more
// is left than there are handles
int check_pool(int halves) {
  for (int handles : {1, 4, 16, 40})
    for (int callers : {1, 4, 5, 16, 24}) {
      const int kept = std::min(16, std::min(handles, callers));
      for (int h = 0; h < handles; ++h) oll::staging_retain();
      int fresh = 0;
      for (int round = 0; round < 2; ++round) {
        const int before = g_mallocs;
        std::vector<oll::Staging *> use;
        for (int c = 0; c < callers; ++c) {
          use.push_back(oll::staging_take(halves));
          if (!use.back() || !use.back()->half[halves - 1]) return std::printf("no staging\n"), 1;
        }
        for (oll::Staging *s : use) oll::staging_give(s);
        fresh = g_mallocs - before;
      }
      if (fresh != halves * (callers - kept) || g_held != halves * kept)
        return std::printf("%d handles, %d callers: %d allocated again, %d held\n", handles, callers,
                           fresh, g_held), 1;
      for (int h = handles - 1; h >= 0; --h) {
        oll::staging_release();
        if (g_held != halves * std::min(h, kept))
          return std::printf("%d buffers left with %d handles\n", g_held, h), 1;
      }
    }
  return 0;
}

// one half, then both of the same, and nothing where the second cannot be had
int check_halves() {
  oll::staging_retain();
  oll::Staging *s = oll::staging_take(1);
  if (!s || g_held != 1) return std::printf("one half: %d held\n", g_held), 1;
  oll::staging_give(s);
  oll::Staging *t = oll::staging_take(2);
  if (t != s || g_held != 2) return std::printf("both halves: %d held\n", g_held), 1;
  oll::staging_give(t);
  oll::Staging *u = oll::staging_take(1), *v = oll::staging_take(1);
  if (u != s || g_held != 3) return std::printf("a second: %d held\n", g_held), 1;
  oll::staging_give(v);
  oll::staging_malloc = [](void **, size_t, unsigned) { return hipErrorOutOfMemory; };
  if (oll::staging_take(2) || g_held != 2) return std::printf("no memory: %d held\n", g_held), 1;
  oll::staging_malloc = hipHostMalloc;
  oll::staging_give(u);
  oll::staging_release();
  if (g_held != 0) return std::printf("%d buffers left\n", g_held), 1;
  return 0;
}

}  // namespace

int main() {
  if (check_copy() || check_pool(1) || check_pool(2) || check_halves()) return 1;
  std::puts("ok");
  return 0;
}
