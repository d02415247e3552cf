// Host check of ollipticid_amd/csrc/staging.cpp with the HIP calls replaced:
// copies that cannot start their threads.  Prints "ok" and exits 0, or what
// fails and exits 1.
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

hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  *p = std::malloc(n);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipHostFree(void *p) {
  std::free(p);
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

}  // namespace

int main() {
  if (check_copy()) return 1;
  std::puts("ok");
  return 0;
}
