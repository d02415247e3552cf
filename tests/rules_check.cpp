// Host check of the launch rules in ollipticid_amd/csrc/kernels.hpp.
// Prints "ok" and exits 0, or the first rule that fails and exits 1.
#include <cstdio>

#include "../ollipticid_amd/csrc/kernels.hpp"

using namespace oll;

namespace {

// a size set by the caller holds for every launch; the default leaves
// launches of few threads to smaller workgroups and never a larger one
int check_sweep_size() {
  const long long lengths[] = {1, 1000, 99999, 100001, 500000, 5000000, 1LL << 33};
  for (long long n : lengths) {
    for (int set = 64; set <= kMaxRowThreads; set += 64)
      if (set != kRowThreads && sweep_size(set, n) != set)
        return std::printf("sweep_size(%d, %lld) = %d\n", set, n, sweep_size(set, n)), 1;
    const int d = sweep_size(kRowThreads, n);
    if (d > kRowThreads || d < 64 || d % 64 != 0 || (n <= 1000 && d != 64) ||
        (n >= 5000000 && d != kRowThreads))
      return std::printf("sweep_size(default, %lld) = %d\n", n, d), 1;
  }
  return 0;
}

}  // namespace

int main() {
  if (check_sweep_size()) return 1;
  std::puts("ok");
  return 0;
}
