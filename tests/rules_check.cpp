// Host check of the launch rules in ollipticid_amd/csrc/kernels.hpp.
// Prints "ok" and exits 0, or the first rule that fails and exits 1.
#include <cstdio>

#include "../ollipticid_amd/csrc/kernels.hpp"

using namespace oll;

namespace {

// a size set by the caller holds for every launch; the default leaves
// launches of few threads to smaller workgroups and never a larger one
int check_sweep_size() {
  // threads a launch -> the default's workgroup: pairs, one point a thread, FP32
  const struct {
    long long n;
    int pairs, one, fp32;
  } want[] = {{1, 64, 64, 64},           {100000, 64, 64, 64},
              {100001, 128, 64, 128},    {200000, 128, 64, 128},
              {200001, 128, 256, 128},   {300000, 128, 256, 128},
              {300001, 128, 256, 256},   {800000, 128, 256, 256},
              {800001, 256, 256, 256},   {1LL << 33, 256, 256, 256}};
  for (const auto &w : want)
    for (int kind = 0; kind < 3; ++kind) {
      const bool mixed = kind == 2;
      const int pts = kind == 0 ? 2 : 1, d = kind == 0 ? w.pairs : (kind == 1 ? w.one : w.fp32);
      for (int set = 64; set <= kMaxRowThreads; set += 64) {
        const int got = sweep_size(set, w.n, mixed, pts);
        if (got != (set == kRowThreads ? d : set))
          return std::printf("sweep_size(%d, %lld, %d, %d) = %d\n", set, w.n, mixed, pts, got), 1;
      }
    }
  return 0;
}

// a coarsest box that the schedule builder takes is one that the launcher
// takes; the cubes are those of up to 21 points an axis
int check_coarse_box() {
  for (int a = 3; a <= 131; ++a)
    for (int b = 3; b <= 131; ++b)
      for (int c = 3; c <= 131; ++c) {
        const int n[3] = {a, b, c};
        const long long size = layout_size(n, 2);
        const bool fits = coarse_box_fits(n, size);
        const bool launches = 2 * (long long)sizeof(double) * size <= kCoarseMostLds &&
                              coarse_colour_slots(n) <= kCoarseMostSlots &&
                              coarse_shell_points(n) <= kCoarseMostShell &&
                              4 * ((a - 2) + (b - 2) + (c - 2)) <= kCoarseMostEdges;
        if (fits != launches || (a == b && b == c && fits != (a <= 21)))
          return std::printf("box %d x %d x %d: fits %d, launches %d\n", a, b, c, fits, launches), 1;
      }
  const int flat[3] = {56, 56, 3};  // 1458 points of a colour, 6484 of the shell
  if (coarse_box_fits(flat, layout_size(flat, 2))) return std::puts("56 x 56 x 3 fits"), 1;
  return 0;
}

}  // namespace

int main() {
  if (check_sweep_size() || check_coarse_box()) return 1;
  std::puts("ok");
  return 0;
}
