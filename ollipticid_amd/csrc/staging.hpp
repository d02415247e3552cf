// Pinned host buffers that calls exchanging arrays with the host borrow.
//
// A call takes one Staging for itself and returns it; kernels read and write
// the buffers over PCIe while the host copies the other half.  A handle
// (hierarchy or engine) has one call at a time, so there is use for one a
// handle; at most kKeep idle ones are kept, no more than there are handles,
// and none once no handle is left.  (16 threads reading 65^3 fields: 70 us a
// call; with 4 kept most calls allocated and freed theirs, 109 us.)  Any
// thread may take one: a Staging has one user at a time and no tie to a device
// or stream.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace oll {

struct Staging {
  static constexpr size_t kBytes = size_t(4) << 20;  // per half
  char *half[2] = {nullptr, nullptr};
};

// the first `halves` of them allocated, the second by the first call that has
// use for it (a call of one piece allocates 4 MiB: 20 us less); null when the
// memory cannot be had: callers then go without (pageable copies, slower)
Staging *staging_take(int halves);
// hipHostMalloc; tests put a failing one in its place
extern hipError_t (*staging_malloc)(void **, size_t, unsigned);
void staging_give(Staging *s);
// a handle begins or ends
void staging_retain();
void staging_release();

// copies of several megabytes by up to kCopyThreads threads: a copy into
// fresh pages is bound by the faults of one thread (204 MB: 43 or 14.7 ms
// with one thread, 4 KiB or 2 MiB pages, 17.2 or 6.1 with four)
void host_copy(void *dst, const void *src, size_t bytes);

}  // namespace oll
