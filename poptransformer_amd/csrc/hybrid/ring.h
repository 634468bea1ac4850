// Which rows of a ring a step of keys reads: whole numbers only, for the kernels and for a check on the host.
#pragma once
#include <hip/hip_runtime.h>

// A step of KEYS keys is read as KEYS / 2 pairs of CH pieces, by 256 threads: a thread's it-th item is `idx` = threadIdx.x + it * 256.  Threads past the
// last item repeat another one's, so that no read needs a branch round it and no key leaves the step.
template <int KEYS, int CH>
struct KeyPairs {
  static constexpr int ITEMS = KEYS / 2 * CH, PER_THREAD = (ITEMS + 255) / 256;
  __host__ __device__ static int piece(int idx) { return idx % CH; }
  __host__ __device__ static int pair(int idx) { return idx / CH % (KEYS / 2); }
};

// The ring row of key k (less than KEYS) of the step that begins at position jt, `first` = jt % ring_len; keys past `last` (not before jt) repeat it.
template <int KEYS>
__host__ __device__ inline int ring_row(int first, int jt, int k, int last, int ring_len) {
  k = first + (jt + k < last ? k : last - jt);
  return k < ring_len ? k : ring_len >= KEYS ? k - ring_len : k % ring_len;
}
