// Roots of unresolved output bytes: the arithmetic of their positions, shared
// by the kernels and their check on the CPU.
#pragma once

#include "deflate_common.h"

namespace hz {

// A root lies 1 to kMaxBack bytes before its byte: the longest back-reference.
// The stripes' ring holds that much output, so that every chain of roots is
// followed there to its end.
constexpr u32 kMaxBack = 32768;
constexpr u32 kNoRoot = 0xffffffffu;  // handed down by emission: a resolved byte

// Positions take more than 32 bits (an output of up to 2^32 - 1 bytes behind a
// dictionary's window), roots are kept in 32: the low bits of a position less
// than 2^32 bytes before the byte at p.  (Roots moved along their chains are of
// unresolved bytes, which lie in the output, not in the window before it.)
__host__ __device__ __forceinline__ u64 root_position(u64 p, u32 root) {
  return p - u32(u32(p) - root);
}

// What emission hands down for a byte whose root is `root`, to root a run of
// it: the byte itself, at `at`, where the root reads as kNoRoot.
__host__ __device__ __forceinline__ u32 handed_root(u32 root, u64 at) {
  return root != kNoRoot ? root : u32(at);
}

// The output cut into at most kStripes stripes of whole tiles, none but the
// last shorter than kMaxBack.  Inside a stripe the kernels count from its
// start: a byte's offset and its root's, from -kMaxBack on, fit 32 bits.
constexpr u32 kStripeTile = 4096;
constexpr u32 kStripes = 256;        // a workgroup per CU
constexpr u64 kStripeMin = 65536;    // output bytes below which a stripe is not cut
struct StripeCut {
  u64 bytes;  // of every stripe but the last
  u32 count;
};
inline StripeCut cut_stripes(u64 total) {
  const u64 most = (total + kStripeMin - 1) / kStripeMin;
  const u64 want = most < kStripes ? most : kStripes;
  const u64 bytes = ((total + want - 1) / want + kStripeTile - 1) / kStripeTile * kStripeTile;
  return {bytes, u32((total + bytes - 1) / bytes)};
}
// The size of the stripe at `start`.
__host__ __device__ __forceinline__ u32 stripe_size(u64 start, u64 bytes, u64 total) {
  return u32(total - start < bytes ? total - start : bytes);
}
// A root's offset from the stripe's start: before it from 2^32 - kMaxBack on.
__host__ __device__ __forceinline__ u32 stripe_offset(u64 start, u32 root) {
  return root - u32(start);
}
__host__ __device__ __forceinline__ bool stripe_before(u32 offset) { return i32(offset) < 0; }

// Roots of the unresolved bytes out[dst, dst + n).  A copy (not `run`) has byte
// dst + j rooted at root + j.  A run of the byte at dst - 1 is rooted as a whole
// at `root`: dst - 1, or the root of that byte, which is taken if it is near
// enough to all of it; a run longer than kMaxBack is rooted in itself from there
// on.  fill(count, root) takes the first bytes, one(j, root) the others (none
// but of such a run).  Returns what roots a run of the last byte.
template <class Fill, class One>
__host__ __device__ __forceinline__ u32 root_range(u64 dst, u32 n, u32 root, bool run,
                                                   const Fill& fill, const One& one) {
  const u32 at = u32(dst);
  u32 last = root + (run ? 0u : n - 1), count = n;
  if (run && at + n - 1 - root > kMaxBack) {
    root = last = at - 1;
    if (n > kMaxBack) {
      count = kMaxBack;
      for (u32 j = kMaxBack; j < n; ++j) one(j, last = at - 1 + j / kMaxBack * kMaxBack);
    }
  }
  fill(count, root);
  return handed_root(last, dst + n - 1);
}

}  // namespace hz
