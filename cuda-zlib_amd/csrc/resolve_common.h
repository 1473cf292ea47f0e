// Roots of unresolved output bytes: the arithmetic of their positions, shared
// by the kernels and their check on the CPU.
#pragma once

#include "deflate_common.h"

namespace hz {

// A root lies 1 to kMaxBack bytes before its byte: the longest back-reference.
// The stripes' ring holds that much output, so that every chain of roots is
// followed there to its end.
constexpr u32 kMaxBack = 32768;

// Roots of the run out[dst, dst + n) of the byte at dst - 1: fill(first, count,
// root) for consecutive pieces.  `root`: dst - 1, or the root of that byte,
// which is taken if it is near enough to the whole run; a run longer than
// kMaxBack is rooted in itself from there on.  Returns the last byte's root.
template <class Fill>
__host__ __device__ __forceinline__ u32 run_roots(u64 dst, u32 n, u32 root, const Fill& fill) {
  if (u32(dst + n - 1) - root > kMaxBack) root = u32(dst - 1);
  for (;;) {
    const u32 reach = kMaxBack + 1 - (u32(dst) - root);
    const u32 m = n < reach ? n : reach;
    fill(dst, m, root);
    n -= m;
    if (!n) return root;
    dst += m;
    root = u32(dst - 1);
  }
}

}  // namespace hz
