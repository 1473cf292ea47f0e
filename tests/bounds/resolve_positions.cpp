// CPU check of the position arithmetic of unresolved output bytes
// (resolve_common.h), compiled for the host with hipcc --offload-host-only.
//
// Usage: resolve_positions <mode>
//   runs  run_roots over chains of runs: no root lies further back than
//         kMaxBack, every chain ends at the byte before the first run, and its
//         links are few
#include <cstdio>
#include <cstring>
#include <vector>

#include "resolve_common.h"

using namespace hz;

namespace {

u32 seed = 12345;
u32 rnd(u32 n) {
  seed = seed * 1664525u + 1013904223u;
  return u32((u64(seed) * n) >> 32);
}

// Runs end to end from `start` on (the first after an unresolved match whose
// last byte is rooted `back` bytes before it), each taking the root of the
// one before as emission hands it down.
int check_runs(u64 start, u32 back, u32 runs, u32 longest) {
  std::vector<u64> root(1, start - 1 - back);  // of position start - 1 + index
  u64 at = start;
  u32 handed = u32(start - 1 - back);
  for (u32 k = 0; k < runs; ++k) {
    const u32 n = 1 + rnd(longest);
    root.resize(root.size() + n, 0);
    handed = run_roots(at, n, handed, [&](u64 first, u32 count, u32 r) {
      for (u32 j = 0; j < count; ++j) {
        const u64 p = first + j;
        root[size_t(p - (start - 1))] = p - u32(u32(p) - r);
      }
    });
    at += n;
    if (at - u32(u32(at) - handed) != root.back()) return 1;
  }
  for (u64 p = start; p < at; ++p) {
    const u64 r = root[size_t(p - (start - 1))];
    if (r >= p || p - r > kMaxBack) return 2;
    if (r >= start - 1) continue;  // its chain is that byte's
    if (r != start - 1 - back) return 3;
  }
  // Links from the last byte to one before the runs: one per kMaxBack bytes,
  // and one per run where the root handed down was out of reach.
  u64 p = at - 1, links = 0;
  while (p >= start) {
    p = root[size_t(p - (start - 1))];
    ++links;
  }
  return links <= (at - start) / (kMaxBack / 2) + 2 ? 0 : 4;
}

int mode_runs() {
  u32 checked = 0;
  for (const u64 start : {u64(40000), (u64(1) << 32) - 100000, (u64(1) << 32) + 5})
    for (const u32 back : {1u, 2u, 258u, 32767u, 32768u})
      for (const u32 longest : {1u, 258u, 32768u, 65535u, 200000u}) {
        const int err = check_runs(start, back, longest < 1000 ? 500 : 9, longest);
        ++checked;
        if (err) {
          printf("runs start=%llu back=%u longest=%u error=%d\n", (unsigned long long)start, back,
                 longest, err);
          return 1;
        }
      }
  printf("runs checked=%u\n", checked);
  return 0;
}

}  // namespace

int main(int argc, char** argv) {
  if (argc < 2) return 2;
  if (!strcmp(argv[1], "runs")) return mode_runs();
  return 2;
}
