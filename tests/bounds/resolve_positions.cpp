// CPU check of the position arithmetic of unresolved output bytes
// (resolve_common.h), compiled for the host with hipcc --offload-host-only.
//
// Usage: resolve_positions <mode>
//   runs  root_range over chains of runs: no root lies further back than
//         kMaxBack, every chain ends at the byte before the first run, and its
//         links are few
//   stripes  the cut of outputs up to 2^32 + 32767 bytes: every position is in
//         one stripe, every root gives its position back (whole, and from its
//         stripe's start), and four-byte accesses end inside the output
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
    u32 calls = 0;
    const auto one = [&](u32 j, u32 r) {
      root[size_t(at + j - (start - 1))] = root_position(at + j, r);
      ++calls;
    };
    handed = root_range(at, n, handed, true, [&](u32 count, u32 r) {
      for (u32 j = 0; j < count; ++j) one(j, r);
    }, one);
    if (calls != n) return 5;
    at += n;
    if (handed == kNoRoot) return 1;
    const u64 h = root_position(at, handed);
    if (h != root.back() && !(u32(root.back()) == kNoRoot && h == at - 1)) return 1;
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
  for (const u64 start : {u64(40000), (u64(1) << 32) - 100000, (u64(1) << 32) + 5, u64(1) << 32,
                          (u64(1) << 32) + 32768})
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

// Position p of an output of `total` bytes, with a root `back` bytes before it.
int check_position(const StripeCut& cut, u64 total, u64 p, u32 back) {
  if (back > p) return 0;
  const u32 root = u32(p - back);
  if (root_position(p, root) != p - back) return 1;
  const u64 start = p / cut.bytes * cut.bytes;
  const u32 size = stripe_size(start, cut.bytes, total);
  const u32 off = u32(p - start);
  if (off >= size) return 2;
  const u32 x = stripe_offset(start, root);
  if (stripe_before(x) != (p - back < start)) return 3;
  if (stripe_before(x)) {
    // The tag of a byte of the window before keeps the offset in 15 bits.
    const u32 tag = (x + kMaxBack) & (kMaxBack - 1);
    if (u32(start) - kMaxBack + tag != root || start - kMaxBack + tag != p - back) return 4;
  } else if (start + x != p - back || x >= off) {
    return 5;
  }
  const u32 q = off & ~3u;  // a thread's four bytes
  if (q + 4 <= size && start + q + 4 > total) return 6;
  return 0;
}

int mode_stripes() {
  const u64 big = u64(1) << 32;
  u64 checked = 0;
  for (const u64 total : {u64(1), u64(4095), u64(65536), u64(65537), u64(131073), u64(300007),
                          u64(16) << 20, (u64(1) << 30) + 1, big - 4, big - 3, big - 2, big - 1, big,
                          big + 1, big + 5, big + 32766, big + 32767}) {
    const StripeCut cut = cut_stripes(total);
    int err = 0;
    if (!cut.count || cut.count > kStripes || cut.bytes % kStripeTile) err = 10;
    if (cut.count > 1 && cut.bytes < kMaxBack) err = 11;
    if ((cut.count - 1) * cut.bytes >= total || cut.count * cut.bytes < total) err = 12;
    u64 sum = 0;
    for (u32 k = 0; !err && k < cut.count; ++k) sum += stripe_size(k * cut.bytes, cut.bytes, total);
    if (!err && sum != total) err = 13;
    // The ends of the first and last stripes and of some between, and the last
    // bytes of the output.
    for (u32 k = 0; !err && k < cut.count; k += k + 3 < cut.count ? 1 + cut.count / 7 : 1)
      for (u64 i = 0; !err && i < 70000; i += 1 + i / 8) {
        const u64 from = k * cut.bytes, to = from + stripe_size(from, cut.bytes, total);
        for (const u32 back : {1u, 2u, 3u, 4u, 255u, 4095u, 4096u, 4097u, 28672u, 32767u, 32768u}) {
          if (!err && from + i < to) err = check_position(cut, total, from + i, back);
          if (!err && i < to - from) err = check_position(cut, total, to - 1 - i, back);
          checked += 2;
        }
      }
    if (err) {
      printf("stripes total=%llu error=%d\n", (unsigned long long)total, err);
      return 1;
    }
  }
  printf("stripes checked=%llu\n", (unsigned long long)checked);
  return 0;
}

}  // namespace

int main(int argc, char** argv) {
  if (argc < 2) return 2;
  if (!strcmp(argv[1], "runs")) return mode_runs();
  if (!strcmp(argv[1], "stripes")) return mode_stripes();
  return 2;
}
