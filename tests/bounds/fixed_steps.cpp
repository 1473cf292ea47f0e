// CPU check of the branch-free steps of fixed-Huffman codes (deflate_common.h:
// fixed_step_entry, fixed_step, fixed_step_within), compiled for the host,
// against fixed_token, which decodes one token with branches.
//
// Every pattern of a step's first 19 bits (a code with its extra bits, or a
// code and a distance symbol), the bits after it random, away from the body's
// end and with the end at every bit up to 45 past the step's start.
#include <cstdio>

#include "deflate_common.h"

using namespace hz;

namespace {

// The step fixed_token's result stands for at bit p, as a serial scan reads it.
u32 expected(u64 bits, u32 p, u32 end) {
  u32 nb, length, value;
  const u32 kind = fixed_token(bits, nb, length, value);
  if (kind == kKindBad) return u32(kBadSymbol) << 6;
  if (p + nb > end) return u32(kTruncated) << 6;
  if (kind != kKindEob) return (nb << 1) | (length << 6);
  const u32 header = u32(bits >> 7) & 7u;
  return (kStepEob | header | (p + 10 > end ? 8u : 0u)) << 6;
}

}  // namespace

int main() {
  u32 seed = 99;
  unsigned long long checked = 0;
  for (u32 low = 0; low < (1u << 19); ++low) {
    seed = seed * 1664525u + 1013904223u;
    const u32 b = low | (seed & ~((1u << 19) - 1));
    const u32 step = fixed_step(b, fixed_step_entry(b & 511u));
    const u32 p = 100 + low % 32, far = ~0u >> 1;
    const u32 want_far = expected(b, p, far);
    if (step != want_far || fixed_step_within(step, p, far) != want_far) {
      printf("steps bits=%x got=%x want=%x\n", b, step, want_far);
      return 1;
    }
    for (u32 end = p; end < p + 45; end += low % 16 ? 1 + low % 7 : 1) {
      const u32 got = fixed_step_within(step, p, end), want = expected(b, p, end);
      ++checked;
      if (got != want) {
        printf("steps bits=%x end=%u got=%x want=%x\n", b, end - p, got, want);
        return 1;
      }
    }
  }
  printf("steps checked=%llu\n", checked);
  return 0;
}
