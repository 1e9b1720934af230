// Checks gl::join_halves (gl_lazy.hpp, host form), the reduction behind the
// linear layers of the hashes and the extension products, against 128-bit
// integer arithmetic: lo + hi 2^32 mod p for every row length, at the edges of
// the halves' range [0, 2^62) and of its words, and on random halves.
#include "../../era-boojum-cuda_amd/csrc/gl_lazy.hpp"

#include <stdio.h>
#include <vector>

using u64 = uint64_t;
using u128 = unsigned __int128;

static u64 state = 0x2545F4914F6CDD1Dull;
static u64 rnd() {
  state ^= state << 13;
  state ^= state >> 7;
  state ^= state << 17;
  return state;
}
static int fails = 0;

template <int N> static void check(const u64 *lo, const u64 *hi) {
  u64 s[N];
  gl::join_halves<N>(s, lo, hi);
  for (int i = 0; i < N; ++i) {
    const u64 want = (u64)((lo[i] + ((u128)hi[i] << 32)) % gl::P);
    if (s[i] % gl::P != want && fails++ < 10)
      printf("FAIL row of %d: %016llx + %016llx 2^32\n", N, (unsigned long long)lo[i], (unsigned long long)hi[i]);
  }
}
static void check_all(const u64 *lo, const u64 *hi) {
  check<1>(lo, hi);
  check<2>(lo, hi);
  check<3>(lo, hi);
  check<4>(lo, hi);
}

int main() {
  const u64 top = 1ull << 62;
  const std::vector<u64> edges{0,         1,         0xFFFFFFFE,          0xFFFFFFFF,          0x100000000,
                               0x100000001, 0x1FFFFFFFF, 1ull << 46,        1ull << 54,          1ull << 61,
                               top - 0x100000000, top - 0x100000001, top - 2, top - 1, 0x3FFFFFFF00000000,
                               0x3FFFFFFF00000001, 0x2AAAAAAA55555555};
  for (u64 a : edges)
    for (u64 b : edges) {
      const u64 lo[4] = {a, b, a ^ b, edges[rnd() % edges.size()]}, hi[4] = {b, b, a, edges[rnd() % edges.size()]};
      check_all(lo, hi);
    }
  for (int r = 0; r < 500000; ++r) {
    u64 lo[4], hi[4];
    for (int i = 0; i < 4; ++i) {
      lo[i] = rnd() >> (2 + rnd() % 40);
      hi[i] = rnd() >> (2 + rnd() % 40);
      if (rnd() % 4 == 0) hi[i] |= 0xFFFFFFFFull;
      if (rnd() % 4 == 0) lo[i] = (lo[i] & 0xFFFFFFFFull) | 0x3FFFFFFF00000000ull;
    }
    check_all(lo, hi);
  }
  if (!fails) printf("ok\n");
  return fails != 0;
}
