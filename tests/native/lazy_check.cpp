// Checks the grouped products and the lazily reduced DFTs (gl_lazy.hpp, host
// form) against 128-bit integer arithmetic: every row length and reduction,
// and every DFT size, direction, order, output form and input form, on values
// at the edges of u64 and of the field and on random ones.
#include "../../era-boojum-cuda_amd/csrc/gl_lazy.hpp"

#include <stdio.h>
#include <vector>

using u64 = uint64_t;
using u128 = unsigned __int128;

static u64 state = 0x9E3779B97F4A7C15ull;
static u64 rnd() {
  state ^= state << 13;
  state ^= state >> 7;
  state ^= state << 17;
  return state;
}
static const u64 EDGES[] = {0ull, 1ull, 2ull, 0xFFFFFFFEull, 0xFFFFFFFFull, 0x100000000ull, 1ull << 48, 1ull << 63,
                            gl::P - 2, gl::P - 1, gl::P, gl::P + 1, ~0ull - 1, ~0ull, 0xFFFFFFFF00000000ull,
                            0xFFFFFFFE00000001ull, 0x00000000FFFF0000ull, 0x8000000080000000ull};
static constexpr int NEDGES = sizeof(EDGES) / sizeof(EDGES[0]);
// edges, words with extreme halves, and uniform words
static u64 value() {
  const u64 r = rnd();
  switch (r % 4) {
  case 0: return EDGES[(r >> 8) % NEDGES];
  case 1: return ((r & 256) ? 0xFFFFFFFF00000000ull : 0) | ((r & 512) ? 0xFFFFFFFFull - (r >> 60) : (r >> 60));
  default: return rnd();
  }
}
static u64 mulmod(u64 a, u64 b) { return (u64)((u128)a * b % gl::P); }
static u64 addmod(u64 a, u64 b) { return (u64)(((u128)a + b) % gl::P); }
static u64 powmod(u64 b, u64 e) {
  u64 r = 1;
  for (; e; e >>= 1, b = mulmod(b, b))
    if (e & 1) r = mulmod(r, b);
  return r;
}
// x + e 2^64 mod p
static u64 lazy_value(u64 x, int e) {
  const u64 t = mulmod((u64)(e < 0 ? -e : e), gl::EPS);
  return addmod(x % gl::P, e < 0 ? (gl::P - t) % gl::P : t);
}

static int fails = 0;
static void fail(const char *what, int a, int b) {
  if (fails++ < 10) printf("FAIL %s %d %d\n", what, a, b);
}

template <int N, gl::Reduce R> static void check_products(const u64 *a, const u64 *b) {
  u64 o[N];
  int32_t e[N] = {};
  gl::mul_row<N, R>(o, a, b, e);
  for (int i = 0; i < N; ++i) {
    if (e[i] < -1 || e[i] > 1) fail("product e", N, R);
    if (lazy_value(o[i], e[i]) != mulmod(a[i] % gl::P, b[i] % gl::P)) fail("product", N, R);
    if (R == gl::CANON && o[i] >= gl::P) fail("product canonical", N, R);
  }
}
template <int N> static void check_rows(const u64 *a, const u64 *b) {
  check_products<N, gl::ANY>(a, b);
  check_products<N, gl::CANON>(a, b);
  check_products<N, gl::LAZY>(a, b);
}

template <int A, bool INV, bool DIT, gl::Reduce R, bool E_IN> static void check_dft(int reps) {
  constexpr int n = 1 << A;
  u64 w = (u64)((u128)1 << 39);
  for (int k = 0; k < 6 - A; ++k) w = mulmod(w, w);
  if (INV) w = powmod(w, gl::P - 2);
  auto brev = [](int i) {
    int r = 0;
    for (int k = 0; k < A; ++k) r |= ((i >> k) & 1) << (A - 1 - k);
    return r;
  };
  for (int rep = 0; rep < reps; ++rep) {
    u64 x[16], in[16];
    int32_t e[16] = {};
    const u64 same = value();
    for (int i = 0; i < 16; ++i) {
      x[i] = rep % 8 == 0 ? same : value();
      if (E_IN) e[i] = rep % 8 == 0 ? (int)(rep / 8 % 3) - 1 : (int)(rnd() % 3) - 1;
      in[i] = lazy_value(x[i], e[i]);
    }
    gl::dft_lazy<A, INV, DIT, R, E_IN>(x, E_IN ? e : nullptr);
    for (int g = 0; g < 16; g += n)
      for (int k = 0; k < n; ++k) {
        u64 want = 0;  // output k (bit-reversed for DIF, whose input is natural)
        for (int i = 0; i < n; ++i) want = addmod(want, mulmod(in[g + (DIT ? brev(i) : i)], powmod(w, (u64)(i * k))));
        const u64 got = x[g + (DIT ? k : brev(k))];
        if (R == gl::CANON ? got != want : got % gl::P != want) fail("dft", A, INV * 8 + DIT * 4 + R * 2 + E_IN);
      }
  }
}
template <int A> static void check_size(int reps) {
  auto forms = [&](auto inv, auto dit) {
    constexpr bool INV = decltype(inv)::value, DIT = decltype(dit)::value;
    check_dft<A, INV, DIT, gl::ANY, false>(reps);
    check_dft<A, INV, DIT, gl::CANON, false>(reps);
    check_dft<A, INV, DIT, gl::ANY, true>(reps);
    check_dft<A, INV, DIT, gl::CANON, true>(reps);
  };
  forms(std::false_type{}, std::false_type{});
  forms(std::false_type{}, std::true_type{});
  forms(std::true_type{}, std::false_type{});
  forms(std::true_type{}, std::true_type{});
}

int main() {
  for (int i = 0; i < NEDGES; ++i)
    for (int j = 0; j < NEDGES; ++j) {
      const u64 a[4] = {EDGES[i], EDGES[j], EDGES[i] ^ EDGES[j], EDGES[(i + j) % NEDGES]};
      const u64 b[4] = {EDGES[j], EDGES[j], EDGES[i], EDGES[(i * j) % NEDGES]};
      check_rows<1>(a, b);
      check_rows<4>(a, b);
    }
  for (int r = 0; r < 200000; ++r) {
    const u64 a[4] = {value(), value(), value(), value()}, b[4] = {value(), value(), value(), value()};
    check_rows<2>(a, b);
    check_rows<3>(a, b);
    check_rows<4>(a, b);
  }
  check_size<1>(600);
  check_size<2>(600);
  check_size<3>(600);
  check_size<4>(600);
  if (!fails) printf("ok\n");
  return fails != 0;
}
