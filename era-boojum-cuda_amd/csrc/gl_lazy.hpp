// Grouped Goldilocks products and lazily reduced radix-2^A DFTs, for gfx950
// (with the same steps on the host, which the CPU tests run).
//
// What bounds this code is instruction issue.  Measured on gfx950: a wave
// issues at most one instruction of any kind per 8 cycles (s_nop, SALU and
// waits included), and a SIMD retires one carry, compare, select, 64-bit or
// multiply-add instruction per 4 cycles and one plain 32-bit add, sub, and,
// or, xor, not, right shift or move per 2.  So the cost is the instruction
// count, and wait states are paid like instructions.
//
// Rows.  An instruction that reads a lane mask (carry, borrow, compare) needs
// two wait states after the VALU instruction that wrote it.  The operations
// below run N independent values in lock step, one instruction of each in
// turn, so for N >= 3 a mask is read at least two instructions after it was
// written and no wait states are spent; rows of 1 or 2 spend them in s_nops.
// As much of a row as can be is one asm block: the compiler counts a block as
// one instruction and would add wait states between two of them, and it does
// not know the masks a block writes, so a block that starts by reading one
// spends the states itself when N < 3 (sub_fold and sub_borrow need not: the
// mask they read comes from the multiply-add t2, and between the two lie the
// move that widens t2's high word and the multiply-add t3, or, where these are
// known when compiling and N < 3, dev::wait_if_known).
//
// Lazy values.  Inside a DFT a value is V = x + e 2^64 with x any u64 and e a
// small signed integer: a sum or difference is three carry instructions
// (12 cycles, against 20-22 for a canonical one), and reductions are paid
// only where a power-of-two twiddle or the end of the DFT needs 64 bits.
// DFTs take any u64 and give any u64 or canonical values.
#pragma once
#include "gl_field.hpp"

#include <utility>

namespace gl {

// Unrolled by the template rather than by the optimizer: the indices are
// compile-time constants on both host and device.
template <class F, int... I> GL_FN void unroll_impl(F &&f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F> GL_FN void unroll(F &&f) { unroll_impl(f, std::make_integer_sequence<int, N>{}); }

GL_FN uint32_t lo32(uint64_t v) { return (uint32_t)v; }
GL_FN uint32_t hi32(uint64_t v) { return (uint32_t)(v >> 32); }
GL_FN uint64_t pair64(uint32_t lo, uint32_t hi) { return ((uint64_t)hi << 32) | lo; }
// Low word of (hi 2^32 + lo) >> s, 0 < s < 32.
GL_FN uint32_t align32(uint32_t hi, uint32_t lo, unsigned s) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_alignbit(hi, lo, s);
#else
  return (uint32_t)(pair64(lo, hi) >> s);
#endif
}

namespace row {

// A lane mask: one bit per lane in an SGPR pair on the device, 0 or 1 on the host.
using Mask = uint64_t;

#if defined(__HIP_DEVICE_COMPILE__)

// Operand lists and instruction lines of a row of N.
#define GL_CAT1(X) X(0)
#define GL_CAT2(X) X(0) X(1)
#define GL_CAT3(X) X(0) X(1) X(2)
#define GL_CAT4(X) X(0) X(1) X(2) X(3)
#define GL_LIST1(X) X(0)
#define GL_LIST2(X) X(0), X(1)
#define GL_LIST3(X) X(0), X(1), X(2)
#define GL_LIST4(X) X(0), X(1), X(2), X(3)
// wait states between a step and one that reads the masks it wrote
#define GL_WAIT1 "s_nop 1\n\t"
#define GL_WAIT2 "s_nop 0\n\t"
#define GL_WAIT3
#define GL_WAIT4

#define GL_OUT(v, i) [v##i] "=&v"(v[i])
#define GL_OUTM(v, i) [v##i] "=&s"(v[i])
#define GL_IN(v, i) [v##i] "v"(v[i])
#define GL_INM(v, i) [v##i] "s"(v[i])
#define GL_OP3(op, r, m, a, b, i) op " %[" #r #i "], %[" #m #i "], %[" #a #i "], " b
#define GL_REF(v, i) "%[" #v #i "]"

#define GL_O_r(i) GL_OUT(r, i)
#define GL_O_r0(i) [lo##i] "=&v"(r0[i])
#define GL_O_r1(i) [hi##i] "=&v"(r1[i])
#define GL_O_n(i) GL_OUT(n, i)
#define GL_O_t(i) GL_OUT(t, i)
#define GL_O_z(i) GL_OUT(z, i)
#define GL_O_c(i) GL_OUTM(c, i)
#define GL_O_k(i) GL_OUTM(k, i)
#define GL_I_a(i) GL_IN(a, i)
#define GL_I_b(i) GL_IN(b, i)
#define GL_I_bs(i) [b##i] "s"(b[i])
#define GL_I_d(i) GL_IN(d, i)
#define GL_I_f(i) GL_IN(f, i)
#define GL_I_h(i) GL_IN(h, i)
#define GL_I_l(i) GL_IN(l, i)
#define GL_I_x0(i) [xl##i] "v"(x0[i])
#define GL_I_x1(i) [xh##i] "v"(x1[i])
#define GL_I_z(i) [z##i] "v"(z[i])
#define GL_I_m(i) GL_INM(m, i)
#define GL_I_w(i) GL_INM(w, i)

// one instruction of each step
#define GL_S_MAD(i) "v_mad_u64_u32 %[r" #i "], %[c" #i "], %[a" #i "], %[b" #i "], %[d" #i "]\n\t"
#define GL_S_EPS(i) "v_mad_u64_u32 %[z" #i "], %[c" #i "], %[f" #i "], -1, %[d" #i "]\n\t"
#define GL_S_SHIFT_E(i) "v_addc_co_u32_e64 %[n" #i "], %[c" #i "], %[b" #i "], 0, %[c" #i "]\n\t"
#define GL_S_GE(i) "v_cmp_le_u64_e64 %[k" #i "], %[p], %[z" #i "]\n\t"
#define GL_S_OR(i) "s_or_b64 %[c" #i "], %[c" #i "], %[k" #i "]\n\t"
#define GL_S_BIT(i) "v_cndmask_b32_e64 %[t" #i "], 0, 1, %[c" #i "]\n\t"
#define GL_S_FOLD(i) "v_mad_u64_u32 %[r" #i "], %[k" #i "], %[t" #i "], -1, %[z" #i "]\n\t"
#define GL_S_YLO(i) "v_subb_co_u32_e64 %[lo" #i "], %[k" #i "], %[xl" #i "], %[h" #i "], %[m" #i "]\n\t"
#define GL_S_YHI(i) "v_subb_co_u32_e64 %[hi" #i "], %[k" #i "], %[xh" #i "], 0, %[k" #i "]\n\t"
#define GL_S_YN(i) "v_subb_co_u32_e64 %[n" #i "], %[k" #i "], %[l" #i "], 0, %[k" #i "]\n\t"
#define GL_S_GE3(i) "v_cmp_le_u64_e64 %[k" #i "], %[p], %[z" #i "]\n\t"
#define GL_S_OR3(i) "s_or_b64 %[k" #i "], %[m" #i "], %[k" #i "]\n\t"
#define GL_S_ONES(i) "v_cndmask_b32_e64 %[t" #i "], 0, -1, %[m" #i "]\n\t"
#define GL_S_ONESK(i) "v_cndmask_b32_e64 %[t" #i "], 0, -1, %[k" #i "]\n\t"
#define GL_S_FLO(i) "v_addc_co_u32_e64 %[lo" #i "], %[k" #i "], %[xl" #i "], %[t" #i "], %[w" #i "]\n\t"
#define GL_S_FHI(i) "v_addc_co_u32_e64 %[hi" #i "], %[k" #i "], %[xh" #i "], 0, %[k" #i "]\n\t"
#define GL_S_ADD(i) "v_add_co_u32_e64 %[r" #i "], %[c" #i "], %[a" #i "], %[b" #i "]\n\t"
#define GL_S_LAZY_E(i) "v_subb_co_u32_e64 %[n" #i "], %[c" #i "], %[t" #i "], 0, %[m" #i "]\n\t"

template <int N> struct Rows;
#define GL_DEFINE_ROWS(N)                                                                                              \
  template <> struct Rows<N> {                                                                                         \
    GL_FN static void mad(uint64_t *r, Mask *c, const uint32_t *a, const uint32_t *b, const uint64_t *d) {             \
      asm(GL_CAT##N(GL_S_MAD) : GL_LIST##N(GL_O_r), GL_LIST##N(GL_O_c)                                                 \
          : GL_LIST##N(GL_I_a), GL_LIST##N(GL_I_b), GL_LIST##N(GL_I_d));                                               \
    }                                                                                                                  \
    GL_FN static void mad_s(uint64_t *r, Mask *c, const uint32_t *a, const uint32_t *b, const uint64_t *d) {           \
      asm(GL_CAT##N(GL_S_MAD) : GL_LIST##N(GL_O_r), GL_LIST##N(GL_O_c)                                                 \
          : GL_LIST##N(GL_I_a), GL_LIST##N(GL_I_bs), GL_LIST##N(GL_I_d));                                              \
    }                                                                                                                  \
    GL_FN static void mad_eps(uint64_t *z, Mask *c, const uint32_t *f, const uint64_t *d) {                            \
      asm(GL_CAT##N(GL_S_EPS) : GL_LIST##N(GL_O_z), GL_LIST##N(GL_O_c) : GL_LIST##N(GL_I_f), GL_LIST##N(GL_I_d));      \
    }                                                                                                                  \
    GL_FN static void add_bit(uint32_t *r, uint32_t *t, const uint32_t *a, const uint32_t *b) {                        \
      Mask c[N];                                                                                                       \
      asm(GL_CAT##N(GL_S_ADD) GL_WAIT##N GL_CAT##N(GL_S_BIT)                                                           \
          : GL_LIST##N(GL_O_r), GL_LIST##N(GL_O_t), GL_LIST##N(GL_O_c) : GL_LIST##N(GL_I_a), GL_LIST##N(GL_I_b));      \
    }                                                                                                                  \
    GL_FN static void mad_eps_carry(uint64_t *z, uint32_t *n, const uint32_t *f, const uint64_t *d,                    \
                                    const uint32_t *b) {                                                               \
      Mask c[N];                                                                                                       \
      asm(GL_CAT##N(GL_S_EPS) GL_WAIT##N GL_CAT##N(GL_S_SHIFT_E)                                                       \
          : GL_LIST##N(GL_O_z), GL_LIST##N(GL_O_n), GL_LIST##N(GL_O_c)                                                 \
          : GL_LIST##N(GL_I_f), GL_LIST##N(GL_I_d), GL_LIST##N(GL_I_b));                                               \
    }                                                                                                                  \
    GL_FN static void mad_eps_lazy(uint64_t *z, uint32_t *n, const uint32_t *f, const uint64_t *d, const Mask *m) {    \
      Mask c[N];                                                                                                       \
      uint32_t t[N];                                                                                                   \
      asm(GL_CAT##N(GL_S_EPS) GL_WAIT##N GL_CAT##N(GL_S_BIT) GL_CAT##N(GL_S_LAZY_E)                                    \
          : GL_LIST##N(GL_O_z), GL_LIST##N(GL_O_n), GL_LIST##N(GL_O_t), GL_LIST##N(GL_O_c)                             \
          : GL_LIST##N(GL_I_f), GL_LIST##N(GL_I_d), GL_LIST##N(GL_I_m));                                               \
    }                                                                                                                  \
    GL_FN static void reduce_any(uint64_t *r, const uint32_t *f, const uint64_t *d) {                                  \
      Mask c[N], k[N];                                                                                                 \
      uint32_t t[N];                                                                                                   \
      uint64_t z[N];                                                                                                   \
      asm(GL_CAT##N(GL_S_EPS) GL_WAIT##N GL_CAT##N(GL_S_BIT) GL_CAT##N(GL_S_FOLD)                                      \
          : GL_LIST##N(GL_O_r), GL_LIST##N(GL_O_z), GL_LIST##N(GL_O_t), GL_LIST##N(GL_O_c), GL_LIST##N(GL_O_k)         \
          : GL_LIST##N(GL_I_f), GL_LIST##N(GL_I_d));                                                                   \
    }                                                                                                                  \
    GL_FN static void reduce_canon(uint64_t *r, const uint32_t *f, const uint64_t *d) {                                \
      Mask c[N], k[N];                                                                                                 \
      uint32_t t[N];                                                                                                   \
      uint64_t z[N];                                                                                                   \
      asm(GL_CAT##N(GL_S_EPS) GL_CAT##N(GL_S_GE) GL_CAT##N(GL_S_OR) GL_CAT##N(GL_S_BIT) GL_CAT##N(GL_S_FOLD)           \
          : GL_LIST##N(GL_O_r), GL_LIST##N(GL_O_z), GL_LIST##N(GL_O_t), GL_LIST##N(GL_O_c), GL_LIST##N(GL_O_k)         \
          : GL_LIST##N(GL_I_f), GL_LIST##N(GL_I_d), [p] "s"(P) : "scc");                                               \
    }                                                                                                                  \
    GL_FN static void sub_fold(uint32_t *r0, uint32_t *r1, uint32_t *n, Mask *k, const uint32_t *x0,                   \
                               const uint32_t *x1, const uint32_t *h, const uint32_t *l, const Mask *m) {              \
      asm(GL_CAT##N(GL_S_YLO) GL_WAIT##N GL_CAT##N(GL_S_YHI) GL_WAIT##N GL_CAT##N(GL_S_YN)                             \
          : GL_LIST##N(GL_O_r0), GL_LIST##N(GL_O_r1), GL_LIST##N(GL_O_n), GL_LIST##N(GL_O_k)                           \
          : GL_LIST##N(GL_I_x0), GL_LIST##N(GL_I_x1), GL_LIST##N(GL_I_h), GL_LIST##N(GL_I_l), GL_LIST##N(GL_I_m));     \
    }                                                                                                                  \
    GL_FN static void sub_borrow(uint32_t *r0, uint32_t *r1, Mask *k, const uint32_t *x0, const uint32_t *x1,          \
                                 const uint32_t *h, const Mask *m) {                                                   \
      asm(GL_CAT##N(GL_S_YLO) GL_WAIT##N GL_CAT##N(GL_S_YHI)                                                           \
          : GL_LIST##N(GL_O_r0), GL_LIST##N(GL_O_r1), GL_LIST##N(GL_O_k)                                               \
          : GL_LIST##N(GL_I_x0), GL_LIST##N(GL_I_x1), GL_LIST##N(GL_I_h), GL_LIST##N(GL_I_m));                         \
    }                                                                                                                  \
    GL_FN static void fold_any(uint32_t *r0, uint32_t *r1, const uint32_t *x0, const uint32_t *x1, const Mask *m,      \
                               const Mask *w) {                                                                        \
      Mask k[N];                                                                                                       \
      uint32_t t[N];                                                                                                   \
      asm(GL_WAIT##N GL_CAT##N(GL_S_ONES) GL_CAT##N(GL_S_FLO) GL_WAIT##N GL_CAT##N(GL_S_FHI)                           \
          : GL_LIST##N(GL_O_r0), GL_LIST##N(GL_O_r1), GL_LIST##N(GL_O_t), GL_LIST##N(GL_O_k)                           \
          : GL_LIST##N(GL_I_x0), GL_LIST##N(GL_I_x1), GL_LIST##N(GL_I_m), GL_LIST##N(GL_I_w));                         \
    }                                                                                                                  \
    GL_FN static void fold_canon(uint32_t *r0, uint32_t *r1, const uint64_t *z, const uint32_t *x0,                    \
                                 const uint32_t *x1, const Mask *m, const Mask *w) {                                   \
      Mask k[N];                                                                                                       \
      uint32_t t[N];                                                                                                   \
      asm(GL_CAT##N(GL_S_GE3) GL_CAT##N(GL_S_OR3) GL_CAT##N(GL_S_ONESK) GL_CAT##N(GL_S_FLO) GL_WAIT##N                 \
              GL_CAT##N(GL_S_FHI)                                                                                      \
          : GL_LIST##N(GL_O_r0), GL_LIST##N(GL_O_r1), GL_LIST##N(GL_O_t), GL_LIST##N(GL_O_k)                           \
          : GL_LIST##N(GL_I_z), GL_LIST##N(GL_I_x0), GL_LIST##N(GL_I_x1), GL_LIST##N(GL_I_m), GL_LIST##N(GL_I_w),      \
            [p] "s"(P) : "scc");                                                                                       \
    }                                                                                                                  \
  };
GL_DEFINE_ROWS(1)
GL_DEFINE_ROWS(2)
GL_DEFINE_ROWS(3)
GL_DEFINE_ROWS(4)

// Two butterflies on lazy values (three words each): s = u + v, d = u - v.
// The masks of one word are read four instructions after they are written.
GL_FN void butterfly2(uint32_t (&s)[2][3], uint32_t (&d)[2][3], const uint32_t (&u)[2][3], const uint32_t (&v)[2][3]) {
  Mask c0, c1, b0, b1;
  asm("v_add_co_u32_e64 %[s00], %[c0], %[u00], %[v00]\n\t"
      "v_add_co_u32_e64 %[s10], %[c1], %[u10], %[v10]\n\t"
      "v_sub_co_u32_e64 %[d00], %[b0], %[u00], %[v00]\n\t"
      "v_sub_co_u32_e64 %[d10], %[b1], %[u10], %[v10]\n\t"
      "v_addc_co_u32_e64 %[s01], %[c0], %[u01], %[v01], %[c0]\n\t"
      "v_addc_co_u32_e64 %[s11], %[c1], %[u11], %[v11], %[c1]\n\t"
      "v_subb_co_u32_e64 %[d01], %[b0], %[u01], %[v01], %[b0]\n\t"
      "v_subb_co_u32_e64 %[d11], %[b1], %[u11], %[v11], %[b1]\n\t"
      "v_addc_co_u32_e64 %[s02], %[c0], %[u02], %[v02], %[c0]\n\t"
      "v_addc_co_u32_e64 %[s12], %[c1], %[u12], %[v12], %[c1]\n\t"
      "v_subb_co_u32_e64 %[d02], %[b0], %[u02], %[v02], %[b0]\n\t"
      "v_subb_co_u32_e64 %[d12], %[b1], %[u12], %[v12], %[b1]"
      : [s00] "=&v"(s[0][0]), [s01] "=&v"(s[0][1]), [s02] "=&v"(s[0][2]), [s10] "=&v"(s[1][0]), [s11] "=&v"(s[1][1]),
        [s12] "=&v"(s[1][2]), [d00] "=&v"(d[0][0]), [d01] "=&v"(d[0][1]), [d02] "=&v"(d[0][2]), [d10] "=&v"(d[1][0]),
        [d11] "=&v"(d[1][1]), [d12] "=&v"(d[1][2]), [c0] "=&s"(c0), [c1] "=&s"(c1), [b0] "=&s"(b0), [b1] "=&s"(b1)
      : [u00] "v"(u[0][0]), [u01] "v"(u[0][1]), [u02] "v"(u[0][2]), [u10] "v"(u[1][0]), [u11] "v"(u[1][1]),
        [u12] "v"(u[1][2]), [v00] "v"(v[0][0]), [v01] "v"(v[0][1]), [v02] "v"(v[0][2]), [v10] "v"(v[1][0]),
        [v11] "v"(v[1][1]), [v12] "v"(v[1][2]));
}

#else

template <int N> struct Rows {
  static uint64_t mad1(uint32_t a, uint32_t b, uint64_t d, Mask &c) {
    const uint64_t r = (uint64_t)a * b + d;
    c = r < d;
    return r;
  }
  static uint32_t sub1(uint32_t a, uint32_t b, Mask &k) {  // a - b - k, k: borrow in and out
    const uint64_t s = (uint64_t)a - b - k;
    k = (s >> 32) & 1;
    return (uint32_t)s;
  }
  static void mad(uint64_t *r, Mask *c, const uint32_t *a, const uint32_t *b, const uint64_t *d) {
    for (int i = 0; i < N; ++i) r[i] = mad1(a[i], b[i], d[i], c[i]);
  }
  static void mad_s(uint64_t *r, Mask *c, const uint32_t *a, const uint32_t *b, const uint64_t *d) { mad(r, c, a, b, d); }
  static void mad_eps(uint64_t *z, Mask *c, const uint32_t *f, const uint64_t *d) {
    for (int i = 0; i < N; ++i) z[i] = mad1(f[i], 0xFFFFFFFFu, d[i], c[i]);
  }
  static void add_bit(uint32_t *r, uint32_t *t, const uint32_t *a, const uint32_t *b) {
    for (int i = 0; i < N; ++i) {
      r[i] = a[i] + b[i];
      t[i] = r[i] < a[i];
    }
  }
  static void mad_eps_carry(uint64_t *z, uint32_t *n, const uint32_t *f, const uint64_t *d, const uint32_t *b) {
    Mask c[N];
    mad_eps(z, c, f, d);
    for (int i = 0; i < N; ++i) n[i] = b[i] + (uint32_t)c[i];
  }
  static void mad_eps_lazy(uint64_t *z, uint32_t *n, const uint32_t *f, const uint64_t *d, const Mask *m) {
    Mask c[N];
    mad_eps(z, c, f, d);
    for (int i = 0; i < N; ++i) n[i] = (uint32_t)c[i] - (uint32_t)m[i];
  }
  static void reduce_any(uint64_t *r, const uint32_t *f, const uint64_t *d) {
    Mask c[N];
    uint64_t z[N];
    mad_eps(z, c, f, d);
    for (int i = 0; i < N; ++i) r[i] = z[i] + c[i] * EPS;
  }
  static void reduce_canon(uint64_t *r, const uint32_t *f, const uint64_t *d) {
    Mask c[N];
    uint64_t z[N];
    mad_eps(z, c, f, d);
    for (int i = 0; i < N; ++i) r[i] = z[i] + (c[i] | (z[i] >= P)) * EPS;
  }
  static void sub_borrow(uint32_t *r0, uint32_t *r1, Mask *k, const uint32_t *x0, const uint32_t *x1, const uint32_t *h,
                         const Mask *m) {
    for (int i = 0; i < N; ++i) {
      k[i] = m[i];
      r0[i] = sub1(x0[i], h[i], k[i]);
      r1[i] = sub1(x1[i], 0, k[i]);
    }
  }
  static void sub_fold(uint32_t *r0, uint32_t *r1, uint32_t *n, Mask *k, const uint32_t *x0, const uint32_t *x1,
                       const uint32_t *h, const uint32_t *l, const Mask *m) {
    sub_borrow(r0, r1, k, x0, x1, h, m);
    for (int i = 0; i < N; ++i) n[i] = sub1(l[i], 0, k[i]);
  }
  static void fold_any(uint32_t *r0, uint32_t *r1, const uint32_t *x0, const uint32_t *x1, const Mask *m, const Mask *w) {
    for (int i = 0; i < N; ++i) {
      const uint64_t r = (((uint64_t)x1[i] << 32) | x0[i]) + m[i] * EPS + w[i];
      r0[i] = (uint32_t)r;
      r1[i] = (uint32_t)(r >> 32);
    }
  }
  static void fold_canon(uint32_t *r0, uint32_t *r1, const uint64_t *z, const uint32_t *x0, const uint32_t *x1,
                         const Mask *m, const Mask *w) {
    Mask g[N];
    for (int i = 0; i < N; ++i) g[i] = m[i] | (z[i] >= P);
    fold_any(r0, r1, x0, x1, g, w);
  }
};

GL_FN void butterfly2(uint32_t (&s)[2][3], uint32_t (&d)[2][3], const uint32_t (&u)[2][3], const uint32_t (&v)[2][3]) {
  for (int i = 0; i < 2; ++i) {
    uint64_t c = 0, b = 0;
    for (int w = 0; w < 3; ++w) {
      c += (uint64_t)u[i][w] + v[i][w];
      s[i][w] = (uint32_t)c;
      c >>= 32;
      const uint64_t t = (uint64_t)u[i][w] - v[i][w] - b;
      d[i][w] = (uint32_t)t;
      b = (t >> 32) & 1;
    }
  }
}

#endif

}  // namespace row

// How a product is returned.
enum Reduce {
  ANY,    // some u64 with the right residue
  CANON,  // the residue in [0, p)
  LAZY,   // x + e 2^64 with e in [-1, 1] (product only: e in `e`)
};

// o[i] = a[i] b[i] mod p for N independent pairs of any u64 (e[i]: LAZY only).
// With the columns of gl::mul, a b = X + l EPS - h - c where X = lo(t0) +
// lo(t2) 2^32, l = lo(t3), h = hi(t3), c the carry out of t2.  Y = X - h - c
// may borrow 2^64 (bw); subtracting EPS for that borrow is one less in the
// factor of the last multiply-add: Z = Y + (l - bw) EPS.  Where l = 0 and
// bw = 1 the factor wraps to 2^32 - 1 (borrow b2), which is 2^32 EPS = -1
// (mod p) too much, so b2 is added back with the final carry-in.  Z's carry
// out (c2) adds EPS: it implies Z <= 2^64 - 2^33, so Z + EPS + b2 < p; and b2
// implies c2.  12 cycles less per product than one-at-a-time gl::mul at four
// waves per SIMD (54 against 66; 49 for ANY), 22 at two waves.
// SGPR: every b[i] is wave-uniform and taken into SGPRs.
template <int N, Reduce R, bool SGPR = false>
GL_FN void mul_row(uint64_t *o, const uint64_t *a, const uint64_t *b, int32_t *e = nullptr) {
  using W = row::Rows<N>;
  uint32_t a1[N], b0[N], b1[N], x0[N], x1[N], l[N], h[N];
  uint64_t t0[N], t1[N], t2[N];
  row::Mask c[N], bw[N], b2[N], c2[N];
  unroll<N>([&](auto k) {
    constexpr int i = decltype(k)::value;
    b0[i] = lo32(b[i]);
    b1[i] = hi32(b[i]);
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (SGPR) {
      b0[i] = __builtin_amdgcn_readfirstlane(b0[i]);
      b1[i] = __builtin_amdgcn_readfirstlane(b1[i]);
    }
#endif
    a1[i] = hi32(a[i]);
    t0[i] = (uint64_t)lo32(a[i]) * b0[i];
    t1[i] = (uint64_t)lo32(a[i]) * b1[i] + (t0[i] >> 32);
  });
  if constexpr (SGPR) W::mad_s(t2, c, a1, b0, t1);
  else W::mad(t2, c, a1, b0, t1);
  unroll<N>([&](auto k) {
    constexpr int i = decltype(k)::value;
    const uint64_t t3 = (uint64_t)a1[i] * b1[i] + (t2[i] >> 32);
    x0[i] = lo32(t0[i]);
    x1[i] = lo32(t2[i]);
    l[i] = lo32(t3);
    h[i] = hi32(t3);
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (N < 3) dev::wait_if_known((uint64_t)a1[i] * b1[i], c[i]);
#endif
  });
  uint32_t y0[N], y1[N];
  uint64_t y[N], z[N];
  auto join = [](uint64_t *v, const uint32_t *v0, const uint32_t *v1) {
    unroll<N>([&](auto k) { v[decltype(k)::value] = pair64(v0[decltype(k)::value], v1[decltype(k)::value]); });
  };
  if constexpr (R == LAZY) {
    uint32_t d[N];
    W::sub_borrow(y0, y1, bw, x0, x1, h, c);
    join(y, y0, y1);
    W::mad_eps_lazy(z, d, l, y, bw);
    unroll<N>([&](auto k) {
      o[decltype(k)::value] = z[decltype(k)::value];
      e[decltype(k)::value] = (int32_t)d[decltype(k)::value];
    });
  } else {
    uint32_t n[N], z0[N], z1[N], r0[N], r1[N];
    W::sub_fold(y0, y1, n, b2, x0, x1, h, l, c);
    join(y, y0, y1);
    W::mad_eps(z, c2, n, y);
    unroll<N>([&](auto k) {
      z0[decltype(k)::value] = lo32(z[decltype(k)::value]);
      z1[decltype(k)::value] = hi32(z[decltype(k)::value]);
    });
    if constexpr (R == CANON) W::fold_canon(r0, r1, z, z0, z1, c2, b2);
    else W::fold_any(r0, r1, z0, z1, c2, b2);
    join(o, r0, r1);
  }
}

// s[i] = lo[i] + hi[i] 2^32 for lo, hi < 2^62 (any u64): hi = h0 + h1 2^32
// gives lo + h1 EPS + h0 2^32, one multiply-add, one addition into the high
// word and its carry.
template <int N> GL_FN void join_halves(uint64_t *s, const uint64_t *lo, const uint64_t *hi) {
  uint32_t z1[N], h0[N], r[N], up[N];
  uint64_t z[N];
  row::Mask drop[N];
  unroll<N>([&](auto k) {
    constexpr int i = decltype(k)::value;
    z[i] = (hi[i] >> 32) * EPS + lo[i];
    z1[i] = hi32(z[i]);
    h0[i] = lo32(hi[i]);
  });
  row::Rows<N>::add_bit(r, up, z1, h0);
  unroll<N>([&](auto k) {
    constexpr int i = decltype(k)::value;
    z[i] = pair64(lo32(z[i]), r[i]);
  });
  row::Rows<N>::mad_eps(s, drop, up, z);
}

// x[i] *= w(i) for i in [FIRST, FIRST + COUNT), in rows of four and one
// shorter row of at least three where that can be had.
template <int FIRST, int COUNT, Reduce R, bool SGPR = false, class F>
GL_FN void mul_each(uint64_t *x, F &&w, int32_t *e = nullptr) {
  constexpr int N = COUNT >= 7 || COUNT == 4 ? 4 : (COUNT > 4 ? 3 : COUNT);
  if constexpr (COUNT > 0) {
    uint64_t b[N];
    unroll<N>([&](auto k) { b[decltype(k)::value] = w(FIRST + decltype(k)::value); });
    mul_row<N, R, SGPR>(x + FIRST, x + FIRST, b, e ? e + FIRST : nullptr);
    mul_each<FIRST + N, COUNT - N, R, SGPR>(x, w, e);
  }
}

// ---- lazily reduced DFTs -------------------------------------------------------

// Bounds of e through a DFT, at compile time: the range of every value's e,
// the bias the DFT's point 0 needs so that every output has e >= 0, and
// whether each twiddled value fits its shift.
struct LazyBounds {
  int lo[16], hi[16];
  bool ok;
};

constexpr unsigned lazy_exp(int lh, int t, bool inv) { return root_pow2_exp((unsigned)(lh + 1), (unsigned)t, inv) % 96u; }
constexpr bool lazy_neg(int lh, int t, bool inv) { return root_pow2_exp((unsigned)(lh + 1), (unsigned)t, inv) >= 96u; }

constexpr void lazy_shift_bounds(LazyBounds &b, int i, unsigned s) {
  if (s == 0) return;
  // |V 2^f / 2^64| must fit a signed 32-bit word, f = s mod 32
  const int f = (int)(s % 32u);
  const int m = (b.hi[i] + 1 > -b.lo[i]) ? b.hi[i] + 1 : -b.lo[i];
  if (((int64_t)m << f) >= (1ll << 31)) b.ok = false;
  b.lo[i] = s < 32 ? 0 : (s < 64 ? -1 : -2);
  b.hi[i] = s < 32 ? 1 : 0;
}

// A: log2 of the DFT; e_in: inputs have e in [-1, 1] (else 0).
constexpr LazyBounds lazy_bounds(int A, bool inv, bool dit, bool e_in, int bias) {
  LazyBounds b{};
  b.ok = true;
  const int n = 1 << A;
  for (int i = 0; i < n; ++i) {
    b.lo[i] = e_in ? -1 : 0;
    b.hi[i] = e_in ? 1 : 0;
  }
  b.lo[0] += bias - 1;  // the borrow of the bias's lower part
  b.hi[0] += bias;
  for (int s = 0; s < A; ++s) {
    const int lh = dit ? s : A - 1 - s, half = 1 << lh;
    for (int k = 0; k < n / 2; ++k) {
      const int t = k % half, i0 = (k / half) * 2 * half + t, i1 = i0 + half;
      const unsigned sh = lazy_exp(lh, t, inv);
      const bool neg = lazy_neg(lh, t, inv);
      if (dit) lazy_shift_bounds(b, i1, sh);
      const int ul = b.lo[i0], uh = b.hi[i0], vl = b.lo[i1], vh = b.hi[i1];
      const int sl = ul + vl, sh2 = uh + vh + 1;
      const bool swap = !dit && neg;
      const int dl = (swap ? vl - uh : ul - vh) - 1, dh = swap ? vh - ul : uh - vl;
      if (dit && neg) {
        b.lo[i0] = dl, b.hi[i0] = dh, b.lo[i1] = sl, b.hi[i1] = sh2;
      } else {
        b.lo[i0] = sl, b.hi[i0] = sh2, b.lo[i1] = dl, b.hi[i1] = dh;
      }
      if (!dit) lazy_shift_bounds(b, i1, sh);
    }
  }
  return b;
}

constexpr int lazy_bias(int A, bool inv, bool dit, bool e_in) {
  const LazyBounds b = lazy_bounds(A, inv, dit, e_in, 1);
  int lo = 0;
  for (int i = 0; i < (1 << A); ++i) lo = b.lo[i] < lo ? b.lo[i] : lo;
  return 1 - lo;
}

// Operands of the multiply-add that gives V 2^S (S = 0 < S < 96) as
// Z + c 2^64 + base 2^64: Z = f EPS + d with carry c.  With f = S mod 32, the
// words of V 2^f are y0, y1 and the signed h:
//   S < 32:   y + h 2^64.  A negative h enters the unsigned product as
//             h + 2^32, and 2^32 EPS = -1, so 1 is put into y's zero low bits.
//   S < 64:   y0 2^32 + y1 2^64 - h = y1 EPS + {~h, y0} - EPS; a negative h
//             makes ~h wrap, which the 1 put into y0's zero low bits restores.
//   S >= 64:  y0 2^64 - y1 - h 2^32 = y0 EPS + {~y1, -h} - EPS, {~y1, -h}
//             read as signed.
// The - EPS is -1 in the new e.
template <unsigned S> GL_FN void shift_operands(uint64_t x, int32_t e, uint32_t &f, uint64_t &d, uint32_t &base) {
  constexpr unsigned F = S % 32u;
  static_assert(F != 0 && S < 96, "");
  const uint32_t x0 = lo32(x), x1 = hi32(x);
  const uint32_t y1 = align32(x1, x0, 32 - F), h = align32((uint32_t)e, x1, 32 - F);
  if constexpr (S < 32) {
    f = h;
    d = pair64((x0 << F) | (h >> 31), y1);
    base = 0;
  } else if constexpr (S < 64) {
    f = y1;
    d = pair64(~h, (x0 << F) | (h >> 31));
    base = 0xFFFFFFFFu;
  } else {
    f = x0 << F;
    d = pair64(~y1, 0u - h);
    base = (uint32_t)((int32_t)(0u - h) >> 31) - 1u;
  }
}

// One level's butterflies over 16 registers (16 >> A DFTs of 2^A points side
// by side), eight of them, two at a time.
template <int A, int LH, bool INV, bool DIT> struct LazyLevel {
  static constexpr int HALF = 1 << LH;
  static constexpr int i0(int k) { return (k / HALF) * 2 * HALF + k % HALF; }
  static constexpr int i1(int k) { return i0(k) + HALF; }
  static constexpr unsigned exp(int k) { return lazy_exp(LH, k % HALF, INV); }
  static constexpr bool neg(int k) { return lazy_neg(LH, k % HALF, INV); }
  // the shifted values among butterflies [4 r, 4 r + 4), in order
  static constexpr int shifts(int r) {
    int n = 0;
    for (int k = 4 * r; k < 4 * r + 4; ++k) n += exp(k) != 0;
    return n;
  }
  static constexpr int shifted(int r, int j) {
    for (int k = 4 * r; k < 4 * r + 4; ++k)
      if (exp(k) != 0 && j-- == 0) return k;
    return -1;
  }

  template <int R> GL_FN static void shift(uint64_t *x, int32_t *e) {
    constexpr int N = shifts(R);
    if constexpr (N > 0) {
      uint32_t f[N], base[N], ne[N];
      uint64_t d[N], z[N];
      unroll<N>([&](auto j) {
        constexpr int J = decltype(j)::value, K = shifted(R, J), I = i1(K);
        shift_operands<exp(K)>(x[I], e[I], f[J], d[J], base[J]);
      });
      row::Rows<N>::mad_eps_carry(z, ne, f, d, base);
      unroll<N>([&](auto j) {
        constexpr int J = decltype(j)::value, I = i1(shifted(R, J));
        x[I] = z[J];
        e[I] = (int32_t)ne[J];
      });
    }
  }

  template <int P2> GL_FN static void butterflies(uint64_t *x, int32_t *e) {
    uint32_t u[2][3], v[2][3], s[2][3], d[2][3];
    unroll<2>([&](auto j) {
      constexpr int J = decltype(j)::value, K = 2 * P2 + J;
      // DIF with a negated twiddle takes v - u; DIT puts u - m first
      constexpr bool swap = !DIT && neg(K);
      constexpr int U = swap ? i1(K) : i0(K), V = swap ? i0(K) : i1(K);
      u[J][0] = lo32(x[U]), u[J][1] = hi32(x[U]), u[J][2] = (uint32_t)e[U];
      v[J][0] = lo32(x[V]), v[J][1] = hi32(x[V]), v[J][2] = (uint32_t)e[V];
    });
    row::butterfly2(s, d, u, v);
    unroll<2>([&](auto j) {
      constexpr int J = decltype(j)::value, K = 2 * P2 + J;
      constexpr bool flip = DIT && neg(K);
      constexpr int S = flip ? i1(K) : i0(K), D = flip ? i0(K) : i1(K);
      x[S] = pair64(s[J][0], s[J][1]);
      e[S] = (int32_t)s[J][2];
      x[D] = pair64(d[J][0], d[J][1]);
      e[D] = (int32_t)d[J][2];
    });
  }

  GL_FN static void run(uint64_t *x, int32_t *e) {
    unroll<2>([&](auto r) {
      constexpr int R = decltype(r)::value;
      if constexpr (DIT) shift<R>(x, e);
      butterflies<2 * R>(x, e);
      butterflies<2 * R + 1>(x, e);
      if constexpr (!DIT) shift<R>(x, e);
    });
  }
};

// 16 >> A in-register DFTs of 2^A points each over x[16] (any u64, plus
// e[i] 2^64 with e in [-1, 1] when E_IN): natural input -> bit-reversed
// output (DIF), or bit-reversed input -> natural output (DIT).  Point 0 of a
// DFT is never twiddled, so K p added to it (K 2^64 in e and K - K 2^32 in x)
// reaches every output once and makes every output's e non-negative; each
// output is then reduced by one multiply-add and a carry.
template <int A, bool INV, bool DIT, Reduce R, bool E_IN = false>
GL_FN void dft_lazy(uint64_t *x, int32_t *e_in = nullptr) {
  static_assert(A >= 1 && A <= 4 && (R == ANY || R == CANON), "");
  constexpr int K = lazy_bias(A, INV, DIT, E_IN);
  static_assert(lazy_bounds(A, INV, DIT, E_IN, K).ok, "a twiddled value may not fit its shift");
  int32_t e[16];
  unroll<16>([&](auto i) {
    constexpr int I = decltype(i)::value;
    if constexpr (E_IN) e[I] = e_in[I];
    else e[I] = 0;
    if constexpr ((I & ((1 << A) - 1)) == 0) {
      constexpr uint64_t KE = (uint64_t)K * EPS;
      e[I] += x[I] < KE ? K - 1 : K;
      x[I] -= KE;
    }
  });
  unroll<A>([&](auto s) {
    constexpr int S = decltype(s)::value;
    LazyLevel<A, DIT ? S : A - 1 - S, INV, DIT>::run(x, e);
  });
  unroll<4>([&](auto r) {
    constexpr int B = 4 * decltype(r)::value;
    uint32_t f[4];
    uint64_t o[4];
    unroll<4>([&](auto j) { f[decltype(j)::value] = (uint32_t)e[B + decltype(j)::value]; });
    if constexpr (R == CANON) row::Rows<4>::reduce_canon(o, f, x + B);
    else row::Rows<4>::reduce_any(o, f, x + B);
    unroll<4>([&](auto j) { x[B + decltype(j)::value] = o[decltype(j)::value]; });
  });
}

}  // namespace gl
