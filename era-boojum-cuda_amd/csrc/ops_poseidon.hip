// Poseidon and Poseidon2 (Goldilocks, width 12 = rate 8 + capacity 4, 8 full
// and 22 partial rounds, S-box x^7) Merkle-tree hashing: leaf hashes of
// column-major matrices, node hashes of digest pairs, and whole trees.
//
// Reference: src/poseidon.rs:129-328 (argument checks, tree layout) and the
// single-thread kernels native/poseidon_single_thread.cu:14-48,
// native/poseidon_single_thread.cuh:18-145, native/poseidon2_single_thread.cu,
// native/poseidon2_single_thread.cuh, native/poseidon_utils.cuh:8-61.  Both
// hashes read the same 360 round constants.
//
// Round constants.  The reference compiles boojum's 360 textbook round
// constants into its kernels and runs the permutation in a fused form derived
// from them at build time (build/poseidon_constants.rs).  Here the caller
// supplies the 360 constants once (bc_poseidon_set_round_constants); the
// library derives the same fused form on the host and keeps it in a
// per-device table that every hashing kernel reads through the scalar cache:
//   - rounds 0-2 and 27-29: textbook (constants, S-box on all 12, MDS);
//   - round 3: its constants and S-box, then the fused constant layer and one
//     dense 12 x 12 matrix (round 3's MDS times the first partial round's
//     dense factor);
//   - 22 partial rounds: S-box on element 0 plus one fused constant, then a
//     sparse matrix (first row and first column plus the identity);
//   - round 26: S-box and MDS only (its constants were moved into the
//     partial rounds).
// Derivation: each partial round's MDS is N = B A with A = diag(1, N^)
// (commutes with the one-element S-box layer) and B = [[1, n^T N^-1],
// [w, I]] sparse; the round before then has N = A M.  Constants move back
// through M^-1: element 0 lands after the previous round's S-box, elements
// 1..11 pass that S-box untouched.
//
// One lane hashes one leaf or node: the permutation is a serial chain of field
// products with no data shared between hashes, at four waves per SIMD (122-128
// registers for Poseidon, 8 more spilled by its leaves; 76 for Poseidon2).  A wave's 64 states take Poseidon's matrix
// products to the matrix cores together (MatMul).  Bound: vector issue slots:
// about 10.3k vector instructions per Poseidon permutation, 60% of them S-box
// products, and 10.4k (cheaper ones) per Poseidon2 permutation, against 64
// bytes absorbed.  With every word reduced to [0, p) in every step, products
// one at a time and sparse partial rounds it was 24.8k and 16.4k; 128 columns
// x 2^20 rows: 10.7 -> 5.5 ms a Poseidon tree, 2^18 leaves of 2 x 93 values:
// 3.28 -> 1.82 ms a Poseidon2 tree.
#include "../../include/boojum_ntt.h"
#include "gl_lazy.hpp"

#include <hip/hip_runtime.h>

#include <stddef.h>
#include <string.h>

#include <mutex>
#include <shared_mutex>
#include <vector>

namespace bc {
namespace {

constexpr int PT = 12, RATE = 8, CAP = 4, ROUNDS = 30, HALF_FULL = 4, PARTIAL = 22;
constexpr unsigned MDS_EXPS[PT] = {0, 0, 1, 0, 3, 5, 1, 8, 12, 3, 16, 10};

// Per-device table (canonical values).
struct PosTable {
  uint64_t rc_full[7][PT];  // textbook constants of rounds 0-3 and 27-29
  uint64_t rcf[PT];         // fused constant layer after round 3's S-box
  uint64_t dense[PT][PT];   // round 3's fused dense matrix
  uint64_t sbox_c[PARTIAL]; // constant after each partial round's S-box
  uint64_t vs[PARTIAL][PT - 1];     // first row (beyond the 1 at [0][0])
  uint64_t w_hats[PARTIAL][PT - 1]; // first column (below [0][0])
  // Poseidon2 (textbook form): constants of the full rounds 0-3 and 26-29,
  // and element 0's constant of each partial round
  uint64_t p2_full[8][PT];
  uint64_t p2_partial[PARTIAL];
};

__device__ PosTable pos_table;

// Constants of the one-lane-per-state permutations (permute, permute2).
//
// Matrix products of Poseidon run on the matrix cores (MatMul below): a matrix's
// operand bytes are in pos_mat, the constant terms of its rows here, as two
// 64-bit halves that also hold the bias MAT_BIAS.
//
// A factor b of a dot product formed on the vector unit is kept as three
// limbs, b = c0 + c1 2^24 + c2 2^48 (c0, c1 < 2^24, c2 < 2^16), so that
// products with a 32-bit half of a state word can be summed in 64 bits without
// carries.
constexpr int LIMBS = 3;
constexpr int BLOCK = 11, BLOCKS = PARTIAL / BLOCK;  // partial rounds are run in blocks of 11
// 2^DOT_BIAS_LOG is added to the low accumulator of every dot product (see
// Dot::value) and taken out of a constant.
constexpr int DOT_BIAS_LOG = 54;
constexpr int MAT_BIAS_LOG = 46;

// Partial rounds in blocks.  With z_j the S-box output of round j of a block
// and s_1..s_11 the other words at the block's start, the words at round r
// are s_i + sum_{j<r} w_j,i z_j, so element 0 after round r is
//   z_r + vs_r . s + sum_{j<r} (vs_r . w_j) z_j + constant,
// and the words 1..11 are only formed at the block's end.  The vs_r . s of all
// rounds are one 11 x 11 matrix product at the block's start, the words at its
// end another; only the sums over z are serial.
struct PosBlock {
  uint64_t start[PT][2];             // constants of the rounds' element 0 (the last row unused)
  uint32_t z[BLOCK][BLOCK][LIMBS];   // [r][j], j < r used
  uint64_t end[PT][2];               // constants of words 1..11 (the last row unused)
};
struct PosFast {
  uint64_t first[PT];       // constants of round 0
  uint64_t mds[7][PT][2];   // behind each MDS: rounds 1-3, then 27-29 and none
  uint64_t dense[PT][2];
  PosBlock block[BLOCKS];
  // Poseidon2: behind the first external matrix and behind each full round's
  // (the constants of the round that follows; element 0 alone before a
  // partial round), and behind each internal matrix (element 0; all of the
  // first closing full round's behind the last)
  uint64_t p2_ext[1 + 2 * HALF_FULL][PT][2];
  uint64_t p2_int[PARTIAL][2];
  uint64_t p2_last[PT][2];
};

// The matrices on the matrix cores.  A constant c multiplies a word by its
// bytes x_b: c x = sum_b (c 2^8b mod p) x_b, and each c 2^8b mod p is written
// as eight signed bytes d_l (balanced digits, of the residue or the residue
// less p), so that row limb l of an output is an integer sum over words and
// bytes of d_l x_b.  The operand is signed, so x_b - 128 goes in, and 128
// times the digits' sum into the row's constant.  12 words of 8 bytes are
// three steps of 32, four outputs of 8 limbs a tile of 32 rows.
enum { MAT_MDS = 0, MAT_DENSE = 1, MAT_BLOCK = 2, MATS = MAT_BLOCK + 2 * BLOCKS };
constexpr int MAT_TILES = 3, MAT_STEPS = 3;
struct PosMat {
  int8_t a[MATS][MAT_TILES][MAT_STEPS][64][16];  // operand bytes of each lane
};

__device__ __align__(16) PosMat pos_mat;
__device__ PosFast pos_fast;

// The table, through an address the optimizer cannot see through: a kernel
// that permutes in a loop then reloads the constants it needs in each pass
// (scalar-cache hits) instead of hoisting them all into more SGPRs than a
// wave has, which spilled them to VGPR lanes.  The address is in the constant
// space: through a plain pointer the loads were per-lane flat ones into
// registers (tree of 2^20 leaves, Poseidon 8.4 -> 6.9 ms and 126 -> 102 VGPRs,
// Poseidon2 2.17 -> 1.97 ms and 26 spilled registers less).
__device__ __forceinline__ const PosFast &table() {
  using Const = const PosFast __attribute__((address_space(4)));
  Const *p = (Const *)&pos_fast;
  asm volatile("" : "+s"(p));
  return *(const PosFast *)p;
}

// x^7 of N words, any u64 in and out.
template <int N> __device__ __forceinline__ void sbox_row(uint64_t *x) {
  uint64_t x2[N], x3[N], x4[N];
  gl::mul_row<N, gl::ANY>(x2, x, x);
  gl::mul_row<N, gl::ANY>(x3, x2, x);
  gl::mul_row<N, gl::ANY>(x4, x2, x2);
  gl::mul_row<N, gl::ANY>(x, x3, x4);
}
__device__ __forceinline__ void sbox_all(uint64_t (&s)[PT]) {
  sbox_row<4>(s);
  sbox_row<4>(s + 4);
  sbox_row<4>(s + 8);
}

// A power of two in an SGPR the optimizer does not know the value of, so that
// a product with it stays one multiply-add into a 64-bit sum (a shift of a
// widened word and an addition otherwise).
__device__ __forceinline__ uint32_t opaque(uint32_t v) {
  asm("" : "+s"(v));
  return v;
}

// Matrix products of the states of a whole wave (every lane of the wave runs
// this, also those without a state of their own).  Lane h's state is column
// h % 32 of one of two 32-column tiles, and a tile's operand wants the first
// two words of a step in lanes 0..31 and the next two in lanes 32..63, for the
// same 32 states: v_permlane32_swap turns two words of all 64 states into
// that for both tiles.  Of the result a lane holds, for its column, limbs 0..3
// of the four outputs (lanes 0..31) or limbs 4..7 (lanes 32..63); two limbs are
// put together (they are below 2^21), the same swap brings the sums of every
// state to its own lane, and the halves are formed with the row's constant
// (which holds a bias that keeps them positive) and reduced once.
//
// The permutation is bound by vector issue slots, and matrix instructions run
// beside those of other waves: an output costs 15 slots here, 28 as an MDS row
// on the vector unit and 82 as a dense row of 11 words.  Poseidon, tree of 2^20
// leaves of 128 words: 6.9 -> 5.5 ms (10.3k vector instructions a permutation
// instead of 15.9k).  Tiles are kept apart for the scheduler: interleaved they
// took 66 registers more than the 128 that four waves a SIMD leave.
struct MatMul {
  using V4 = int __attribute__((ext_vector_type(4)));
  using V16 = int __attribute__((ext_vector_type(16)));
  static constexpr uint32_t SIGNS = 0x80808080u;
  V4 x[MAT_STEPS][2];
  __device__ __forceinline__ explicit MatMul(const uint64_t (&w)[PT]) {
#pragma unroll
    for (int st = 0; st < MAT_STEPS; ++st)
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const uint64_t a = w[4 * st + d / 2], b = w[4 * st + 2 + d / 2];
        const auto r = __builtin_amdgcn_permlane32_swap((d % 2 ? gl::hi32(a) : gl::lo32(a)) ^ SIGNS,
                                                        (d % 2 ? gl::hi32(b) : gl::lo32(b)) ^ SIGNS, false, false);
        x[st][0][d] = (int)r[0];
        x[st][1][d] = (int)r[1];
      }
  }
  // The words of step st again (the swap is its own inverse).
  __device__ __forceinline__ void words(uint64_t *w, int st) const {
    uint32_t h[2][4];
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const auto r = __builtin_amdgcn_permlane32_swap((uint32_t)x[st][0][d], (uint32_t)x[st][1][d], false, false);
      h[0][d] = r[0] ^ SIGNS;
      h[1][d] = r[1] ^ SIGNS;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = gl::pair64(h[i / 2][2 * (i % 2)], h[i / 2][2 * (i % 2) + 1]);
  }
  // y[q] = output 4 tile + q, + add[q]
  template <bool ADD = false>
  __device__ __forceinline__ void tile(uint64_t *y, int mat, int tile, const uint64_t (*k)[2],
                                       const uint64_t *add = nullptr) const {
    const V4 *a = (const V4 *)&pos_mat.a[mat][tile][0][threadIdx.x % 64][0];
    V16 acc[2] = {};
#pragma unroll
    for (int st = 0; st < MAT_STEPS; ++st) {
      const V4 op = a[st * 64];
      acc[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(op, x[st][0], acc[0], 0, 0, 0);
      acc[1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(op, x[st][1], acc[1], 0, 0, 0);
    }
    // vector registers, so that the row constant may be the scalar operand
    int32_t one = 1, c16 = 1 << 16;
    asm("" : "+v"(one), "+v"(c16));
    uint64_t h[2][4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      // two limbs at a time, before the swap: |l| < 2^21
      int32_t l[2][2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const auto r = __builtin_amdgcn_permlane32_swap(
            (uint32_t)acc[0][4 * q + 2 * i] + ((uint32_t)acc[0][4 * q + 2 * i + 1] << 8),
            (uint32_t)acc[1][4 * q + 2 * i] + ((uint32_t)acc[1][4 * q + 2 * i + 1] << 8), false, false);
        l[0][i] = (int32_t)r[0];
        l[1][i] = (int32_t)r[1];
      }
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        int64_t v = (int64_t)l[w][1] * c16 + (int64_t)k[4 * tile + q][w];
        v += (int64_t)l[w][0] * one;
        if constexpr (ADD) v += (uint64_t)(w ? gl::hi32(add[q]) : gl::lo32(add[q])) * (uint32_t)one;
        h[w][q] = (uint64_t)v;
      }
    }
    gl::join_halves<4>(y, h[0], h[1]);
    __builtin_amdgcn_sched_barrier(0);
  }
  __device__ __forceinline__ void all(uint64_t *y, int mat, const uint64_t (*k)[2]) const {
#pragma unroll
    for (int t = 0; t < MAT_TILES; ++t) tile(y + 4 * t, mat, t, k);
  }
};

// A dot product of state words with table constants: six 64-bit sums, one
// multiply-add per word half and limb.  At most BLOCK terms, so the sums stay
// below 2^61 (limbs of 24 bits) and 2^53 (16 bits).
struct Dot {
  uint64_t p0, p1 = 0, p2 = 0, q0, q1 = 0, q2 = 0;
  __device__ __forceinline__ explicit Dot(uint64_t start)  // the sum's first term, less the bias
      : p0(gl::pair64(gl::lo32(start), 1u << (DOT_BIAS_LOG - 32))), q0(gl::hi32(start)) {}
  __device__ __forceinline__ void mac(uint64_t a, const uint32_t *c) {
    const uint64_t a0 = gl::lo32(a), a1 = gl::hi32(a);
    p0 += a0 * c[0];
    p1 += a0 * c[1];
    p2 += a0 * c[2];
    q0 += a1 * c[0];
    q1 += a1 * c[1];
    q2 += a1 * c[2];
  }
  __device__ __forceinline__ void add(uint64_t a, uint32_t one) {  // one: opaque(1)
    p0 += (uint64_t)gl::lo32(a) * one;
    q0 += (uint64_t)gl::hi32(a) * one;
  }
  // p0 + p1 2^24 + p2 2^48 + (q0 + q1 2^24 + q2 2^48) 2^32, by weight:
  // l + u 2^32 + v 2^64 + w 2^96 = (l - v - w) + (u + v) 2^32.  The bias in p0
  // keeps l - v - w >= 0 (v < 2^53, w < 2^37).  lo < 2^62, hi < 2^62.
  __device__ __forceinline__ void halves(uint64_t &lo, uint64_t &hi, uint32_t c24, uint32_t c16) const {
    const uint64_t l = p0 + (uint64_t)gl::lo32(p1) * c24;
    const uint64_t u = q0 + (uint64_t)gl::hi32(p1) * c24 + (uint64_t)gl::lo32(p2) * c16 + (uint64_t)gl::lo32(q1) * c24;
    const uint64_t v = (uint64_t)gl::hi32(q1) * c24 + (uint64_t)gl::hi32(p2) * c16 + (uint64_t)gl::lo32(q2) * c16;
    const uint64_t w = (uint64_t)gl::hi32(q2) * c16 + v;
    lo = l - w;
    hi = u + v;
  }
};

// One dot product's value (any u64).
__device__ __forceinline__ uint64_t dot_value(const Dot &d, uint32_t c24, uint32_t c16) {
  uint64_t lo, hi, r;
  d.halves(lo, hi, c24, c16);
  gl::join_halves<1>(&r, &lo, &hi);
  return r;
}

// The permutation on any u64 words, giving any u64 words.  Only the four words
// read next are formed by the last MDS: the capacity (capacity_out; a sponge
// overwrites the rate), else words 0..3, the digest.
__device__ __forceinline__ void permute(uint64_t (&s)[PT], bool capacity_out) {
  const PosFast &t = table();
#pragma unroll
  for (int i = 0; i < PT; ++i) {
    // s + constant: the constant is below p, so one carry is all there can be
    const uint64_t v = s[i] + t.first[i];
    s[i] = v + (v < s[i] ? gl::EPS : 0ull);
  }
#pragma unroll 1
  for (int r = 0; r < HALF_FULL - 1; ++r) {
    sbox_all(s);
    MatMul(s).all(s, MAT_MDS, t.mds[r]);
  }
  sbox_all(s);
  MatMul(s).all(s, MAT_DENSE, t.dense);
  const uint32_t c24 = opaque(1u << 24), c16 = opaque(1u << 16), one = opaque(1u);
#pragma unroll 1
  for (int b = 0; b < BLOCKS; ++b) {
    const PosBlock &blk = t.block[b];
    uint64_t first[4], z[PT], w[PT];
#pragma unroll
    for (int i = 1; i < PT; ++i) w[i - 1] = s[i];
    w[PT - 1] = 0;
    const MatMul start(w);
#pragma unroll
    for (int r = 0; r < BLOCK; ++r) {
      if (r % 4 == 0) start.tile(first, MAT_BLOCK + 2 * b, r / 4, blk.start);
      z[r] = s[0];
      sbox_row<1>(z + r);
      Dot d(first[r % 4]);
#pragma unroll
      for (int j = 0; j < r; ++j) d.mac(z[j], blk.z[r][j]);
      d.add(z[r], one);
      s[0] = dot_value(d, c24, c16);
    }
    z[PT - 1] = 0;
    const MatMul end(z);
#pragma unroll
    for (int tl = 0; tl < MAT_TILES; ++tl) {
      start.words(w + 4 * tl, tl);
      end.tile<true>(w + 4 * tl, MAT_BLOCK + 2 * b + 1, tl, blk.end, w + 4 * tl);
    }
#pragma unroll
    for (int i = 1; i < PT; ++i) s[i] = w[i - 1];
  }
#pragma unroll 1
  for (int r = 0; r < 3; ++r) {
    sbox_all(s);
    MatMul(s).all(s, MAT_MDS, t.mds[3 + r]);
  }
  sbox_all(s);
  uint64_t y[CAP];
  const MatMul m(s);
  if (capacity_out) {
    m.tile(y, MAT_MDS, RATE / CAP, t.mds[6]);
#pragma unroll
    for (int i = 0; i < CAP; ++i) s[RATE + i] = y[i];
  } else {
    m.tile(y, MAT_MDS, 0, t.mds[6]);
#pragma unroll
    for (int i = 0; i < CAP; ++i) s[i] = y[i];
  }
}

// ---- Poseidon2 (native/poseidon2_single_thread.cu:7-24,
// native/poseidon2_single_thread.cuh:12-66): external matrix M_E = circ(2 M4,
// M4, M4) over the three 4-tiles, internal matrix M_I = J + diag(2^mu_i).
constexpr unsigned P2_MU[PT] = {4, 14, 11, 8, 0, 5, 2, 9, 13, 6, 3, 12};

// M4 = [[5,7,1,3],[4,6,1,1],[1,3,5,7],[1,1,4,6]] on one tile of 64-bit sums, by
// the addition chain of eprint 2023/323 Appendix B (8 shifted additions).
__device__ __forceinline__ void m4_tile(uint64_t *x) {
  const uint64_t t0 = x[0] + x[1];
  const uint64_t t1 = x[2] + x[3];
  const uint64_t t2 = (x[1] << 1) + t1;
  const uint64_t t3 = (x[3] << 1) + t0;
  const uint64_t t4 = (t1 << 2) + t3;
  const uint64_t t5 = (t0 << 2) + t2;
  x[0] = t3 + t5;
  x[1] = t5;
  x[2] = t2 + t4;
  x[3] = t4;
}

// acc + a * c, kept from being put together with others of the same factor.
__device__ __forceinline__ uint64_t mad_keep(uint32_t a, uint32_t c, uint64_t acc) {
  uint64_t r = acc + (uint64_t)a * c;
  asm("" : "+v"(r));
  return r;
}

// The external matrix plus constants: M4 on each tile plus the sum of the
// tiles.  The two 32-bit halves of the words go through the additions apart
// (below 2^39) and each word is reduced once; halves are added to 64-bit sums
// as products with 1, since as addends they would need a zeroed upper register
// each.
__device__ __forceinline__ void m_ext(uint64_t (&s)[PT], const uint64_t (*k)[2]) {
  const uint32_t one = opaque(1u);
  uint64_t h[2][PT];
#pragma unroll
  for (int w = 0; w < 2; ++w) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint64_t sum = w ? gl::hi32(s[j]) : gl::lo32(s[j]);
#pragma unroll
      for (int g = 4; g < PT; g += 4) sum = mad_keep(w ? gl::hi32(s[g + j]) : gl::lo32(s[g + j]), one, sum);
#pragma unroll
      for (int g = 0; g < PT; g += 4) h[w][g + j] = mad_keep(w ? gl::hi32(s[g + j]) : gl::lo32(s[g + j]), one, sum);
    }
#pragma unroll
    for (int g = 0; g < PT; g += 4) m4_tile(h[w] + g);
#pragma unroll
    for (int i = 0; i < PT; ++i) h[w][i] += k[i][w];
  }
  gl::unroll<3>([&](auto g) {
    constexpr int G = 4 * decltype(g)::value;
    gl::join_halves<4>(s + G, h[0] + G, h[1] + G);
  });
}

// 1, 2^mu_i and 2^2mu_i in SGPRs, each of a value of its own to the optimizer
// (products with the same factor would be put together behind a sum).
struct P2Factors {
  uint32_t one[PT], d[PT], dd[PT];
  __device__ __forceinline__ P2Factors() {
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      one[i] = 1u;
      d[i] = 1u << P2_MU[i];
      dd[i] = 1u << (2 * P2_MU[i]);
      asm volatile("" : "+s"(one[i]), "+s"(d[i]), "+s"(dd[i]));
    }
  }
};

// Two partial rounds but for the first one's S-box.  M_I x = sum(x) + D x with
// D = diag(2^mu), so with S = sum(x), z the S-box of element 0 after the first
// matrix, and T the sum of the other elements after it,
//   u_0 = S + D_0 x_0 (+ k0),  T = 11 S + sum_{i>0} D_i x_i,
//   y_0 = T + z + D_0 z (+ k1),  y_i = T + z + D_i S + D_i^2 x_i:
// only element 0 is reduced between the two.  The halves go apart, below
// 2^61.
__device__ __forceinline__ void two_partial_rounds(uint64_t (&s)[PT], const P2Factors &f, const uint64_t *k0,
                                                   const uint64_t *k1, const uint64_t (*last)[2]) {
  uint64_t S[2], h[2][PT], u[2], z;
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    S[w] = w ? gl::hi32(s[0]) : gl::lo32(s[0]);
#pragma unroll
    for (int i = 1; i < PT; ++i) S[w] += (uint64_t)(w ? gl::hi32(s[i]) : gl::lo32(s[i])) * f.one[i];
    u[w] = S[w] + k0[w] + (uint64_t)(w ? gl::hi32(s[0]) : gl::lo32(s[0])) * f.d[0];
  }
  gl::join_halves<1>(&z, u, u + 1);
  sbox_row<1>(&z);
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    uint64_t t = (S[w] << 3) + S[w];
    t = (S[w] << 1) + t;
#pragma unroll
    for (int i = 1; i < PT; ++i) t += (uint64_t)(w ? gl::hi32(s[i]) : gl::lo32(s[i])) * f.d[i];
    const uint32_t zw = w ? gl::hi32(z) : gl::lo32(z);
    t += (uint64_t)zw * f.one[0];
    h[w][0] = t + (uint64_t)zw * f.d[0];
    if (!last) h[w][0] += k1[w];
    // S by 2^4, 2^8, 2^12: a product with D_i is a shift by up to 3 in the addition
    uint64_t sh[4] = {S[w]};
#pragma unroll
    for (int g = 1; g < 4; ++g) {
      sh[g] = sh[g - 1] << 4;
      asm("" : "+v"(sh[g]));
    }
#pragma unroll
    for (int i = 1; i < PT; ++i)
      h[w][i] = (sh[P2_MU[i] / 4] << (P2_MU[i] % 4)) + t + (uint64_t)(w ? gl::hi32(s[i]) : gl::lo32(s[i])) * f.dd[i];
    if (last) {
#pragma unroll
      for (int i = 0; i < PT; ++i) h[w][i] += last[i][w];
    }
  }
  gl::unroll<3>([&](auto g) {
    constexpr int G = 4 * decltype(g)::value;
    gl::join_halves<4>(s + G, h[0] + G, h[1] + G);
  });
}

__device__ __forceinline__ void permute2(uint64_t (&s)[PT], bool) {
  const PosFast &t = table();
  m_ext(s, t.p2_ext[0]);
#pragma unroll 1
  for (int r = 0; r < HALF_FULL; ++r) {
    sbox_all(s);
    m_ext(s, t.p2_ext[1 + r]);
  }
  const P2Factors f;
#pragma unroll 1
  for (int k = 0; k < PARTIAL - 2; k += 2) {
    sbox_row<1>(s);
    two_partial_rounds(s, f, t.p2_int[k], t.p2_int[k + 1], nullptr);
  }
  sbox_row<1>(s);
  two_partial_rounds(s, f, t.p2_int[PARTIAL - 2], nullptr, t.p2_last);
#pragma unroll 1
  for (int r = 0; r < HALF_FULL; ++r) {
    sbox_all(s);
    m_ext(s, t.p2_ext[1 + HALF_FULL + r]);
  }
}

template <int H> __device__ __forceinline__ void permute_h(uint64_t (&s)[PT], bool capacity_out) {
  if constexpr (H == 0) permute(s, capacity_out);
  else permute2(s, capacity_out);
}

// native/poseidon_utils.cuh:8-42: leaf g absorbs the values (row r, column c)
// at values[g rows + r + c rows count] in the order c rows + r, 8 at a time
// into state[0..8] (the last chunk zero-padded), permuting after each chunk.
template <int H>
__global__ __launch_bounds__(256, 4) void poseidon_leaves_kernel(const uint64_t *__restrict__ values,
                                                              uint64_t *__restrict__ results, uint32_t rows,
                                                              uint32_t cols, uint32_t count, bool load_intermediate,
                                                              bool store_intermediate) {
  // a wave's lanes all take part in its matrix products, so lanes past the end
  // hash the last leaf again and store nothing
  const uint32_t lane_leaf = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t g = lane_leaf < count ? lane_leaf : count - 1;
  uint64_t s[PT];
#pragma unroll
  for (int i = 0; i < PT; ++i) s[i] = 0;
  if (load_intermediate) {
#pragma unroll
    for (int i = 0; i < CAP; ++i) s[RATE + i] = results[g + (uint64_t)i * count];
  }
  const uint64_t col_stride = (uint64_t)rows * count;
  const uint64_t *base = values + (uint64_t)g * rows;
  const uint64_t total = (uint64_t)rows * cols;
  uint32_t r = 0, c = 0;  // position of `off` = c rows + r
  for (uint64_t off = 0; off < total; off += RATE) {
#pragma unroll
    for (int i = 0; i < RATE; ++i) {
      s[i] = c < cols ? base[r + c * col_stride] : 0ull;
      if (++r == rows) {
        r = 0;
        ++c;
      }
    }
    // the next chunk overwrites the rate, so only the capacity is read on
    permute_h<H>(s, store_intermediate || off + RATE < total);
  }
  if (lane_leaf >= count) return;
#pragma unroll
  for (int i = 0; i < CAP; ++i)
    results[g + (uint64_t)i * count] = gl::canon(store_intermediate ? s[RATE + i] : s[i]);
}

// native/poseidon_utils.cuh:44-61: node g hashes children 2g, 2g + 1 of the
// layer below (4 columns of 2 count digests): state[i] = left[i],
// state[4 + i] = right[i], capacity zero.
template <int H>
__global__ __launch_bounds__(256, 4) void poseidon_nodes_kernel(const uint64_t *__restrict__ values,
                                                             uint64_t *__restrict__ results, uint32_t count) {
  const uint32_t lane_node = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t g = lane_node < count ? lane_node : count - 1;
  uint64_t s[PT];
#pragma unroll
  for (int i = 0; i < CAP; ++i) {
    const uint64_t *pair = values + 2 * ((uint64_t)g + (uint64_t)i * count);
    s[i] = pair[0];
    s[CAP + i] = pair[1];
    s[RATE + i] = 0;
  }
  permute_h<H>(s, false);
  if (lane_node >= count) return;
#pragma unroll
  for (int i = 0; i < CAP; ++i) results[g + (uint64_t)i * count] = gl::canon(s[i]);
}

// ---- cooperative hashing: one state over 16 lanes ------------------------------
// A small layer is one dependent permutation chain per lane, whatever its
// size: 10-12k instructions at one per 8 cycles, the rate of a wave alone on
// its SIMD.  Here lane j of a 16-lane row owns state element j (lanes 12-15
// hold values nobody reads), so a lane runs one S-box and one matrix row per
// round.  Sums over the row are taken on 22-bit limbs with row rotations
// (plain 32-bit additions, 12 instructions for the 16 lanes); the MDS row and
// the 4-tiles gather their words through the wave's LDS, a round's constants
// come from LDS.  Used for layers and leaf sets of at most COOP_MAX (the
// reference likewise switches to cooperative kernels for small layers,
// src/poseidon.rs:71,279-283).  Four permutations a leaf, 16 lanes against
// one: Poseidon 64 / 119 us at 2^13, 107 / 118 at 2^14, 193 / 121 at 2^15;
// Poseidon2 49 / 91 us at 2^13, 86 / 91 at 2^14, 158 / 92 at 2^15.
constexpr uint32_t COOP_LANES = 16;
constexpr uint32_t COOP_MAX = 1u << 14;
constexpr uint32_t COOP_NT = 512, COOP_GROUPS = COOP_NT / COOP_LANES;  // two waves per SIMD issue side by side

// A lane's part of a Poseidon partial round: its row and column entries (0 and
// 1 for element 0) and, by halves, what the S-box's constant c adds (c itself
// for element 0, else w c).
struct PartialLane {
  uint64_t v, w, k[2];
};
__device__ PartialLane pos_partial_lanes[PARTIAL][PT];

// A row's words in LDS, twice in a row so that word (j + i) mod 12 is at j + i.
struct CoopLds {
  PosTable t;
  PartialLane partial[PARTIAL][PT];
  // constants behind Poseidon2's partial rounds, by halves (0 but for element 0
  // and the last round)
  uint64_t p2_add[PARTIAL][PT][2];
  uint64_t words[COOP_GROUPS][2 * PT];
};

// The wave's LDS accesses run in program order; this keeps the compiler from
// moving them across.
__device__ __forceinline__ void coop_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int CTRL> __device__ __forceinline__ uint32_t dpp(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true);
}
constexpr int ROW_ROR = 0x120, ROW_NEWBCAST = 0x150;  // rotate by n inside a row of 16; lane n to the whole row

// Element 0's value to every lane of the row.
__device__ __forceinline__ uint64_t row_first(uint64_t v) {
  return gl::pair64(dpp<ROW_NEWBCAST>(gl::lo32(v)), dpp<ROW_NEWBCAST>(gl::hi32(v)));
}

// v in limbs of 22, 22 and 20 bits; keep is the 22-bit mask, 0 in lanes whose
// value must not count.
struct Limbs {
  uint32_t a, b, c;
  __device__ __forceinline__ Limbs(uint64_t v, uint32_t keep)
      : a(gl::lo32(v) & keep), b(gl::align32(gl::hi32(v), gl::lo32(v), 22) & keep), c((gl::hi32(v) >> 12) & keep) {}
  template <int N> __device__ __forceinline__ void add_ror() {
    a += dpp<ROW_ROR + N>(a);
    b += dpp<ROW_ROR + N>(b);
    c += dpp<ROW_ROR + N>(c);
  }
  // lo + hi 2^32 += a + b 2^22 + c 2^44 (limbs below 2^32)
  __device__ __forceinline__ void add_to(uint64_t &lo, uint64_t &hi) const {
    lo += (uint64_t)b * opaque(1u << 22) + a;
    hi += (uint64_t)c * opaque(1u << 12);
  }
};

// x^7, the cube and the fourth power side by side.
__device__ __forceinline__ uint64_t coop_sbox(uint64_t x) {
  uint64_t s, a[2], b[2], c[2], r;
  gl::mul_row<1, gl::ANY>(&s, &x, &x);
  a[0] = a[1] = s;
  b[0] = x;
  b[1] = s;
  gl::mul_row<2, gl::ANY>(c, a, b);
  gl::mul_row<1, gl::ANY>(&r, &c[0], &c[1]);
  return r;
}

// Partial rounds: the S-box of element 0 with the sum over the row in its
// waits.  A mask written by a vector instruction may be read two instructions
// later at the earliest (and a rotation reads a register two instructions
// after its write), and a wave alone on its SIMD pays a full issue slot for
// every s_nop that fills such a gap: 27 of 119 slots in a Poseidon2 round.
// The sum does not depend on the S-box's end, so its instructions stand there
// (103 slots; a Poseidon2 tree of 2^11 leaves, one permutation each, 122 -> 111
// us; 128 with the same sum ahead of the S-box).  Poseidon: 168 -> 131 slots,
// four permutations a leaf 63.9 -> 57.8 us at 2^10 leaves.
#define BC_ROR(v, n) "v_add_u32_dpp %[" #v "], %[" #v "], %[" #v "] row_ror:" #n " row_mask:0xf bank_mask:0xf bound_ctrl:1\n"
// A product's 32-bit steps, as in mul_row: u v0 + ..., the middle sum with its
// carry, and the top half.
__device__ __forceinline__ uint64_t coop_mid(uint64_t u, uint64_t v, uint64_t &p, uint64_t &carry) {
  p = (uint64_t)gl::lo32(u) * gl::lo32(v);
  uint64_t t = (uint64_t)gl::lo32(u) * gl::hi32(v) + gl::hi32(p);
  asm("v_mad_u64_u32 %0, %1, %2, %3, %4" : "=v"(t), "=s"(carry) : "v"(gl::hi32(u)), "v"(gl::lo32(v)), "v"(t));
  return t;
}
__device__ __forceinline__ uint64_t coop_top(uint64_t t, uint64_t u, uint64_t v) {
  return (uint64_t)gl::hi32(u) * gl::hi32(v) + gl::hi32(t);
}

// Poseidon2:
// rest.lo + rest.hi 2^32 becomes (k_lo + k_hi 2^32) + mu x + the sum of x over
// the lanes with keep set, the sum on limbs a, b, c of 22, 22 and 20 bits; its
// b and c are left to be added.
struct RestSum {
  uint64_t lo, hi;
  uint32_t b, c;
};
__device__ __forceinline__ uint64_t coop_sbox_rest(uint64_t x, uint32_t keep, uint32_t mu, uint64_t k_lo, uint64_t k_hi,
                                                   RestSum &rest) {
  const uint32_t x0 = gl::lo32(x), x1 = gl::hi32(x);
  uint32_t a, b, c;
  uint64_t p, q, t, v, m, n;
  uint32_t e0, e1, r2, f, g0, g1;
  // the square
  t = coop_mid(x, x, p, m);
  q = coop_top(t, x, x);
  asm("s_nop 0\n"
      "v_subb_co_u32_e64 %[e0], %[m], %[p0], %[q1], %[m]\n"
      "v_and_b32 %[a], %[x0], %[keep]\n"
      "v_alignbit_b32 %[b], %[x1], %[x0], 22\n"
      "v_subb_co_u32_e64 %[e1], %[m], %[t0], 0, %[m]\n"
      "v_lshrrev_b32 %[c], 12, %[x1]\n"
      "v_and_b32 %[b], %[b], %[keep]\n"
      "v_subb_co_u32_e64 %[r2], %[m], %[q0], 0, %[m]\n"
      : [e0] "=&v"(e0), [e1] "=&v"(e1), [r2] "=&v"(r2), [a] "=&v"(a), [b] "=&v"(b), [c] "=&v"(c), [m] "+s"(m)
      : [p0] "v"(gl::lo32(p)), [q1] "v"(gl::hi32(q)), [t0] "v"(gl::lo32(t)), [q0] "v"(gl::lo32(q)), [x0] "v"(x0),
        [x1] "v"(x1), [keep] "v"(keep));
  uint64_t w;  // masks nobody reads
  asm("v_mad_u64_u32 %[v], %[n], %[r2], -1, %[e]\n"
      "v_and_b32 %[c], %[c], %[keep]\n"
      "v_mad_u64_u32 %[lo], %[w], %[x0], %[mu], %[k]\n"
      "v_cndmask_b32_e64 %[f], 0, -1, %[n]\n"
      : [v] "=&v"(v), [n] "=&s"(n), [w] "=&s"(w), [f] "=&v"(f), [c] "+v"(c), [lo] "=&v"(rest.lo)
      : [r2] "v"(r2), [e] "v"(gl::pair64(e0, e1)), [keep] "v"(keep), [x0] "v"(x0), [mu] "v"(mu), [k] "v"(k_lo));
  uint32_t s0, s1;
  asm("v_addc_co_u32_e64 %[s0], %[m], %[v0], %[f], %[m]\n" BC_ROR(a, 8) BC_ROR(b, 8)
      "v_addc_co_u32_e64 %[s1], %[m], %[v1], 0, %[m]\n"
      : [s0] "=&v"(s0), [s1] "=&v"(s1), [m] "+s"(m), [a] "+v"(a), [b] "+v"(b)
      : [v0] "v"(gl::lo32(v)), [v1] "v"(gl::hi32(v)), [f] "v"(f));
  // the cube and the fourth power
  uint64_t p2, q2, t2, v2, m2, n2;
  uint32_t d0, d1, h2, f2;
  t = coop_mid(gl::pair64(s0, s1), x, p, m);
  t2 = coop_mid(gl::pair64(s0, s1), gl::pair64(s0, s1), p2, m2);
  q = coop_top(t, gl::pair64(s0, s1), x);
  q2 = coop_top(t2, gl::pair64(s0, s1), gl::pair64(s0, s1));
  asm("v_subb_co_u32_e64 %[e0], %[m], %[p0], %[q1], %[m]\n"
      "v_subb_co_u32_e64 %[d0], %[m2], %[p20], %[q21], %[m2]\n" BC_ROR(c, 8)
      "v_subb_co_u32_e64 %[e1], %[m], %[t0], 0, %[m]\n"
      "v_subb_co_u32_e64 %[d1], %[m2], %[t20], 0, %[m2]\n" BC_ROR(a, 4)
      "v_subb_co_u32_e64 %[r2], %[m], %[q0], 0, %[m]\n"
      "v_subb_co_u32_e64 %[h2], %[m2], %[q20], 0, %[m2]\n"
      : [e0] "=&v"(e0), [e1] "=&v"(e1), [r2] "=&v"(r2), [d0] "=&v"(d0), [d1] "=&v"(d1), [h2] "=&v"(h2), [a] "+v"(a),
        [c] "+v"(c), [m] "+s"(m), [m2] "+s"(m2)
      : [p0] "v"(gl::lo32(p)), [q1] "v"(gl::hi32(q)), [t0] "v"(gl::lo32(t)), [q0] "v"(gl::lo32(q)),
        [p20] "v"(gl::lo32(p2)), [q21] "v"(gl::hi32(q2)), [t20] "v"(gl::lo32(t2)), [q20] "v"(gl::lo32(q2)));
  asm("v_mad_u64_u32 %[v], %[n], %[r2], -1, %[e]\n"
      "v_mad_u64_u32 %[v2], %[n2], %[h2], -1, %[d]\n" BC_ROR(b, 4)
      "v_cndmask_b32_e64 %[f], 0, -1, %[n]\n"
      "v_cndmask_b32_e64 %[f2], 0, -1, %[n2]\n"
      : [v] "=&v"(v), [n] "=&s"(n), [f] "=&v"(f), [v2] "=&v"(v2), [n2] "=&s"(n2), [f2] "=&v"(f2), [b] "+v"(b)
      : [r2] "v"(r2), [e] "v"(gl::pair64(e0, e1)), [h2] "v"(h2), [d] "v"(gl::pair64(d0, d1)));
  asm("v_addc_co_u32_e64 %[s0], %[m], %[v0], %[f], %[m]\n"
      "v_addc_co_u32_e64 %[g0], %[m2], %[v20], %[f2], %[m2]\n" BC_ROR(c, 4)
      "v_addc_co_u32_e64 %[s1], %[m], %[v1], 0, %[m]\n"
      "v_addc_co_u32_e64 %[g1], %[m2], %[v21], 0, %[m2]\n"
      : [s0] "=&v"(s0), [s1] "=&v"(s1), [g0] "=&v"(g0), [g1] "=&v"(g1), [m] "+s"(m), [m2] "+s"(m2), [c] "+v"(c)
      : [v0] "v"(gl::lo32(v)), [v1] "v"(gl::hi32(v)), [f] "v"(f), [v20] "v"(gl::lo32(v2)), [v21] "v"(gl::hi32(v2)),
        [f2] "v"(f2));
  // their product
  t = coop_mid(gl::pair64(s0, s1), gl::pair64(g0, g1), p, m);
  q = coop_top(t, gl::pair64(s0, s1), gl::pair64(g0, g1));
  asm("s_nop 0\n"
      "v_subb_co_u32_e64 %[e0], %[m], %[p0], %[q1], %[m]\n" BC_ROR(a, 2) BC_ROR(b, 2)
      "v_subb_co_u32_e64 %[e1], %[m], %[t0], 0, %[m]\n" BC_ROR(c, 2) BC_ROR(a, 1)
      "v_subb_co_u32_e64 %[r2], %[m], %[q0], 0, %[m]\n"
      : [e0] "=&v"(e0), [e1] "=&v"(e1), [r2] "=&v"(r2), [a] "+v"(a), [b] "+v"(b), [c] "+v"(c), [m] "+s"(m)
      : [p0] "v"(gl::lo32(p)), [q1] "v"(gl::hi32(q)), [t0] "v"(gl::lo32(t)), [q0] "v"(gl::lo32(q)));
  asm("v_mad_u64_u32 %[v], %[n], %[r2], -1, %[e]\n" BC_ROR(b, 1) BC_ROR(c, 1)
      "v_cndmask_b32_e64 %[f], 0, -1, %[n]\n"
      : [v] "=&v"(v), [n] "=&s"(n), [f] "=&v"(f), [b] "+v"(b), [c] "+v"(c)
      : [r2] "v"(r2), [e] "v"(gl::pair64(e0, e1)));
  // the last two wait for the rotations that read s0 and s1 next
  asm("v_addc_co_u32_e64 %[s0], %[m], %[v0], %[f], %[m]\n"
      "v_mad_u64_u32 %[lo], %[w], %[a], 1, %[lo]\n"
      "v_mad_u64_u32 %[hi], %[w], %[x1], %[mu], %[k]\n"
      "v_addc_co_u32_e64 %[s1], %[m], %[v1], 0, %[m]\n"
      "s_nop 1\n"
      : [s0] "=&v"(s0), [s1] "=&v"(s1), [m] "+s"(m), [w] "=&s"(w), [lo] "+v"(rest.lo), [hi] "=&v"(rest.hi)
      : [v0] "v"(gl::lo32(v)), [v1] "v"(gl::hi32(v)), [f] "v"(f), [a] "v"(a), [x1] "v"(x1), [mu] "v"(mu), [k] "v"(k_hi));
  rest.b = b;
  rest.c = c;
  return gl::pair64(s0, s1);
}

// Poseidon: the S-box of element 0, and the sum of v x over the lanes with keep
// set as limbs a, b, c (whose last rotations are left).  acc.lo + acc.hi 2^32
// becomes (k_lo + k_hi 2^32) + f x (f: 0 or 1).
struct TermSum {
  uint64_t lo, hi;
  uint32_t a, b, c;
};
__device__ __forceinline__ uint64_t coop_sbox_terms(uint64_t x, uint64_t vx, uint32_t keep, uint32_t fx, uint64_t k_lo,
                                                    uint64_t k_hi, TermSum &acc) {
  const uint32_t x0 = gl::lo32(x), x1 = gl::hi32(x);
  uint64_t p, q, t, v, m, n, p2, q2, t2, v2, m2, n2, w;  // w: masks nobody reads
  uint32_t e0, e1, r2, f, s0, s1, d0, d1, h2, f2, g0, g1, a, b, c;
  // the square and the term
  t = coop_mid(x, x, p, m);
  t2 = coop_mid(vx, x, p2, m2);
  q = coop_top(t, x, x);
  q2 = coop_top(t2, vx, x);
  asm("v_subb_co_u32_e64 %[e0], %[m], %[p0], %[q1], %[m]\n"
      "v_subb_co_u32_e64 %[d0], %[m2], %[p20], %[q21], %[m2]\n"
      "v_mad_u64_u32 %[lo], %[w], %[x0], %[fx], %[kl]\n"
      "v_subb_co_u32_e64 %[e1], %[m], %[t0], 0, %[m]\n"
      "v_subb_co_u32_e64 %[d1], %[m2], %[t20], 0, %[m2]\n"
      "v_mad_u64_u32 %[hi], %[w], %[x1], %[fx], %[kh]\n"
      "v_subb_co_u32_e64 %[r2], %[m], %[q0], 0, %[m]\n"
      "v_subb_co_u32_e64 %[h2], %[m2], %[q20], 0, %[m2]\n"
      : [e0] "=&v"(e0), [e1] "=&v"(e1), [r2] "=&v"(r2), [d0] "=&v"(d0), [d1] "=&v"(d1), [h2] "=&v"(h2),
        [lo] "=&v"(acc.lo), [hi] "=&v"(acc.hi), [m] "+s"(m), [m2] "+s"(m2), [w] "=&s"(w)
      : [p0] "v"(gl::lo32(p)), [q1] "v"(gl::hi32(q)), [t0] "v"(gl::lo32(t)), [q0] "v"(gl::lo32(q)),
        [p20] "v"(gl::lo32(p2)), [q21] "v"(gl::hi32(q2)), [t20] "v"(gl::lo32(t2)), [q20] "v"(gl::lo32(q2)),
        [x0] "v"(x0), [x1] "v"(x1), [fx] "v"(fx), [kl] "v"(k_lo), [kh] "v"(k_hi));
  asm("v_mad_u64_u32 %[v], %[n], %[r2], -1, %[e]\n"
      "v_mad_u64_u32 %[v2], %[n2], %[h2], -1, %[d]\n"
      "s_nop 0\n"
      "v_cndmask_b32_e64 %[f], 0, -1, %[n]\n"
      "v_cndmask_b32_e64 %[f2], 0, -1, %[n2]\n"
      : [v] "=&v"(v), [n] "=&s"(n), [f] "=&v"(f), [v2] "=&v"(v2), [n2] "=&s"(n2), [f2] "=&v"(f2)
      : [r2] "v"(r2), [e] "v"(gl::pair64(e0, e1)), [h2] "v"(h2), [d] "v"(gl::pair64(d0, d1)));
  asm("v_addc_co_u32_e64 %[s0], %[m], %[v0], %[f], %[m]\n"
      "v_addc_co_u32_e64 %[g0], %[m2], %[v20], %[f2], %[m2]\n"
      "s_nop 0\n"
      "v_addc_co_u32_e64 %[s1], %[m], %[v1], 0, %[m]\n"
      "v_addc_co_u32_e64 %[g1], %[m2], %[v21], 0, %[m2]\n"
      : [s0] "=&v"(s0), [s1] "=&v"(s1), [g0] "=&v"(g0), [g1] "=&v"(g1), [m] "+s"(m), [m2] "+s"(m2)
      : [v0] "v"(gl::lo32(v)), [v1] "v"(gl::hi32(v)), [f] "v"(f), [v20] "v"(gl::lo32(v2)), [v21] "v"(gl::hi32(v2)),
        [f2] "v"(f2));
  const uint64_t sq = gl::pair64(s0, s1);
  const uint32_t y0 = g0, y1 = g1;  // the term
  // the cube and the fourth power
  t = coop_mid(sq, x, p, m);
  t2 = coop_mid(sq, sq, p2, m2);
  q = coop_top(t, sq, x);
  q2 = coop_top(t2, sq, sq);
  asm("v_subb_co_u32_e64 %[e0], %[m], %[p0], %[q1], %[m]\n"
      "v_subb_co_u32_e64 %[d0], %[m2], %[p20], %[q21], %[m2]\n"
      "v_and_b32 %[a], %[y0], %[keep]\n"
      "v_subb_co_u32_e64 %[e1], %[m], %[t0], 0, %[m]\n"
      "v_subb_co_u32_e64 %[d1], %[m2], %[t20], 0, %[m2]\n"
      "v_alignbit_b32 %[b], %[y1], %[y0], 22\n"
      "v_subb_co_u32_e64 %[r2], %[m], %[q0], 0, %[m]\n"
      "v_subb_co_u32_e64 %[h2], %[m2], %[q20], 0, %[m2]\n"
      : [e0] "=&v"(e0), [e1] "=&v"(e1), [r2] "=&v"(r2), [d0] "=&v"(d0), [d1] "=&v"(d1), [h2] "=&v"(h2), [a] "=&v"(a),
        [b] "=&v"(b), [m] "+s"(m), [m2] "+s"(m2)
      : [p0] "v"(gl::lo32(p)), [q1] "v"(gl::hi32(q)), [t0] "v"(gl::lo32(t)), [q0] "v"(gl::lo32(q)),
        [p20] "v"(gl::lo32(p2)), [q21] "v"(gl::hi32(q2)), [t20] "v"(gl::lo32(t2)), [q20] "v"(gl::lo32(q2)),
        [y0] "v"(y0), [y1] "v"(y1), [keep] "v"(keep));
  asm("v_mad_u64_u32 %[v], %[n], %[r2], -1, %[e]\n"
      "v_mad_u64_u32 %[v2], %[n2], %[h2], -1, %[d]\n"
      "v_lshrrev_b32 %[c], 12, %[y1]\n"
      "v_cndmask_b32_e64 %[f], 0, -1, %[n]\n"
      "v_cndmask_b32_e64 %[f2], 0, -1, %[n2]\n"
      : [v] "=&v"(v), [n] "=&s"(n), [f] "=&v"(f), [v2] "=&v"(v2), [n2] "=&s"(n2), [f2] "=&v"(f2), [c] "=&v"(c)
      : [r2] "v"(r2), [e] "v"(gl::pair64(e0, e1)), [h2] "v"(h2), [d] "v"(gl::pair64(d0, d1)), [y1] "v"(y1));
  asm("v_addc_co_u32_e64 %[s0], %[m], %[v0], %[f], %[m]\n"
      "v_addc_co_u32_e64 %[g0], %[m2], %[v20], %[f2], %[m2]\n"
      "v_and_b32 %[b], %[b], %[keep]\n"
      "v_addc_co_u32_e64 %[s1], %[m], %[v1], 0, %[m]\n"
      "v_addc_co_u32_e64 %[g1], %[m2], %[v21], 0, %[m2]\n"
      : [s0] "=&v"(s0), [s1] "=&v"(s1), [g0] "=&v"(g0), [g1] "=&v"(g1), [m] "+s"(m), [m2] "+s"(m2), [b] "+v"(b)
      : [v0] "v"(gl::lo32(v)), [v1] "v"(gl::hi32(v)), [f] "v"(f), [v20] "v"(gl::lo32(v2)), [v21] "v"(gl::hi32(v2)),
        [f2] "v"(f2), [keep] "v"(keep));
  // their product
  const uint64_t cube = gl::pair64(s0, s1), fourth = gl::pair64(g0, g1);
  t = coop_mid(cube, fourth, p, m);
  q = coop_top(t, cube, fourth);
  asm("s_nop 0\n"
      "v_subb_co_u32_e64 %[e0], %[m], %[p0], %[q1], %[m]\n"
      "v_and_b32 %[c], %[c], %[keep]\n" BC_ROR(a, 8)
      "v_subb_co_u32_e64 %[e1], %[m], %[t0], 0, %[m]\n" BC_ROR(b, 8) BC_ROR(c, 8)
      "v_subb_co_u32_e64 %[r2], %[m], %[q0], 0, %[m]\n"
      : [e0] "=&v"(e0), [e1] "=&v"(e1), [r2] "=&v"(r2), [a] "+v"(a), [b] "+v"(b), [c] "+v"(c), [m] "+s"(m)
      : [p0] "v"(gl::lo32(p)), [q1] "v"(gl::hi32(q)), [t0] "v"(gl::lo32(t)), [q0] "v"(gl::lo32(q)), [keep] "v"(keep));
  asm("v_mad_u64_u32 %[v], %[n], %[r2], -1, %[e]\n" BC_ROR(a, 4) BC_ROR(b, 4)
      "v_cndmask_b32_e64 %[f], 0, -1, %[n]\n"
      : [v] "=&v"(v), [n] "=&s"(n), [f] "=&v"(f), [a] "+v"(a), [b] "+v"(b)
      : [r2] "v"(r2), [e] "v"(gl::pair64(e0, e1)));
  // the rotations behind the last instruction also stand before the broadcast
  // of s0 and s1, which waits as they do
  asm("v_addc_co_u32_e64 %[s0], %[m], %[v0], %[f], %[m]\n" BC_ROR(c, 4) BC_ROR(a, 2)
      "v_addc_co_u32_e64 %[s1], %[m], %[v1], 0, %[m]\n" BC_ROR(b, 2) BC_ROR(c, 2) BC_ROR(a, 1) BC_ROR(b, 1) BC_ROR(c, 1)
      : [s0] "=&v"(s0), [s1] "=&v"(s1), [m] "+s"(m), [a] "+v"(a), [b] "+v"(b), [c] "+v"(c)
      : [v0] "v"(gl::lo32(v)), [v1] "v"(gl::hi32(v)), [f] "v"(f));
  acc.a = a;
  acc.b = b;
  acc.c = c;
  return gl::pair64(s0, s1);
}
#undef BC_ROR

// a b + lo + hi 2^32, any u64, for the sums of a partial round: in a lane of
// words 1..11 lo, hi <= 2^33 - 2 (two 32-bit terms) and the low word of a is
// below 2^32 - 1 (derive_lanes), so a0 b0 + lo and a0 b1 + hi + (a0 b0 + lo) / 2^32
// stay below 2^64; in lane 0 a = 1 and lo, hi < 2^52.
__device__ __forceinline__ uint64_t coop_mul_add(uint64_t a, uint64_t b, uint64_t lo, uint64_t hi) {
  const uint64_t p = (uint64_t)gl::lo32(a) * gl::lo32(b) + lo;
  uint64_t t = (uint64_t)gl::lo32(a) * gl::hi32(b) + (hi + gl::hi32(p));
  uint64_t m, n, v;
  asm("v_mad_u64_u32 %0, %1, %2, %3, %4" : "=v"(t), "=s"(m) : "v"(gl::hi32(a)), "v"(gl::lo32(b)), "v"(t));
  const uint64_t q = coop_top(t, a, b);
  uint32_t e0, e1, r2, f, s0, s1;
  asm("s_nop 0\n"
      "v_subb_co_u32_e64 %[e0], %[m], %[p0], %[q1], %[m]\n"
      "s_nop 1\n"
      "v_subb_co_u32_e64 %[e1], %[m], %[t0], 0, %[m]\n"
      "s_nop 1\n"
      "v_subb_co_u32_e64 %[r2], %[m], %[q0], 0, %[m]\n"
      : [e0] "=&v"(e0), [e1] "=&v"(e1), [r2] "=&v"(r2), [m] "+s"(m)
      : [p0] "v"(gl::lo32(p)), [q1] "v"(gl::hi32(q)), [t0] "v"(gl::lo32(t)), [q0] "v"(gl::lo32(q)));
  asm("v_mad_u64_u32 %[v], %[n], %[r2], -1, %[e]\n"
      "s_nop 1\n"
      "v_cndmask_b32_e64 %[f], 0, -1, %[n]\n"
      : [v] "=&v"(v), [n] "=&s"(n), [f] "=&v"(f)
      : [r2] "v"(r2), [e] "v"(gl::pair64(e0, e1)));
  asm("v_addc_co_u32_e64 %[s0], %[m], %[v0], %[f], %[m]\n"
      "s_nop 1\n"
      "v_addc_co_u32_e64 %[s1], %[m], %[v1], 0, %[m]\n"
      : [s0] "=&v"(s0), [s1] "=&v"(s1), [m] "+s"(m)
      : [v0] "v"(gl::lo32(v)), [v1] "v"(gl::hi32(v)), [f] "v"(f));
  return gl::pair64(s0, s1);
}

// lo + hi 2^32 (both below 2^62), any u64.
__device__ __forceinline__ uint64_t coop_join(uint64_t lo, uint64_t hi) {
  uint64_t r;
  gl::join_halves<1>(&r, &lo, &hi);
  return r;
}

// a + b for b below p, any u64.
__device__ __forceinline__ uint64_t add_const(uint64_t a, uint64_t b) {
  const uint64_t v = a + b;
  return v + (v < a ? gl::EPS : 0ull);
}

// One lane's view of the cooperative permutations: element j of the state
// whose words are staged in w.
struct Coop {
  const PosTable &t;
  const PartialLane (&partial)[PARTIAL][PT];
  const uint64_t (&p2_add)[PARTIAL][PT][2];
  uint64_t *w;      // the row's 2 PT words in LDS
  uint32_t j, jj;   // lane of the row; table row (lanes 12-15 reuse row 11)
  uint32_t keep;    // 22-bit mask, 0 in lanes 12-15
  __device__ __forceinline__ Coop(CoopLds &l, uint32_t lane, uint32_t group)
      : t(l.t), partial(l.partial), p2_add(l.p2_add), w(l.words[group]), j(lane), jj(lane < PT ? lane : PT - 1), keep(lane < PT ? 0x3FFFFFu : 0u) {}

  __device__ __forceinline__ void stage(uint64_t x) const {
    coop_sync();  // the row's earlier reads come first
    if (j < PT) w[j] = w[j + PT] = x;
    coop_sync();
  }

  // The MDS row plus the next round's constant k.
  __device__ __forceinline__ uint64_t mds_row(uint64_t x, uint64_t k) const {
    stage(x);
    uint64_t lo = gl::lo32(k), hi = gl::hi32(k);
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      const uint64_t v = w[jj + i];
      const uint32_t c = opaque(1u << MDS_EXPS[i]);
      lo += (uint64_t)gl::lo32(v) * c;
      hi += (uint64_t)gl::hi32(v) * c;
    }
    return coop_join(lo, hi);
  }

  __device__ __forceinline__ void permute(uint64_t &x) const {
    x = add_const(x, t.rc_full[0][jj]);
#pragma unroll 1
    for (int r = 1; r < HALF_FULL; ++r) x = mds_row(coop_sbox(x), t.rc_full[r][jj]);
    {
      stage(add_const(coop_sbox(x), t.rcf[jj]));
      gl::Acc acc;
#pragma unroll
      for (int c = 0; c < PT; ++c) gl::mac(acc, w[c], t.dense[jj][c]);
      x = gl::acc_reduce(acc);
    }
    // element 0 becomes z + sum_i vs_i x_i, element i becomes x_i + w_i z
    const uint32_t keep_rest = j ? keep : 0u, fx = j ? 1u : 0u;
    const uint32_t g0 = j ? 0u : 1u, g22 = j ? 0u : 1u << 22, g12 = j ? 0u : 1u << 12;
#pragma unroll 1
    for (int k = 0; k < PARTIAL; ++k) {
      const PartialLane &pl = partial[k][jj];
      TermSum acc;
      const uint64_t z = row_first(coop_sbox_terms(x, pl.v, keep_rest, fx, pl.k[0], pl.k[1], acc));
      acc.lo += (uint64_t)acc.a * g0;
      acc.lo += (uint64_t)acc.b * g22;
      acc.hi += (uint64_t)acc.c * g12;
      x = coop_mul_add(pl.w, z, acc.lo, acc.hi);
    }
#pragma unroll 1
    for (int r = 0; r < 3; ++r) x = mds_row(coop_sbox(x), t.rc_full[HALF_FULL + r][jj]);
    x = mds_row(coop_sbox(x), 0);
  }

  // (J + I) (x) M4 on the three tiles: each word plus the sum over the tiles,
  // then the 4 x 4 row, on limbs, plus the constant k (with 32-bit products, a
  // quarter of the 24-bit ones' rate, the tree above took 109 us, now 107).
  __device__ __forceinline__ uint64_t m_ext_row(uint64_t x, const uint32_t *m4row, uint64_t k) const {
    Limbs l(x, keep), s = l;
    s.add_ror<8>();
    s.add_ror<4>();
    l.a += s.a;
    l.b += s.b;
    l.c += s.c;
    auto row = [&](uint32_t v) {  // four limbs below 2^22: 24-bit products; the row sums to at most 16
      return __umul24(m4row[0], dpp<0x00>(v)) + __umul24(m4row[1], dpp<0x55>(v)) + __umul24(m4row[2], dpp<0xAA>(v)) +
             __umul24(m4row[3], dpp<0xFF>(v));
    };
    l.a = row(l.a);
    l.b = row(l.b);
    l.c = row(l.c);
    uint64_t lo = gl::lo32(k), hi = gl::hi32(k);
    l.add_to(lo, hi);
    return coop_join(lo, hi);
  }

  __device__ __forceinline__ void permute2(uint64_t &x) const {
    constexpr uint32_t M4[4][4] = {{5, 7, 1, 3}, {4, 6, 1, 1}, {1, 3, 5, 7}, {1, 1, 4, 6}};
    uint32_t m4row[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const uint32_t q = j & 3u;
      m4row[c] = q == 0 ? M4[0][c] : (q == 1 ? M4[1][c] : (q == 2 ? M4[2][c] : M4[3][c]));
    }
    uint32_t mu = 0;  // of the lane's own word in the rest sum: none for element 0
#pragma unroll
    for (int i = 1; i < PT; ++i) mu = jj == (uint32_t)i ? 1u << P2_MU[i] : mu;
    const uint32_t keep_rest = j ? keep : 0u, z_factor = j ? 1u : 1u + (1u << P2_MU[0]);
    uint32_t s22 = 1u << 22, s12 = 1u << 12;
    asm volatile("" : "+s"(s22), "+s"(s12));
    // the constants of the next round ride on each matrix
    x = m_ext_row(x, m4row, t.p2_full[0][jj]);
#pragma unroll 1
    for (int r = 1; r < HALF_FULL; ++r) x = m_ext_row(coop_sbox(x), m4row, t.p2_full[r][jj]);
    x = m_ext_row(coop_sbox(x), m4row, j ? 0ull : t.p2_partial[0]);
#pragma unroll 1
    for (int k = 0; k < PARTIAL; ++k) {
      // y_0 = rest + (1 + 2^mu_0) z, y_i = rest + mu_i x_i + z
      const uint64_t *kp = p2_add[k][jj];
      RestSum rest;
      const uint64_t z = row_first(coop_sbox_rest(x, keep_rest, mu, kp[0], kp[1], rest));
      rest.lo += (uint64_t)rest.b * s22 + (uint64_t)gl::lo32(z) * z_factor;
      rest.hi += (uint64_t)rest.c * s12 + (uint64_t)gl::hi32(z) * z_factor;
      x = coop_join(rest.lo, rest.hi);
    }
#pragma unroll 1
    for (int r = 1; r < HALF_FULL; ++r) x = m_ext_row(coop_sbox(x), m4row, t.p2_full[HALF_FULL + r][jj]);
    x = m_ext_row(coop_sbox(x), m4row, 0);
  }

  template <int H> __device__ __forceinline__ void permute_h(uint64_t &x) const {
    if constexpr (H == 0) permute(x);
    else permute2(x);
  }
};

template <int H> __device__ __forceinline__ void coop_stage_table(CoopLds &l) {
  if constexpr (H == 0) {
    const uint64_t *src = (const uint64_t *)&pos_table;
    uint64_t *dst = (uint64_t *)&l.t;
    for (uint32_t i = threadIdx.x; i < offsetof(PosTable, p2_full) / sizeof(uint64_t); i += blockDim.x) dst[i] = src[i];
    src = (const uint64_t *)&pos_partial_lanes;
    dst = (uint64_t *)&l.partial;
    for (uint32_t i = threadIdx.x; i < sizeof l.partial / sizeof(uint64_t); i += blockDim.x) dst[i] = src[i];
    return;
  }
  if (threadIdx.x < 2 * HALF_FULL * PT) (&l.t.p2_full[0][0])[threadIdx.x] = (&pos_table.p2_full[0][0])[threadIdx.x];
  if (threadIdx.x == 0) l.t.p2_partial[0] = pos_table.p2_partial[0];
  for (uint32_t i = threadIdx.x; i < PARTIAL * PT; i += blockDim.x) {
    const uint32_t r = i / PT, j = i % PT;
    const uint64_t k = r == PARTIAL - 1 ? pos_table.p2_full[HALF_FULL][j] : (j ? 0ull : pos_table.p2_partial[r + 1]);
    l.p2_add[r][j][0] = gl::lo32(k);
    l.p2_add[r][j][1] = gl::hi32(k);
  }
}

// Climbs `layers` node layers from a workgroup's COOP_GROUPS digests in LDS,
// the first of `count` nodes (digests past a short layer's end are not read).
// Layer l's digests go to its place behind the layers before it.
template <int H>
__device__ __forceinline__ void coop_climb(const Coop &c, uint64_t (&digest)[COOP_GROUPS][CAP], uint64_t *results,
                                           uint32_t count, uint32_t layers, uint32_t group, uint32_t j) {
  uint32_t active = COOP_GROUPS;
  for (; layers; --layers) {
    __syncthreads();
    active /= 2;
    const uint64_t g = (uint64_t)blockIdx.x * active + group;
    uint64_t x = 0;
    if (j < 2 * CAP && group < active) x = digest[2 * group + (j >> 2)][j & 3u];
    __syncthreads();
    if (group < active && g < count) {
      c.permute_h<H>(x);
      if (j < CAP) {
        const uint64_t d = gl::canon(x);
        results[g + (uint64_t)j * count] = d;
        digest[group][j] = d;
      }
    }
    results += (uint64_t)CAP * count;
    count /= 2;
  }
}

// `layers` consecutive node layers, the first of `count` nodes: a workgroup
// hashes COOP_GROUPS nodes of the first layer and climbs from their digests, so
// one launch takes up to log2(COOP_GROUPS) + 1 layers (count is a multiple of
// COOP_GROUPS or below it and a power of two when layers > 1).
constexpr uint32_t COOP_MAX_LAYERS = 6;
static_assert(COOP_GROUPS == 1u << (COOP_MAX_LAYERS - 1), "");
template <int H>
__global__ __launch_bounds__(COOP_NT) void poseidon_nodes_coop_kernel(const uint64_t *__restrict__ values,
                                                                      uint64_t *__restrict__ results, uint32_t count,
                                                                      uint32_t layers) {
  __shared__ CoopLds lds;
  __shared__ uint64_t digest[COOP_GROUPS][CAP];
  coop_stage_table<H>(lds);
  const uint32_t group = threadIdx.x / COOP_LANES, j = threadIdx.x % COOP_LANES;
  const uint64_t g = (uint64_t)blockIdx.x * COOP_GROUPS + group;
  // element j: left[j] (j < 4), right[j - 4] (4 <= j < 8), capacity 0
  uint64_t x = 0;
  if (j < 2 * CAP && g < count) x = values[2 * (g + (uint64_t)(j & 3u) * count) + (j >> 2)];
  __syncthreads();
  const Coop c(lds, j, group);
  if (g < count) {
    c.permute_h<H>(x);
    if (j < CAP) {
      const uint64_t d = gl::canon(x);
      results[g + (uint64_t)j * count] = d;
      digest[group][j] = d;
    }
  }
  coop_climb<H>(c, digest, results + (uint64_t)CAP * count, count / 2, layers - 1, group, j);
}

// Cooperative leaves (src/poseidon.rs:194-216): the absorption of
// poseidon_leaves_kernel with one state over a 16-lane row; for each chunk,
// lane j < 8 takes position off + j (= c rows + r) into state element j, read
// one chunk ahead.  Then up to log2(COOP_GROUPS) node layers (count as above).
template <int H>
__global__ __launch_bounds__(COOP_NT) void poseidon_leaves_coop_kernel(const uint64_t *__restrict__ values,
                                                                       uint64_t *__restrict__ results,
                                                                       uint32_t log_rows, uint32_t cols, uint32_t count,
                                                                       bool load_intermediate,
                                                                       bool store_intermediate, uint32_t layers) {
  __shared__ CoopLds lds;
  __shared__ uint64_t digest[COOP_GROUPS][CAP];
  coop_stage_table<H>(lds);
  const uint32_t group = threadIdx.x / COOP_LANES, j = threadIdx.x % COOP_LANES;
  const uint64_t g = (uint64_t)blockIdx.x * COOP_GROUPS + group;
  const uint64_t rows = 1ull << log_rows;
  const uint64_t col_stride = rows * count;
  const uint64_t *base = values + g * rows;
  const uint64_t total = rows * cols;
  const bool on = g < count;
  auto chunk = [&](uint64_t off) -> uint64_t {
    const uint64_t k = off + j;
    return on && j < RATE && k < total ? base[(k & (rows - 1)) + (k >> log_rows) * col_stride] : 0ull;
  };
  uint64_t x = 0, next = chunk(0);
  if (on && load_intermediate && j >= RATE && j < PT) x = results[g + (uint64_t)(j - RATE) * count];
  __syncthreads();
  const Coop c(lds, j, group);
  if (on) {  // whole rows together
    for (uint64_t off = 0; off < total; off += RATE) {
      if (j < RATE) x = next;
      next = chunk(off + RATE);
      c.permute_h<H>(x);
    }
    // the digest is state[0..4], the stored capacity state[8..12]
    x = gl::canon(x);
    if (store_intermediate) {
      if (j >= RATE && j < PT) results[g + (uint64_t)(j - RATE) * count] = x;
    } else if (j < CAP) {
      results[g + (uint64_t)j * count] = x;
      digest[group][j] = x;
    }
  }
  coop_climb<H>(c, digest, results + (uint64_t)CAP * count, count / 2, layers, group, j);
}

// ---- Merkle openings: row and path gathers (native/poseidon_common.cu:9-37) --

// result[col][i rpi + r] = values[col][indexes[i] rpi + r] for r < rpi =
// 2^log_rpi; rows past the source (an index out of range) are skipped, the
// destination left as it was.  x: destination rows, y: columns.
__global__ __launch_bounds__(256) void gather_rows_kernel(const uint32_t *__restrict__ indexes, uint64_t dst_rows,
                                                          uint32_t log_rpi, const uint64_t *__restrict__ values,
                                                          uint64_t values_stride, uint64_t values_rows,
                                                          uint64_t *__restrict__ results, uint64_t results_stride,
                                                          uint32_t cols) {
  const uint64_t dst = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (dst >= dst_rows) return;
  const uint64_t src = ((uint64_t)indexes[dst >> log_rpi] << log_rpi) + (dst & ((1ull << log_rpi) - 1));
  if (src >= values_rows) return;
  for (uint32_t c = blockIdx.y; c < cols; c += gridDim.y) results[c * results_stride + dst] = values[c * values_stride + src];
}

// Siblings along each index's path: for layer l < layers, column c (of 4) and
// index i, results[l count 4 + c count + i] = the layer-l digest element c of
// node (indexes[i] >> l) ^ 1.  Layer l of the tree buffer starts at
// 4 (2^(L+1) - 2^(L+1-l)) and holds 4 columns of 2^(L-l) (L = log2 leaves).
__global__ __launch_bounds__(256) void gather_merkle_paths_kernel(const uint32_t *__restrict__ indexes,
                                                                  uint32_t count, const uint64_t *__restrict__ values,
                                                                  uint32_t log_leaves, uint64_t *__restrict__ results) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const uint32_t c = blockIdx.y, l = blockIdx.z;
  const uint64_t leaf = indexes[i];
  if (leaf >> log_leaves) return;  // index out of range: nothing to gather
  const uint64_t layer_off = ((uint64_t)CAP << (log_leaves + 1)) - ((uint64_t)CAP << (log_leaves + 1 - l));
  const uint64_t src = layer_off + ((uint64_t)c << (log_leaves - l)) + ((leaf >> l) ^ 1ull);
  results[(uint64_t)l * count * CAP + (uint64_t)count * c + i] = values[src];
}

// ---- host: the fused form ---------------------------------------------------

using Mat = std::vector<uint64_t>;  // row-major n x n

uint64_t mds_entry(int r, int c) { return 1ull << MDS_EXPS[((c - r) % PT + PT) % PT]; }

bool invert(Mat a, int n, Mat &out) {
  out.assign((size_t)n * n, 0);
  for (int i = 0; i < n; ++i) out[(size_t)i * n + i] = 1;
  for (int col = 0; col < n; ++col) {
    int piv = -1;
    for (int r = col; r < n && piv < 0; ++r)
      if (a[(size_t)r * n + col]) piv = r;
    if (piv < 0) return false;
    for (int j = 0; j < n; ++j) {
      std::swap(a[(size_t)col * n + j], a[(size_t)piv * n + j]);
      std::swap(out[(size_t)col * n + j], out[(size_t)piv * n + j]);
    }
    const uint64_t iv = gl::inv(a[(size_t)col * n + col]);
    for (int j = 0; j < n; ++j) {
      a[(size_t)col * n + j] = gl::mul(a[(size_t)col * n + j], iv);
      out[(size_t)col * n + j] = gl::mul(out[(size_t)col * n + j], iv);
    }
    for (int r = 0; r < n; ++r) {
      const uint64_t f = a[(size_t)r * n + col];
      if (r == col || !f) continue;
      for (int j = 0; j < n; ++j) {
        a[(size_t)r * n + j] = gl::sub(a[(size_t)r * n + j], gl::mul(f, a[(size_t)col * n + j]));
        out[(size_t)r * n + j] = gl::sub(out[(size_t)r * n + j], gl::mul(f, out[(size_t)col * n + j]));
      }
    }
  }
  return true;
}

void mat_vec(const Mat &m, const uint64_t *v, uint64_t *out) {
  for (int r = 0; r < PT; ++r) {
    uint64_t acc = 0;
    for (int c = 0; c < PT; ++c) acc = gl::add(acc, gl::mul(m[(size_t)r * PT + c], v[c]));
    out[r] = acc;
  }
}

bool derive(const uint64_t *rc_in, PosTable &t) {
  uint64_t rc[ROUNDS * PT];
  for (int i = 0; i < ROUNDS * PT; ++i) rc[i] = gl::canon(rc_in[i]);
  Mat m((size_t)PT * PT), minv;
  for (int r = 0; r < PT; ++r)
    for (int c = 0; c < PT; ++c) m[(size_t)r * PT + c] = mds_entry(r, c);
  if (!invert(m, PT, minv)) return false;
  for (int r = 0; r < HALF_FULL; ++r)
    for (int i = 0; i < PT; ++i) t.rc_full[r][i] = rc[r * PT + i];
  for (int r = 0; r < 3; ++r)
    for (int i = 0; i < PT; ++i) t.rc_full[HALF_FULL + r][i] = rc[(HALF_FULL + PARTIAL + 1 + r) * PT + i];
  for (int r = 0; r < HALF_FULL; ++r)
    for (int i = 0; i < PT; ++i) {
      t.p2_full[r][i] = rc[r * PT + i];
      t.p2_full[HALF_FULL + r][i] = rc[(HALF_FULL + PARTIAL + r) * PT + i];
    }
  for (int k = 0; k < PARTIAL; ++k) t.p2_partial[k] = rc[(HALF_FULL + k) * PT];
  // constants of round 26, then of each partial round, moved backwards
  uint64_t cur[PT], e[PT];
  for (int i = 0; i < PT; ++i) cur[i] = rc[(HALF_FULL + PARTIAL) * PT + i];
  for (int k = HALF_FULL + PARTIAL - 1; k >= HALF_FULL; --k) {
    mat_vec(minv, cur, e);
    t.sbox_c[k - HALF_FULL] = e[0];
    for (int i = 0; i < PT; ++i) cur[i] = i ? gl::add(rc[k * PT + i], e[i]) : rc[k * PT + i];
  }
  mat_vec(minv, cur, t.rcf);
  // matrices
  Mat n = m;
  for (int k = HALF_FULL + PARTIAL - 1; k >= HALF_FULL; --k) {
    const int pr = k - HALF_FULL;
    Mat nh((size_t)(PT - 1) * (PT - 1)), nhinv;
    for (int i = 0; i < PT - 1; ++i)
      for (int j = 0; j < PT - 1; ++j) nh[(size_t)i * (PT - 1) + j] = n[(size_t)(i + 1) * PT + j + 1];
    if (!invert(nh, PT - 1, nhinv)) return false;
    for (int j = 0; j < PT - 1; ++j) {
      uint64_t acc = 0;
      for (int i = 0; i < PT - 1; ++i) acc = gl::add(acc, gl::mul(n[i + 1], nhinv[(size_t)i * (PT - 1) + j]));
      t.vs[pr][j] = acc;
      t.w_hats[pr][j] = n[(size_t)(j + 1) * PT];
    }
    Mat next((size_t)PT * PT);
    for (int c = 0; c < PT; ++c) next[c] = m[c];
    for (int r = 1; r < PT; ++r)
      for (int c = 0; c < PT; ++c) {
        uint64_t acc = 0;
        for (int i = 1; i < PT; ++i)
          acc = gl::add(acc, gl::mul(nh[(size_t)(r - 1) * (PT - 1) + i - 1], m[(size_t)i * PT + c]));
        next[(size_t)r * PT + c] = acc;
      }
    n.swap(next);
  }
  for (int r = 0; r < PT; ++r)
    for (int c = 0; c < PT; ++c) t.dense[r][c] = n[(size_t)r * PT + c];
  return true;
}

// c in limbs of 24, 24 and 16 bits.
void set_limbs(uint32_t *out, uint64_t c) {
  out[0] = (uint32_t)(c & 0xFFFFFF);
  out[1] = (uint32_t)((c >> 24) & 0xFFFFFF);
  out[2] = (uint32_t)(c >> 48);
}
void set_halves(uint64_t (*out)[2], const uint64_t *c, int n = PT) {
  for (int i = 0; i < n; ++i) {
    out[i][0] = (uint32_t)c[i];
    out[i][1] = c[i] >> 32;
  }
}

// Eight signed bytes d_l with sum d_l 2^8l = c mod p.  The balanced digits of
// a residue up to 0x7F7F...7F end without a carry; of a larger one they carry
// out 2^64, and the residue less p (whose digits those of c + 2^64 - p are)
// takes its place.
void signed_bytes(int8_t *d, uint64_t c) {
  uint64_t v = c > 0x7F7F7F7F7F7F7F7Full ? c + gl::EPS : c;  // c - p mod 2^64
  for (int l = 0; l < 8; ++l) {
    d[l] = (int8_t)(uint8_t)v;
    v = (v >> 8) + (d[l] < 0 ? 1 : 0);
  }
}

// Operand bytes and row constants of the matrix rows[o][w] (o < 12, w < 12)
// plus constants k[o] (see PosMat).
void set_mat(PosMat &m, int mat, uint64_t (*kout)[2], int outputs, const uint64_t (*rows)[PT], const uint64_t *k) {
  for (int o = 0; o < outputs; ++o) {
    uint64_t kv = k[o];
    for (int w = 0; w < PT; ++w) {
      uint64_t c = rows[o][w];
      kv = gl::add(kv, gl::mul(c, 0x8080808080808080ull));
      for (int b = 0; b < 8; ++b) {
        int8_t d[8];
        signed_bytes(d, c);
        // the word's byte is byte `at` of lanes 32 half + row in its step
        const int st = w / 4, half = (w % 4) / 2, at = 8 * (w % 2) + b;
        for (int l = 0; l < 8; ++l) m.a[mat][o / 4][st][32 * half + 8 * (o % 4) + l][at] = d[l];
        c = gl::mul(c, 256);
      }
    }
    const uint64_t bias = 1ull << MAT_BIAS_LOG;
    kv = gl::sub(kv, gl::mul(bias, 1 + (1ull << 32)));
    kout[o][0] = bias + (uint32_t)kv;
    kout[o][1] = bias + (kv >> 32);
  }
}

// False if a column entry does not suit coop_mul_add (the MDS matrix alone
// decides that, not the round constants).
bool derive_lanes(const PosTable &t, PartialLane (*lanes)[PT]) {
  for (int k = 0; k < PARTIAL; ++k)
    for (int j = 0; j < PT; ++j) {
      PartialLane &l = lanes[k][j];
      l.v = j ? t.vs[k][j - 1] : 0;
      l.w = j ? t.w_hats[k][j - 1] : 1;
      if ((uint32_t)l.w == 0xFFFFFFFFu) return false;
      const uint64_t c = gl::mul(l.w, t.sbox_c[k]);
      l.k[0] = (uint32_t)c;
      l.k[1] = c >> 32;
    }
  return true;
}

// The one-lane forms' tables from the fused one.
void derive_fast(const PosTable &t, PosFast &f, PosMat &m) {
  uint64_t rows[PT][PT], k[PT];
  for (int i = 0; i < PT; ++i) f.first[i] = t.rc_full[0][i];
  for (int r = 0; r < PT; ++r)
    for (int c = 0; c < PT; ++c) rows[r][c] = mds_entry(r, c);
  for (int i = 0; i < 7; ++i) {
    for (int r = 0; r < PT; ++r) k[r] = i < 3 ? t.rc_full[1 + i][r] : (i < 6 ? t.rc_full[HALF_FULL + i - 3][r] : 0);
    set_mat(m, MAT_MDS, f.mds[i], PT, rows, k);
  }
  // dense (v + rcf): the fused constant layer becomes each row's constant
  for (int r = 0; r < PT; ++r) {
    k[r] = 0;
    for (int c = 0; c < PT; ++c) k[r] = gl::add(k[r], gl::mul(t.dense[r][c], t.rcf[c]));
  }
  set_mat(m, MAT_DENSE, f.dense, PT, t.dense, k);
  // z_j below is the S-box output without its constant sbox_c
  for (int b = 0; b < BLOCKS; ++b) {
    PosBlock &blk = f.block[b];
    const int k0 = b * BLOCK;
    memset(rows, 0, sizeof rows);
    for (int r = 0; r < BLOCK; ++r) {
      // the bias of the round's sum over z comes out of its first term
      k[r] = gl::sub(t.sbox_c[k0 + r], 1ull << DOT_BIAS_LOG);
      for (int i = 0; i < PT - 1; ++i) rows[r][i] = t.vs[k0 + r][i];
      for (int j = 0; j < r; ++j) {
        uint64_t c = 0;
        for (int i = 0; i < PT - 1; ++i) c = gl::add(c, gl::mul(t.vs[k0 + r][i], t.w_hats[k0 + j][i]));
        set_limbs(blk.z[r][j], c);
        k[r] = gl::add(k[r], gl::mul(c, t.sbox_c[k0 + j]));
      }
    }
    set_mat(m, MAT_BLOCK + 2 * b, blk.start, BLOCK, rows, k);
    memset(rows, 0, sizeof rows);
    for (int i = 0; i < PT - 1; ++i) {
      k[i] = 0;
      for (int j = 0; j < BLOCK; ++j) {
        rows[i][j] = t.w_hats[k0 + j][i];
        k[i] = gl::add(k[i], gl::mul(t.w_hats[k0 + j][i], t.sbox_c[k0 + j]));
      }
    }
    set_mat(m, MAT_BLOCK + 2 * b + 1, blk.end, PT - 1, rows, k);
  }
  for (int r = 0; r < HALF_FULL; ++r) set_halves(f.p2_ext[r], t.p2_full[r]);
  set_halves(f.p2_ext[HALF_FULL], t.p2_partial, 1);
  for (int k = 0; k + 1 < PARTIAL; ++k) set_halves(&f.p2_int[k], t.p2_partial + k + 1, 1);
  set_halves(f.p2_last, t.p2_full[HALF_FULL]);
  for (int r = 1; r < HALF_FULL; ++r) set_halves(f.p2_ext[HALF_FULL + r], t.p2_full[HALF_FULL + r]);
}

constexpr int MAX_DEVICES = 64;
// Every hashing entry point holds this lock shared from its readiness check
// through its launches; replacing the table holds it exclusively.  So no
// hashing kernel is queued between the wait for queued work and the copy of
// the new table, on any stream or thread.
std::shared_mutex pos_mu;
bool pos_ready[MAX_DEVICES];

// Caller holds pos_mu (shared or exclusive).
int require_table() {
  int dev = 0;
  const hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) return err;
  if (dev < 0 || dev >= MAX_DEVICES) return BC_ERROR_INVALID_VALUE;
  return pos_ready[dev] ? BC_SUCCESS : BC_ERROR_NOT_INITIALIZED;
}

using TableUse = std::shared_lock<std::shared_mutex>;

// Whether a layer's inputs share memory with what the layers above it write.
// They then have to be read before those layers start, in a launch of their own.
bool overlap(const uint64_t *a, uint64_t a_len, const uint64_t *b, uint64_t b_len) {
  return (uintptr_t)a < (uintptr_t)(b + b_len) && (uintptr_t)b < (uintptr_t)(a + a_len);
}

// COOP: always the cooperative kernel; otherwise the cooperative kernel for
// at most COOP_MAX leaves and one thread per leaf above.
template <int H, bool COOP>
int launch_leaves(const uint64_t *values, uint64_t *results, uint32_t log_rows, uint32_t cols, uint32_t count,
                  bool load, bool store, hipStream_t s) {
  if (count == 0) return BC_SUCCESS;
  if (COOP || count <= COOP_MAX) {
    poseidon_leaves_coop_kernel<H><<<dim3((count + COOP_GROUPS - 1) / COOP_GROUPS), dim3(COOP_NT), 0, s>>>(
        values, results, log_rows, cols, count, load, store, 0);
  } else {
    poseidon_leaves_kernel<H><<<dim3((count + 255) / 256), dim3(256), 0, s>>>(values, results, 1u << log_rows, cols,
                                                                             count, load, store);
  }
  return hipGetLastError();
}

// Node layers [values -> results], the first of `count` nodes (layers > 1: a
// power of two).  COOP: always the cooperative kernel (the reference's
// launch_cooperative_nodes_kernel); otherwise the cooperative kernel, several
// layers to a launch, for layers of at most COOP_MAX nodes, and one
// thread per node above.
template <int H, bool COOP = false>
int launch_nodes(const uint64_t *values, uint64_t *results, uint32_t count, uint32_t layers, hipStream_t s) {
  while (layers && count) {
    uint32_t n = 1;
    if (COOP || count <= COOP_MAX) {
      n = layers < COOP_MAX_LAYERS ? layers : COOP_MAX_LAYERS;
      if (overlap(values, 2ull * CAP * count, results + (uint64_t)CAP * count, (uint64_t)CAP * count)) n = 1;
      poseidon_nodes_coop_kernel<H>
          <<<dim3((count + COOP_GROUPS - 1) / COOP_GROUPS), dim3(COOP_NT), 0, s>>>(values, results, count, n);
    } else {
      poseidon_nodes_kernel<H><<<dim3((count + 255) / 256), dim3(256), 0, s>>>(values, results, count);
    }
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
    for (layers -= n; n; --n) {
      values = results;
      results += (uint64_t)CAP * count;
      count /= 2;
    }
  }
  return BC_SUCCESS;
}

// The entry points of both hashes share these (src/poseidon.rs is generic
// over the hash in the same way).

template <int H, bool COOP = false>
int leaves_impl(const uint64_t *values, uint64_t values_len, uint64_t *results, uint64_t results_len,
                uint32_t log_rows_per_hash, bool load_intermediate, bool store_intermediate, void *stream) {
  // src/poseidon.rs:139-155
  if (log_rows_per_hash >= 32 || results_len % CAP != 0) return BC_ERROR_INVALID_VALUE;
  const uint64_t count = results_len / CAP;
  if (count == 0) return values_len == 0 ? BC_SUCCESS : BC_ERROR_INVALID_VALUE;
  if (!values || !results || count > 0xFFFFFFFFull) return BC_ERROR_INVALID_VALUE;
  const uint64_t rows = 1ull << log_rows_per_hash;
  if (values_len % (count * rows) != 0) return BC_ERROR_INVALID_VALUE;
  const uint64_t cols = values_len / (count * rows);
  if (cols > 0xFFFFFFFFull || rows * cols > 0xFFFFFFFFull) return BC_ERROR_INVALID_VALUE;
  if (store_intermediate && (rows * cols) % RATE != 0) return BC_ERROR_INVALID_VALUE;
  const int rc = require_table();
  if (rc != BC_SUCCESS) return rc;
  return launch_leaves<H, COOP>(values, results, log_rows_per_hash, (uint32_t)cols, (uint32_t)count,
                                load_intermediate, store_intermediate, (hipStream_t)stream);
}

template <int H, bool COOP = false>
int nodes_impl(const uint64_t *values, uint64_t values_len, uint64_t *results, uint64_t results_len, void *stream) {
  // src/poseidon.rs:224-232
  if (values_len % RATE != 0 || results_len % CAP != 0 || values_len != 2 * results_len)
    return BC_ERROR_INVALID_VALUE;
  const uint64_t count = results_len / CAP;
  if (count == 0) return BC_SUCCESS;
  if (!values || !results || count > 0xFFFFFFFFull) return BC_ERROR_INVALID_VALUE;
  const int rc = require_table();
  if (rc != BC_SUCCESS) return rc;
  return launch_nodes<H, COOP>(values, results, (uint32_t)count, 1, (hipStream_t)stream);
}

template <int H>
int tree_nodes_impl(const uint64_t *values, uint64_t values_len, uint64_t *results, uint64_t results_len,
                    uint32_t layers_count, void *stream) {
  // src/poseidon.rs:262-286: each layer halves; its nodes fill the first half
  // of what remains of `results`
  if (layers_count == 0) return BC_SUCCESS;
  if (values_len % RATE != 0 || values_len != results_len) return BC_ERROR_INVALID_VALUE;
  const uint64_t nodes = values_len / RATE;  // of the first layer
  if (nodes == 0 || (nodes & (nodes - 1)) != 0) return BC_ERROR_INVALID_VALUE;
  if (layers_count > 64 || (layers_count > 1 && (values_len >> (layers_count - 1)) < RATE))
    return BC_ERROR_INVALID_VALUE;
  const int rc = require_table();
  if (rc != BC_SUCCESS) return rc;
  if (!values || !results || nodes > 0xFFFFFFFFull) return BC_ERROR_INVALID_VALUE;
  return launch_nodes<H>(values, results, (uint32_t)nodes, layers_count, (hipStream_t)stream);
}

template <int H>
int tree_impl(const uint64_t *values, uint64_t values_len, uint64_t *results, uint64_t results_len,
              uint32_t log_rows_per_hash, uint32_t layers_count, void *stream) {
  // src/poseidon.rs:311-328: the leaf digests fill the first half of
  // `results`, the node layers the rest
  if (layers_count == 0 || results_len % (2 * CAP) != 0) return BC_ERROR_INVALID_VALUE;
  const uint64_t leaves = results_len / (2 * CAP);
  if (leaves == 0 || layers_count - 1 >= 64 || (1ull << (layers_count - 1)) > leaves ||
      values_len % leaves != 0)
    return BC_ERROR_INVALID_VALUE;
  const uint64_t half = results_len / 2;
  // few leaves: their launch also takes the first node layers, one launch and
  // one staging of the tables less.  Trees of one permutation a leaf, Poseidon /
  // Poseidon2, with and without: 2^9 leaves 116 / 85 and 121 / 90 us, 2^11 141 /
  // 103 and 143 / 106, 2^13 167 / 123 and 170 / 126; at 2^14 the workgroups of
  // the leaves no longer start at once and hold the climb up: 196 / 150 and 191 /
  // 144 (five permutations 298 / 228 and 283 / 215).
  const uint64_t rows = 1ull << (log_rows_per_hash & 31u), total = values_len / leaves;
  if (layers_count > 1 && leaves >= 2 && leaves <= COOP_MAX / 2 && (leaves & (leaves - 1)) == 0 && values && results &&
      log_rows_per_hash < 32 && total % rows == 0 && total <= 0xFFFFFFFFull &&
      !overlap(values, values_len, results + half, half)) {
    const int rc = require_table();
    if (rc != BC_SUCCESS) return rc;
    constexpr uint32_t MAX_CLIMB = COOP_MAX_LAYERS - 1;
    const uint32_t climb = layers_count - 1 < MAX_CLIMB ? layers_count - 1 : MAX_CLIMB;
    const uint32_t count = (uint32_t)leaves;
    poseidon_leaves_coop_kernel<H>
        <<<dim3((count + COOP_GROUPS - 1) / COOP_GROUPS), dim3(COOP_NT), 0, (hipStream_t)stream>>>(
            values, results, log_rows_per_hash, (uint32_t)(total >> log_rows_per_hash), count, false, false, climb);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
    // layer l (l = 0: the leaves) has count >> l digests behind the layers before it
    for (uint32_t l = 0; l < climb; ++l) results += (uint64_t)CAP * (count >> l);
    return launch_nodes<H>(results, results + (uint64_t)CAP * (count >> climb), count >> (climb + 1),
                           layers_count - 1 - climb, (hipStream_t)stream);
  }
  const int e = leaves_impl<H>(values, values_len, results, half, log_rows_per_hash, false, false, stream);
  if (e != BC_SUCCESS) return e;
  return tree_nodes_impl<H>(results, half, results + half, half, layers_count - 1, stream);
}

}  // namespace

size_t poseidon_table_words() { return sizeof(PosTable) / sizeof(uint64_t); }

}  // namespace bc

extern "C" int bc_poseidon_set_round_constants(const uint64_t *round_constants) {
  using namespace bc;
  if (!round_constants) return BC_ERROR_INVALID_VALUE;
  int dev = 0;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) return err;
  if (dev < 0 || dev >= MAX_DEVICES) return BC_ERROR_INVALID_VALUE;
  PosTable t{};
  if (!derive(round_constants, t)) return BC_ERROR_INVALID_VALUE;
  PosFast f{};
  std::vector<PosMat> m(1);
  derive_fast(t, f, m[0]);
  PartialLane lanes[PARTIAL][PT];
  if (!derive_lanes(t, lanes)) return BC_ERROR_INVALID_VALUE;
  std::unique_lock<std::shared_mutex> lk(pos_mu);
  // hashing kernels already queued on any stream of this device read the
  // table: let them finish before it changes (no new ones can be queued
  // while the lock is held)
  err = hipDeviceSynchronize();
  if (err != hipSuccess) return err;
  pos_ready[dev] = false;  // until all tables are new
  err = hipMemcpyToSymbol(HIP_SYMBOL(pos_table), &t, sizeof t, 0, hipMemcpyHostToDevice);
  if (err != hipSuccess) return err;
  err = hipMemcpyToSymbol(HIP_SYMBOL(pos_fast), &f, sizeof f, 0, hipMemcpyHostToDevice);
  if (err != hipSuccess) return err;
  err = hipMemcpyToSymbol(HIP_SYMBOL(pos_partial_lanes), lanes, sizeof lanes, 0, hipMemcpyHostToDevice);
  if (err != hipSuccess) return err;
  err = hipMemcpyToSymbol(HIP_SYMBOL(pos_mat), &m[0], sizeof m[0], 0, hipMemcpyHostToDevice);
  if (err != hipSuccess) return err;
  err = hipDeviceSynchronize();
  if (err != hipSuccess) return err;
  pos_ready[dev] = true;
  return BC_SUCCESS;
}

extern "C" int bc_poseidon_fused_table(const uint64_t *round_constants, uint64_t *out, uint64_t out_words) {
  using namespace bc;
  if (!round_constants || !out || out_words < poseidon_table_words()) return BC_ERROR_INVALID_VALUE;
  PosTable t{};
  if (!derive(round_constants, t)) return BC_ERROR_INVALID_VALUE;
  memcpy(out, &t, sizeof t);
  return BC_SUCCESS;
}

extern "C" int bc_poseidon_leaves(const uint64_t *values, uint64_t values_len, uint64_t *results,
                                  uint64_t results_len, uint32_t log_rows_per_hash, bool load_intermediate,
                                  bool store_intermediate, void *stream) {
  const bc::TableUse use(bc::pos_mu);
  return bc::leaves_impl<0>(values, values_len, results, results_len, log_rows_per_hash, load_intermediate,
                            store_intermediate, stream);
}

extern "C" int bc_poseidon_nodes(const uint64_t *values, uint64_t values_len, uint64_t *results,
                                 uint64_t results_len, void *stream) {
  const bc::TableUse use(bc::pos_mu);
  return bc::nodes_impl<0>(values, values_len, results, results_len, stream);
}

extern "C" int bc_poseidon_build_merkle_tree_nodes(const uint64_t *values, uint64_t values_len, uint64_t *results,
                                                   uint64_t results_len, uint32_t layers_count, void *stream) {
  const bc::TableUse use(bc::pos_mu);
  return bc::tree_nodes_impl<0>(values, values_len, results, results_len, layers_count, stream);
}

extern "C" int bc_poseidon_build_merkle_tree(const uint64_t *values, uint64_t values_len, uint64_t *results,
                                             uint64_t results_len, uint32_t log_rows_per_hash,
                                             uint32_t layers_count, void *stream) {
  const bc::TableUse use(bc::pos_mu);
  return bc::tree_impl<0>(values, values_len, results, results_len, log_rows_per_hash, layers_count, stream);
}

extern "C" int bc_poseidon2_leaves(const uint64_t *values, uint64_t values_len, uint64_t *results,
                                   uint64_t results_len, uint32_t log_rows_per_hash, bool load_intermediate,
                                   bool store_intermediate, void *stream) {
  const bc::TableUse use(bc::pos_mu);
  return bc::leaves_impl<1>(values, values_len, results, results_len, log_rows_per_hash, load_intermediate,
                            store_intermediate, stream);
}

extern "C" int bc_poseidon2_nodes(const uint64_t *values, uint64_t values_len, uint64_t *results,
                                  uint64_t results_len, void *stream) {
  const bc::TableUse use(bc::pos_mu);
  return bc::nodes_impl<1>(values, values_len, results, results_len, stream);
}

extern "C" int bc_poseidon2_build_merkle_tree_nodes(const uint64_t *values, uint64_t values_len, uint64_t *results,
                                                    uint64_t results_len, uint32_t layers_count, void *stream) {
  const bc::TableUse use(bc::pos_mu);
  return bc::tree_nodes_impl<1>(values, values_len, results, results_len, layers_count, stream);
}

extern "C" int bc_poseidon2_build_merkle_tree(const uint64_t *values, uint64_t values_len, uint64_t *results,
                                              uint64_t results_len, uint32_t log_rows_per_hash,
                                              uint32_t layers_count, void *stream) {
  const bc::TableUse use(bc::pos_mu);
  return bc::tree_impl<1>(values, values_len, results, results_len, log_rows_per_hash, layers_count, stream);
}

extern "C" int bc_poseidon_leaves_cooperative(const uint64_t *values, uint64_t values_len, uint64_t *results,
                                              uint64_t results_len, uint32_t log_rows_per_hash,
                                              bool load_intermediate, bool store_intermediate, void *stream) {
  const bc::TableUse use(bc::pos_mu);
  return bc::leaves_impl<0, true>(values, values_len, results, results_len, log_rows_per_hash, load_intermediate,
                                  store_intermediate, stream);
}

extern "C" int bc_poseidon2_leaves_cooperative(const uint64_t *values, uint64_t values_len, uint64_t *results,
                                               uint64_t results_len, uint32_t log_rows_per_hash,
                                               bool load_intermediate, bool store_intermediate, void *stream) {
  const bc::TableUse use(bc::pos_mu);
  return bc::leaves_impl<1, true>(values, values_len, results, results_len, log_rows_per_hash, load_intermediate,
                                  store_intermediate, stream);
}

extern "C" int bc_poseidon_nodes_cooperative(const uint64_t *values, uint64_t values_len, uint64_t *results,
                                             uint64_t results_len, void *stream) {
  const bc::TableUse use(bc::pos_mu);
  return bc::nodes_impl<0, true>(values, values_len, results, results_len, stream);
}

extern "C" int bc_poseidon2_nodes_cooperative(const uint64_t *values, uint64_t values_len, uint64_t *results,
                                              uint64_t results_len, void *stream) {
  const bc::TableUse use(bc::pos_mu);
  return bc::nodes_impl<1, true>(values, values_len, results, results_len, stream);
}

extern "C" int bc_gather_rows(const uint32_t *indexes, uint32_t indexes_count, uint32_t log_rows_per_index,
                              const uint64_t *values, uint64_t values_stride, uint64_t values_rows, uint64_t *results,
                              uint64_t results_stride, uint64_t results_rows, uint32_t cols, void *stream) {
  using namespace bc;
  // src/poseidon.rs:337-346
  if (log_rows_per_index >= 32) return BC_ERROR_INVALID_VALUE;
  if (results_rows != ((uint64_t)indexes_count << log_rows_per_index)) return BC_ERROR_INVALID_VALUE;
  if (results_rows == 0 || cols == 0) return BC_SUCCESS;
  if (!indexes || !values || !results || values_stride < values_rows || results_stride < results_rows)
    return BC_ERROR_INVALID_VALUE;
  const uint64_t blocks = (results_rows + 255) / 256;
  if (blocks > 0x7FFFFFFFull) return BC_ERROR_INVALID_VALUE;
  gather_rows_kernel<<<dim3((uint32_t)blocks, cols < 65535 ? cols : 65535), dim3(256), 0, (hipStream_t)stream>>>(
      indexes, results_rows, log_rows_per_index, values, values_stride, values_rows, results, results_stride, cols);
  return hipGetLastError();
}

extern "C" int bc_gather_merkle_paths(const uint32_t *indexes, uint32_t indexes_count, const uint64_t *values,
                                      uint64_t values_len, uint64_t *results, uint64_t results_len,
                                      uint32_t layers_count, void *stream) {
  using namespace bc;
  // src/poseidon.rs:367-382
  if (values_len % CAP != 0) return BC_ERROR_INVALID_VALUE;
  const uint64_t values_count = values_len / CAP;
  if (values_count == 0 || (values_count & (values_count - 1)) != 0) return BC_ERROR_INVALID_VALUE;
  const uint32_t log_values = (uint32_t)__builtin_ctzll(values_count);
  if (log_values == 0) return BC_ERROR_INVALID_VALUE;
  const uint32_t log_leaves = log_values - 1;
  if (layers_count >= log_leaves) return BC_ERROR_INVALID_VALUE;
  if ((uint64_t)indexes_count * layers_count * CAP != results_len) return BC_ERROR_INVALID_VALUE;
  if (indexes_count == 0 || layers_count == 0) return BC_SUCCESS;
  if (!indexes || !values || !results) return BC_ERROR_INVALID_VALUE;
  gather_merkle_paths_kernel<<<dim3((indexes_count + 255) / 256, CAP, layers_count), dim3(256), 0,
                               (hipStream_t)stream>>>(indexes, indexes_count, values, log_leaves, results);
  return hipGetLastError();
}
