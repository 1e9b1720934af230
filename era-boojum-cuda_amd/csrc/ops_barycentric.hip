// Barycentric evaluation of polynomials given on the coset domain
// {coset * omega_N^i}: Lagrange coefficients at a point x, then many columns
// evaluated against them.  Reference: src/barycentric.rs:83-280 (host) and
// native/barycentric.cu:10-156 (kernels).
//
//   common = coset (x^N - coset^N) / (N coset^N)          (barycentric.cu:12-21)
//   L_i    = common / (x omega_N^-i - coset)               (barycentric.cu:44-86)
//   eval_p = sum_i L_i y_{i,p}                             (barycentric.cu:104-156
//                                                           + the reference's
//                                                           final column sums)
// x and the coefficients are base-field or extension (F_p[u]/(u^2 - 7))
// values; the columns y are base or extension.  Layouts are the reference's:
// extension vectors and matrix columns are "double vectors" (the c0 plane,
// then the c1 plane, each N long); extension evaluations are (c0, c1) pairs.
//
// The evaluation is one pass over the columns, so it is bound by HBM reads
// (8 or 16 bytes per element) and by the VALU cost of one field product per
// base element.  Products are accumulated unreduced (gl::mac: 4 multiply-adds
// and a carry chain) and reduced once per lane and column.  A wave reads a
// column tile with 16-byte loads (a whole wave per column for long columns:
// 1 KiB contiguous per load instruction), and every lane keeps its rows'
// coefficients in registers for all the columns it visits; per-tile partial
// sums are then added per column by a second small kernel (the sum is exact
// in the field, so the order does not change the result).
#include "../../include/boojum_ntt.h"
#include "gl_ext.hpp"
#include "gl_lazy.hpp"
#include "ntt_device.hpp"

#include <mutex>

namespace bc {

Tables current_tables(bool &ok);  // ntt_api.hip

namespace {

// ---- Lagrange coefficients ---------------------------------------------------

constexpr uint32_t LC_NT = 256;  // threads per workgroup
constexpr uint32_t LC_B = 4;     // coefficients per thread

// N products side by side, in the base field (c1 unused) or in the extension:
// any u64 components in and out.  The extension's four component products of
// a pair are one row; a0 b0 + 7 a1 b1 and a0 b1 + a1 b0 are summed by 32-bit
// halves and reduced once.
template <bool EXT, int N>
__device__ __forceinline__ void pmul(gl::E2 *r, const gl::E2 *a, const gl::E2 *b) {
  if constexpr (!EXT) {
    uint64_t x[N], y[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      x[i] = a[i].c0;
      y[i] = b[i].c0;
    }
    gl::mul_row<N, gl::ANY>(x, x, y);
#pragma unroll
    for (int i = 0; i < N; ++i) r[i] = {x[i], 0};
  } else {
    gl::unroll<N>([&](auto k) {
      constexpr int i = decltype(k)::value;
      uint64_t x[4] = {a[i].c0, a[i].c1, a[i].c0, a[i].c1}, y[4] = {b[i].c0, b[i].c1, b[i].c1, b[i].c0};
      gl::mul_row<4, gl::ANY>(x, x, y);
      uint64_t lo[2], hi[2], o[2];
      lo[0] = (uint64_t)gl::lo32(x[1]) * gl::E2_NON_RESIDUE + gl::lo32(x[0]);
      hi[0] = (uint64_t)gl::hi32(x[1]) * gl::E2_NON_RESIDUE + gl::hi32(x[0]);
      lo[1] = (uint64_t)gl::lo32(x[2]) + gl::lo32(x[3]);
      hi[1] = (uint64_t)gl::hi32(x[2]) + gl::hi32(x[3]);
      gl::join_halves<2>(o, lo, hi);
      r[i] = {o[0], o[1]};
    });
  }
}
template <bool EXT> __device__ __forceinline__ gl::E2 pmul1(gl::E2 a, gl::E2 b) {
  gl::E2 r;
  pmul<EXT, 1>(&r, &a, &b);
  return r;
}

// Thread t of workgroup b owns outputs i = 1024 b + 256 j + t (j < 4; stores
// coalesced for each j) with denominators d = x omega_N^-idx - coset (idx = i,
// or brev(i) when the output is bit-reversed); padding outputs (i >= N) use
// d = 1.  All 1024 denominators of the workgroup share ONE field inversion
// through a product tree: each thread multiplies its four (keeping prefix
// products); wave 0 takes the 256 thread products, four to a lane, and
// multiplies them up a binary tree of 63 nodes kept in LDS, inverts the root,
// multiplies in the common factor and goes back down: a child's inverse is
// its parent's times its sibling's product.  Each thread ends with common /
// (its own product) and peels off its four coefficients with its prefix
// products.  The common factor is
//   coset (x^N - coset^N) / (N coset^N) = (x^N - coset^N) f,
// with coset^N and f = coset / (N coset^N) from the host (they depend on
// coset and N only); wave 1 squares x log N times while wave 0 climbs the tree
// and inverts, and workgroup 0 stores the common factor for the caller, as the
// reference's first kernel does.
//
// Bound: the serial chain (8 tree products, an inversion of 72 products, 8
// products down), at one instruction per 8 cycles of a wave.  With a workgroup
// barrier per level, two products a node on the way down, the squarings ahead
// of the tree and products one at a time an extension call took 26 us at 2^10
// and 42 us at 2^20.
template <bool EXT>
__global__ __launch_bounds__(LC_NT) void bary_coeffs_kernel(Tables tab, const uint64_t *x, uint64_t *common_out,
                                                            uint64_t coset, uint64_t coset_n, uint64_t f,
                                                            uint64_t *coeffs, uint32_t log_count, bool bit_reverse) {
  __shared__ gl::E2 leaf[LC_NT];  // thread products, then their inverses times the common factor
  __shared__ gl::E2 tree[128];    // node i's children are 2 i and 2 i + 1; lane l of wave 0 is node 64 + l
  __shared__ gl::E2 common;
  const uint32_t t = threadIdx.x;
  const uint64_t count = 1ull << log_count;
  const gl::E2 xv{gl::canon(x[0]), EXT ? gl::canon(x[1]) : 0ull};

  const uint64_t base = (uint64_t)blockIdx.x * (LC_NT * LC_B) + t;
  uint64_t w[LC_B];
#pragma unroll
  for (uint32_t j = 0; j < LC_B; ++j) {
    const uint64_t i = base + (uint64_t)j * LC_NT;
    const uint32_t idx = bit_reverse ? (log_count ? __builtin_bitreverse32((uint32_t)i) >> (32 - log_count) : 0u)
                                     : (uint32_t)i;
    w[j] = i < count ? pow_w(tab, 0u - (log_count ? idx << (32 - log_count) : 0u)) : 0ull;  // omega_N^-idx
  }
  gl::E2 d[LC_B], pre[LC_B];
  {
    uint64_t p0[LC_B], p1[LC_B], xs0[LC_B], xs1[LC_B];
#pragma unroll
    for (uint32_t j = 0; j < LC_B; ++j) {
      xs0[j] = xv.c0;
      xs1[j] = xv.c1;
    }
    gl::mul_row<LC_B, gl::CANON>(p0, w, xs0);
    if constexpr (EXT) gl::mul_row<LC_B, gl::CANON>(p1, w, xs1);
#pragma unroll
    for (uint32_t j = 0; j < LC_B; ++j) {
      const bool in = base + (uint64_t)j * LC_NT < count;
      d[j] = {in ? gl::sub(p0[j], coset) : 1ull, EXT && in ? p1[j] : 0ull};
    }
  }
  pre[0] = {1, 0};
  pre[1] = d[0];
#pragma unroll
  for (uint32_t j = 2; j < LC_B; ++j) pre[j] = pmul1<EXT>(pre[j - 1], d[j - 1]);
  leaf[t] = pmul1<EXT>(pre[LC_B - 1], d[LC_B - 1]);
  __syncthreads();

  auto wave_sync = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  gl::E2 q[4], pairs[2], root_inv{0, 0};
  if (t < 64) {
#pragma unroll
    for (int k = 0; k < 4; ++k) q[k] = leaf[4 * t + k];
    const gl::E2 l[2] = {q[0], q[2]}, r[2] = {q[1], q[3]};
    pmul<EXT, 2>(pairs, l, r);
    gl::E2 v = pmul1<EXT>(pairs[0], pairs[1]);
    tree[64 + t] = v;
    for (uint32_t n = 32; n; n >>= 1) {
      wave_sync();
      if (t < n) {
        v = pmul1<EXT>(tree[2 * (n + t)], tree[2 * (n + t) + 1]);
        tree[n + t] = v;
      }
    }
    if (t == 0) {
      v = {gl::canon(v.c0), gl::canon(v.c1)};
      if constexpr (EXT) root_inv = gl::e2_inv(v);
      else root_inv = {gl::inv(v.c0), 0};
    }
  } else if (t < 128) {
    gl::E2 xn = xv;
    for (uint32_t i = 0; i < log_count; ++i) xn = pmul1<EXT>(xn, xn);
    if (t == 64) {
      common = {gl::mul(gl::sub(gl::canon(xn.c0), coset_n), f), EXT ? gl::mul(xn.c1, f) : 0ull};
      if (blockIdx.x == 0) {
        common_out[0] = common.c0;
        if constexpr (EXT) common_out[1] = common.c1;
      }
    }
  }
  __syncthreads();
  if (t < 64) {
    if (t == 0) tree[1] = pmul1<EXT>(root_inv, common);
    for (uint32_t n = 2; n <= 64; n <<= 1) {
      wave_sync();
      // child n + t takes its parent's inverse times its sibling's product;
      // every child has read its sibling before the products are replaced
      gl::E2 v{0, 0};
      if (t < n) v = pmul1<EXT>(tree[(n + t) >> 1], tree[(n + t) ^ 1]);
      wave_sync();
      if (t < n) tree[n + t] = v;
    }
    const gl::E2 self = tree[64 + t];
    const gl::E2 halves_in[2] = {self, self}, other[2] = {pairs[1], pairs[0]};
    gl::E2 halves[2];
    pmul<EXT, 2>(halves, halves_in, other);
    const gl::E2 in[4] = {halves[0], halves[0], halves[1], halves[1]}, sib[4] = {q[1], q[0], q[3], q[2]};
    gl::E2 out[4];
    pmul<EXT, 4>(out, in, sib);
#pragma unroll
    for (int k = 0; k < 4; ++k) leaf[4 * t + k] = out[k];
  }
  __syncthreads();

  // common / (d_0 d_1 d_2 d_3) of this thread
  gl::E2 rest = leaf[t];
#pragma unroll
  for (uint32_t j = LC_B; j-- > 0;) {
    const uint64_t i = base + (uint64_t)j * LC_NT;
    const gl::E2 a[2] = {rest, rest}, b[2] = {pre[j], d[j]};
    gl::E2 o[2];
    if (j) pmul<EXT, 2>(o, a, b);
    else o[0] = rest;
    rest = o[1];
    if (i < count) {
      coeffs[i] = gl::canon(o[0].c0);
      if constexpr (EXT) coeffs[count + i] = gl::canon(o[0].c1);
    }
  }
}

// ---- batch evaluation ----------------------------------------------------------

enum Kind : uint32_t { BASE_AT_BASE = 0, BASE_AT_EXT = 1, EXT_AT_EXT = 2 };

constexpr uint32_t BE_NT = 256;  // 4 independent waves
constexpr uint32_t BE_WAVES = BE_NT / 64;

struct U2 {
  uint64_t x, y;
};

// Two consecutive elements; one 16-byte load when the buffer allows it.  The
// columns are read once, so the loads are non-temporal (7-9% faster for the
// base-at-base and extension batches).
template <bool ALIGNED> __device__ __forceinline__ U2 load2(const uint64_t *p) {
  if constexpr (ALIGNED) {
    typedef uint64_t v2u64 __attribute__((ext_vector_type(2)));
    const v2u64 v = __builtin_nontemporal_load(reinterpret_cast<const v2u64 *>(p));
    return {v.x, v.y};
  } else {
    return {__builtin_nontemporal_load(p), __builtin_nontemporal_load(p + 1)};
  }
}

__device__ __forceinline__ uint64_t shfl_xor64(uint64_t v, int m) {
  const uint32_t lo = __shfl_xor((int)(uint32_t)v, m), hi = __shfl_xor((int)(uint32_t)(v >> 32), m);
  return ((uint64_t)hi << 32) | lo;
}

// Tile shape: LPC lanes share a column and read it with 16-byte loads, so a
// wave load instruction covers 64 / LPC columns, 16 LPC contiguous bytes
// each; each lane issues K such loads per column (and per plane for
// extension columns), so a wave tile is 2 LPC K rows.  PREFETCH issues the
// next column pass's loads before the current pass's arithmetic.
template <uint32_t LPC, uint32_t K, bool PREFETCH> struct EvalShape {
  static constexpr uint32_t lpc = LPC, k = K, rows = 2 * LPC * K, cols = 64 / LPC;
  static constexpr bool prefetch = PREFETCH;
  static_assert(LPC >= 1 && LPC <= 64 && 64 % LPC == 0 && K >= 1, "shape");
};

// Tile shapes per kind, from a sweep on MI355X over 256 columns of 2^20 and
// 2^16 rows: wide contiguous runs per column (64 lanes x 16 B = 1 KiB per
// load instruction) read fastest.  `large` serves columns of at least 2^18
// rows, `mid` shorter ones above COLUMN_MAX_ROWS.
template <uint32_t KIND> struct Shapes;
template <> struct Shapes<BASE_AT_BASE> {
  using large = EvalShape<64, 16, false>;  // 2048-row tiles
  using mid = EvalShape<64, 4, true>;      // 512
};
template <> struct Shapes<BASE_AT_EXT> {
  using large = EvalShape<64, 8, false>;  // 1024
  using mid = EvalShape<16, 4, false>;    // 128
};
template <> struct Shapes<EXT_AT_EXT> {
  using large = EvalShape<64, 4, true>;  // 512
  using mid = EvalShape<64, 4, true>;
};
constexpr uint64_t BE_LARGE_COUNT = 1ull << 18;

// Wave w of workgroup b evaluates tile t = 4 b + w (rows [R t, R t + R),
// R = S::rows) for column passes blockIdx.y, blockIdx.y + gridDim.y, ...;
// lane l reads column cols pass + l / LPC at rows R t + 2 LPC k + 2 (l % LPC)
// + {0, 1}.  The sum over a column's LPC lanes is written to
// partial[column][t] (one element, or a (c0, c1) pair for extension
// results).  Waves share nothing, so a wave past the last tile returns.
template <uint32_t KIND, bool ALIGNED, class S>
__global__ __launch_bounds__(BE_NT) void bary_eval_tiles_kernel(const uint64_t *ys, const uint64_t *coeffs,
                                                                uint64_t count, uint32_t num_polys,
                                                                uint64_t *partial, uint64_t tiles) {
  constexpr bool CEXT = KIND != BASE_AT_BASE;
  constexpr bool YEXT = KIND == EXT_AT_EXT;
  constexpr uint32_t LPC = S::lpc, K = S::k, COLS = S::cols, STEP = 2 * LPC;
  const uint32_t lane = threadIdx.x & 63;
  const uint64_t tile = (uint64_t)blockIdx.x * BE_WAVES + (threadIdx.x >> 6);
  if (tile >= tiles) return;
  const uint32_t g = lane / LPC, q = lane % LPC;
  const uint64_t row0 = tile * S::rows + 2 * q;

  uint64_t l0[2 * K], l1[CEXT ? 2 * K : 1];
#pragma unroll
  for (uint32_t k = 0; k < K; ++k) {
    const U2 v = load2<ALIGNED>(coeffs + row0 + STEP * k);
    l0[2 * k] = v.x;
    l0[2 * k + 1] = v.y;
    if constexpr (CEXT) {
      const U2 w = load2<ALIGNED>(coeffs + count + row0 + STEP * k);
      l1[2 * k] = w.x;
      l1[2 * k + 1] = w.y;
    }
  }

  const uint64_t col_elems = YEXT ? 2 * count : count;
  U2 y0[K], y1[YEXT ? K : 1];
  auto load_pass = [&](uint32_t pass, U2 (&d0)[K], U2 (&d1)[YEXT ? K : 1]) {
    const uint32_t c = pass * COLS + g;
    if (c < num_polys) {
      const uint64_t *col = ys + (uint64_t)c * col_elems + row0;
#pragma unroll
      for (uint32_t k = 0; k < K; ++k) {
        d0[k] = load2<ALIGNED>(col + STEP * k);
        if constexpr (YEXT) d1[k] = load2<ALIGNED>(col + count + STEP * k);
      }
    }
  };
  uint32_t pass = blockIdx.y;
  if constexpr (S::prefetch)
    if (pass * COLS < num_polys) load_pass(pass, y0, y1);
  for (; pass * COLS < num_polys; pass += gridDim.y) {
    const uint32_t c = pass * COLS + g;
    const bool valid = c < num_polys;
    const uint32_t next = pass + gridDim.y;
    U2 n0[K], n1[YEXT ? K : 1];
    if constexpr (S::prefetch) {
      if (next * COLS < num_polys) load_pass(next, n0, n1);
    } else {
      load_pass(pass, y0, y1);
    }
    // KIND 0: a0 = sum l0 y.  KIND 1: a0 = sum l0 y, a1 = sum l1 y.
    // KIND 2: a0 = sum l0 y0, a1 = sum (l0 y1 + l1 y0), a2 = sum l1 y1.
    gl::Acc a0, a1, a2;
    if (valid) {
#pragma unroll
      for (uint32_t k = 0; k < K; ++k) {
        gl::mac(a0, y0[k].x, l0[2 * k]);
        gl::mac(a0, y0[k].y, l0[2 * k + 1]);
        if constexpr (CEXT) {
          gl::mac(a1, y0[k].x, l1[2 * k]);
          gl::mac(a1, y0[k].y, l1[2 * k + 1]);
        }
        if constexpr (YEXT) {
          gl::mac(a1, y1[k].x, l0[2 * k]);
          gl::mac(a1, y1[k].y, l0[2 * k + 1]);
          gl::mac(a2, y1[k].x, l1[2 * k]);
          gl::mac(a2, y1[k].y, l1[2 * k + 1]);
        }
      }
    }
    uint64_t s0 = gl::acc_reduce(a0), s1 = CEXT ? gl::acc_reduce(a1) : 0ull;
    if constexpr (YEXT) s0 = gl::add(s0, gl::mul_by_non_residue(gl::acc_reduce(a2)));
#pragma unroll
    for (int m = 1; m < (int)LPC; m <<= 1) {
      s0 = gl::add(s0, shfl_xor64(s0, m));
      if constexpr (CEXT) s1 = gl::add(s1, shfl_xor64(s1, m));
    }
    if (valid && q == 0) {
      if constexpr (CEXT) {
        uint64_t *dst = partial + 2 * ((uint64_t)c * tiles + tile);
        dst[0] = s0;
        dst[1] = s1;
      } else {
        partial[(uint64_t)c * tiles + tile] = s0;
      }
    }
    if constexpr (S::prefetch) {
#pragma unroll
      for (uint32_t k = 0; k < K; ++k) {
        y0[k] = n0[k];
        if constexpr (YEXT) y1[k] = n1[k];
      }
    }
  }
}

// One workgroup per column: the column's tile sums added up.
template <bool EXT>
__global__ __launch_bounds__(BE_NT) void bary_eval_final_kernel(const uint64_t *partial, uint64_t tiles,
                                                                uint64_t *evals) {
  __shared__ uint64_t s[2][BE_WAVES];
  const uint64_t c = blockIdx.x;
  const uint64_t *src = partial + (EXT ? 2 : 1) * c * tiles;
  uint64_t s0 = 0, s1 = 0;
  for (uint64_t t = threadIdx.x; t < tiles; t += BE_NT) {
    if constexpr (EXT) {
      s0 = gl::add(s0, src[2 * t]);
      s1 = gl::add(s1, src[2 * t + 1]);
    } else {
      s0 = gl::add(s0, src[t]);
    }
  }
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) {
    s0 = gl::add(s0, shfl_xor64(s0, m));
    if constexpr (EXT) s1 = gl::add(s1, shfl_xor64(s1, m));
  }
  const uint32_t wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    s[0][wave] = s0;
    s[1][wave] = s1;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    uint64_t r0 = s[0][0], r1 = s[1][0];
    for (uint32_t w = 1; w < BE_WAVES; ++w) {
      r0 = gl::add(r0, s[0][w]);
      r1 = gl::add(r1, s[1][w]);
    }
    if constexpr (EXT) {
      evals[2 * c] = r0;
      evals[2 * c + 1] = r1;
    } else {
      evals[c] = r0;
    }
  }
}

// Few rows (N >= 2, a power of two): one workgroup per column sums it in one
// launch, without partial sums in memory.  Bound by the chain of loads, products
// and the sum over lanes.
template <uint32_t KIND, bool ALIGNED, uint32_t THREADS>
__global__ __launch_bounds__(THREADS) void bary_eval_column_kernel(const uint64_t *ys, const uint64_t *coeffs,
                                                                   uint32_t count, uint64_t *evals) {
  constexpr bool CEXT = KIND != BASE_AT_BASE;
  constexpr bool YEXT = KIND == EXT_AT_EXT;
  constexpr uint32_t WAVES = THREADS / 64;
  __shared__ uint64_t part[2][WAVES];
  const uint64_t c = blockIdx.x;
  const uint64_t *col = ys + c * (YEXT ? 2 : 1) * count;
  gl::Acc a0, a1, a2;
  for (uint32_t r = 2 * threadIdx.x; r < count; r += 2 * THREADS) {
    const U2 l = load2<ALIGNED>(coeffs + r), y = load2<ALIGNED>(col + r);
    gl::mac(a0, y.x, l.x);
    gl::mac(a0, y.y, l.y);
    if constexpr (CEXT) {
      const U2 m = load2<ALIGNED>(coeffs + count + r);
      gl::mac(a1, y.x, m.x);
      gl::mac(a1, y.y, m.y);
      if constexpr (YEXT) {
        const U2 z = load2<ALIGNED>(col + count + r);
        gl::mac(a1, z.x, l.x);
        gl::mac(a1, z.y, l.y);
        gl::mac(a2, z.x, m.x);
        gl::mac(a2, z.y, m.y);
      }
    }
  }
  uint64_t s0 = gl::acc_reduce(a0), s1 = CEXT ? gl::acc_reduce(a1) : 0ull;
  if constexpr (YEXT) s0 = gl::add(s0, gl::mul_by_non_residue(gl::acc_reduce(a2)));
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) {
    s0 = gl::add(s0, shfl_xor64(s0, m));
    if constexpr (CEXT) s1 = gl::add(s1, shfl_xor64(s1, m));
  }
  if constexpr (WAVES > 1) {
    if ((threadIdx.x & 63) == 0) {
      part[0][threadIdx.x >> 6] = s0;
      part[1][threadIdx.x >> 6] = s1;
    }
    __syncthreads();
    s0 = part[0][0];
    s1 = part[1][0];
#pragma unroll
    for (uint32_t w = 1; w < WAVES; ++w) {
      s0 = gl::add(s0, part[0][w]);
      if constexpr (CEXT) s1 = gl::add(s1, part[1][w]);
    }
  }
  if (threadIdx.x == 0) {
    if constexpr (CEXT) {
      evals[2 * c] = s0;
      evals[2 * c + 1] = s1;
    } else {
      evals[c] = s0;
    }
  }
}

// N < 32 (or N < 128 and many columns): one thread per column sums its N
// products directly.
template <uint32_t KIND>
__global__ void bary_eval_small_kernel(const uint64_t *ys, const uint64_t *coeffs, uint32_t count,
                                       uint32_t num_polys, uint64_t *evals) {
  constexpr bool CEXT = KIND != BASE_AT_BASE;
  constexpr bool YEXT = KIND == EXT_AT_EXT;
  const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= num_polys) return;
  const uint64_t *col = ys + (uint64_t)c * (YEXT ? 2 : 1) * count;
  gl::Acc a0, a1, a2;
  for (uint32_t r = 0; r < count; ++r) {
    const uint64_t y0 = col[r];
    gl::mac(a0, y0, coeffs[r]);
    if constexpr (CEXT) gl::mac(a1, y0, coeffs[count + r]);
    if constexpr (YEXT) {
      const uint64_t y1 = col[count + r];
      gl::mac(a1, y1, coeffs[r]);
      gl::mac(a2, y1, coeffs[count + r]);
    }
  }
  uint64_t s0 = gl::acc_reduce(a0);
  if constexpr (YEXT) s0 = gl::add(s0, gl::mul_by_non_residue(gl::acc_reduce(a2)));
  if constexpr (CEXT) {
    evals[2 * c] = s0;
    evals[2 * c + 1] = gl::acc_reduce(a1);
  } else {
    evals[c] = s0;
  }
}

int finish() {
  const hipError_t err = hipGetLastError();
  return err == hipSuccess ? BC_SUCCESS : (int)err;
}

bool power_of_two(uint64_t v) { return v && !(v & (v - 1)); }

// Tiles of a column (each gives one partial sum) for the shape that serves N
// rows, and so the partial sums a caller provides room for (short columns,
// which take none now, keep the room they were given).
constexpr uint32_t MIN_TILE_ROWS = 128;
template <uint32_t KIND> uint32_t tile_rows(uint64_t count) {
  using T = Shapes<KIND>;
  if (count >= BE_LARGE_COUNT && count >= T::large::rows) return T::large::rows;
  if (count >= T::mid::rows) return T::mid::rows;
  return count >= MIN_TILE_ROWS ? MIN_TILE_ROWS : 0;
}

uint64_t eval_tiles(uint32_t kind, uint64_t count) {
  const uint32_t rows = kind == BASE_AT_BASE  ? tile_rows<BASE_AT_BASE>(count)
                        : kind == BASE_AT_EXT ? tile_rows<BASE_AT_EXT>(count)
                                              : tile_rows<EXT_AT_EXT>(count);
  return rows ? count / rows : 0;
}

// Workgroups of one tile-kernel variant resident on the current device (CUs x
// workgroups per CU at its register use), queried once per device.
template <uint32_t KIND, class S> uint32_t resident_wgs() {
  constexpr int MAX_DEVICES = 64;
  static std::mutex mu;
  static uint32_t cache[MAX_DEVICES] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return 768;
  std::lock_guard<std::mutex> lk(mu);
  if (!cache[dev]) {
    int cus = 0, per_cu = 0;
    const bool ok = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
                    hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, bary_eval_tiles_kernel<KIND, true, S>,
                                                                 BE_NT, 0) == hipSuccess &&
                    cus > 0 && per_cu > 0;
    cache[dev] = ok ? (uint32_t)(cus * per_cu) : 768u;
  }
  return cache[dev];
}

// Launch grid: tiles x column-pass groups, about `target` workgroups (more
// for the short-column shapes, whose tiles are few).
template <uint32_t KIND, class S>
void launch_tiles(const uint64_t *ys, const uint64_t *coeffs, uint64_t count, uint32_t num_polys, uint64_t *partial,
                  uint64_t *evals, uint64_t target, hipStream_t s) {
  constexpr bool OUT_EXT = KIND != BASE_AT_BASE;
  const uint64_t tiles = count / S::rows;
  const uint64_t gx = (tiles + BE_WAVES - 1) / BE_WAVES;
  const uint32_t passes = (num_polys + S::cols - 1) / S::cols;
  uint64_t gy = (target + gx - 1) / gx;
  if (gy > passes) gy = passes;
  if (gy > 65535) gy = 65535;
  const dim3 grid((uint32_t)gx, (uint32_t)gy);
  const bool aligned = !(((uintptr_t)ys | (uintptr_t)coeffs) & 15);
  if (aligned)
    bary_eval_tiles_kernel<KIND, true, S><<<grid, BE_NT, 0, s>>>(ys, coeffs, count, num_polys, partial, tiles);
  else
    bary_eval_tiles_kernel<KIND, false, S><<<grid, BE_NT, 0, s>>>(ys, coeffs, count, num_polys, partial, tiles);
  bary_eval_final_kernel<OUT_EXT><<<dim3(num_polys), BE_NT, 0, s>>>(partial, tiles, evals);
}

// Columns of 32..1024 rows take the column kernel, below 128 rows while the
// columns are few.  Coefficients and evaluations at an extension point, column
// kernel against the others: 20 columns of 2^5 / 2^6 / 2^8 / 2^10 / 2^12 rows
// 18.2 / 18.4 / 18.8 / 19.9 / 23.9 us against 19.8 / 23.9 / 20.4 / 21.2 / 22.0
// (2^3: 18.6 against 16.6), 40000 columns of 2^7 / 2^8 rows 34 / 40 against 74 /
// 82 us, of 2^5 32 against 24, 4000 of 2^10 28 against 31.  Evaluations alone,
// base columns at base points / extension columns: 20 columns of 2^6 and 2^10
// rows 7.0 and 7.1 / 7.1 and 7.0 us against 8.0 and 10.3 / 14.1 and 10.4, 4000 of
// 2^10 7.3 / 16.8 against 10.3 / 22.8, 40000 of 2^7 11.6 / 24 against 32.6 / 68.
constexpr uint64_t COLUMN_MIN_ROWS = 32, COLUMN_MAX_ROWS = 1024;
constexpr uint32_t COLUMN_FEW = 8192;
bool column_path(uint64_t count, uint32_t num_polys) {
  return count >= COLUMN_MIN_ROWS && count <= COLUMN_MAX_ROWS && (count >= 128 || num_polys <= COLUMN_FEW);
}

bool overlap(const uint64_t *a, uint64_t a_len, const uint64_t *b, uint64_t b_len) {
  return (uintptr_t)a < (uintptr_t)(b + b_len) && (uintptr_t)b < (uintptr_t)(a + a_len);
}

// Evaluations that go over columns or coefficients other workgroups still read
// are kept in the partial sums, one to a column, until all have been read
// (from MIN_TILE_ROWS on, where callers provide these).
template <uint32_t KIND>
void launch_column(const uint64_t *ys, const uint64_t *coeffs, uint32_t count, uint32_t num_polys, uint64_t *partial,
                   uint64_t *evals, hipStream_t s) {
  constexpr uint64_t YW = KIND == EXT_AT_EXT ? 2 : 1, W = KIND == BASE_AT_BASE ? 1 : 2;
  const bool hold = count >= MIN_TILE_ROWS && (overlap(evals, W * num_polys, ys, YW * count * num_polys) ||
                                               overlap(evals, W * num_polys, coeffs, W * count));
  uint64_t *sums = hold ? partial : evals;
  const bool aligned = !(((uintptr_t)ys | (uintptr_t)coeffs) & 15);
  auto go = [&](auto threads) {
    constexpr uint32_t N = decltype(threads)::value;
    if (aligned) bary_eval_column_kernel<KIND, true, N><<<dim3(num_polys), N, 0, s>>>(ys, coeffs, count, sums);
    else bary_eval_column_kernel<KIND, false, N><<<dim3(num_polys), N, 0, s>>>(ys, coeffs, count, sums);
  };
  if (count <= 512) go(std::integral_constant<uint32_t, 64>{});
  else go(std::integral_constant<uint32_t, 256>{});
  if (hold) bary_eval_final_kernel<KIND != BASE_AT_BASE><<<dim3(num_polys), BE_NT, 0, s>>>(sums, 1, evals);
}

template <uint32_t KIND>
void launch_eval(const uint64_t *ys, const uint64_t *coeffs, uint64_t count, uint32_t num_polys, uint64_t *partial,
                 uint64_t *evals, hipStream_t s) {
  using T = Shapes<KIND>;
  if (column_path(count, num_polys))
    launch_column<KIND>(ys, coeffs, (uint32_t)count, num_polys, partial, evals, s);
  else if (count < COLUMN_MAX_ROWS)
    bary_eval_small_kernel<KIND><<<dim3((num_polys + 255) / 256), 256, 0, s>>>(ys, coeffs, (uint32_t)count,
                                                                               num_polys, evals);
  else if (count >= BE_LARGE_COUNT)  // about three whole rounds of resident workgroups
    launch_tiles<KIND, typename T::large>(ys, coeffs, count, num_polys, partial, evals,
                                          3ull * resident_wgs<KIND, typename T::large>(), s);
  else
    launch_tiles<KIND, typename T::mid>(ys, coeffs, count, num_polys, partial, evals, 8192, s);
}

}  // namespace
}  // namespace bc

extern "C" int bc_barycentric_precompute(bool ext, const uint64_t *x, uint64_t *common_factor, uint64_t coset,
                                         uint64_t *coeffs, uint64_t count, bool bit_reverse, void *stream) {
  using namespace bc;
  if (!x || !common_factor || !coeffs || !power_of_two(count) || count > (1ull << 31)) return BC_ERROR_INVALID_VALUE;
  bool ok = false;
  const Tables tab = current_tables(ok);
  if (!ok) return BC_ERROR_NOT_INITIALIZED;
  const uint32_t log_count = (uint32_t)__builtin_ctzll(count);
  hipStream_t s = (hipStream_t)stream;
  // coset^N and f = coset / (N coset^N): host arithmetic on two scalars
  const uint64_t c = gl::canon(coset);
  const uint64_t cn = gl::sqn(c, log_count);
  const uint64_t f = gl::mul(c, gl::inv(gl::mul(count, cn)));
  const dim3 grid((uint32_t)((count + LC_NT * LC_B - 1) / (LC_NT * LC_B)));
  if (ext)
    bary_coeffs_kernel<true><<<grid, LC_NT, 0, s>>>(tab, x, common_factor, c, cn, f, coeffs, log_count, bit_reverse);
  else
    bary_coeffs_kernel<false><<<grid, LC_NT, 0, s>>>(tab, x, common_factor, c, cn, f, coeffs, log_count, bit_reverse);
  return finish();
}

extern "C" int bc_batch_eval_temp_sizes(uint32_t kind, uint64_t stride, uint32_t num_polys, size_t *partial_elems,
                                        size_t *final_bytes) {
  using namespace bc;
  if (kind > EXT_AT_EXT || !power_of_two(stride) || stride > (1ull << 31) || !partial_elems || !final_bytes)
    return BC_ERROR_INVALID_VALUE;
  const uint64_t tiles = eval_tiles(kind, stride);
  *partial_elems = (size_t)num_polys * (tiles ? tiles : 1);
  *final_bytes = 0;
  return BC_SUCCESS;
}

extern "C" int bc_batch_eval(uint32_t kind, const uint64_t *ys, uint64_t stride, uint32_t num_polys,
                             const uint64_t *coeffs, uint64_t *temp_partial, size_t temp_partial_elems,
                             void *temp_final, size_t temp_final_bytes, uint64_t *evals, void *stream) {
  using namespace bc;
  (void)temp_final;
  (void)temp_final_bytes;
  size_t need = 0, need_final = 0;
  if (bc_batch_eval_temp_sizes(kind, stride, num_polys, &need, &need_final) != BC_SUCCESS)
    return BC_ERROR_INVALID_VALUE;
  if (num_polys == 0) return BC_SUCCESS;
  if (!ys || !coeffs || !evals || (eval_tiles(kind, stride) && (!temp_partial || temp_partial_elems < need)))
    return BC_ERROR_INVALID_VALUE;
  hipStream_t s = (hipStream_t)stream;
  switch (kind) {
  case BASE_AT_BASE: launch_eval<BASE_AT_BASE>(ys, coeffs, stride, num_polys, temp_partial, evals, s); break;
  case BASE_AT_EXT: launch_eval<BASE_AT_EXT>(ys, coeffs, stride, num_polys, temp_partial, evals, s); break;
  default: launch_eval<EXT_AT_EXT>(ys, coeffs, stride, num_polys, temp_partial, evals, s); break;
  }
  return finish();
}
