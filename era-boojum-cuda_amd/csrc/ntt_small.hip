// Transforms of one wave, 4 values per lane: columns of 2..128 points
// (ntt_short_kernel, below), and the latency path for a few columns of
// 2^13..2^16 points (the single-column case of the reference's benches) as two
// launches of one-wave workgroups, each wave holding 256 values.
//
// The pass kernels of ntt_fast.hip give each thread 16 values of a 4096-point
// tile, so one 2^16 column is 16 workgroups per pass and the call takes one
// workgroup's serial work.  Here the transform is split h + 8: the top pass
// runs 256 2^h-point sub-DFTs over the top index bits (stride 256, with the
// pass twist omega_n^(r * brev(j))), 2^(8-h) to a wave, the bottom pass
// 256-point sub-DFTs over consecutive points, one to a wave; each lane does
// four values' work.
//
// One wave's 256-point DIF, point j = 64 i + l at lane l, register i:
//   stage 1: radix 4 over j bits 7..6 (registers), twist omega_256^(l k1);
//   exchange 1: register bits <-> lane bits 4, 5 (v_permlane16/32_swap);
//   stage 2: radix 4 over j bits 5..4, twist omega_64^((l & 15) k2);
//   exchange 2: register bits <-> lane bits 2, 3 (through the wave's LDS);
//   stage 3: radix 4 over j bits 3..2, twist omega_16^((l & 3) k3);
//   exchange 3: register bits <-> lane bits 0, 1 (through the wave's LDS);
//   stage 4: radix 4 over j bits 1..0,
// where k_s = brev2(register) after the stage's radix-4 DIF.  Every exchange
// transposes two register bits with two lane bits, so lane l, register i ends
// at the bit-reversed output position 4 l + i (the wave stores 32 contiguous
// bytes per lane).  DIT (bit-reversed input) is the transpose: the same
// stages, twists and exchanges in reverse order.
#include "ntt_device.hpp"
#include "ntt_internal.hpp"

namespace bc {
namespace {

constexpr uint32_t SW = 64;  // threads per workgroup: one wave

__device__ __forceinline__ uint32_t brev2(uint32_t i) { return ((i & 1u) << 1) | (i >> 1); }

// omega_{2^s}^e (e < 2^s, s <= 16) from the coarse table: omega_{2^32}^(e 2^(32-s))
__device__ __forceinline__ uint64_t root(const Tables &tab, uint32_t s, uint32_t e, bool inv) {
  const uint32_t m = (1u << s) - 1u;
  const uint32_t k = inv ? ((0u - e) & m) : (e & m);
  return tab.w_coarse[k << (16u - s)];
}

// Transposes register bits 0, 1 with lane bits 4, 5 of four 64-bit values:
// v_permlane16_swap exchanges the odd 16-lane rows of its first operand with
// the even rows of its second, v_permlane32_swap the upper 32 lanes of the
// first with the lower 32 of the second.
__device__ __forceinline__ void swap_lane45(uint64_t *x) {
  auto sw16 = [](uint64_t &a, uint64_t &b) {
    const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)a, (uint32_t)b, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((uint32_t)(a >> 32), (uint32_t)(b >> 32), false, false);
    a = ((uint64_t)hi[0] << 32) | lo[0];
    b = ((uint64_t)hi[1] << 32) | lo[1];
  };
  auto sw32 = [](uint64_t &a, uint64_t &b) {
    const auto lo = __builtin_amdgcn_permlane32_swap((uint32_t)a, (uint32_t)b, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((uint32_t)(a >> 32), (uint32_t)(b >> 32), false, false);
    a = ((uint64_t)hi[0] << 32) | lo[0];
    b = ((uint64_t)hi[1] << 32) | lo[1];
  };
  sw16(x[0], x[1]);
  sw16(x[2], x[3]);
  sw32(x[0], x[2]);
  sw32(x[1], x[3]);
}

// Transposes register bits 0, 1 with lane bits B, B + 1 through `buf` (256
// words of this wave's LDS).
template <int B> __device__ __forceinline__ void swap_lanes_lds(uint64_t *x, uint64_t *buf, uint32_t l) {
#pragma unroll
  for (int i = 0; i < 4; ++i) buf[i * SW + l] = x[i];
  __syncthreads();
  const uint32_t src_reg = (l >> B) & 3u, lane_rest = l & ~(3u << B);
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = buf[src_reg * SW + (lane_rest | ((uint32_t)i << B))];
}

struct WaveLds {
  uint64_t ex2[4 * SW];
  uint64_t ex3[4 * SW];
};

// The lower LN levels of a wave's 256-point transform: 2^(8-LN) transforms of
// 2^LN points.  Position p of the wave's 256 values is point p mod 2^LN of
// transform p / 2^LN; at stage s register i of lane l holds the position with
// register bits at B = 6 - 2s, and the stages above the transforms' length
// (and the exchanges behind them) fall away.  With odd LN the first stage is
// radix 2 over its lower bit.
template <int LN, bool INV, bool DIT> struct WaveDft {
  static constexpr int S0 = 4 - (LN + 1) / 2;
  static constexpr int FIRST = DIT ? 3 : S0, LAST = DIT ? S0 : 3;  // stages of the inputs and the outputs
  uint32_t l;
  uint64_t tw[3][3];  // twists of registers 1..3 behind (DIT: before) the stages
  __device__ __forceinline__ WaveDft(const Tables &tab, uint32_t lane) : l(lane) {
    static_for<3 - S0>([&](auto k) {
      constexpr int S = S0 + decltype(k)::value, B = 6 - 2 * S;
      const uint32_t rp = l & ((1u << B) - 1u);
      if constexpr (S == S0 && LN % 2) {
        tw[S][0] = root(tab, B + 1, rp, INV);
      } else {
#pragma unroll
        for (int i = 1; i < 4; ++i) tw[S][i - 1] = root(tab, B + 2, rp * brev2((uint32_t)i), INV);
      }
    });
  }
  __device__ __forceinline__ uint32_t pos(int s, int i) const {
    const int b = 6 - 2 * s;
    return ((l >> b) << (b + 2)) | ((uint32_t)i << b) | (l & ((1u << b) - 1u));
  }
  template <int S> __device__ __forceinline__ void twist(uint64_t *x) const {
    if constexpr (S == 3) return;
    else if constexpr (S == S0 && LN % 2) {
      x[1] = gl::mul(x[1], tw[S][0]);
      x[3] = gl::mul(x[3], tw[S][0]);
    } else {
#pragma unroll
      for (int i = 1; i < 4; ++i) x[i] = gl::mul(x[i], tw[S][i - 1]);
    }
  }
  template <int S> __device__ __forceinline__ static void dft(uint64_t *x) {
    constexpr int A = S == S0 && LN % 2 ? 1 : 2;
#pragma unroll
    for (int g = 0; g < 4; g += 1 << A) {
      if constexpr (DIT) dft_dit<A, INV>(x + g);
      else dft_dif<A, INV>(x + g);
    }
  }
  // between stages S and S + 1, either way
  template <int S> __device__ __forceinline__ void exchange(uint64_t *x, WaveLds &sh) const {
    if constexpr (S == 0) swap_lane45(x);
    else if constexpr (S == 1) swap_lanes_lds<2>(x, sh.ex2, l);
    else if constexpr (S == 2) swap_lanes_lds<0>(x, sh.ex3, l);
  }
  // canonical values in, canonical values out
  __device__ __forceinline__ void run(uint64_t *x, WaveLds &sh) const {
    static_for<4 - S0>([&](auto k) {
      constexpr int K = decltype(k)::value, S = DIT ? 3 - K : S0 + K;
      if constexpr (DIT) {
        if constexpr (K > 0) exchange<S>(x, sh);
        twist<S>(x);
        dft<S>(x);
      } else {
        dft<S>(x);
        twist<S>(x);
        if constexpr (S < 3) exchange<S>(x, sh);
      }
    });
  }
};

// Top pass of a 2^(LH+8)-point column: workgroup (group of 2^(8-LH)
// consecutive r, column), a 2^LH-point sub-DFT over the points j 256 + r for
// each r, with the pass twist omega_n^(r brev(j)) (n^-1 folded in for inverse
// transforms) behind it (DIT: before).
template <int LH, bool INV, bool DIT>
__global__ __launch_bounds__(SW) void ntt_small_top_kernel(FastArgs a) {
  __shared__ WaveLds sh;
  // workgroups are dispatched round-robin over the 8 XCDs: keep the
  // workgroups whose r share a 128-byte line on one XCD (one L2)
  const uint32_t r0 = (((blockIdx.x & 7u) << (LH - 3)) | (blockIdx.x >> 3)) << (8 - LH);
  const uint64_t c = blockIdx.y;
  const uint64_t *in = a.in + c * a.stride_in + r0;
  uint64_t *out = a.out + c * a.stride_out + r0;
  using W = WaveDft<LH, INV, DIT>;
  const W w(a.tab, threadIdx.x);
  auto at = [&](int s, int i) -> uint64_t {
    const uint32_t p = w.pos(s, i);
    return ((uint64_t)(p & ((1u << LH) - 1u)) << 8) + (p >> LH);
  };
  constexpr int TS = 3;  // the stage at the twisted end
  uint64_t pt[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t p = w.pos(TS, i), k = brev_bits(p & ((1u << LH) - 1u), LH);
    uint32_t e = ((r0 + (p >> LH)) * k) << (24 - LH);
    if (INV) e = 0u - e;
    pt[i] = pow_w(a.tab, e);
    if (INV) pt[i] = gl::mul(pt[i], a.n_inv);
  }
  uint64_t x[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = in[at(W::FIRST, i)];
  if constexpr (!DIT) {
    if (a.first) {
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = gl::canon(x[i]);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = gl::mul(x[i], pt[i]);
  }
  w.run(x, sh);
#pragma unroll
  for (int i = 0; i < 4; ++i) out[at(W::LAST, i)] = DIT ? x[i] : gl::mul(x[i], pt[i]);
}

// Bottom pass (sub-DFTs over index bits 7..0): workgroup (block, column),
// 256 consecutive points.
template <bool INV, bool DIT>
__global__ __launch_bounds__(SW) void ntt_small_bottom_kernel(FastArgs a) {
  __shared__ WaveLds sh;
  const uint64_t c = blockIdx.y, b = blockIdx.x;
  const uint64_t *in = a.in + c * a.stride_in + (b << 8);
  uint64_t *out = a.out + c * a.stride_out + (b << 8);
  using W = WaveDft<8, INV, DIT>;
  const W w(a.tab, threadIdx.x);
  uint64_t x[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = in[w.pos(W::FIRST, i)];
  if (a.first) {
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = gl::canon(x[i]);
  }
  w.run(x, sh);
#pragma unroll
  for (int i = 0; i < 4; ++i) out[w.pos(W::LAST, i)] = x[i];
}

template <int LH, bool INV, bool DIT> hipError_t launch_pair(const FastArgs &top, const FastArgs &bottom, hipStream_t s) {
  const dim3 grid(1u << LH, top.num_cols);
  if constexpr (!DIT) {
    ntt_small_top_kernel<LH, INV, false><<<grid, SW, 0, s>>>(top);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
    ntt_small_bottom_kernel<INV, false><<<grid, SW, 0, s>>>(bottom);
  } else {
    ntt_small_bottom_kernel<INV, true><<<grid, SW, 0, s>>>(bottom);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
    ntt_small_top_kernel<LH, INV, true><<<grid, SW, 0, s>>>(top);
  }
  return hipGetLastError();
}

// `first` reads the caller's input, `second` works in place on the output.
template <int LH>
hipError_t launch_small_h(const FastArgs &first, const FastArgs &second, bool bitrev_inputs, bool inverse,
                          hipStream_t s) {
  if (!bitrev_inputs)
    return inverse ? launch_pair<LH, true, false>(first, second, s) : launch_pair<LH, false, false>(first, second, s);
  return inverse ? launch_pair<LH, true, true>(second, first, s) : launch_pair<LH, false, true>(second, first, s);
}

// Columns of 2^LN points, LN = 1..7, 2^(8-LN) columns to a wave.
//
// A small call is bound by one wave's serial work behind the launch: 256
// columns of 2^4 / 2^7 points took 8.7-14 / 12-17 us as 4096-point tiles of
// 256 threads with 16 values each, 6.5-7 us here, about a call's time on the
// host.  Large ones are bound by memory in pieces of columns: 2^26 values in
// columns of 2^4 / 2^7 305-514 / 399-614 -> 262-344 / 327-490 us.
constexpr uint32_t SHORT_WAVES = 4;  // waves a workgroup of many-column calls has
template <int LN, bool INV, bool DIT>
__global__ __launch_bounds__(SHORT_WAVES * SW) void ntt_short_kernel(FastArgs a) {
  __shared__ WaveLds sh[SHORT_WAVES];
  const uint64_t col0 = ((uint64_t)blockIdx.x * (blockDim.x / SW) + threadIdx.x / SW) << (8 - LN);
  using W = WaveDft<LN, INV, DIT>;
  const W w(a.tab, threadIdx.x % SW);
  uint64_t x[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t p = w.pos(W::FIRST, i), j = p & ((1u << LN) - 1u);
    const uint64_t c = col0 + (p >> LN);
    x[i] = c < a.num_cols ? gl::canon(a.in[c * a.stride_in + j]) : 0ull;
  }
  if (!INV && a.log_ext) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t j = w.pos(W::FIRST, i) & ((1u << LN) - 1u);
      x[i] = gl::mul(x[i], coset_pow(a.tab, a.coset_exp, DIT ? brev_bits(j, LN) : j, false));
    }
  }
  w.run(x, sh[threadIdx.x / SW]);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t p = w.pos(W::LAST, i), j = p & ((1u << LN) - 1u);
    const uint64_t c = col0 + (p >> LN);
    if (c >= a.num_cols) continue;
    uint64_t v = x[i];
    if (INV) {
      v = gl::mul(v, a.n_inv);
      if (a.log_ext) v = gl::mul(v, coset_pow(a.tab, a.coset_exp, DIT ? j : brev_bits(j, LN), true));
    }
    a.out[c * a.stride_out + j] = gl::canon(v);
  }
}

template <int LN> hipError_t launch_short_ln(const FastArgs &all, bool inverse, bool dit, hipStream_t s) {
  // A launch takes fewer than 2^32 threads: 2^33 values at a time, a whole
  // number of workgroups of SHORT_WAVES waves.
  constexpr uint64_t MAX_COLS = 1ull << (33 - LN);
  for (uint64_t col = 0; col < all.num_cols; col += MAX_COLS) {
    FastArgs a = all;
    a.in += col * a.stride_in;
    a.out += col * a.stride_out;
    a.num_cols = (uint32_t)(all.num_cols - col < MAX_COLS ? all.num_cols - col : MAX_COLS);
    // one-wave workgroups until the chip has four on every SIMD
    const uint64_t waves = ((uint64_t)a.num_cols + (1u << (8 - LN)) - 1) >> (8 - LN);
    const uint32_t per_wg = waves > 4096 ? SHORT_WAVES : 1;
    const dim3 grid((uint32_t)((waves + per_wg - 1) / per_wg)), block(per_wg * SW);
    if (inverse) {
      if (dit) ntt_short_kernel<LN, true, true><<<grid, block, 0, s>>>(a);
      else ntt_short_kernel<LN, true, false><<<grid, block, 0, s>>>(a);
    } else {
      if (dit) ntt_short_kernel<LN, false, true><<<grid, block, 0, s>>>(a);
      else ntt_short_kernel<LN, false, false><<<grid, block, 0, s>>>(a);
    }
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
  }
  return hipSuccess;
}

}  // namespace

hipError_t launch_short(const FastArgs &a, bool inverse, bool bitrev_inputs, hipStream_t s) {
  switch (a.log_n) {
  case 1: return launch_short_ln<1>(a, inverse, bitrev_inputs, s);
  case 2: return launch_short_ln<2>(a, inverse, bitrev_inputs, s);
  case 3: return launch_short_ln<3>(a, inverse, bitrev_inputs, s);
  case 4: return launch_short_ln<4>(a, inverse, bitrev_inputs, s);
  case 5: return launch_short_ln<5>(a, inverse, bitrev_inputs, s);
  case 6: return launch_short_ln<6>(a, inverse, bitrev_inputs, s);
  case 7: return launch_short_ln<7>(a, inverse, bitrev_inputs, s);
  default: return hipErrorInvalidValue;
  }
}

bool small_path_applies(uint32_t log_n, uint32_t num_cols, uint32_t log_ext, const TuneParams &tp) {
  if (log_n < SMALL_MIN_LOG_N || log_n > SMALL_LOG_N || log_ext != 0 || num_cols < 1 || num_cols > 65535) return false;
  // an entry that shapes the 4096-point passes of a shorter column asks for them
  const bool shaped = log_n != SMALL_LOG_N && (tp.contig_log || tp.strided_bpw || tp.contig_grid);
  return tp.tile_log == 8 || (tp.tile_log == 0 && !shaped && num_cols <= (1u << SMALL_LOG_POINTS) >> log_n);
}

hipError_t launch_small(const Tables &tab, const uint64_t *inputs, uint64_t *outputs, uint32_t log_n,
                        uint32_t num_cols, uint64_t stride_in, uint64_t stride_out, bool bitrev_inputs, bool inverse,
                        hipStream_t s) {
  FastArgs a{};
  a.tab = tab;
  a.num_cols = num_cols;
  a.log_n = log_n;
  a.n_inv = gl::inv((1ull << log_n) % gl::P);
  FastArgs first = a, second = a;
  first.in = inputs;
  first.stride_in = stride_in;
  first.out = outputs;
  first.stride_out = stride_out;
  first.first = 1;
  second.in = outputs;
  second.stride_in = stride_out;
  second.out = outputs;
  second.stride_out = stride_out;
  second.first = 0;
  switch (log_n) {
  case 13: return launch_small_h<5>(first, second, bitrev_inputs, inverse, s);
  case 14: return launch_small_h<6>(first, second, bitrev_inputs, inverse, s);
  case 15: return launch_small_h<7>(first, second, bitrev_inputs, inverse, s);
  case 16: return launch_small_h<8>(first, second, bitrev_inputs, inverse, s);
  default: return hipErrorInvalidValue;
  }
}

}  // namespace bc
