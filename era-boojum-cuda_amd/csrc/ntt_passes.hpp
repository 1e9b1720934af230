// Register-resident NTT pass bodies for gfx950 (device code shared by the
// standalone pass kernels and the ragged persistent kernel).
//
// Semantics (reference: src/ntt.rs:527-583 and native/ntt.cu:105-122):
//   forward:  X_k = sum_i x_i s^i w^(ik)
//   inverse:  y_i = n^-1 s^-i sum_k x_k w^(-ik)
// with w = omega_n, s = g * omega_{n 2^ext}^coset when log_ext > 0 (else 1).
// n2b: natural input, bit-reversed output; b2n: bit-reversed input, natural
// output.
//
// Decomposition.  A transform of 2^L points is split into HBM passes
// L = h_0 + h_1 + ... (plan_passes).  In n2b order pass p works inside blocks
// of N = 2^(L - h_0 - ... - h_{p-1}) points.  Writing an index inside a block
// as i = j * R + r (R = N / H, H = 2^h_p), the pass runs, for every r, an
// H-point natural->bit-reversed DFT over j (root omega_H), then multiplies the
// value at position j by the twist omega_N^(r * brev(j)).  The next pass then
// works on blocks of R contiguous points.  This is the four-step recursion of
// the DFT; the last pass has R = 1 and no twist.
//
// b2n is the transpose of n2b: the same diagonal twists and the same
// symmetric sub-DFTs applied in the reverse order, so passes run last-first,
// each pass applies its twist before its sub-DFT, and sub-DFTs use the
// bit-reversed-input (decimation in time) form.
//
// Two tile shapes cover
// every pass of a transform with log_n >= 8:
//
//   contig<h>  (8 <= h <= 12): R = 1, the last pass in n2b order.  A tile is
//              4096 consecutive points = 2^(12-h) sub-DFTs.  Levels of radix
//              16, 16 and 2^(h-8) run in registers, with LDS exchanges
//              between them; for plain and n^-1 passes the one between
//              levels 1 and 2 (and in b2n the load regrouping) stays inside
//              a wave, with no workgroup barrier.
//   strided<h> (4 <= h <= 8):  R >= 16, every other pass.  A tile is
//              2^(12-h) consecutive r times the h-point sub-DFT, so each row of
//              the tile is >= 128 contiguous bytes.  Levels of radix 16 and
//              2^(h-4), one LDS exchange (none for h = 4).
//
// Every workgroup has 256 threads holding 16 values each.  Global loads go
// straight into the first level's registers and the last level stores from
// registers.  Column values are read and written once per pass, so those
// loads and stores are non-temporal (`nt`: streamed past the caches, which
// keep the twiddle tables); measured 2% faster per 256 x 2^20 call than
// ordinary loads and stores.  Per-thread level twists depend only on the
// thread and are computed once per workgroup; the strided pass twist depends
// on the tile's r range, so a workgroup walks several (column, block) pairs
// that share it and computes it once.  n2b runs levels top-down (DIF), b2n
// bottom-up (DIT) as the transpose.
#pragma once
#include "gl_lazy.hpp"
#include "ntt_device.hpp"

#include <stddef.h>

namespace bc {
namespace pass {

constexpr uint32_t NT = 256;  // threads per workgroup

// Padded LDS index: one pad slot per 16 keeps stride-16 accesses on distinct banks.
__device__ __forceinline__ uint32_t pidx(uint32_t e) { return e + (e >> 4); }
constexpr uint32_t LDS_PADDED = TILE + TILE / 16;

// Level-twist table of a radix-16 level in blocks of M = 2^LM points: entry
// (i - 1) * S + rp = omega_M^(+-rp * brev4(i)), S = M / 16.
template <int LM, bool INV> __device__ __forceinline__ const uint64_t *lvl_table(const Tables &tab) {
  return tab.lvl_tw + (INV ? LVL_TW_BLOCK : 0u) + lvl_tw_offset(LM);
}

// Copies a level-twist table into LDS (once per workgroup).
template <int LM, bool INV> __device__ __forceinline__ void stage_level_twists(uint64_t *dst, const Tables &tab) {
  constexpr uint32_t LEN = 15u << (LM - 4);
  const uint64_t *src = lvl_table<LM, INV>(tab);
  for (uint32_t k = threadIdx.x; k < LEN; k += NT) dst[k] = src[k];
}

// x[i] *= tw[(i - 1) * S + rp] for i = 1..15 (tw in LDS).
template <int LM, gl::Reduce R>
__device__ __forceinline__ void level_twist_lds(uint64_t *x, const uint64_t *tw, uint32_t rp, int32_t *e = nullptr) {
  constexpr uint32_t S = 1u << (LM - 4);
  gl::mul_each<1, 15, R>(x, [&](int i) { return tw[(i - 1) * S + rp]; }, e);
}

// x[i] *= base * part[i] for all 16 points.
template <gl::Reduce R> __device__ __forceinline__ void coset_twist(uint64_t *x, uint64_t base, const uint64_t *part) {
  gl::unroll<4>([&](auto r) {
    constexpr int B = 4 * decltype(r)::value;
    uint64_t f[4] = {part[B], part[B + 1], part[B + 2], part[B + 3]};
    const uint64_t b[4] = {base, base, base, base};
    gl::mul_row<4, gl::ANY>(f, f, b);
    gl::mul_row<4, R>(x + B, x + B, f);
  });
}

// -------------------------------------------------------------------------
// contig<h>

// Tile element e of thread t's group g, point i, at level L (width A) of an
// h-point sub-DFT whose levels are 4, 4, h - 8.
template <int LH, int L, int A> __device__ __forceinline__ uint32_t celem(uint32_t t, int g, int i) {
  constexpr int C = 4 * L, LM = LH - C, LS = LM - A;
  const uint32_t gi = t + NT * (uint32_t)g;
  const uint32_t rp = gi & ((1u << LS) - 1u);
  const uint32_t b = (gi >> LS) & ((1u << C) - 1u);
  const uint32_t qb = gi >> (LH - A);
  return (qb << LH) + (b << LM) + ((uint32_t)i << LS) + rp;
}

// Coset scaling (MODE_LDE_IN: s^idx on the inputs; MODE_LDE_OUT: n^-1 s^-idx
// on the outputs).  A thread's 16 points sit at indices idx0 + part(i) whose
// parts use bits the thread's base index leaves zero, so s^(idx0 + part(i)) =
// s^idx0 * s^part(i): the 16 part factors are computed once per workgroup
// (into LDS, by threads 0..15) and each thread computes one power per tile.
template <int MODE> __device__ __forceinline__ uint64_t coset_scale_pow(const FastArgs &a, uint32_t idx) {
  return coset_pow(a.tab, a.coset_exp, idx, MODE == MODE_LDE_OUT);
}
template <int MODE> __device__ __forceinline__ uint64_t coset_part_factor(const FastArgs &a, uint32_t part) {
  const uint64_t v = coset_scale_pow<MODE>(a, part);
  return MODE == MODE_LDE_OUT ? gl::mul(a.n_inv, v) : v;
}

// Level twists with a coset factor folded in (strided passes): group rp's
// twists become tw * c(rp) with c(rp) = s^(+-rp 2^log_r), and dst0[rp] = c(rp)
// scales the group's point 0, whose twist is 1.
template <int LM, bool INV, int MODE>
__device__ __forceinline__ void stage_level_twists_coset(uint64_t *dst, uint64_t *dst0, const FastArgs &a,
                                                         uint32_t log_r) {
  constexpr uint32_t S = 1u << (LM - 4), LEN = 15u * S;
  const uint64_t *src = lvl_table<LM, INV>(a.tab);
  for (uint32_t k = threadIdx.x; k < LEN; k += NT)
    dst[k] = gl::mul(src[k], coset_scale_pow<MODE>(a, (k & (S - 1u)) << log_r));
  if (threadIdx.x < S) dst0[threadIdx.x] = coset_scale_pow<MODE>(a, threadIdx.x << log_r);
}

// Column values are loaded and stored through buffer descriptors: a wave-
// uniform base, a 32-bit per-thread offset that does not change, and the rest
// of the address in a scalar offset, so that the 16 accesses of a tile need no
// vector address arithmetic (three instructions and a wait state per pair of
// loads before).  Accesses are non-temporal.
__device__ __forceinline__ uint64_t uniform64(uint64_t v) {
  return gl::pair64(__builtin_amdgcn_readfirstlane((uint32_t)v), __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32)));
}
struct Buf {
  static constexpr int RAW_32 = 0x00020000;  // word 3: raw buffer, 32-bit data format
  static constexpr int NT = 2;               // cache policy: non-temporal
  using V2 = uint32_t __attribute__((ext_vector_type(2)));
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ Buf(const uint64_t *base, uint32_t bytes)
      : r(__builtin_amdgcn_make_buffer_rsrc((void *)uniform64((uint64_t)base), 0, (int)bytes, RAW_32)) {}
  __device__ __forceinline__ uint64_t load(uint32_t voff, uint32_t soff) const {
    const V2 v = __builtin_amdgcn_raw_buffer_load_b64(r, (int)voff, (int)soff, NT);
    return gl::pair64(v.x, v.y);
  }
  __device__ __forceinline__ void store(uint64_t x, uint32_t voff, uint32_t soff) const {
    V2 v;
    v.x = (uint32_t)x;
    v.y = (uint32_t)(x >> 32);
    __builtin_amdgcn_raw_buffer_store_b64(v, r, (int)voff, (int)soff, NT);
  }
};

// A pointer read from memory, known to point to global memory (a generic
// pointer's accesses also wait on LDS).
template <class T> __device__ __forceinline__ T *global_ptr(T *p) {
  return (T *)(__attribute__((address_space(1))) T *)(uint64_t)p;
}

// One launch for the first pass of all cosets of an LDE (a.coset_log):
// workgroup `wg` of `wgs` takes coset c and workgroup index `rest` of the
// coset's own wgs >> coset_log.  Workgroups go round-robin to the 8 XCDs, so
// the cosets of one index are put 8 apart: they run on one XCD at about the
// same time and read the same coefficients (4.51 -> 4.35 ms per 128 x 2^20
// blowup-4 LDE with the later passes in one launch each; ordinary loads
// instead of non-temporal ones made no difference).
__device__ __forceinline__ uint32_t coset_split(FastArgs &a, uint32_t wg, uint32_t wgs) {
  const uint32_t lb = a.coset_log, own = wgs >> lb;
  uint32_t c, rest;
  if (own % 8 == 0) {
    c = (wg >> 3) & ((1u << lb) - 1u);
    rest = ((wg >> (3 + lb)) << 3) | (wg & 7u);
  } else {
    c = wg & ((1u << lb) - 1u);
    rest = wg >> lb;
  }
  a.coset_exp = c << (32u - a.log_n - a.log_ext);
  a.out += (uint64_t)(a.coset_brev ? brev_bits(c, lb) : c) << a.log_n;
  return rest;
}

// Column addressing: one matrix (base + c * stride) for the standalone
// launches, or a per-column pointer table (CT) for ragged job groups; the
// table does not change during a launch, and for a uniform c its entry is a
// scalar load.
template <bool CT> __device__ __forceinline__ const uint64_t *in_col(const FastArgs &a, uint64_t c) {
  if constexpr (CT) return global_ptr((const uint64_t *)((const __attribute__((address_space(4))) uint64_t *)(uint64_t)a.cols)[2 * c]);
  else return a.in + c * a.stride_in;
}
template <bool CT> __device__ __forceinline__ uint64_t *out_col(const FastArgs &a, uint64_t c) {
  if constexpr (CT) return global_ptr((uint64_t *)((const __attribute__((address_space(4))) uint64_t *)(uint64_t)a.cols)[2 * c + 1]);
  else return a.out + c * a.stride_out;
}
static_assert(sizeof(ColPtrs) == 16 && offsetof(ColPtrs, in) == 0 && offsetof(ColPtrs, out) == 8, "");

// Addressing of a contiguous-pass tile: 4096 consecutive points of one column
// (position pos0 of column col), or (MC: single-pass transforms shorter than
// 4096) 2^(12-h) whole columns from col0 on.
template <int LH, bool MC> struct ContigTile {
  uint64_t col;
  uint32_t pos0, col0;
  __device__ __forceinline__ ContigTile(const FastArgs &a, uint32_t tile) {
    if constexpr (!MC) {
      const uint32_t sh = a.log_n - TILE_LOG;
      col = tile >> sh;
      pos0 = (tile & ((1u << sh) - 1u)) << TILE_LOG;
      col0 = 0;
    } else {
      col0 = tile << (12 - LH);
      col = 0;
      pos0 = 0;
    }
  }
  __device__ __forceinline__ uint32_t pos(uint32_t e) const {
    if constexpr (MC) return e & ((1u << LH) - 1u);
    else return pos0 + e;
  }
};

// Wave-region mappings of a 4096-point tile, used from level 1 on when a
// transform has three register levels.  Tile bits 10-11 are the wave index in
// the level-1 mapping (celem<LH, 1, 4> for every 9 <= LH <= 12), so each wave
// then owns the 1024 points (and LDS slots) w * 1024 + [0, 1024):
//   wl_run: thread t holds 16 consecutive points t * 16 + k (the last level's
//           2^(LH-8)-point runs, grouped by k's low bits);
//   wl_row: register i of lane l of wave w holds point w * 1024 + i * 64 + l
//           (coalesced: 64 consecutive points per register).
__device__ __forceinline__ uint32_t wl_run(uint32_t t, int k) { return (t << 4) + (uint32_t)k; }
__device__ __forceinline__ uint32_t wl_row(uint32_t t, int i) {
  return ((t >> 6) << 10) + ((uint32_t)i << 6) + (t & 63u);
}

// Orders one wave's LDS accesses across its lanes.  A wave's LDS operations
// execute in program order, so this only keeps the compiler from moving LDS
// loads and stores across it; no workgroup barrier is involved.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Loads a tile's 16 values per thread in the level-0 mapping (lanes on
// consecutive points), or (ROW) in the wl_row mapping.
template <int LH, bool MC, bool CT, bool ROW = false>
__device__ __forceinline__ void contig_load(const FastArgs &a, uint32_t tile, uint32_t t, uint64_t *x) {
  const ContigTile<LH, MC> ct(a, tile);
  if constexpr (!MC) {
    const Buf in(in_col<CT>(a, ct.col) + ct.pos0, TILE * 8);
    const uint32_t v = (ROW ? wl_row(t, 0) : celem<LH, 0, 4>(t, 0, 0)) * 8;
    constexpr uint32_t STEP = ROW ? 64 * 8 : 8u << (LH - 4);
#pragma unroll
    for (uint32_t i = 0; i < 16; ++i) x[i] = in.load(v + i * STEP % 4096, i * STEP / 4096 * 4096);
  } else {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const uint32_t e = celem<LH, 0, 4>(t, 0, i), c = ct.col0 + (e >> LH);
      x[i] = c < a.num_cols ? __builtin_nontemporal_load(in_col<CT>(a, c) + (e & ((1u << LH) - 1u))) : 0ull;
    }
  }
}

// Stores a tile's 16 values per thread from the level-0 mapping.
template <int LH, bool MC, bool CT>
__device__ __forceinline__ void contig_store(const FastArgs &a, const ContigTile<LH, MC> &ct, uint32_t t,
                                             const uint64_t *x) {
  if constexpr (!MC) {
    const Buf out(out_col<CT>(a, ct.col) + ct.pos0, TILE * 8);
    const uint32_t v = celem<LH, 0, 4>(t, 0, 0) * 8;
    constexpr uint32_t STEP = 8u << (LH - 4);
#pragma unroll
    for (uint32_t i = 0; i < 16; ++i) out.store(x[i], v + i * STEP % 4096, i * STEP / 4096 * 4096);
  } else {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const uint32_t e = celem<LH, 0, 4>(t, 0, i), c = ct.col0 + (e >> LH);
      if (c < a.num_cols) __builtin_nontemporal_store(x[i], out_col<CT>(a, c) + (e & ((1u << LH) - 1u)));
    }
  }
}

// LDS a pass needs: the padded tile plus a staged level-twist table.
constexpr uint32_t LDS_TW_LEN = 15u << 4;  // largest staged table (M = 256)
struct PassLds {
  uint64_t tile[LDS_PADDED];
  uint64_t tw[LDS_TW_LEN];
  uint64_t cf[16];  // coset part factors (LDE modes)
  uint64_t cr[16];  // coset factors of the strided level-0 groups (LDE modes)
};

// Runs tiles tile_begin, tile_begin + step, ... < tile_end of a contiguous
// pass.  Called by a whole workgroup; ends with a barrier.
template <int LH, bool INV, bool DIT, int MODE, bool MC, bool CT = false>
__device__ __forceinline__ void contig_run(const FastArgs &a, PassLds &sh, uint32_t tile_begin, uint32_t tile_end,
                                           uint32_t step) {
  constexpr int NL = LH > 8 ? 3 : 2;
  constexpr int A2 = NL == 3 ? LH - 8 : 4;  // width of the third level
  constexpr int G2 = 16 >> A2;              // third-level groups per thread
  constexpr int LL = NL - 1, AL = NL == 3 ? A2 : 4, GL = 16 >> AL;  // last level
  // WL: with three levels and no coset factors, the exchange between levels 1
  // and 2 stays inside each wave's own 1024 points (wl_run) and needs no
  // workgroup barrier.  b2n also loads in the wl_row mapping, so its
  // regrouping exchange is wave-local too (two barriers per tile instead of
  // four); n2b keeps its store in the level-0 mapping (three barriers), which
  // measured faster than wl_row stores.
  constexpr bool WL = NL == 3 && !MC && (MODE == MODE_NONE || MODE == MODE_NINV);
  uint64_t *lds = sh.tile;
  uint64_t *tw1 = sh.tw;
  const uint32_t t = threadIdx.x;
  // LDS slots of a thread's 16 points in the fixed mappings, as one base and
  // a constant stride, so that they are addressed with immediate offsets
  // instead of 16 loop-invariant address registers per mapping:
  // pidx(e0 + i 2^S) = pidx(e0) + i (2^S + 2^(S-4)) when S >= 4 and bits
  // S..S+3 of e0 are zero (level 0: S = h - 4; level 1: S = h - 8, so h = 12
  // only; wl_row: S = 6; wl_run: consecutive slots).
  uint64_t *const s0b = lds + pidx(celem<LH, 0, 4>(t, 0, 0));
  uint64_t *const s1b = lds + pidx(celem<LH, 1, 4>(t, 0, 0));
  uint64_t *const srunb = lds + pidx(wl_run(t, 0));
  uint64_t *const srowb = lds + pidx(wl_row(t, 0));
  auto s0 = [&](int i) -> uint64_t & { return s0b[i * ((1 << (LH - 4)) + (1 << (LH - 8)))]; };
  auto s1 = [&](int i) -> uint64_t & {
    if constexpr (LH >= 12) return s1b[i * ((1 << (LH - 8)) + (1 << (LH - 12)))];
    else return lds[pidx(celem<LH, 1, 4>(t, 0, i))];
  };
  auto srun = [&](int k) -> uint64_t & { return srunb[k]; };
  auto srow = [&](int i) -> uint64_t & { return srowb[i * 68]; };

  // level-0 twists: 15 per thread.  The plain n2b pass keeps them in
  // registers: read at each use they wait, in order, behind the prefetch of
  // the next tile (5-9% slower on 256 x 2^20).  b2n uses them last, when the
  // prefetch has landed, and the coset and multi-column forms would spill;
  // these read the (cache-resident) level table each time, which keeps 30
  // VGPRs free.
  const uint64_t *tw0 = lvl_table<LH, INV>(a.tab) + (t & ((1u << (LH - 4)) - 1u));
  constexpr bool TW_REGS = WL && !DIT && !CT;
  uint64_t twr[16];
  if constexpr (TW_REGS) {
#pragma unroll
    for (int i = 1; i < 16; ++i) twr[i] = tw0[(i - 1) << (LH - 4)];
  }
  // level-1 twists (at most 240 entries) in LDS
  if constexpr (NL == 3) stage_level_twists<LH - 4, INV>(tw1, a.tab);
  const uint32_t rp1 = t & ((1u << (LH - 8)) - 1u);
  // coset part factors: point i of the level-0 mapping is at tile position
  // pos(e_0) + i 2^(LH-4); the scaled index is that position, or its log_n-bit
  // reversal (DIT inputs, DIF outputs), whose part is brev4(i) 2^(log_n-LH)
  constexpr bool SC = MODE == MODE_LDE_IN || MODE == MODE_LDE_OUT;
  constexpr bool SC_BREV = (MODE == MODE_LDE_IN) == DIT;
  if constexpr (SC) {
    if (t < 16) {
      const uint32_t part = SC_BREV ? (brev_bits(t, 4) << (a.log_n - LH)) : (t << (LH - 4));
      sh.cf[t] = coset_part_factor<MODE>(a, part);
    }
  }

  // b2n with WL loads in the wl_row mapping, everything else in level 0's
  constexpr bool ROW_LOAD = WL && DIT;
  uint32_t tile = __builtin_amdgcn_readfirstlane(tile_begin);
  tile_end = __builtin_amdgcn_readfirstlane(tile_end);
  uint64_t pf[16];
  if (tile < tile_end) contig_load<LH, MC, CT, ROW_LOAD>(a, tile, t, pf);
  __syncthreads();  // tw1 and coset part factors staged

  for (; tile < tile_end; tile += step) {
    const ContigTile<LH, MC> ct(a, tile);
    uint64_t x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = pf[i];
    {
      const uint32_t next = tile + step;
      if (next < tile_end) contig_load<LH, MC, CT, ROW_LOAD>(a, next, t, pf);  // prefetch: in flight during this tile's math
    }
    uint64_t cfb = 0;  // coset factor of the thread's point 0 in this tile
    if constexpr (SC) {
      const uint32_t pos = ct.pos(celem<LH, 0, 4>(t, 0, 0));
      cfb = coset_scale_pow<MODE>(a, SC_BREV ? brev_bits(pos, a.log_n) : pos);
    }
    if constexpr (MODE == MODE_LDE_IN) coset_twist<gl::ANY>(x, cfb, sh.cf);

    // Values between levels are any u64; the pass's last operation on each
    // makes it canonical (this pass writes the caller's outputs in n2b, and in
    // single-pass b2n calls).
    constexpr bool SCALE_OUT = MODE == MODE_NINV || MODE == MODE_LDE_OUT;
    constexpr gl::Reduce LAST = SCALE_OUT ? gl::ANY : gl::CANON;
    auto scale_out = [&](uint64_t *v) {
      if constexpr (MODE == MODE_NINV) gl::mul_each<0, 16, gl::CANON>(v, [&](int) { return a.n_inv; });
      if constexpr (MODE == MODE_LDE_OUT) coset_twist<gl::CANON>(v, cfb, sh.cf);
    };
    auto tw0_at = [&](int i) { return TW_REGS ? twr[i] : tw0[(i - 1) << (LH - 4)]; };
    if constexpr (!DIT) {
      gl::dft_lazy<4, INV, false, gl::ANY>(x);
      gl::mul_each<1, 15, gl::ANY>(x, tw0_at);
#pragma unroll
      for (int i = 0; i < 16; ++i) s0(i) = x[i];
      __syncthreads();
#pragma unroll
      for (int i = 0; i < 16; ++i) x[i] = s1(i);
      if constexpr (WL) {
        gl::dft_lazy<4, INV, false, gl::ANY>(x);
        level_twist_lds<LH - 4, gl::ANY>(x, tw1, rp1);
        // each thread rewrites the slots it read, inside its wave's region
#pragma unroll
        for (int i = 0; i < 16; ++i) s1(i) = x[i];
        wave_lds_sync();
#pragma unroll
        for (int k = 0; k < 16; ++k) x[k] = srun(k);
        gl::dft_lazy<A2, INV, false, LAST>(x);
#pragma unroll
        for (int k = 0; k < 16; ++k) srun(k) = x[k];
        __syncthreads();  // the level-0 mapping crosses waves
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] = s0(i);
        scale_out(x);
        contig_store<LH, MC, CT>(a, ct, t, x);
      } else if constexpr (NL == 3) {
        gl::dft_lazy<4, INV, false, gl::ANY>(x);
        level_twist_lds<LH - 4, gl::ANY>(x, tw1, rp1);
#pragma unroll
        for (int i = 0; i < 16; ++i) s1(i) = x[i];
        __syncthreads();
#pragma unroll
        for (int g = 0; g < G2; ++g)
#pragma unroll
          for (int i = 0; i < (1 << A2); ++i) x[g * (1 << A2) + i] = lds[pidx(celem<LH, 2, A2>(t, g, i))];
        gl::dft_lazy<A2, INV, false, LAST>(x);
      } else {
        gl::dft_lazy<4, INV, false, LAST>(x);
      }
      // regroup the last level's runs into the coalesced level-0 mapping
      // through LDS (each thread rewrites the slots it read, so no barrier
      // is needed before the write), then store
      if constexpr (!WL) {
#pragma unroll
        for (int g = 0; g < GL; ++g)
#pragma unroll
          for (int i = 0; i < (1 << AL); ++i) lds[pidx(celem<LH, LL, AL>(t, g, i))] = x[g * (1 << AL) + i];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] = s0(i);
        scale_out(x);
        contig_store<LH, MC, CT>(a, ct, t, x);
      }
    } else {
      int32_t e[16];
      e[0] = 0;  // point 0 of a level takes no twist
      if constexpr (WL) {
        // loaded in the wl_row mapping: regroup into runs inside the wave's region
#pragma unroll
        for (int i = 0; i < 16; ++i) srow(i) = x[i];
        wave_lds_sync();
#pragma unroll
        for (int k = 0; k < 16; ++k) x[k] = srun(k);
        gl::dft_lazy<A2, INV, true, gl::ANY>(x);
#pragma unroll
        for (int k = 0; k < 16; ++k) srun(k) = x[k];
        wave_lds_sync();
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] = s1(i);
        level_twist_lds<LH - 4, gl::LAZY>(x, tw1, rp1, e);
        gl::dft_lazy<4, INV, true, gl::ANY, true>(x, e);
      } else {
        // regroup the coalesced load into the last level's runs through LDS
#pragma unroll
        for (int i = 0; i < 16; ++i) s0(i) = x[i];
        __syncthreads();
#pragma unroll
        for (int g = 0; g < GL; ++g)
#pragma unroll
          for (int i = 0; i < (1 << AL); ++i) x[g * (1 << AL) + i] = lds[pidx(celem<LH, LL, AL>(t, g, i))];
        if constexpr (NL == 3) {
          gl::dft_lazy<A2, INV, true, gl::ANY>(x);
#pragma unroll
          for (int g = 0; g < G2; ++g)
#pragma unroll
            for (int i = 0; i < (1 << A2); ++i) lds[pidx(celem<LH, 2, A2>(t, g, i))] = x[g * (1 << A2) + i];
          __syncthreads();
#pragma unroll
          for (int i = 0; i < 16; ++i) x[i] = s1(i);
          level_twist_lds<LH - 4, gl::LAZY>(x, tw1, rp1, e);
          gl::dft_lazy<4, INV, true, gl::ANY, true>(x, e);
        } else {
          gl::dft_lazy<4, INV, true, gl::ANY>(x);
        }
      }
      // each thread rewrites the slots it read; the level-0 mapping crosses waves
#pragma unroll
      for (int i = 0; i < 16; ++i) s1(i) = x[i];
      __syncthreads();
#pragma unroll
      for (int i = 0; i < 16; ++i) x[i] = s0(i);
      gl::mul_each<1, 15, gl::LAZY>(x, tw0_at, e);
      gl::dft_lazy<4, INV, true, LAST, true>(x, e);
      scale_out(x);
      contig_store<LH, MC, CT>(a, ct, t, x);
    }
    __syncthreads();  // LDS is reused by the next tile
  }
}

// -------------------------------------------------------------------------
// strided<h>

// Runs (column, block) pairs [p_begin, p_end) at r-range rho of a strided
// pass.  Called by a whole workgroup; ends with a barrier.
template <int LH, bool INV, bool DIT, int MODE, bool CT = false>
__device__ __forceinline__ void strided_run(const FastArgs &a, PassLds &sh, uint32_t rho, uint64_t p_begin,
                                            uint64_t p_end) {
  constexpr int LT = 12 - LH;         // log2 sub-DFTs (consecutive r) per tile
  constexpr int T = 1 << LT;
  constexpr int NL = LH > 4 ? 2 : 1;
  constexpr int A1 = NL == 2 ? LH - 4 : 4;  // second level width
  constexpr int G1 = 16 >> A1;
  constexpr int LS0 = LH - 4;               // level-0 stride (log2)
  uint64_t *lds = sh.tile;
  uint64_t *tw0 = sh.tw;
  const uint32_t t = threadIdx.x;
  const uint32_t log_r = a.log_N - LH;
  rho = __builtin_amdgcn_readfirstlane(rho);
  const uint32_t r0 = rho << LT;

  // level-0 mapping: q = t % T, rp = t / T, j = i * 2^LS0 + rp
  const uint32_t q0 = t & (T - 1u), rp0 = t >> LT;
  // last-level mapping (level 1, or level 0 when h = 4): q = gi % T, b = gi / T, j = b * 2^A1 + i
  auto lastj = [&](int g, int i) -> uint32_t {
    if constexpr (NL == 2) return (((t + NT * (uint32_t)g) >> LT) << A1) + (uint32_t)i;
    else return ((uint32_t)i << LS0) + rp0;
  };
  auto lastq = [&](int g) -> uint32_t {
    if constexpr (NL == 2) return (t + NT * (uint32_t)g) & (T - 1u);
    else return q0;
  };
  // Element offsets from the block base (r0 included).  Level-0 mapping:
  // base0 + i * step0; last-level mapping: basel(g) + i * stepl.
  const uint32_t log_step0 = LS0 + log_r, log_stepl = NL == 2 ? log_r : log_step0;
  const uint64_t base0 = ((uint64_t)rp0 << log_r) + q0;
  auto basel = [&](int g) -> uint64_t {
    if constexpr (NL == 2) return ((uint64_t)lastj(g, 0) << log_r) + lastq(g);
    else return base0;
  };

  // Coset scaling (this is the top pass: one block per column).  The point of
  // level-0 slot i sits at column position i 2^(log_N - 4) + rp 2^log_r + r
  // (r = r0 + q), and its factor s^(+-pos) splits into three parts, each
  // folded where it costs no extra multiply per point: s^(+-r) is common to
  // the whole sub-DFT at r and joins its pass twist; s^(+-rp 2^log_r) is
  // common to one level-0 DFT and joins that level's twists (plus point 0);
  // s^(+-i 2^(log_N - 4)) multiplies slot i (n2b inputs, b2n outputs) from a
  // 16-entry LDS table.  n^-1 of the inverse coset transform joins the pass
  // twist.
  constexpr bool SC = MODE == MODE_LDE_IN || MODE == MODE_LDE_OUT;
  if constexpr (NL == 2) {
    if constexpr (SC) stage_level_twists_coset<LH, INV, MODE>(tw0, sh.cr, a, log_r);
    else stage_level_twists<LH, INV>(tw0, a.tab);
  }
  if constexpr (SC) {
    if (t < 16) sh.cf[t] = coset_scale_pow<MODE>(a, t << (a.log_N - 4));
  }

  // pass twist omega_N^(r brev_h(j)) in the last-level mapping, with n^-1 and
  // the coset factor of r folded in.  T <= 256, so r = r0 + q is the same for
  // all of a thread's values, and their j differ in four bits: register k =
  // (g, i) has bits i at the bottom of j and bits g at its top.  So the 16
  // twists are the thread's own power times the subset products of four
  // powers omega_N^(r 2^m): five table powers and 15 products a workgroup
  // instead of 16 powers and up to 48 products.
  uint64_t pt[16];
  {
    const uint32_t r = r0 + lastq(0);
    auto power = [&](uint32_t k) {  // omega_N^(+-r k)
      const uint32_t e = (r * k) << (32u - a.log_N);
      return pow_w(a.tab, INV ? 0u - e : e);
    };
    pt[0] = power(brev_bits(lastj(0, 0), LH));
    if constexpr (MODE == MODE_NINV || MODE == MODE_LDE_OUT) pt[0] = gl::mul(pt[0], a.n_inv);
    if constexpr (SC) pt[0] = gl::mul(pt[0], coset_scale_pow<MODE>(a, r));
    // register bit m is bit m of j (m < A1: i; h = 4: the slot's bit m + LS0)
    // or, for g, bit h - 4 + m
    gl::unroll<4>([&](auto m) {
      constexpr int B = decltype(m)::value, N = 1 << B;
      constexpr int JBIT = NL == 2 ? (B < A1 ? B : LH - 4 + B) : LS0 + B;
      const uint64_t f = power(1u << (LH - 1 - JBIT));
      const uint64_t fs[4] = {f, f, f, f};
      gl::unroll<(N + 3) / 4>([&](auto c) {
        constexpr int C = 4 * decltype(c)::value, R = N < 4 ? N : 4;
        gl::mul_row<R, gl::ANY>(pt + N + C, pt + C, fs);
      });
    });
  }

  const uint32_t blocks_per_col_log = a.log_n - a.log_N;
  // offset of pair p's r-range inside its column
  auto pair_pos = [&](uint64_t p) -> uint64_t {
    return ((p & ((1ull << blocks_per_col_log) - 1ull)) << a.log_N) + r0;
  };
  // One pair's 16 values in the level-0 (DIF loads, DIT stores) or last-level
  // mapping.  Blocks of up to 2^28 points (2 GiB) are addressed through a
  // buffer descriptor, longer ones, whose offsets pass 32 bits, with pointers.
  const bool buffered = a.log_N <= 28;
  const uint32_t block_bytes = buffered ? (uint32_t)(((1ull << a.log_N) - r0) * 8) : 0u;
  auto load = [&](uint64_t p, uint64_t *v) {
    const uint64_t *in = in_col<CT>(a, p >> blocks_per_col_log) + pair_pos(p);
    if (buffered) {
      const Buf b(in, block_bytes);
      if constexpr (!DIT) {
#pragma unroll
        for (uint32_t k = 0; k < 16; ++k) v[k] = b.load((uint32_t)base0 * 8, k << (log_step0 + 3));
      } else {
#pragma unroll
        for (int g = 0; g < G1; ++g)
#pragma unroll
          for (uint32_t i = 0; i < (1u << A1); ++i)
            v[g * (1 << A1) + i] = b.load((uint32_t)basel(g) * 8, i << (log_stepl + 3));
      }
    } else if constexpr (!DIT) {
#pragma unroll
      for (uint64_t k = 0; k < 16; ++k) v[k] = __builtin_nontemporal_load(in + base0 + (k << log_step0));
    } else {
#pragma unroll
      for (int g = 0; g < G1; ++g)
#pragma unroll
        for (uint64_t i = 0; i < (1u << A1); ++i)
          v[g * (1 << A1) + i] = __builtin_nontemporal_load(in + basel(g) + (i << log_stepl));
    }
  };
  auto store = [&](uint64_t p, const uint64_t *v) {
    uint64_t *out = out_col<CT>(a, p >> blocks_per_col_log) + pair_pos(p);
    if (buffered) {
      const Buf b(out, block_bytes);
      if constexpr (DIT) {
#pragma unroll
        for (uint32_t k = 0; k < 16; ++k) b.store(v[k], (uint32_t)base0 * 8, k << (log_step0 + 3));
      } else {
#pragma unroll
        for (int g = 0; g < G1; ++g)
#pragma unroll
          for (uint32_t i = 0; i < (1u << A1); ++i)
            b.store(v[g * (1 << A1) + i], (uint32_t)basel(g) * 8, i << (log_stepl + 3));
      }
    } else if constexpr (DIT) {
#pragma unroll
      for (uint64_t k = 0; k < 16; ++k) __builtin_nontemporal_store(v[k], out + base0 + (k << log_step0));
    } else {
#pragma unroll
      for (int g = 0; g < G1; ++g)
#pragma unroll
        for (uint64_t i = 0; i < (1u << A1); ++i)
          __builtin_nontemporal_store(v[g * (1 << A1) + i], out + basel(g) + (i << log_stepl));
    }
  };

  p_begin = uniform64(p_begin);
  p_end = uniform64(p_end);
  constexpr bool PREFETCH = !CT;
  uint64_t pf[16];
  if constexpr (PREFETCH) {
    if (p_begin < p_end) load(p_begin, pf);
  }
  __syncthreads();  // tw0 and coset factors staged
  for (uint64_t p = p_begin; p < p_end; ++p) {
    uint64_t x[16];
    if constexpr (PREFETCH) {
#pragma unroll
      for (int i = 0; i < 16; ++i) x[i] = pf[i];
      if (p + 1 < p_end) load(p + 1, pf);  // in flight during this pair's math
    } else {
      load(p, x);
    }
    if constexpr (!DIT) {
      if constexpr (MODE == MODE_LDE_IN) gl::mul_each<1, 15, gl::ANY, true>(x, [&](int i) { return sh.cf[i]; });
      gl::dft_lazy<4, INV, false, gl::ANY>(x);
      if constexpr (NL == 2) {
        level_twist_lds<LH, gl::ANY>(x, tw0, rp0);
        if constexpr (SC) x[0] = gl::mul(x[0], sh.cr[rp0]);
        // LDS row-major by j: element (q, j) at j * T + q
#pragma unroll
        for (int i = 0; i < 16; ++i) lds[((((uint32_t)i << LS0) + rp0) << LT) + q0] = x[i];
        __syncthreads();
#pragma unroll
        for (int g = 0; g < G1; ++g)
#pragma unroll
          for (int i = 0; i < (1 << A1); ++i) x[g * (1 << A1) + i] = lds[(lastj(g, i) << LT) + lastq(g)];
        __syncthreads();  // the next iteration rewrites LDS
        gl::dft_lazy<A1, INV, false, gl::ANY>(x);
      }
      // a later pass reads these, so any u64 will do
      gl::mul_each<0, 16, gl::ANY>(x, [&](int k) { return pt[k]; });
      store(p, x);
    } else {
      // outputs are canonical: this may be the call's last pass
      constexpr gl::Reduce LAST = MODE == MODE_LDE_OUT ? gl::ANY : gl::CANON;
      int32_t e[16];
      gl::mul_each<0, 16, gl::LAZY>(x, [&](int k) { return pt[k]; }, e);
      if constexpr (NL == 2) {
        gl::dft_lazy<A1, INV, true, gl::ANY, true>(x, e);
#pragma unroll
        for (int g = 0; g < G1; ++g)
#pragma unroll
          for (int i = 0; i < (1 << A1); ++i) lds[(lastj(g, i) << LT) + lastq(g)] = x[g * (1 << A1) + i];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] = lds[((((uint32_t)i << LS0) + rp0) << LT) + q0];
        __syncthreads();
        level_twist_lds<LH, gl::LAZY>(x, tw0, rp0, e);
        e[0] = 0;
        if constexpr (SC) x[0] = gl::mul(x[0], sh.cr[rp0]);
      }
      gl::dft_lazy<4, INV, true, LAST, true>(x, e);
      if constexpr (MODE == MODE_LDE_OUT) {
        x[0] = gl::canon(x[0]);
        gl::mul_each<1, 15, gl::CANON, true>(x, [&](int i) { return sh.cf[i]; });
      }
      store(p, x);
    }
  }
  __syncthreads();  // LDS (tile and staged twists) is reused by the caller's next unit
}

}  // namespace pass
}  // namespace bc
