// Standalone launches of the NTT pass kernels (one kernel per pass); the
// pass bodies and their math are in ntt_passes.hpp.
#include "ntt_passes.hpp"

#include <mutex>

namespace bc {
namespace {
using namespace pass;

// Register bounds: three workgroups per CU for the n2b variants and the
// 12-bit b2n ones, two for the shorter b2n ones, some of which need more (up to
// 204 VGPRs).  The 12-bit kernels take 150-168 VGPRs without spills; n2b ones
// of 10 and 11 bits spill up to 6 dwords.  Four per CU spills 18-20 dwords in
// the 12-bit kernels and ran 4-5% slower.
template <int LH, bool INV, bool DIT, int MODE, bool MC>
__global__ __launch_bounds__(NT, DIT && LH != 12 ? 2 : 3) void
    ntt_contig_kernel(FastArgs a) {
  __shared__ PassLds sh;
  uint32_t wg = blockIdx.x, wgs = gridDim.x;
  if constexpr (MODE == MODE_LDE_IN && !MC) {
    if (a.coset_log) {
      wg = coset_split(a, wg, wgs);
      wgs >>= a.coset_log;
    }
  }
  contig_run<LH, INV, DIT, MODE, MC>(a, sh, wg, a.tiles, wgs);
}

// No form spills VGPRs.  n2b h = 7 and 8 take 155-166 and are bounded to three
// workgroups per CU (at two the compiler takes more: 5-6% slower on 256 x
// 2^20).  The others are bounded to two: h = 5 and 6 and the inverse coset forms
// need 171-196 and run two, plain h = 4 (139-147) and plain b2n h = 7 and 8 (167
// and 163) run three under that bound as well.
template <int LH, bool INV, bool DIT, int MODE>
__global__ __launch_bounds__(NT, LH >= 7 && !DIT ? 3 : 2) void ntt_strided_kernel(FastArgs a) {
  __shared__ PassLds sh;
  const uint64_t total = (uint64_t)a.num_cols << (a.log_n - a.log_N);
  const uint64_t p_begin = (uint64_t)blockIdx.y * a.blocks_per_wg;
  const uint64_t p_end = p_begin + a.blocks_per_wg < total ? p_begin + a.blocks_per_wg : total;
  uint32_t rho = blockIdx.x;
  if constexpr (MODE == MODE_LDE_IN) {
    if (a.coset_log) rho = coset_split(a, rho, gridDim.x);
  }
  strided_run<LH, INV, DIT, MODE>(a, sh, rho, p_begin, p_end);
}

// -------------------------------------------------------------------------
// launch dispatch (only the (direction, mode) pairs the planner can ask for)

template <int LH, bool INV, bool DIT, bool MC>
hipError_t contig_mode(const FastArgs &a, int mode, dim3 grid, hipStream_t s) {
  switch (mode) {
  case MODE_NONE: ntt_contig_kernel<LH, INV, DIT, MODE_NONE, MC><<<grid, NT, 0, s>>>(a); break;
  case MODE_NINV: ntt_contig_kernel<LH, INV, DIT, MODE_NINV, MC><<<grid, NT, 0, s>>>(a); break;
  case MODE_LDE_IN: ntt_contig_kernel<LH, INV, DIT, MODE_LDE_IN, MC><<<grid, NT, 0, s>>>(a); break;
  case MODE_LDE_OUT: ntt_contig_kernel<LH, INV, DIT, MODE_LDE_OUT, MC><<<grid, NT, 0, s>>>(a); break;
  default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <int LH, bool MC>
hipError_t contig_dir(const FastArgs &a, bool inv, bool dit, int mode, dim3 grid, hipStream_t s) {
  // forward transforms never scale outputs; inverse ones never scale inputs
  if (inv ? mode == MODE_LDE_IN : (mode == MODE_NINV || mode == MODE_LDE_OUT)) return hipErrorInvalidValue;
  if (inv) return dit ? contig_mode<LH, true, true, MC>(a, mode, grid, s) : contig_mode<LH, true, false, MC>(a, mode, grid, s);
  return dit ? contig_mode<LH, false, true, MC>(a, mode, grid, s) : contig_mode<LH, false, false, MC>(a, mode, grid, s);
}

template <int LH, bool INV, bool DIT>
hipError_t strided_mode(const FastArgs &a, int mode, dim3 grid, hipStream_t s) {
  switch (mode) {
  case MODE_NONE: ntt_strided_kernel<LH, INV, DIT, MODE_NONE><<<grid, NT, 0, s>>>(a); break;
  case MODE_NINV:
    if constexpr (INV) { ntt_strided_kernel<LH, INV, DIT, MODE_NINV><<<grid, NT, 0, s>>>(a); break; }
    return hipErrorInvalidValue;
  case MODE_LDE_IN:
    if constexpr (!INV && !DIT) { ntt_strided_kernel<LH, INV, DIT, MODE_LDE_IN><<<grid, NT, 0, s>>>(a); break; }
    return hipErrorInvalidValue;
  case MODE_LDE_OUT:
    if constexpr (INV && DIT) { ntt_strided_kernel<LH, INV, DIT, MODE_LDE_OUT><<<grid, NT, 0, s>>>(a); break; }
    return hipErrorInvalidValue;
  default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <int LH>
hipError_t strided_dir(const FastArgs &a, bool inv, bool dit, int mode, dim3 grid, hipStream_t s) {
  if (inv) return dit ? strided_mode<LH, true, true>(a, mode, grid, s) : strided_mode<LH, true, false>(a, mode, grid, s);
  return dit ? strided_mode<LH, false, true>(a, mode, grid, s) : strided_mode<LH, false, false>(a, mode, grid, s);
}

// Default grid of the contiguous pass: eight whole rounds of resident
// workgroups.  The tile loop is grid-strided, and a SIMD with three waves
// issues from them unevenly (two share an issue slot that the third has to
// itself), so the work has to be handed out in several rounds: two rounds
// were 3-8% slower on 256 x 2^20, a part-filled last round 4%.
// Queried once per device and direction: the n2b and b2n 12-bit kernels may
// differ in register use and so in workgroups per CU.
constexpr int MAX_DEVICES = 64;
std::mutex g_grid_mu;
uint32_t g_grid[MAX_DEVICES][2] = {};

uint32_t default_contig_grid(bool dit) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return 6144;
  std::lock_guard<std::mutex> lk(g_grid_mu);
  uint32_t &g = g_grid[dev][dit ? 1 : 0];
  if (!g) {
    int cus = 0, per_cu = 0;
    const bool ok =
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
        (dit ? hipOccupancyMaxActiveBlocksPerMultiprocessor(
                   &per_cu, ntt_contig_kernel<12, false, true, MODE_NONE, false>, NT, 0)
             : hipOccupancyMaxActiveBlocksPerMultiprocessor(
                   &per_cu, ntt_contig_kernel<12, false, false, MODE_NONE, false>, NT, 0)) == hipSuccess &&
        cus > 0 && per_cu > 0;
    g = ok ? (uint32_t)(8 * cus * per_cu) : 6144u;
  }
  return g;
}

}  // namespace

hipError_t launch_contig(const FastArgs &a, int log_h, bool inverse, bool dit, int mode, uint32_t max_wgs,
                         hipStream_t stream) {
  if (a.tiles == 0) return hipSuccess;
  if (max_wgs == 0) max_wgs = default_contig_grid(dit);
  uint32_t wgs = a.tiles < max_wgs ? a.tiles : max_wgs;
  if (a.coset_log) {  // the cap is for all cosets together
    const uint32_t cap = (max_wgs >> a.coset_log) > 8 ? max_wgs >> a.coset_log : 8;
    wgs = (a.tiles < cap ? a.tiles : cap) << a.coset_log;
  }
  const dim3 grid(wgs);
  if (a.log_n < TILE_LOG) {  // single pass over whole columns, several per tile
    switch (log_h) {
    case 8: return contig_dir<8, true>(a, inverse, dit, mode, grid, stream);
    case 9: return contig_dir<9, true>(a, inverse, dit, mode, grid, stream);
    case 10: return contig_dir<10, true>(a, inverse, dit, mode, grid, stream);
    case 11: return contig_dir<11, true>(a, inverse, dit, mode, grid, stream);
    default: return hipErrorInvalidValue;
    }
  }
  switch (log_h) {
  case 9: return contig_dir<9, false>(a, inverse, dit, mode, grid, stream);
  case 10: return contig_dir<10, false>(a, inverse, dit, mode, grid, stream);
  case 11: return contig_dir<11, false>(a, inverse, dit, mode, grid, stream);
  case 12: return contig_dir<12, false>(a, inverse, dit, mode, grid, stream);
  default: return hipErrorInvalidValue;
  }
}

hipError_t launch_strided(const FastArgs &a, int log_h, bool inverse, bool dit, int mode, uint32_t positions,
                          uint32_t groups, hipStream_t stream) {
  if (positions == 0 || groups == 0) return hipSuccess;
  if (groups > 65535) return hipErrorInvalidConfiguration;
  const dim3 grid(positions, groups);
  switch (log_h) {
  case 4: return strided_dir<4>(a, inverse, dit, mode, grid, stream);
  case 5: return strided_dir<5>(a, inverse, dit, mode, grid, stream);
  case 6: return strided_dir<6>(a, inverse, dit, mode, grid, stream);
  case 7: return strided_dir<7>(a, inverse, dit, mode, grid, stream);
  case 8: return strided_dir<8>(a, inverse, dit, mode, grid, stream);
  default: return hipErrorInvalidValue;
  }
}

}  // namespace bc
