// Cells, cubes and boxes shared by the sampling kernels (nsfps_runs.hip,
// nsfps_small.hip).
#pragma once

#include "nsfps_device.h"

#pragma clang fp contract(off)

namespace nsfps {

__device__ __forceinline__ uint32_t pack_cell(uint32_t x, uint32_t y, uint32_t z) {
  return x | (y << 10) | (z << 20);
}

// Squared distance from q to the nearest point of the box lo..hi, in the
// operation order of sqdist.  Rounding is monotonic, so it never exceeds
// sqdist of q and a point in the box: when it is >= every distance of the
// box's points, q lowers none of them (a point is lowered by a strictly
// smaller distance).  NaN when q has a NaN coordinate.
__device__ __forceinline__ float box_bound(float qx, float qy, float qz, float lx, float ly,
                                           float lz, float hx, float hy, float hz) {
  const float qv[3] = {qx, qy, qz}, lv[3] = {lx, ly, lz}, hv[3] = {hx, hy, hz};
  float g[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float below = lv[a] - qv[a], above = qv[a] - hv[a];
    const float gg = below > above ? below : above;
    g[a] = gg > 0.f ? gg : 0.f;
  }
  return (g[0] * g[0] + g[1] * g[1]) + g[2] * g[2];
}

// Cells packed 11 bits per axis (x | y << 11 | z << 22): bits 10 and 21 stay
// clear and act as guards, so lo <= c <= hi on all three axes takes two
// subtractions.  cg = pack11(c) | kGuards, c11 = pack11(c), hig = pack11(hi) |
// kGuards.  Per axis, cg - lo keeps its guard bit (or, for z, does not borrow)
// exactly when c >= lo, and hig - c11 likewise when c <= hi.
constexpr uint32_t kGuards = (1u << 10) | (1u << 21);

__device__ __forceinline__ uint32_t pack11(uint32_t c10) {
  return (c10 & 1023u) | (((c10 >> 10) & 1023u) << 11) | ((c10 >> 20) << 22);
}

__device__ __forceinline__ uint32_t in_box11(uint32_t cg, uint32_t c11, uint32_t lo,
                                             uint32_t hig) {
  uint32_t t1, t2;
  const bool b1 = __builtin_usub_overflow(cg, lo, &t1);
  const bool b2 = __builtin_usub_overflow(hig, c11, &t2);
  return (uint32_t)(((t1 & t2 & kGuards) == kGuards) & !b1 & !b2);
}

// Cube corners of a sample: cell qc, half-widths h, clipped to the grid.
__device__ __forceinline__ void cube_corners(uint32_t qc, uint32_t h, uint32_t b0, uint32_t b1,
                                             uint32_t b2, uint32_t &lo_c, uint32_t &hi_c) {
  const uint32_t qcx = qc & 1023u, qcy = (qc >> 10) & 1023u, qcz = qc >> 20;
  const uint32_t g0 = h & 1023u, g1 = (h >> 10) & 1023u, g2 = h >> 20;
  lo_c = pack_cell(qcx > g0 ? qcx - g0 : 0u, qcy > g1 ? qcy - g1 : 0u, qcz > g2 ? qcz - g2 : 0u);
  hi_c = pack_cell(min(qcx + g0, b0 - 1), min(qcy + g1, b1 - 1), min(qcz + g2, b2 - 1));
}

// Cube half-width of a sample with distance D on axis a (src/yuezu_fps.cpp:
// 564-570), clipped to blocks - 1 (at or beyond the grid it selects the same
// cells).  The half-width is monotone in D: below the last of the range's
// thresholds it is the number of thresholds <= D (no square root or
// division); above it, the reference's arithmetic (correctly rounded sqrtf
// and division, as on the host that derived the thresholds).
__device__ __forceinline__ uint32_t half_axis(const RangeDev &r, int a, float D) {
  uint32_t h = 0;
#pragma unroll
  for (uint32_t k = 0; k < kCubeThr; ++k) h += D >= r.cube_thr[a][k] ? 1u : 0u;
  if (h == kCubeThr) h = min((uint32_t)cube_half(D, r.bsize[a], r.blocks[a]), r.blocks[a] - 1);
  return h;
}

// The three half-widths packed 10 bits per axis.
__device__ __forceinline__ uint32_t packed_halves(const RangeDev &r, float D) {
  return half_axis(r, 0, D) | (half_axis(r, 1, D) << 10) | (half_axis(r, 2, D) << 20);
}

// The first three thresholds of every axis, in scalar registers.  Below the
// third of every axis (half-widths of at most 2: the common case once cubes
// are small) the packed half-widths take two comparisons per axis.
struct SmallHalves {
  float t[3][3];
  __device__ __forceinline__ explicit SmallHalves(const RangeDev &r) {
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int k = 0; k < 3; ++k) t[a][k] = r.cube_thr[a][k];
  }
  __device__ __forceinline__ bool covers(float D) const {
    return D < t[0][2] && D < t[1][2] && D < t[2][2];
  }
  __device__ __forceinline__ uint32_t packed(float D) const {
    uint32_t h = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a)
      h |= ((D >= t[a][0] ? 1u : 0u) + (D >= t[a][1] ? 1u : 0u)) << (10 * a);
    return h;
  }
};

// Cube of a sample at a point of cell c11 (pack11) with distance D: corners
// {pack11(lo), pack11(hi) | guards}.
__device__ __forceinline__ uint2 sample_cube(const RangeDev &r, uint32_t c11, float D) {
  const SmallHalves sh(r);
  uint32_t h;
  if (sh.covers(D)) h = sh.packed(D);
  else h = packed_halves(r, D);
  const uint32_t cc = (c11 & 1023u) | (((c11 >> 11) & 1023u) << 10) | ((c11 >> 22) << 20);
  uint32_t lo_c, hi_c;
  cube_corners(cc, h, r.blocks[0], r.blocks[1], r.blocks[2], lo_c, hi_c);
  return make_uint2(pack11(lo_c), pack11(hi_c) | kGuards);
}

// The bits of v at the set positions of mask, lowest first.
__device__ __forceinline__ uint32_t deposit_bits(uint32_t v, uint32_t mask) {
  uint32_t r = 0, k = 0;
  for (uint32_t m = mask; m; m &= m - 1, ++k) r |= ((v >> k) & 1u) ? m & (0u - m) : 0u;
  return r;
}

// The Morton code of a cell (pack11) from the code bits of each axis, and a
// cell of its bucket inside a cube: with shared buckets a sample updates
// every point of every bucket of its cube's cells (src/yuezu_fps.cpp:413,
// 573-597).
__device__ inline bool bucket_in_cube(const RangeDev &r, uint32_t c11, uint2 cube) {
  const uint32_t own = deposit_bits(c11 & 1023u, r.cmask[0]) |
                       deposit_bits((c11 >> 11) & 1023u, r.cmask[1]) |
                       deposit_bits(c11 >> 22, r.cmask[2]);
  for (uint64_t code = own % r.T; code < (1ull << r.cbits); code += r.T) {
    const uint32_t x = extract_bits((uint32_t)code, r.cmask[0]);
    const uint32_t y = extract_bits((uint32_t)code, r.cmask[1]);
    const uint32_t z = extract_bits((uint32_t)code, r.cmask[2]);
    if (x >= r.blocks[0] || y >= r.blocks[1] || z >= r.blocks[2]) continue;
    const uint32_t a = x | (y << 11) | (z << 22);
    if (in_box11(a | kGuards, a, cube.x, cube.y)) return true;
  }
  return false;
}

}  // namespace nsfps
