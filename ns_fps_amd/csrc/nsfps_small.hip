// Clouds of at most kSmallMaxPoints points (gfx950): one workgroup per cloud
// sorts it (k_small_sort) and one samples it from start to end
// (k_small_sample), every point in registers and no pass over memory between
// samples (the kernels of 16 points a thread, above 8,192, keep some of them
// in scratch memory: 128 registers a thread are too few, and the compiler
// spills 100 of the sort's and 36 of the sampling's).
//
// The sampling goes in rounds.  Let B be a threshold that leaves at most
// kSmallList points whose keys (min-distance, then lower logical rank) are at
// or above it, and call two of them in conflict when their squared distance
// is below the larger of their min-distances: only then can either lower the
// other.  A listed point that conflicts with none of a larger key is a sample
// with the key it has: every point of a larger key is listed, those not
// sampled yet are too far to lower it, and those sampled have been applied.
// Its cube (src/yuezu_fps.cpp:560-597) may be applied to every point at once,
// since a point of a larger key that it could lower would be in conflict with
// it.  The largest key never has a conflict above it, so each round samples
// at least one point.  The samples' order is the order of their keys; the
// sampling ends when m of them lie above every key left, or only points at
// distance 0 are left (src/yuezu_fps.cpp:705-706), and one sort orders them.
// A CPU model of the rounds: 18 for 256 of 1,024 points, 33 for 1,000 of the
// 10,000-point quickstart, 63 for 4,096 of a 16,384-point cloud.
//
// Against the general engine's launches per round (build, update, gather and
// run kernels), per call on one MI355X, device-resident: 1,024 points -> 256
// 269 -> 136 us, 8,192 -> 1,024 of a cube 634 -> 427, 32 clouds of 1,024 -> 512
// 433 -> 190 us, 64 clouds of 16,384 -> 4,096 1,809 -> 1,370 us; the
// quickstart's 10,000 -> 1,000 hardly gains (639 -> 627).  Tie-heavy clouds
// sampled to a half lose: an 8,192-point lattice -> 4,096 2.2 -> 2.8 ms.
#include <hip/hip_runtime.h>

#include <float.h>

#include "nsfps_box.h"
#include "nsfps_device.h"
#include "nsfps_launch.h"

namespace nsfps {

constexpr uint32_t kSmThreads = 1024, kSmWaves = kSmThreads / 64, kSmLog = 10;
static_assert(kSmThreads == 1u << kSmLog, "a histogram bin per thread");
// Listed points per round, at most: all pairs of the list meet on one CU, so
// its cost grows with the square, while longer lists save few rounds (the
// quickstart takes 33 at 128 entries and 30 without a limit).
constexpr uint32_t kSmallList = 128;
static_assert(kSmallMaxPoints == 16 * kSmThreads && kSmallMaxPoints <= (1u << 14), "14-bit rows");
static_assert(kSmallList % 64 == 0 && kSmallList <= 256, "list groups of a wave");

// ------------------------------------------------------------------- sort

// compute_bbox's range of the bounds (order-preserving integers lo, hi) as
// k_range_of_bounds derives it: lanes 0 .. 3 kCubeThr - 1 of one wave search
// a threshold each.
__device__ __forceinline__ void range_of_bounds(const uint32_t *lo, const uint32_t *hi,
                                                RangeDev &r, float *bounds, uint32_t lane) {
  constexpr float kEps = 1e-6f;  // BOUNDARY_EPS, src/yuezu_fps.h:43-45
#pragma unroll
  for (uint32_t a = 0; a < 3; ++a) {
    const bool any = lo[a] <= hi[a];
    const float mn = (any ? float_of(lo[a]) : 0.f) - kEps;
    const float mx = (any ? float_of(hi[a]) : 0.f) + kEps;
    const float bs = (mx - mn) / (float)r.blocks[a];
    if (lane < kCubeThr) r.cube_thr[a][lane] = cube_threshold_dev(bs, r.blocks[a], lane + 1);
    if (lane == 0) {
      r.mn[a] = mn;
      r.hiclamp[a] = mx - kEps;
      r.bsize[a] = bs;
      r.inv_bs[a] = 1.0f / bs;
      bounds[2 * a] = mn;
      bounds[2 * a + 1] = mx;
    }
  }
}

// Stable sort of n elements by `bits` key bits above the 14-bit payload; lane
// l of wave w holds elements 64 R w + 64 r + l.  The ranking is k_seg_sort's:
// 8 key bits a pass, a wave's elements in order by ballots.  The sorted
// elements are left in s_el.
template <uint32_t R>
__device__ __forceinline__ void sort_elements(uint32_t *el, uint32_t n, uint32_t bits,
                                              uint32_t *s_el, uint32_t (*s_cnt)[256],
                                              uint32_t *s_sum) {
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t first = wave * 64u * R + lane;
  const uint64_t lt = lane ? (~0ull >> (64 - lane)) : 0ull;
  for (uint32_t shift = 0; shift < bits; shift += 8) {
    for (uint32_t i = tid; i < kSmWaves * 256u; i += kSmThreads) (&s_cnt[0][0])[i] = 0u;
    __syncthreads();
    uint32_t rnk[R];
#pragma unroll
    for (uint32_t r = 0; r < R; ++r) {
      const bool valid = first + 64u * r < n;
      const uint32_t d = (el[r] >> (14 + shift)) & 255u;
      uint64_t peers = __ballot(valid);
#pragma unroll
      for (uint32_t b = 0; b < 8; ++b) {
        const uint64_t m = __ballot((d >> b) & 1u);
        peers &= ((d >> b) & 1u) ? m : ~m;
      }
      const uint32_t before = (uint32_t)__popcll(peers & lt);
      const uint32_t at = valid ? s_cnt[wave][d] : 0u;
      rnk[r] = at + before;
      // all lanes read their base before a leader writes (in-order LDS, one wave)
      __builtin_amdgcn_s_waitcnt(0xc07f);
      if (valid && before == 0) s_cnt[wave][d] = at + (uint32_t)__popcll(peers);
      __builtin_amdgcn_s_waitcnt(0xc07f);
    }
    __syncthreads();
    uint32_t tot = 0;
    if (tid < 256u)
      for (uint32_t w = 0; w < kSmWaves; ++w) tot += s_cnt[w][tid];
    uint32_t all;
    uint32_t at = block_excl_scan<kSmWaves>(tot, s_sum, &all);
    if (tid < 256u) {
      for (uint32_t w = 0; w < kSmWaves; ++w) {
        const uint32_t k = s_cnt[w][tid];
        s_cnt[w][tid] = at;
        at += k;
      }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t r = 0; r < R; ++r)
      if (first + 64u * r < n) s_el[s_cnt[wave][(el[r] >> (14 + shift)) & 255u] + rnk[r]] = el[r];
    __syncthreads();
    if (shift + 8 < bits) {
#pragma unroll
      for (uint32_t r = 0; r < R; ++r) el[r] = first + 64u * r < n ? s_el[first + 64u * r] : 0u;
      __syncthreads();
    }
  }
}

// cell_axis with the range's values in scalar registers (the same operations).
struct CellRange {
  float mn[3], hi[3], inv[3];
  uint32_t last[3];
  __device__ __forceinline__ explicit CellRange(const RangeDev &r) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      mn[a] = uni(r.mn[a]);
      hi[a] = uni(r.hiclamp[a]);
      inv[a] = uni(r.inv_bs[a]);
      last[a] = uniform(r.blocks[a]) - 1;
    }
  }
  __device__ __forceinline__ uint32_t axis(int a, float v) const {
    const float c = std_max(mn[a], std_min(v, hi[a]));
    return min((uint32_t)((c - mn[a]) * inv[a]), last[a]);
  }
};

constexpr uint32_t kSpatialBits = 16;  // two passes of the sort

// One cloud's points in the logical order (by bucket, then input row: rank and
// row tables), and the order they are stored in.  That is the logical order
// too where it keeps 64 consecutive points together in space; where a bucket
// holds more than 64 points (all of the 10,000-point quickstart's lie in 8),
// or holds points of several cells, a second sort puts them in the Morton
// order of a grid of 2^16 cells over their box.  The points are read once and stay in
// registers until they are stored in place (read again in order instead, three
// scattered words a point, the kernel took 70 us for 16,384 points).
template <uint32_t R, bool ONE>
__device__ __forceinline__ void sort_cloud(const SmallDev &c, SmallDev *dst, SmallDev *first_dev) {
  __shared__ uint32_t s_el[kSmThreads * R];
  __shared__ uint16_t s_rank[kSmThreads * R], s_pos[kSmThreads * R];  // by row
  __shared__ uint32_t s_cnt[kSmWaves][256];
  __shared__ uint32_t s_lut[3][1024];
  __shared__ uint32_t s_sum[kSmWaves], s_bad, s_spatial;
  __shared__ uint32_t s_lo[kSmWaves][3], s_hi[kSmWaves][3];
  __shared__ RangeDev s_r;
  __shared__ float s_b[6];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t n = c.n, bbox = c.bbox;
  const NSFPS_GLOBAL float *const xyz = gptr(c.xyz);
  if (tid == 0) {
    s_bad = 0;
    s_spatial = 0;
    s_r = c.r;
  }
  float p[R][3];
  bool bad = false;
  const uint32_t first = wave * 64u * R + lane;
#pragma unroll
  for (uint32_t r = 0; r < R; ++r) {
    const uint32_t e = first + 64u * r;
#pragma unroll
    for (uint32_t a = 0; a < 3; ++a) {
      p[r][a] = e < n ? xyz[3u * e + a] : 0.f;
      bad = bad || !isfinite(p[r][a]);
    }
  }
  __syncthreads();
  if (bad) atomicOr(&s_bad, 1u);
#pragma unroll
  for (uint32_t a = 0; a < 3; ++a) {
    uint32_t l = 0xffffffffu, h = 0u;
#pragma unroll
    for (uint32_t r = 0; r < R; ++r) {
      if (first + 64u * r < n && isfinite(p[r][a])) {
        l = min(l, ord_of(p[r][a]));
        h = max(h, ord_of(p[r][a]));
      }
    }
    l = wave_min_u32(l);
    h = wave_max_u32(h);
    if (lane == 0) {
      s_lo[wave][a] = l;
      s_hi[wave][a] = h;
    }
  }
  __syncthreads();
  uint32_t lo[3], hi[3];  // the points' box
#pragma unroll
  for (uint32_t a = 0; a < 3; ++a) {
    lo[a] = wave_min_u32(s_lo[lane % kSmWaves][a]);
    hi[a] = wave_max_u32(s_hi[lane % kSmWaves][a]);
  }
  if (bbox && wave == 0) {
    range_of_bounds(lo, hi, s_r, s_b, lane);
    // a range that check_range refuses: the call reports it
    if (lane < 3 && !(isfinite(s_b[2 * lane]) && isfinite(s_b[2 * lane + 1]) &&
                      s_b[2 * lane + 1] > s_b[2 * lane]))
      atomicOr(&s_bad, 2u);
    if (lane < 6) gptr(c.st)->bounds[lane] = s_b[lane];
  }
  // the bits of an axis value at their places in the Morton code
  for (uint32_t a = 0; a < 3; ++a) {
    if (tid < s_r.blocks[a]) s_lut[a][tid] = deposit_bits(tid, s_r.cmask[a]);
  }
  __syncthreads();
  const bool stop = s_bad != 0;
  if (tid < sizeof(RangeDev) / 4 && (ONE || bbox))
    reinterpret_cast<uint32_t *>(&dst->r)[tid] = reinterpret_cast<const uint32_t *>(&s_r)[tid];
  if (tid == 0) {
    if (ONE) {
      dst->n = n;
      dst->m = c.m;
      dst->out = c.out;
      dst->pts = c.pts;
      dst->rows = c.rows;
      dst->st = c.st;
      dst->any_bad = s_bad;
    } else if (s_bad) {
      atomicOr(&first_dev->any_bad, s_bad);
    }
    gptr(c.st)->bad = s_bad;
    gptr(c.st)->len = 0;
    gptr(c.st)->rounds = 0;
    gptr(c.st)->err = 0;
  }
  if (stop) return;
  const CellRange cells(s_r);
  const bool bijective = uniform(s_r.bijective) != 0;
  const uint32_t buckets = uniform(s_r.T);
  uint32_t el[R];
#pragma unroll
  for (uint32_t r = 0; r < R; ++r) {
    const uint32_t e = first + 64u * r;
    const uint32_t code = s_lut[0][cells.axis(0, p[r][0])] | s_lut[1][cells.axis(1, p[r][1])] |
                          s_lut[2][cells.axis(2, p[r][2])];
    el[r] = e < n ? ((bijective ? code : code % buckets) << 14) | e : 0u;
  }
  uint32_t bits = 1;
  while ((1u << bits) < buckets) ++bits;
  bool spatial = false;
  while (true) {  // one copy of the sort's code: most of it runs once, so its length counts
    sort_elements<R>(el, n, bits, s_el, s_cnt, s_sum);
    if (spatial) break;
    // rows by rank and ranks by row; whether some bucket holds more than a
    // leaf's points
#pragma unroll 1
    for (uint32_t q = tid; q < n; q += kSmThreads) {
      const uint32_t e = s_el[q];
      s_rank[e & 0x3fffu] = (uint16_t)q;
      gptr(c.rows)[q] = (uint16_t)(e & 0x3fffu);
      if (!bijective || (q + 64 < n && (s_el[q + 64] >> 14) == (e >> 14))) s_spatial = 1;
    }
    __syncthreads();
    spatial = n > 64 && uniform(s_spatial) != 0;
    if (!spatial) break;
    // kSpatialBits code bits, the next one always to the axis whose cells are
    // longest (at most 10 an axis); the order alone depends on this
    float mn[3], sc[3], cell[3];
    uint32_t mask[3] = {0, 0, 0}, have[3] = {0, 0, 0};
#pragma unroll
    for (uint32_t a = 0; a < 3; ++a) {
      mn[a] = float_of(lo[a]);
      cell[a] = float_of(hi[a]) - mn[a];
      sc[a] = cell[a] > 0.f ? 0.9999f / cell[a] : 0.f;
    }
    for (uint32_t k = kSpatialBits; k-- > 0;) {
      uint32_t best = have[0] < 10 ? 0u : have[1] < 10 ? 1u : 2u;
#pragma unroll
      for (uint32_t a = 1; a < 3; ++a)
        if (have[a] < 10 && cell[a] > (best == 0 ? cell[0] : best == 1 ? cell[1] : cell[2])) best = a;
#pragma unroll
      for (uint32_t a = 0; a < 3; ++a) {
        if (a == best) {
          mask[a] |= 1u << k;
          cell[a] *= 0.5f;
          ++have[a];
        }
      }
    }
#pragma unroll
    for (uint32_t a = 0; a < 3; ++a) {
      sc[a] *= (float)(1u << have[a]);
      s_lut[a][tid] = deposit_bits(tid, mask[a]);
    }
    __syncthreads();
#pragma unroll
    for (uint32_t r = 0; r < R; ++r) {
      const uint32_t e = first + 64u * r;
      uint32_t code = 0;
#pragma unroll
      for (uint32_t a = 0; a < 3; ++a) {
        const float f = (p[r][a] - mn[a]) * sc[a];
        code |= s_lut[a][(uint32_t)fminf(fmaxf(f, 0.f), (float)((1u << have[a]) - 1u))];
      }
      el[r] = e < n ? (code << 14) | e : 0u;
    }
    bits = kSpatialBits;
  }
  if (spatial) {
#pragma unroll 1
    for (uint32_t q = tid; q < n; q += kSmThreads) s_pos[s_el[q] & 0x3fffu] = (uint16_t)q;
    __syncthreads();
  }
#pragma unroll
  for (uint32_t r = 0; r < R; ++r) {
    const uint32_t e = first + 64u * r;
    if (e < n) {
      const uint32_t rank = s_rank[e], q = spatial ? s_pos[e] : rank;
      gptr(c.pts)[q] = make_float4(p[r][0], p[r][1], p[r][2], __uint_as_float(rank));
      if (e == 0) {
        gptr(c.st)->pos0 = q;
        gptr(c.st)->rank0 = rank;
      }
    }
  }
}

// one: the cloud's parameters when there is a single cloud (they are left in
// devs[0] for the sampling); otherwise devs[blockIdx.x].
template <uint32_t R>
__global__ __launch_bounds__(kSmThreads) void k_small_sort1(SmallDev one, SmallDev *devs) {
  sort_cloud<R, true>(one, devs, devs);
}
template <uint32_t R>
__global__ __launch_bounds__(kSmThreads) void k_small_sort(SmallDev *devs) {
  sort_cloud<R, false>(devs[blockIdx.x], devs + blockIdx.x, devs);
}

// ----------------------------------------------------------------- sample


// A point is updated by a sample when the sample's cube holds its cell, or
// with shared buckets another cell of its bucket.
__device__ bool in_cube(const RangeDev &r, float x, float y, float z, uint2 cube) {
  const uint32_t c11 =
      pack11(pack_cell(cell_axis(r, 0, x), cell_axis(r, 1, y), cell_axis(r, 2, z)));
  if (in_box11(c11 | kGuards, c11, cube.x, cube.y)) return true;
  return r.bijective == 0u && bucket_in_cube(r, c11, cube);
}

// The cube of sample p (distance p.w) certainly holds the cell of every point
// nearer to it than p.w: such a point lies within `reach` of p on each axis
// (rounding included: half an ulp of a product, or half the smallest
// subnormal), and cell_axis is monotone.  The cube's half-width is the
// distance in blocks rounded up, so only rounding at a cell's edge can fail.
__device__ __forceinline__ bool cube_certain(const RangeDev &r, float4 p, uint2 cube) {
  const float reach = sqrtf(p.w) * 1.00001f + 1e-22f;
  const float v[3] = {p.x, p.y, p.z};
  bool ok = true;
#pragma unroll
  for (uint32_t a = 0; a < 3; ++a) {
    const uint32_t lo = (cube.x >> (11 * a)) & 1023u, hi = (cube.y >> (11 * a)) & 1023u;
    ok = ok && cell_axis(r, a, v[a] - reach) >= lo && cell_axis(r, a, v[a] + reach) <= hi;
  }
  return ok;
}

// Up to S points per thread: wave w holds the leaves w K .. w K + K - 1 (64
// consecutive points each; K = leaves / waves, rounded up), point s of lane l
// being point l of leaf w K + s.  Lane l also keeps the box and the largest
// min-distance of the wave's leaf l % S, so that one step tests 64 / S picks
// against all of the wave's leaves.
//
// Bound by one CU's vector units: of some 40,000 cycles a round at S = 16,
// 11,000 go to the threshold and the list and 9,000 to 13,000 to waiting for
// the wave whose leaves most samples reach.  Sixteen waves measured faster
// than eight with twice the slots each, and than four; leaves in stretches per
// wave faster than dealt out in turn, which spreads the samples but gives
// every wave all of them to test.
template <uint32_t S>
__global__ __launch_bounds__(kSmThreads) void k_small_sample(const SmallDev *__restrict__ devs,
                                                             uint32_t m_over,
                                                             int32_t *out_over) {
  constexpr uint32_t N = S * kSmThreads, kPer = 64 / S, kCertain = 0xffffffffu;
  constexpr uint32_t kBinsPer = 4096 / kSmThreads;  // the final sort's bins
  static_assert(S == 1 || S == 2 || S == 4 || S == 8 || S == 16, "points per thread");
  __shared__ uint32_t s_sd[N];  // samples: distance bits,
  __shared__ uint16_t s_sp[N];  //   logical rank
  // the rounds' buffers, and after them the final sort's
  struct Round {
    float4 lp[kSmallList];    // list: x, y, z, distance
    float4 pp[kSmallList];    // the round's samples: x, y, z, and kCertain or their number (bits)
    uint2 pc[kSmallList];     // list: cubes
    uint32_t lc[kSmallList];  //   kCertain, or the entry's number when its cube has to be looked at
    uint32_t lq[kSmallList];  //   logical ranks
    uint32_t lf[kSmallList];  //   in conflict with a larger key
    uint32_t hist[kSmThreads];
    float4 near[kSmWaves][kSmallList];  // the samples that reach a wave's box
    unsigned long long mask[kSmWaves][S];  // of 64 of those, the ones that reach a leaf's
  };
  struct Final {
    uint32_t bin[4096 + 4];
    uint16_t at[N];
  };
  __shared__ union {
    Round r;
    Final f;
  } u;
  __shared__ RangeDev s_r;
  __shared__ uint32_t s_wmax[kSmWaves], s_wn[kSmWaves], s_wc[kSmWaves];
  __shared__ uint32_t s_n, s_a, s_above, s_x[2];
  const SmallDev &c = devs[blockIdx.x];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t n = c.n, m = m_over ? m_over : c.m;
  NSFPS_GLOBAL SmallStatus &st = *gptr(c.st);
  const NSFPS_GLOBAL float4 *const pts = gptr(c.pts);
  // a call with a cloud that it refuses writes no row of any (uniform)
  if (gptr(devs)->any_bad) return;
  const uint32_t pos0 = st.pos0, rank0 = st.rank0;
  const uint32_t lpw = ((n + 63u) / 64u + kSmWaves - 1) / kSmWaves;  // leaves per wave, <= S
  if (tid < sizeof(RangeDev) / 4)
    reinterpret_cast<uint32_t *>(&s_r)[tid] = reinterpret_cast<const uint32_t *>(&c.r)[tid];
  float x[S], y[S], z[S];
  uint32_t rk[(S + 1) / 2];  // logical ranks, two a word
  uint32_t d[S];  // min-distance bits (non-negative floats order like their bits)
#pragma unroll
  for (uint32_t s = 0; s < S; ++s) {
    const uint32_t i = (wave * lpw + s) * 64u + lane;
    const float4 p = pts[s < lpw && i < n ? i : 0u];
    x[s] = p.x;
    y[s] = p.y;
    z[s] = p.z;
    if (s % 2 == 0) rk[s / 2] = __float_as_uint(p.w);
    else rk[s / 2] |= __float_as_uint(p.w) << 16;
  }
  const float4 p0 = pts[pos0];
  const auto rank_of = [&](uint32_t s) { return s % 2 ? rk[s / 2] >> 16 : rk[s / 2] & 0xffffu; };
  if (tid == 0) {
    s_sd[0] = 0xffffffffu;  // the first sample: input row 0
    s_sp[0] = (uint16_t)rank0;
    s_n = s_a = s_above = 0;
  }
  __syncthreads();
  // the first sample reaches every point (src/yuezu_fps.cpp:431-438); then
  // each leaf's box and largest distance, and the wave's
  float blo[3] = {INFINITY, INFINITY, INFINITY}, bhi[3] = {-INFINITY, -INFINITY, -INFINITY};
  uint32_t lmax = 0;
#pragma unroll
  for (uint32_t s = 0; s < S; ++s) {
    const bool in = s < lpw && (wave * lpw + s) * 64u + lane < n;
    const float dd = sqdist(x[s], y[s], z[s], p0.x, p0.y, p0.z);
    d[s] = in ? __float_as_uint(dd < FLT_MAX ? dd : FLT_MAX) : 0u;
    const float v[3] = {x[s], y[s], z[s]};
#pragma unroll
    for (uint32_t a = 0; a < 3; ++a) {
      const uint32_t l = wave_min_u32(in ? ord_of(v[a]) : 0xffffffffu);
      const uint32_t h = wave_max_u32(in ? ord_of(v[a]) : 0u);
      if (lane % S == s && l <= h) {
        blo[a] = float_of(l);
        bhi[a] = float_of(h);
      }
    }
    const uint32_t mx = wave_max_u32(d[s]);
    if (lane % S == s) lmax = mx;
    __builtin_amdgcn_sched_barrier(0);  // one leaf after another: their registers would add up
  }
  float wlo[3], whi[3];
#pragma unroll
  for (uint32_t a = 0; a < 3; ++a) {
    wlo[a] = float_of(wave_min_u32(ord_of(blo[a])));
    whi[a] = float_of(wave_max_u32(ord_of(bhi[a])));
  }
  uint32_t wmax = wave_max_u32(lmax);
  if (lane == 0) s_wmax[wave] = wmax;
  uint32_t T = 1, sh = 31 - kSmLog, rounds = 0, lcap = 64;
  bool ok = false;
  __syncthreads();
  for (; rounds < N + 2; ++rounds) {
    const uint32_t kmax = wave_max_u32(s_wmax[lane % kSmWaves]);
    if (kmax == 0) {  // only points at distance 0 are left
      ok = true;
      break;
    }
    if (T >= m) {  // done once m samples lie above every key left
      uint32_t k = 0;
      for (uint32_t i = tid; i < T; i += kSmThreads) k += s_sd[i] > kmax ? 1u : 0u;
      k = rdlane(wave_incl_scan(k), 63);
      if (lane == 0 && k) atomicAdd(&s_above, k);
      __syncthreads();
      if (uniform(s_above) >= m) {
        ok = true;
        break;
      }
    }
    // ---- threshold: histograms of the distances below kref, refined inside
    // the bin where the list would overflow
    uint32_t thr, kref = kmax, cap = lcap, taken = 0, sft = sh;
    bool tie = false;
    while (true) {
      u.r.hist[tid] = 0;
      __syncthreads();
      if (tid == 0) s_above = 0;
      const uint64_t wide = (uint64_t)kSmThreads << sft;
      const uint32_t low = wide > kref ? 0u : kref - (uint32_t)wide + 1u;  // lowest distance counted
      const uint64_t some = __ballot(lane < S && lmax >= max(low, 1u));
#pragma unroll
      for (uint32_t s = 0; s < S; ++s) {
        if ((some >> s) & 1u) {
          if (d[s] - max(low, 1u) <= kref - max(low, 1u))
            atomicAdd(&u.r.hist[(kref - d[s]) >> sft], 1u);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      __syncthreads();
      const uint32_t h = u.r.hist[tid];
      uint32_t tot;
      const uint32_t pre = block_excl_scan<kSmWaves>(h, s_wn, &tot);
      if (tot <= cap) {
        if (low <= 1u || taken + tot >= lcap / 4) {
          thr = max(low, 1u);
          break;
        }
        sft = min(sft + 3u, 31 - kSmLog);  // too few: a wider window
        __syncthreads();           // s_wn is read
        continue;
      }
      if (pre <= cap && pre + h > cap) {
        s_x[0] = tid;
        s_x[1] = pre;
      }
      __syncthreads();
      const uint32_t bs = uniform(s_x[0]), before = uniform(s_x[1]);
      if (taken + before >= lcap / 4 || sft == 0) {
        if (taken + before) {
          thr = kref - (bs << sft) + 1u;
        } else {  // more points than the list holds share the largest distance
          thr = kref - bs;
          tie = true;
        }
        break;
      }
      taken += before;
      cap -= before;
      kref -= bs << sft;
      sft = sft >= kSmLog ? sft - kSmLog : 0u;
    }
    {
      const uint32_t bl = 32u - (uint32_t)__builtin_clz((kmax - thr) | 1u);
      sh = bl > kSmLog - 1 ? min(bl - (kSmLog - 1), 31 - kSmLog) : 0u;  // one to two spans next time
    }
    // ---- list
    // entries: distance >= thr, and in a tie rank < rtop (the smallest ranks
    // are the largest keys): rtop is found by halving the ranks' range until
    // at most kSmallList and at least one lie below it
    uint32_t cnt = 0, rtop = kSmallMaxPoints;
    if (tie) {
      uint32_t rlo = 0;  // no entry's rank is below rlo, more than the list's are below rtop
      while (true) {
        const uint32_t mid = (rlo + rtop + 1) / 2;
        uint32_t k = 0;
#pragma unroll
        for (uint32_t s = 0; s < S; ++s)
          k += (uint32_t)__popcll(__ballot(d[s] >= thr && rank_of(s) < mid));
        if (lane == 0) s_wc[wave] = k;
        __syncthreads();
        uint32_t all = 0;
        for (uint32_t w = 0; w < kSmWaves; ++w) all += s_wc[w];
        __syncthreads();
        if (all > kSmallList) {
          rtop = mid;
        } else if (all) {
          rtop = mid;
          break;
        } else {
          rlo = mid;
        }
      }
    }
    const uint64_t high = __ballot(lane < S && lmax >= thr);  // leaves with entries
#pragma unroll
    for (uint32_t s = 0; s < S; ++s)
      if ((high >> s) & 1u)
        cnt += (uint32_t)__popcll(__ballot(d[s] >= thr && (!tie || rank_of(s) < rtop)));
    uint32_t base = 0;
    if (lane == 0 && cnt) base = atomicAdd(&s_n, cnt);
    base = rdlane(base, 0);
    if (cnt) {
#pragma unroll
      for (uint32_t s = 0; s < S; ++s) {
        if (!((high >> s) & 1u)) continue;
        const bool in = d[s] >= thr && (!tie || rank_of(s) < rtop);
        const uint64_t take = __ballot(in);
        const uint32_t i = base + lanes_below(take);
        if (in && i < kSmallList) {  // always below it
          u.r.lp[i] = make_float4(x[s], y[s], z[s], __uint_as_float(d[s]));
          u.r.lq[i] = rank_of(s);
          u.r.lf[i] = 0;
        }
        base += (uint32_t)__popcll(take);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __syncthreads();
    // ---- conflicts: a wave's lanes hold 64 entries and meet a share of the
    // list; the last waves find the entries' cubes meanwhile
    const uint32_t L = min(uniform(s_n), kSmallList);
    const uint32_t groups = (L + 63) / 64, parts = (kSmWaves - groups) / groups;
    static_assert(kSmWaves >= 2 * (kSmallList / 64), "waves for the conflicts and the cubes");
    if (wave < groups * parts) {
      const uint32_t g = wave % groups, i = g * 64u + lane, part = wave / groups;
      const uint32_t per = (L + parts - 1) / parts;
      const uint32_t q0 = part * per, q1 = min(q0 + per, L);
      const float4 me = u.r.lp[i];
      const uint32_t mq = u.r.lq[i];
      bool blocked = false;
#pragma unroll 4
      for (uint32_t q = q0; q < q1; ++q) {
        const float4 o = u.r.lp[q];
        const uint32_t oq = u.r.lq[q];
        const bool above = (o.w > me.w) | ((o.w == me.w) & (oq < mq));
        blocked |= above & (sqdist(me.x, me.y, me.z, o.x, o.y, o.z) < o.w);
      }
      if (blocked && i < L) u.r.lf[i] = 1;
    } else if (wave >= kSmWaves - groups) {
      const uint32_t i = (wave - (kSmWaves - groups)) * 64u + lane;
      if (i < L) {
        const float4 p = u.r.lp[i];
        const uint2 cube =
            sample_cube(s_r, pack11(pack_cell(cell_axis(s_r, 0, p.x), cell_axis(s_r, 1, p.y),
                                              cell_axis(s_r, 2, p.z))), p.w);
        u.r.pc[i] = cube;
        u.r.lc[i] = cube_certain(s_r, p, cube) ? kCertain : i;
      }
    }
    __syncthreads();
    // ---- the round's samples
    if (tid == 0) s_n = 0;
    if (wave < groups) {
      const bool acc = tid < L && u.r.lf[tid] == 0u;
      const uint64_t bal = __ballot(acc);
      uint32_t at = 0;
      if (lane == 0 && bal) at = atomicAdd(&s_a, (uint32_t)__popcll(bal));
      at = rdlane(at, 0) + lanes_below(bal);
      if (acc) {
        const float4 p = u.r.lp[tid];
        u.r.pp[at] = make_float4(p.x, p.y, p.z, __uint_as_float(u.r.lc[tid]));
        if (T + at < N) {  // always: a point is sampled once
          s_sd[T + at] = __float_as_uint(p.w);
          s_sp[T + at] = (uint16_t)u.r.lq[tid];
        }
      }
    }
    __syncthreads();
    const uint32_t A = uniform(s_a);
    // ---- applied to every point: the samples that reach the wave's box, and
    // of those, 64 at a time (one a lane), the ones that reach each leaf's
    uint32_t nn = 0;
    for (uint32_t b = 0; b < A; b += 64) {
      const float4 q = u.r.pp[min(b + lane, A - 1)];
      const bool reach = b + lane < A &&
                         !(box_bound(q.x, q.y, q.z, wlo[0], wlo[1], wlo[2], whi[0], whi[1], whi[2]) >=
                           __uint_as_float(wmax));
      const uint64_t bal = __ballot(reach);
      if (reach) u.r.near[wave][nn + lanes_below(bal)] = q;
      nn += (uint32_t)__popcll(bal);
    }
    uint32_t touched = 0;
    for (uint32_t b = 0; b < nn; b += 64) {
      const uint32_t cn = min(nn - b, 64u);
      const float4 a = u.r.near[wave][b + min(lane, cn - 1)];
      if (lane < S) u.r.mask[wave][lane] = 0;
#pragma unroll 2
      for (uint32_t j0 = 0; j0 < cn; j0 += kPer) {
        const uint32_t j = j0 + lane / S;
        const float4 q = u.r.near[wave][b + min(j, cn - 1)];
        if (j < cn && !(box_bound(q.x, q.y, q.z, blo[0], blo[1], blo[2], bhi[0], bhi[1], bhi[2]) >=
                        __uint_as_float(lmax)))
          atomicOr(&u.r.mask[wave][lane % S], 1ull << j);
      }
      const uint64_t mm = u.r.mask[wave][lane % S];
      const uint64_t sure = __ballot(__float_as_uint(a.w) == kCertain);
      const uint32_t mlo = (uint32_t)(mm & sure), mhi = (uint32_t)((mm & sure) >> 32);
#pragma unroll
      for (uint32_t s = 0; s < S; ++s) {
        uint64_t t = ((uint64_t)rdlane(mhi, s) << 32) | rdlane(mlo, s);
        if (t) touched |= 1u << s;
        while (t) {  // two a trip (a last one alone is taken twice: min is idempotent)
          const uint32_t j = (uint32_t)__builtin_ctzll(t);
          t &= t - 1;
          const uint32_t k = t ? (uint32_t)__builtin_ctzll(t) : j;
          t &= t - 1;
          const float ax = __uint_as_float(rdlane(__float_as_uint(a.x), j));
          const float ay = __uint_as_float(rdlane(__float_as_uint(a.y), j));
          const float az = __uint_as_float(rdlane(__float_as_uint(a.z), j));
          const float bx = __uint_as_float(rdlane(__float_as_uint(a.x), k));
          const float by = __uint_as_float(rdlane(__float_as_uint(a.y), k));
          const float bz = __uint_as_float(rdlane(__float_as_uint(a.z), k));
          d[s] = min(d[s], min(__float_as_uint(sqdist(x[s], y[s], z[s], ax, ay, az)),
                               __float_as_uint(sqdist(x[s], y[s], z[s], bx, by, bz))));
        }
        __builtin_amdgcn_sched_barrier(0);  // the masks are read one leaf at a time
      }
      // the samples whose cubes have to be looked at, one point at a time
      for (uint64_t t = ~sure & (cn < 64 ? (1ull << cn) - 1 : ~0ull); t; t &= t - 1) {
        const uint32_t j = (uint32_t)__builtin_ctzll(t);
        const float4 q = make_float4(__uint_as_float(rdlane(__float_as_uint(a.x), j)),
                                     __uint_as_float(rdlane(__float_as_uint(a.y), j)),
                                     __uint_as_float(rdlane(__float_as_uint(a.z), j)), 0.f);
        const uint2 cube = u.r.pc[rdlane(__float_as_uint(a.w), j)];
        for (uint64_t k = __ballot(lane < S && ((mm >> j) & 1u)); k; k &= k - 1) {
          const uint32_t s0 = (uint32_t)__builtin_ctzll(k);
          float px = 0.f, py = 0.f, pz = 0.f;
          uint32_t dp = 0;
#pragma unroll
          for (uint32_t s = 0; s < S; ++s) {
            px = s == s0 ? x[s] : px;
            py = s == s0 ? y[s] : py;
            pz = s == s0 ? z[s] : pz;
            dp = s == s0 ? d[s] : dp;
          }
          const uint32_t dd = __float_as_uint(sqdist(px, py, pz, q.x, q.y, q.z));
          if (dd < dp && in_cube(s_r, px, py, pz, cube)) dp = dd;
#pragma unroll
          for (uint32_t s = 0; s < S; ++s) d[s] = s == s0 ? dp : d[s];
          touched |= 1u << s0;
        }
      }
    }
    if (touched) {
#pragma unroll
      for (uint32_t s = 0; s < S; ++s) {
        // unless a point still has the leaf's largest distance
        if (((touched >> s) & 1u) && !__ballot(d[s] >= rdlane(lmax, s))) {
          const uint32_t mx = wave_max_u32(d[s]);
          if (lane % S == s) lmax = mx;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      wmax = wave_max_u32(lmax);
    }
    if (lane == 0) s_wmax[wave] = wmax;
    T += A;
    lcap = 2 * A > 64 ? kSmallList : 64;  // few of a longer list would be samples
    __syncthreads();
    if (tid == 0) s_a = 0;  // read by all; the next round adds after its barriers
  }
  // ---- the samples in key order: bins of the distance bits (a logarithmic
  // scale), then each sample's place among its bin's; sample 0 stays first
  __syncthreads();
  T = min(T, N);
  uint32_t mx = 0, mn = 0;
  for (uint32_t i = 1 + tid; i < T; i += kSmThreads) {
    mx = max(mx, s_sd[i]);
    mn = max(mn, ~s_sd[i]);
  }
  mx = wave_max_u32(mx);
  mn = wave_max_u32(mn);
  if (lane == 0) {
    s_wn[wave] = mx;
    s_wc[wave] = mn;
  }
  for (uint32_t j = tid; j < 4096 + 4; j += kSmThreads) u.f.bin[j] = 0;
  if (tid == 0) s_above = 0;
  __syncthreads();
  mx = wave_max_u32(s_wn[lane % kSmWaves]);
  mn = ~wave_max_u32(s_wc[lane % kSmWaves]);
  const uint32_t span = mx > mn ? mx - mn : 1u;
  const uint32_t fs = 32u - (uint32_t)__builtin_clz(span) > 12u ? 20u - (uint32_t)__builtin_clz(span) : 0u;
  uint32_t bin[S], at[S];
#pragma unroll
  for (uint32_t s = 0; s < S; ++s) {
    const uint32_t i = 1 + s * kSmThreads + tid;
    bin[s] = at[s] = 0;
    if (i < T) {
      bin[s] = (mx - s_sd[i]) >> fs;
      at[s] = atomicAdd(&u.f.bin[bin[s]], 1u);
    }
  }
  __syncthreads();
  {
    uint32_t v[kBinsPer], sum = 0, tot, big = 0;
#pragma unroll
    for (uint32_t j = 0; j < kBinsPer; ++j) {
      v[j] = u.f.bin[kBinsPer * tid + j];
      sum += v[j];
      big = max(big, v[j]);
    }
    if (big > 256u) s_above = 1;
    uint32_t pre = block_excl_scan<kSmWaves>(sum, s_wn, &tot);
#pragma unroll
    for (uint32_t j = 0; j < kBinsPer; ++j) {
      u.f.bin[kBinsPer * tid + j] = pre;
      pre += v[j];
    }
    if (tid == 0) u.f.bin[4096] = tot;
  }
  __syncthreads();
  const auto above = [&](uint32_t da, uint32_t pa, uint32_t db, uint32_t pb) -> bool {
    return da > db || (da == db && pa < pb);
  };
  if (uniform(s_above) == 0u) {
#pragma unroll
    for (uint32_t s = 0; s < S; ++s)
      if (1 + s * kSmThreads + tid < T) u.f.at[u.f.bin[bin[s]] + at[s]] = (uint16_t)(1 + s * kSmThreads + tid);
    __syncthreads();
#pragma unroll
    for (uint32_t s = 0; s < S; ++s) {
      const uint32_t i = 1 + s * kSmThreads + tid;
      if (i < T) {
        const uint32_t b0 = u.f.bin[bin[s]], b1 = u.f.bin[bin[s] + 1], di = s_sd[i], pi = s_sp[i];
        uint32_t r = b0;
        if (b0 < m)
          for (uint32_t j = b0; j < b1; ++j) {
            const uint32_t o = u.f.at[j];
            r += above(s_sd[o], s_sp[o], di, pi) ? 1u : 0u;
          }
        at[s] = 1 + r;
      }
    }
  } else {
    // many equal distances (lattices): a bitonic sort of the sample numbers;
    // numbers past the samples sort last
    for (uint32_t i = tid; i < N; i += kSmThreads) u.f.at[i] = (uint16_t)i;
    __syncthreads();
    for (uint32_t k = 2; k <= N; k <<= 1) {
      for (uint32_t j = k >> 1; j; j >>= 1) {
        for (uint32_t t = tid; t < N / 2; t += kSmThreads) {
          const uint32_t a = ((t & ~(j - 1)) << 1) | (t & (j - 1)), b = a | j;
          const uint32_t ea = u.f.at[a], eb = u.f.at[b];
          bool first = ea < eb;  // ea belongs ahead of eb
          if (ea < T && eb < T) first = above(s_sd[ea], s_sp[ea], s_sd[eb], s_sp[eb]);
          if (first != ((a & k) == 0)) {
            u.f.at[a] = (uint16_t)eb;
            u.f.at[b] = (uint16_t)ea;
          }
        }
        __syncthreads();
      }
    }
  }
  const NSFPS_GLOBAL uint16_t *const rows = gptr(c.rows);
  NSFPS_GLOBAL int32_t *const out = gptr(out_over ? out_over : c.out);
  if (uniform(s_above) == 0u) {
#pragma unroll
    for (uint32_t s = 0; s < S; ++s) {
      const uint32_t i = 1 + s * kSmThreads + tid;
      if (i < T && at[s] < m) out[at[s]] = (int32_t)rows[s_sp[i]];
    }
    if (tid == 0) out[0] = 0;
  } else {
    for (uint32_t r = tid; r < min(T, m); r += kSmThreads)
      out[r] = (int32_t)rows[s_sp[u.f.at[r]]];
  }
  if (tid == 0) {
    st.len = min(T, m);
    st.rounds = rounds;
    st.err = ok ? 0u : 1u;
  }
}

// -------------------------------------------------------------- launchers

hipError_t preload_small_kernels() {
  return func_attributes(k_small_sort1<1>, k_small_sort1<2>, k_small_sort1<4>, k_small_sort1<8>,
                         k_small_sort1<16>, k_small_sort<1>, k_small_sort<2>, k_small_sort<4>,
                         k_small_sort<8>, k_small_sort<16>, k_small_sample<1>, k_small_sample<2>,
                         k_small_sample<4>, k_small_sample<8>, k_small_sample<16>);
}

// The smallest power of two of 1,024-point slots that holds n points.
static uint32_t slots_of(uint32_t n) {
  uint32_t s = 1;
  while (s * kSmThreads < n) s *= 2;
  return s;
}

hipError_t launch_small_sort(const SmallDev *one, SmallDev *devs, uint32_t nclouds, uint32_t n,
                             hipStream_t st) {
  if (n == 0 || n > kSmallMaxPoints || nclouds == 0 || (one && nclouds != 1))
    return hipErrorInvalidValue;
  switch (slots_of(n)) {
#define NSFPS_SORT(R)                                              \
  case R:                                                          \
    if (one) k_small_sort1<R><<<1, kSmThreads, 0, st>>>(*one, devs); \
    else k_small_sort<R><<<nclouds, kSmThreads, 0, st>>>(devs);    \
    break;
    NSFPS_SORT(1)
    NSFPS_SORT(2)
    NSFPS_SORT(4)
    NSFPS_SORT(8)
    NSFPS_SORT(16)
#undef NSFPS_SORT
  }
  return hipGetLastError();
}

hipError_t launch_small_sample(const SmallDev *devs, uint32_t nclouds, uint32_t n, uint32_t m,
                               int32_t *out, hipStream_t st) {
  if (n == 0 || n > kSmallMaxPoints || nclouds == 0) return hipErrorInvalidValue;
  switch (slots_of(n)) {
#define NSFPS_SAMPLE(R)                                              \
  case R:                                                            \
    k_small_sample<R><<<nclouds, kSmThreads, 0, st>>>(devs, m, out); \
    break;
    NSFPS_SAMPLE(1)
    NSFPS_SAMPLE(2)
    NSFPS_SAMPLE(4)
    NSFPS_SAMPLE(8)
    NSFPS_SAMPLE(16)
#undef NSFPS_SAMPLE
  }
  return hipGetLastError();
}

}  // namespace nsfps
