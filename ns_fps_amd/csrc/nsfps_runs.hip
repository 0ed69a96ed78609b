// Round-based sampling engine (gfx950).
//
// Keys (min-distance bits << 32 | ~logical rank) only ever decrease, and the
// reference takes the point of the largest key each time
// (src/yuezu_fps.cpp:703-722).  Take a threshold key B and the list of every
// point whose key is >= B, and call two points in conflict when their squared
// distance is below the larger of their min-distances: only then can either
// lower the other.  A listed point that conflicts with none of a larger key
// is a sample with the key it has (k_accept gives the proof); all such points
// of a list are settled at once, over the whole chip, and the samples' order
// is the order of their keys, found once at the end.  The sampling ends when
// m samples have keys above every key left, or only points at distance 0 are
// left.
//
// A grid-wide pass applies a round's samples to every point (each sample's
// cube update, src/yuezu_fps.cpp:560-597).  min() of exact fp32 distances
// commutes, so a point's distance has the same bits as after the reference's
// one-by-one updates by the time its key counts.  The same pass rebuilds the
// leaf and level-1 keys and histograms the keys for the next threshold.
// Only the keys: the samples come from the list, so the winners' positions
// (leaf_pos, l1_pos, which the tree engine keeps) are not maintained.
//
// One round, in stream order:
//   k_update     samples -> points, leaf and level-1 keys, key histogram
//   k_refine x2  finer histograms inside the crossing bin, only when needed
//   k_gather     threshold B (<= list_cap keys above it), list of those points
//   k_accept     the list's conflicts: its samples and their cubes
// and after the last one k_sort_rounds and k_order, the samples' order.
// The first round's only sample is input row 0 with a cube covering the whole
// grid: the reference's first full pass (src/yuezu_fps.cpp:431-438).
//
// What bounds it: the rounds' launches (three of 5 to 17 us each; the points
// that a round touches are read from cache) times the rounds.  They are few:
// samples settle as soon as the few larger keys near them have, so a round of
// 4,096 listed points settles some 900 to 2,200.  Per call on one MI355X, device-resident,
// against lists sampled one after another by one workgroup: 120,000-point
// scan -> 16,384 (47 rounds) 3.65 -> 1.28 ms, 1M-point cube -> 65,536 (75)
// 7.02 -> 2.56, the same on 30^3 cells 10.6 -> 3.83, 8M clustered points ->
// 524,288 (243) 59 -> 16.0, 1M -> 524,288 (236) 38 -> 7.2.  Few samples, and
// the middle ones of many clouds, gain nothing: 17,000 Gaussian points -> 64
// 320 -> 292 us, -> 256 425 -> 442; 64 clouds of 17,000 -> 265 0.98 -> 1.15 ms,
// of 65,536 -> 4,096 3.3 -> 3.8.
//
// The cube test compares cell coordinates.  Where cells share buckets (block
// counts that are not powers of two: the Morton code is taken modulo the
// block count, src/yuezu_fps.cpp:413, 592) a point is updated when the cube
// holds any cell of its bucket, so every kernel tests each cell of a bucket
// (the ALIAS variants).
#include <hip/hip_runtime.h>

#include "nsfps_box.h"
#include "nsfps_device.h"
#include "nsfps_launch.h"

namespace nsfps {

constexpr uint32_t kPassThreads = 1024;  // grid-wide passes: one level-1 node per workgroup
constexpr uint32_t kPassWaves = kPassThreads / 64;
constexpr uint32_t kLeavesPerWave = kFan / kPassWaves;
constexpr uint32_t kMaxShift = 52;  // kHistBins << 52 covers the whole u64 key range
// Workgroups per cloud of the refinement and gather passes, and of a launch's
// clouds together (each replays the selection from 16 KB of histogram, and
// takes up to kGatherNodes nodes at a time): 64 clouds of 65,536 points ->
// 4,096 4.24 ms per call with one a node, 3.78 at 256 a launch (3.62 at 128,
// where 17,000 Gaussian points x 64 -> 265 lose 3 %).
constexpr uint32_t kSparseGroups = 128, kSparseLaunch = 256;
constexpr uint32_t kGatherNodes = 16;    // nodes per list-range claim of the gather pass
constexpr uint32_t kGatherHold = 4;      // hot leaves per wave whose points stay in registers

// Work counters of the grid-wide passes (profile words, summed over rounds):
// leaves whose points the update pass reads and those points, and the same
// for the gather pass.
enum : uint32_t { kCtUpLeaves = 24, kCtUpPoints, kCtGaLeaves, kCtGaPoints };
// The update pass's phase clocks (s_memrealtime ticks summed over the
// workgroups that update a node): run state, node and picks; the leaves; the
// node key and the histogram's flush; and those workgroups.
enum : uint32_t { kUpTPicks = 32, kUpTLeaves, kUpTFlush, kUpGroups };
// Finer update-pass clocks: the first reads, clearing the histogram, finding
// the touched leaves, and their points' reads (parts of the two above); the
// gather pass's: the selection's replay, the leaf records, the held points
// and the list range's claim, the writes; and its workgroups.
enum : uint32_t {
  kUpTLoad = 40, kUpTZero, kUpTHits, kUpTPts,
  kGaTSel = 44, kGaTLeaf, kGaTClaim, kGaTWrite, kGaGroups,
  // per update workgroup, over its waves: the latest and the summed times
  // from the picks' barrier to the points' arrival and to the leaf loop's end
  kUpWPtsMax = 49, kUpWPtsSum, kUpWLoopMax, kUpWLoopSum,
  // leaves the update pass reads because a pick touches them, and their points
  kCtUpHitLeaves = 53, kCtUpHitPoints,
  // per update workgroup, over its waves: the latest and the summed times of
  // finding the touched leaves
  kUpWHitsMax = 55, kUpWHitsSum,
  // keys inside the update pass's histogram window (summed over rounds), and
  // the list entries gathered
  kGaWinKeys = 57, kGaListed, kGaWinMax
};

// Level-1 node g's key: the largest of l1_key and the node's parts (in a call
// whose update pass is split, l1_key is zero and the parts hold the largest
// keys of the node's quarters; otherwise the parts are zero).  In the split
// update pass a workgroup reads its siblings' parts while they may write
// them: the parts are read and written as relaxed agent-scope atomics (each
// 64-bit word whole, no order needed: either value of a part bounds its
// quarter's points, distances only falling).  There one wave reads the key
// for its whole workgroup, which leaves ahead of a barrier by it.
__device__ __forceinline__ uint64_t node_key(const CloudDev &c, uint32_t g) {
  NSFPS_GLOBAL uint64_t *const pp = gptr(c.l1_part) + (size_t)g * kUpdateSplit;
  uint64_t k = gptr(c.l1_key)[g];
#pragma unroll
  for (uint32_t s = 0; s < kUpdateSplit; ++s) {
    const uint64_t v = __hip_atomic_load(pp + s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    k = v > k ? v : k;
  }
  return k;
}

// Histogram window of a selection pass: nb bins of 2^S keys each, bin 0 ending
// at kref.  Lowest key inside the window (kHistBins bins at kMaxShift hold
// every key: the product wraps to 0, and w to the largest key):
__device__ __forceinline__ uint64_t window_lo(uint64_t kref, uint32_t S, uint32_t nb = kHistBins) {
  const uint64_t w = ((uint64_t)nb << S) - 1;
  return kref >= w ? kref - w : 0;
}

__device__ __forceinline__ uint32_t key_bin(uint64_t key, uint64_t kref, uint32_t S,
                                            uint32_t nb = kHistBins) {
  if (key > kref) return kNone;
  const uint64_t b = (kref - key) >> S;
  return b < nb ? (uint32_t)b : kNone;
}

// The key histograms (kHists of kHistBins each): the update pass counts
// histogram 0, the refinement passes histograms 1 and 2.
__device__ __forceinline__ NSFPS_GLOBAL uint32_t *hist_set(const CloudDev &c) {
  return gptr(c.hist);
}

// Threshold selection, replayed identically by every workgroup that needs it.
// A histogram over window (kref, S) gives the first bin where the cumulative
// count exceeds the free capacity; the bins before it are taken.  If they
// fill less than half of it, that crossing bin is histogrammed again 12 bits
// finer by the next refinement pass.  The update pass counts one window below
// kref0 (shift s0, set from the previous round's key span).  A window that
// holds fewer keys than the list takes all of them: the run is shorter, and
// the next round's window, sized from this round's span, is 4x wider.  When
// nothing fits (more than kListCap keys share the finest bin) or the window is
// empty, the threshold is the maximum key.
struct Sel {
  uint64_t kref;
  uint64_t bkey;     // resolved threshold
  uint32_t S;
  uint32_t cap;      // capacity left
  uint32_t total;    // entries taken so far
  uint32_t state;    // 0: refinement pass `pass` needed, 1: resolved, 2: use the maximum key
  uint32_t pass;
  uint32_t win;      // keys inside the update pass's histogram window
  uint64_t ktop;     // no key is above this (0 when the window is empty)
};

struct Step {
  uint32_t tot;     // keys in the window
  uint32_t bs;      // crossing bin, kNone when tot <= cap
  uint32_t before;  // keys in the bins before it
  uint32_t first;   // first bin that holds a key, kNone when none does
};

// Block-wide, all kPassThreads threads; sc holds kPassWaves + 3 words of LDS.
// h: this thread's four bins of the histogram.
__device__ Step hist_step(uint4 h, uint32_t cap, uint32_t *sc) {
  const uint32_t tid = threadIdx.x;
  uint32_t tot;
  const uint32_t pre = block_excl_scan<kPassWaves>(h.x + h.y + h.z + h.w, sc, &tot);
  const uint32_t bins[4] = {h.x, h.y, h.z, h.w};
  uint32_t c = pre;
#pragma unroll
  for (uint32_t j = 0; j < 4; ++j) {
    if (c <= cap && c + bins[j] > cap) {  // exactly one bin crosses
      sc[kPassWaves] = 4 * tid + j;
      sc[kPassWaves + 1] = c;
    }
    if (c == 0 && bins[j]) sc[kPassWaves + 2] = 4 * tid + j;  // one thread, once
    c += bins[j];
  }
  __syncthreads();
  Step st;
  st.tot = tot;
  st.bs = tot <= cap ? kNone : sc[kPassWaves];
  st.before = tot <= cap ? 0u : sc[kPassWaves + 1];
  st.first = tot ? sc[kPassWaves + 2] : kNone;
  __syncthreads();
  return st;
}
__device__ Step hist_step(const uint32_t *H, uint32_t cap, uint32_t *sc) {
  return hist_step(gptr(reinterpret_cast<const uint4 *>(H))[threadIdx.x], cap, sc);
}

// Replays the selection from the update pass's histograms and the first
// `avail - 1` refinement histograms; `passes` refinement passes run this
// round, so the threshold is forced at step `passes` (forced is set when that
// rule, not the histograms, ended the selection with a list under a quarter
// full).  h0: this thread's bins of the update pass's histogram, when the
// caller read them already.
__device__ Sel sel_replay(const CloudDev &c, uint32_t avail, uint32_t passes, uint32_t *sc,
                          bool *forced = nullptr, const uint4 *h0 = nullptr) {
  const NSFPS_GLOBAL RunState &rs = *gptr(c.rs);
  Sel s;
  s.kref = rs.kref0;
  s.bkey = 0;
  s.S = rs.s0;
  s.cap = min(max(rs.cap, 1u), kListCap);
  const uint32_t cap0 = s.cap;
  s.total = 0;
  s.state = 0;
  s.pass = 0;
  const uint32_t *H0 = c.hist;
  Step st = h0 ? hist_step(*h0, s.cap, sc) : hist_step(H0, s.cap, sc);
  s.win = st.tot;
  s.ktop = st.first == kNone ? 0ull : s.kref - ((uint64_t)st.first << s.S);
  for (uint32_t p = 0;; ++p) {
    if (st.bs == kNone) {  // the whole window fits
      s.total += st.tot;
      s.bkey = window_lo(s.kref, s.S, p ? kHistBins : rs.nb);
      s.state = s.total ? 1u : 2u;
      return s;
    }
    s.total += st.before;
    if (st.before >= s.cap / 2 || s.S == 0 || p == passes) {
      // forced, and the list under a quarter full: refinement would have paid
      if (forced) *forced = st.before < s.cap / 2 && s.S != 0 && s.total < cap0 / 4;
      s.bkey = s.kref - ((uint64_t)st.bs << s.S) + 1;  // keys above bin bs
      s.state = s.total ? 1u : 2u;
      return s;
    }
    s.cap -= st.before;
    s.kref -= (uint64_t)st.bs << s.S;
    s.S = s.S >= 12 ? s.S - 12 : 0;
    if (p + 1 >= avail) {
      s.pass = p + 1;
      return s;
    }
    st = hist_step(H0 + (1 + p) * kHistBins, s.cap, sc);
  }
}

__device__ __forceinline__ const NSFPS_GLOBAL RunState &rstate(const CloudDev &c) {
  return *gptr(c.rs);
}

// ------------------------------------------------------------ the samples

// By one workgroup of the update pass: the last list's settled entries join
// the samples (keys and rows), with a log entry per round: the samples
// before it, the smallest threshold up to it and the largest key in it.
__device__ void record_samples(const CloudDev &c, uint32_t par, uint32_t *sc) {
  const uint32_t tid = threadIdx.x;
  NSFPS_GLOBAL RunState &rs = *gptr(c.rs);
  const uint32_t nl = min(rs.nl[par ^ 1u], kListCap), base = rs.ntaken, nlog = rs.nlog;
  const uint64_t bkey = rs.bkey, bmin = rs.bmin, ktop = rs.ktop;
  // a list sampled one after another is recorded by the accept pass
  const uint32_t done = *gptr(c.done) | rs.seq;
  constexpr uint32_t kSlots = kListCap / kPassThreads;
  bool take[kSlots];
  float4 p[kSlots];
  uint2 r[kSlots];
  uint32_t n = 0;
#pragma unroll
  for (uint32_t s = 0; s < kSlots; ++s) {
    const uint32_t i = kSlots * tid + s;
    p[s] = gptr(c.list_p)[i];
    r[s] = gptr(c.list_r)[i];
    take[s] = i < nl && gptr(c.list_f)[i] == 0u;
    n += take[s] ? 1u : 0u;
  }
  if (done) return;
  uint32_t total;
  uint32_t at = base + block_excl_scan<kPassWaves>(n, sc, &total);
#pragma unroll
  for (uint32_t s = 0; s < kSlots; ++s) {
    if (take[s]) {
      if (at < c.n) {
        gptr(c.smp_d)[at] = __float_as_uint(p[s].w);
        gptr(c.smp_lo)[at] = ~r[s].x;
        gptr(c.smp_row)[at] = r[s].y;
      } else {
        rs.err = 2;  // cannot happen (a point is settled once)
      }
      ++at;
    }
  }
  if (tid == 0) {
    const uint64_t b = bkey < bmin ? bkey : bmin;
    rs.bmin = b;
    rs.ntaken = base + total;
    *gptr(c.iter) = min(base + total, c.m);
    rs.cap = min(max(kListGrow * total, kListMin), c.list_cap);
    // a full log's last entry stands for all later rounds
    const uint32_t i = nlog < c.log_cap ? nlog : c.log_cap - 1;
    gptr(c.log_bmin)[i] = b;
    if (nlog < c.log_cap) {
      gptr(c.log_ktop)[i] = ktop;
      gptr(c.log_start)[i] = base;
      rs.nlog = nlog + 1;
    }
  }
}

// ------------------------------------------------------------ update pass

// Applies the picks of the last run to the points of level-1 node blockIdx.x,
// rewrites the keys of the touched leaves and of the node, and counts the keys
// inside the histogram window.  A pick takes part in a node only when its
// cube overlaps the node's cells and it may lower one of the node's points:
// its least squared distance to the node's box (box_bound) is below the
// largest distance of those points, which the node's key holds (the
// reference's cube rule, src/yuezu_fps.cpp:560-597, also visits points no
// pick lowers; skipping them changes no distance).  Leaves no pick touches
// whose key lies below the window keep their key and are not read.  A leaf
// keeps its key too when no pick lowers the point that holds it (keys only
// decrease), so its maximum is searched only otherwise.  Reads that do not depend on each other are
// issued together: the wave's leaf records with the run state and the node's
// record, a pick's cube with its position, and the points of every leaf of
// the wave that needs reading.  PROF: counts the leaves and points it reads.
// ALIAS: cells share buckets, and a pick touches a leaf when its cube holds
// any cell of the leaf's bucket (src/yuezu_fps.cpp:573-597 updates every point
// of every bucket of the cube's cells); nodes are screened by the corners of
// those cells.  SPLIT: the node's leaves are split over SPLIT workgroups, each
// storing the largest key of its leaves as one of the
// node's parts (node_key reads the node's key back as the largest part).
// MIXED: a leaf is a run of 64 slots of the logical order and may hold
// several buckets (one cell each); a pick lowers a point only when the point's
// own cell lies in the cube (the reference's rule, point by point).
template <bool PROF, bool ALIAS, uint32_t SPLIT, bool MIXED>
__global__ __launch_bounds__(kPassThreads) __attribute__((amdgpu_num_sgpr(60), amdgpu_waves_per_eu(8, 8))) void k_update(
    const CloudDev *__restrict__ clouds, uint32_t round) {
  static_assert(!(ALIAS && MIXED), "leaves of several buckets need one cell per bucket");
  __shared__ uint32_t s_hist[kHistBins];
  __shared__ float4 s_pp[kPickLds];
  __shared__ uint2 s_pc[kPickLds];  // the picks' cube corners: pack11(lo), pack11(hi) | kGuards
  __shared__ uint16_t s_more[kListCap - kPickLds];  // the node's picks past kPickLds
  __shared__ uint64_t s_lk[kFan];
  __shared__ uint64_t s_nkey;  // SPLIT: the node's key as wave 0 read it
  __shared__ uint32_t s_np;
  __shared__ uint32_t s_ct[4];  // PROF: leaves and points read by the workgroup, and of them touched
  __shared__ uint32_t s_wt[PROF ? 3 * kPassWaves : 1];  // PROF: per-wave clocks
  const CloudDev &c = clouds[blockIdx.y];
  const uint32_t par = round & 1u;
  if (blockIdx.x + 1 == gridDim.x) {  // the last workgroup records the last list's samples
    if (round) record_samples(c, par, s_hist);
    return;
  }
  // SPLIT workgroups per node: this one takes leaves sub * kFan / SPLIT ..
  constexpr uint32_t kLPW = kLeavesPerWave / SPLIT;  // leaves per wave
  static_assert(kLPW >= 1 && kLPW * SPLIT == kLeavesPerWave, "whole leaves per wave");
  const uint32_t g = blockIdx.x / SPLIT, sub = blockIdx.x % SPLIT;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint64_t ut0 = PROF ? __builtin_amdgcn_s_memrealtime() : 0;
  // this wave's leaves: lane k < kLPW holds leaf leaf0 + k's record
  const uint32_t leaf0 = g * kFan + sub * (kFan / SPLIT) + wave * kLPW;
  uint64_t mkey = 0;
  uint32_t mcell = 0, mst = 0, mcnt = 0;
  float4 mlo = make_float4(0.f, 0.f, 0.f, 0.f), mhi = mlo;
  if (lane < kLPW && leaf0 + lane < c.nleaves) {
    mkey = gptr(c.leaf_key)[leaf0 + lane];
    if (!MIXED && !ALIAS) mcell = gptr(c.leaf_cell)[leaf0 + lane];
    const uint2 sc = gptr(c.leaf_sc)[leaf0 + lane];
    mst = sc.x;
    mcnt = sc.y;
    mlo = gptr(c.leaf_lo)[leaf0 + lane];
    mhi = gptr(c.leaf_hi)[leaf0 + lane];
  }
  const NSFPS_GLOBAL RunState &rs = rstate(c);
  const uint32_t done = *gptr(c.done);
  const uint32_t npicks = min(rs.nl[par ^ 1u], kListCap);
  const uint64_t kref = rs.kref0;
  const uint32_t S = rs.s0;
  const uint32_t gn = g < c.nl1 ? g : 0u;  // read unconditionally, used only if g < nl1
  // split: a sibling workgroup may have written its part already; either value
  // bounds this workgroup's points (distances only fall), but every wave has
  // to take the same one (s_nkey)
  uint64_t nkey = 0;
  if (SPLIT == 1) nkey = gptr(c.l1_key)[gn];
  else if (wave == 0) nkey = node_key(c, gn);
  uint32_t clo, chi;
  uint64_t uta = 0, utb = 0, utc = 0, utd = 0;
  // the node's box of points (x > its hi x: no points)
  const float4 nlo = gptr(c.l1_lo)[gn], nhi = gptr(c.l1_hi)[gn];
  // the cells of this wave's leaves' buckets: lane i < kLPW * na
  // holds word i of the wave's stretch of leaf_al
  const uint32_t na = ALIAS ? c.r.na : 1u;
  uint32_t mal = kNoCell;
  if (ALIAS) {
    const uint2 cb = gptr(c.l1_cbox)[gn];
    if (lane < kLPW * na && leaf0 + lane / na < c.nleaves)
      mal = gptr(c.leaf_al)[(size_t)leaf0 * na + lane];
    pin_sgpr(done, npicks, kref, S, nkey, cb.x, cb.y, nlo.x, nlo.y, nlo.z, nhi.x, nhi.y,
             nhi.z);
    if (g >= c.nl1 || done || cb.x == kNone) return;  // finished, or no points
    if (PROF) uta = __builtin_amdgcn_s_memrealtime();
    clo = cb.x;
    chi = cb.y;
  } else {
    // the run state and the node's record are read together, ahead of the exit
    pin_sgpr(done, npicks, kref, S, nkey, nlo.x, nlo.y, nlo.z, nhi.x, nhi.y, nhi.z);
    if (g >= c.nl1 || done || nlo.x > nhi.x) return;  // finished, or no points
    if (PROF) uta = __builtin_amdgcn_s_memrealtime();
    clo = pack_cell(cell_axis(c.r, 0, nlo.x), cell_axis(c.r, 1, nlo.y), cell_axis(c.r, 2, nlo.z));
    chi = pack_cell(cell_axis(c.r, 0, nhi.x), cell_axis(c.r, 1, nhi.y), cell_axis(c.r, 2, nhi.z));
  }
  const uint32_t nb = rs.nb;
  const uint64_t wlo = window_lo(kref, S, nb);
  // the node's cell range in the picks' box-test form
  const uint32_t clo11 = pack11(clo), chi11g = pack11(chi) | kGuards;
  for (uint32_t j = tid; j < kHistBins; j += kPassThreads) s_hist[j] = 0;
  if (tid == 0) s_np = 0;
  if (SPLIT > 1 && tid == 0) s_nkey = nkey;
  if (PROF && tid < 4) s_ct[tid] = 0;
  __syncthreads();
  if (SPLIT > 1) nkey = uni(s_nkey);
  if (PROF) utb = __builtin_amdgcn_s_memrealtime();
  // every thread's list entries are read together (entries past the list are
  // stale and unused)
  constexpr uint32_t kPickSlots = kListCap / kPassThreads;
  uint2 pcb[kPickSlots];
  float4 ppp[kPickSlots];
  uint32_t ppf[kPickSlots];
#pragma unroll
  for (uint32_t s = 0; s < kPickSlots; ++s) {
    if (s == 0 || s * kPassThreads < npicks) {
      pcb[s] = gptr(c.list_c)[s * kPassThreads + tid];
      ppp[s] = gptr(c.list_p)[s * kPassThreads + tid];
      ppf[s] = gptr(c.list_f)[s * kPassThreads + tid];
    }
  }
#pragma unroll
  for (uint32_t s = 0; s < kPickSlots; ++s) {
    const uint32_t i = s * kPassThreads + tid;
    if (s * kPassThreads >= npicks) break;  // uniform
    // a settled entry (a pick) whose cube overlaps the node's cells (cube lo
    // <= node hi and node lo <= cube hi on every axis: the guard test of
    // in_box11 crosswise), and that may lower one of its points (the node
    // key holds their largest distance)
    if (i < npicks && ppf[s] == 0u && in_box11(pcb[s].y, pcb[s].x, clo11, chi11g) &&
        !(box_bound(ppp[s].x, ppp[s].y, ppp[s].z, nlo.x, nlo.y, nlo.z, nhi.x, nhi.y, nhi.z) >=
          __uint_as_float((uint32_t)(nkey >> 32)))) {
      const uint32_t k = atomicAdd(&s_np, 1u);
      if (k < kPickLds) {
        s_pp[k] = make_float4(ppp[s].x, ppp[s].y, ppp[s].z, 0.f);
        s_pc[k] = pcb[s];
      } else {
        s_more[k - kPickLds] = (uint16_t)i;
      }
    }
  }
  __syncthreads();
  const uint32_t nall = s_np;
  const uint64_t ut1 = PROF ? __builtin_amdgcn_s_memrealtime() : 0;
  if (nall == 0 && nkey < wlo) return;  // nothing changes, nothing to count
  // which leaves a pick may lower a point of (hm: the first 64 picks), and
  // which must be read
  uint32_t st[kLPW], cnt[kLPW];
  uint64_t okey[kLPW], hm[kLPW];
  bool hit[kLPW], need[kLPW];
  uint32_t nsel = min(nall, kPickLds);
#pragma unroll
  for (uint32_t k = 0; k < kLPW; ++k) {
    okey[k] = ((uint64_t)rdlane((uint32_t)(mkey >> 32), k) << 32) | rdlane((uint32_t)mkey, k);
    st[k] = rdlane(mst, k);
    cnt[k] = rdlane(mcnt, k);
  }
  // A pick takes part in leaf k only if its squared distance to the leaf's
  // box (in sqdist's operation order, so never above a point's distance) is
  // below the leaf key's distance, the largest of its points: otherwise it
  // lowers none of them.
  const auto may_lower = [&](uint32_t k, float4 q) -> bool {
    return !(box_bound(q.x, q.y, q.z, __uint_as_float(rdlane(__float_as_uint(mlo.x), k)),
                       __uint_as_float(rdlane(__float_as_uint(mlo.y), k)),
                       __uint_as_float(rdlane(__float_as_uint(mlo.z), k)),
                       __uint_as_float(rdlane(__float_as_uint(mhi.x), k)),
                       __uint_as_float(rdlane(__float_as_uint(mhi.y), k)),
                       __uint_as_float(rdlane(__float_as_uint(mhi.z), k))) >=
             __uint_as_float((uint32_t)(okey[k] >> 32)));
  };
  // A pick of this cube updates the lane's point (lanes of leaf k): the cube
  // holds the cell of the point's bucket.  A pick nearer to a point than the
  // point's distance nearly always passes, so this is looked at only for
  // those; with shared buckets a leaf's box can span the grid, and the test
  // (any cell of the bucket) goes ahead of the points.
  const auto in_cube = [&](uint32_t k, uint32_t pc11, uint2 cube) -> bool {
    if (ALIAS) return true;
    const uint32_t a0 = MIXED ? pc11 : pack11(rdlane(mcell, k));
    return in_box11(a0 | kGuards, a0, cube.x, cube.y) != 0;
  };
  const auto touches = [&](uint32_t k, uint32_t i) -> bool {
    if (!ALIAS) return true;
    const uint2 cube = s_pc[i];
    uint32_t in = 0;
    for (uint32_t a = 0; a < na; ++a) {
      const uint32_t a0 = pack11(rdlane(mal, k * na + a));
      in |= in_box11(a0 | kGuards, a0, cube.x, cube.y);
    }
    return in != 0;
  };
  // kPickLds picks at a time: a node rarely has more (few nodes, many
  // samples a round), and the last of these passes counts the keys
  for (uint32_t ch = 0;;) {
  const bool last = nall - ch <= kPickLds;
  const bool in0 = lane < nsel;
  const float4 pp0 = s_pp[lane];  // past nsel: stale LDS, masked out
#pragma unroll
  for (uint32_t k = 0; k < kLPW; ++k) {
    hm[k] = __ballot(in0 && touches(k, lane) && may_lower(k, pp0));
    bool h = hm[k] != 0;
    for (uint32_t cb = 64; cb < nsel && !h; cb += 64)
      h = __ballot((cb + lane < nsel) && touches(k, cb + lane) && may_lower(k, s_pp[cb + lane])) != 0;
    hit[k] = h;
    need[k] = leaf0 + k < c.nleaves && (h || (last && okey[k] >= wlo));
  }
  if (PROF) {
    utc = __builtin_amdgcn_s_memrealtime();
    if (lane == 0) s_wt[2 * kPassWaves + wave] = (uint32_t)(utc - ut1);
  }
  if (PROF && lane == 0) {
    uint32_t nl = 0, npt = 0, nh = 0, nhp = 0;
#pragma unroll
    for (uint32_t k = 0; k < kLPW; ++k) {
      nl += need[k] ? 1u : 0u;
      npt += need[k] ? cnt[k] : 0u;
      nh += need[k] && hit[k] ? 1u : 0u;
      nhp += need[k] && hit[k] ? cnt[k] : 0u;
    }
    if (nl) {
      atomicAdd(&s_ct[0], nl);
      atomicAdd(&s_ct[1], npt);
      atomicAdd(&s_ct[2], nh);
      atomicAdd(&s_ct[3], nhp);
    }
  }
  float4 p[kLPW];
  uint32_t rk[kLPW];  // logical ranks
  // every lane loads, without a branch, so that the four leaves' loads are in
  // flight together; a lane without a point of a needed leaf reads slot 0
  // (one line for the whole wave) and its values are never used: every use
  // below is guarded by lane < cnt
#pragma unroll
  for (uint32_t k = 0; k < kLPW; ++k) {
    const uint32_t idx = need[k] && lane < cnt[k] ? st[k] + lane : 0u;
    p[k] = gptr(c.P4)[idx];
    rk[k] = gptr(c.R)[idx];
  }
  if (PROF) {  // wait for the points (profiled build only)
#pragma unroll
    for (uint32_t k = 0; k < kLPW; ++k) pin_vgpr(p[k].x, rk[k]);
    utd = __builtin_amdgcn_s_memrealtime();
    if (lane == 0) s_wt[wave] = (uint32_t)(utd - ut1);
  }
  // each leaf's stores are issued as soon as it is worked out, so that they
  // overlap the next leaves' work (deferring them all to the end measured
  // 0.23 ms slower per call on the 1M uniform cube)
#pragma unroll
  for (uint32_t k = 0; k < kLPW; ++k) {
    const uint32_t li = wave * kLPW + k;
    uint64_t key = 0;
    if (leaf0 + k < c.nleaves) {
      // unchanged unless the point holding the key is lowered below
      key = okey[k];
      if (need[k]) {
        const bool act = lane < cnt[k];
        const uint32_t lo = ~rk[k];
        float d = p[k].w;
        if (hit[k]) {
          // MIXED: this point's own cell (pack11), the cell its bucket is
          uint32_t pc11 = 0;
          if (MIXED)
            pc11 = pack11(pack_cell(cell_axis(c.r, 0, p[k].x), cell_axis(c.r, 1, p[k].y),
                                    cell_axis(c.r, 2, p[k].z)));
          for (uint32_t cb = 0; cb < nsel; cb += 64) {
            uint64_t m = cb == 0 ? hm[k]
                                 : __ballot((cb + lane < nsel) && touches(k, cb + lane) &&
                                            may_lower(k, s_pp[cb + lane]));
            while (m) {
              const uint32_t j = (uint32_t)__ffsll((long long)m) - 1;
              m &= m - 1;
              const float4 q = s_pp[cb + j];
              const float dd = sqdist(p[k].x, p[k].y, p[k].z, q.x, q.y, q.z);
              if (__ballot(dd < d)) {
                const uint2 qc = s_pc[cb + j];
                d = dd < d && in_cube(k, pc11, qc) ? dd : d;
              }
            }
          }
          const bool lowered = act && d < p[k].w;
          if (lowered) ((NSFPS_GLOBAL float *)gptr(c.P4 + st[k] + lane))[3] = d;
          if (__ballot(lowered && lo == (uint32_t)okey[k])) {
            const uint32_t hi = act ? __float_as_uint(d) : 0u;
            uint32_t mh;
            const uint32_t wl = key_winner(hi, lo, act, mh);
            key = ((uint64_t)mh << 32) | rdlane(lo, wl);  // the leaf has points: wl < 64
            if (lane == 0) gptr(c.leaf_key)[leaf0 + k] = key;
          }
        }
        if (act && last) {
          const uint32_t hi = __float_as_uint(d);
          const uint32_t b = key_bin(((uint64_t)hi << 32) | lo, kref, S, nb);
          if (b != kNone) atomicAdd(&s_hist[b], 1u);
        }
      }
    }
    okey[k] = key;
    if (lane == 0) s_lk[li] = key;
  }
  if (last) break;
  ch += kPickLds;
  nsel = min(nall - ch, kPickLds);
  __syncthreads();  // every wave is through with the picks before
  if (tid < nsel) {
    const uint32_t i = s_more[ch - kPickLds + tid];
    const float4 pp = gptr(c.list_p)[i];
    s_pp[tid] = make_float4(pp.x, pp.y, pp.z, 0.f);
    s_pc[tid] = gptr(c.list_c)[i];
  }
  __syncthreads();
  }
  if (PROF && lane == 0) s_wt[kPassWaves + wave] = (uint32_t)(__builtin_amdgcn_s_memrealtime() - ut1);
  __syncthreads();
  const uint64_t ut2 = PROF ? __builtin_amdgcn_s_memrealtime() : 0;
  if (wave == 0 && SPLIT == 1) {
    const uint64_t k = s_lk[lane];
    uint32_t mh;
    const uint32_t wl = key_winner((uint32_t)(k >> 32), (uint32_t)k, true, mh);
    if (lane == 0) gptr(c.l1_key)[g] = ((uint64_t)mh << 32) | (uint32_t)s_lk[wl];
  } else if (wave == 0) {
    // this quarter's largest key (keys are unique: the rank is their low word)
    const uint64_t part = wave_max_u64(lane < kFan / SPLIT ? s_lk[lane] : 0ull);
    if (lane == 0)
      __hip_atomic_store(gptr(c.l1_part) + (size_t)g * SPLIT + sub, part, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
  }
  NSFPS_GLOBAL uint32_t *H = hist_set(c);
  for (uint32_t j = tid; j < kHistBins; j += kPassThreads) {
    const uint32_t v = s_hist[j];
    if (v) atomicAdd(&H[j], v);
  }
  if (PROF && tid == 0) {
    const uint64_t ut3 = __builtin_amdgcn_s_memrealtime();
    unsigned long long *pw = (unsigned long long *)gptr(c.prof);
    atomicAdd(pw + kUpTPicks, (unsigned long long)(ut1 - ut0));
    atomicAdd(pw + kUpTLeaves, (unsigned long long)(ut2 - ut1));
    atomicAdd(pw + kUpTFlush, (unsigned long long)(ut3 - ut2));
    atomicAdd(pw + kUpGroups, 1ull);
    atomicAdd(pw + kUpTLoad, (unsigned long long)(uta - ut0));
    atomicAdd(pw + kUpTZero, (unsigned long long)(utb - uta));
    atomicAdd(pw + kUpTHits, (unsigned long long)(utc - ut1));
    atomicAdd(pw + kUpTPts, (unsigned long long)(utd - utc));
    uint32_t pmax = 0, psum = 0, lmax = 0, lsum = 0, hmax = 0, hsum = 0;
    for (uint32_t w = 0; w < kPassWaves; ++w) {
      hmax = max(hmax, s_wt[2 * kPassWaves + w]);
      hsum += s_wt[2 * kPassWaves + w];
      pmax = max(pmax, s_wt[w]);
      psum += s_wt[w];
      lmax = max(lmax, s_wt[kPassWaves + w]);
      lsum += s_wt[kPassWaves + w];
    }
    atomicAdd(pw + kUpWPtsMax, (unsigned long long)pmax);
    atomicAdd(pw + kUpWPtsSum, (unsigned long long)psum);
    atomicAdd(pw + kUpWLoopMax, (unsigned long long)lmax);
    atomicAdd(pw + kUpWLoopSum, (unsigned long long)lsum);
    atomicAdd(pw + kUpWHitsMax, (unsigned long long)hmax);
    atomicAdd(pw + kUpWHitsSum, (unsigned long long)hsum);
    atomicAdd(pw + kCtUpLeaves, (unsigned long long)s_ct[0]);
    atomicAdd(pw + kCtUpPoints, (unsigned long long)s_ct[1]);
    atomicAdd(pw + kCtUpHitLeaves, (unsigned long long)s_ct[2]);
    atomicAdd(pw + kCtUpHitPoints, (unsigned long long)s_ct[3]);
  }
}

// ------------------------------------------------------- refinement passes

// Refinement pass `pass` (1 or 2): counts the keys inside the window the
// selection replayed from the earlier histograms asks for; does nothing when
// the threshold is already resolved.  Few workgroups, each striding over the
// level-1 nodes: the pass is usually skipped, and then costs little more than
// its launch.
__global__ __launch_bounds__(kPassThreads) void k_refine(const CloudDev *__restrict__ clouds,
                                                         uint32_t pass, uint32_t passes) {
  __shared__ uint32_t s_hist[kHistBins];
  __shared__ uint32_t s_sc[kPassWaves + 3];
  const CloudDev &c = clouds[blockIdx.y];
  if (blockIdx.x >= c.nl1 || *gptr(c.done)) return;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const Sel s = sel_replay(c, pass, passes, s_sc);
  if (s.state != 0 || s.pass != pass) return;
  const uint64_t wlo = window_lo(s.kref, s.S);
  for (uint32_t j = tid; j < kHistBins; j += kPassThreads) s_hist[j] = 0;
  __syncthreads();
  for (uint32_t g = blockIdx.x; g < c.nl1; g += gridDim.x) {
    if (node_key(c, g) < wlo) continue;
    for (uint32_t k = 0; k < kLeavesPerWave; ++k) {
      const uint32_t leaf = g * kFan + wave * kLeavesPerWave + k;
      if (leaf >= c.nleaves || gptr(c.leaf_key)[leaf] < wlo) continue;
      const uint2 sc = gptr(c.leaf_sc)[leaf];
      const uint32_t st = sc.x, cnt = sc.y;
      if (lane < cnt) {
        const float d = ((const NSFPS_GLOBAL float *)gptr(c.P4 + st + lane))[3];
        const uint32_t rank = gptr(c.R)[st + lane];
        const uint32_t b = key_bin(((uint64_t)__float_as_uint(d) << 32) | ~rank, s.kref, s.S);
        if (b != kNone) atomicAdd(&s_hist[b], 1u);
      }
    }
  }
  __syncthreads();
  NSFPS_GLOBAL uint32_t *H = hist_set(c) + pass * kHistBins;
  for (uint32_t j = tid; j < kHistBins; j += kPassThreads) {
    const uint32_t v = s_hist[j];
    if (v) atomicAdd(&H[j], v);
  }
}

// ------------------------------------------------------------- gather pass

__device__ __forceinline__ uint32_t bit_length(uint64_t v) { return v ? 64u - __clzll(v) : 0u; }

// Resolves the threshold from the histograms and appends every point whose key
// is >= it to the list.  When no threshold below the maximum fits the list
// (more than kListCap keys inside the finest bin), the threshold is the
// maximum key itself: a run of one sample.  Few workgroups, each striding over
// the level-1 nodes; most nodes hold no key above the threshold.  PROF: counts
// the hot leaves whose points it reads and those points.  Its first workgroup
// also finds the sampling's end: when m samples have keys above every key
// left, or only points at distance 0 are left (src/yuezu_fps.cpp:705-706).
// may_seq: the accept pass that follows can take samples one after another.
// The end is left in rs.fin, which no workgroup of this launch tests; the
// accept pass tests fin and writes done, which none of its own tests.  With
// one word for both, waves of one workgroup could read it before and after
// the write, and those that went on would scan LDS words that the others
// never wrote.
template <bool PROF>
__global__ __launch_bounds__(kPassThreads) void k_gather(const CloudDev *__restrict__ clouds,
                                                         uint32_t passes, uint32_t par,
                                                         uint32_t may_seq) {
  __shared__ uint32_t s_sc[kPassWaves + 3];
  __shared__ uint64_t s_wk[kPassWaves];
  const CloudDev &c = clouds[blockIdx.y];
  const uint64_t gt0 = PROF ? __builtin_amdgcn_s_memrealtime() : 0;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  // Reads that depend on nothing read before them go out together with the
  // run state: the update pass's histogram bins and the first node chunk's
  // leaf records.
  const uint4 h0 = gptr(reinterpret_cast<const uint4 *>(c.hist))[tid];
  const auto leaf_of = [&](uint32_t c0, uint32_t &gq) {
    gq = c0 + (lane / kLeavesPerWave) * gridDim.x;
    return gq * kFan + wave * kLeavesPerWave + lane % kLeavesPerWave;
  };
  uint64_t lkey = 0;
  uint32_t lst = 0, lcnt = 0;
  const auto read_leaf = [&](uint32_t c0) {
    uint32_t gq;
    const uint32_t lf = leaf_of(c0, gq);
    lkey = 0;
    lst = lcnt = 0;
    if (gq < c.nl1 && lf < c.nleaves) {
      lkey = gptr(c.leaf_key)[lf];
      const uint2 sc = gptr(c.leaf_sc)[lf];
      lst = sc.x;
      lcnt = sc.y;
    }
  };
  read_leaf(blockIdx.x);
  NSFPS_GLOBAL RunState &rs = *gptr(c.rs);
  if (blockIdx.x >= c.nl1 || *gptr(c.done)) {
    // done: the accept pass, which sets it, tests fin
    if (blockIdx.x == 0 && tid == 0) rs.fin = 1;
    return;
  }
  uint64_t gt1 = 0, gt2 = 0, gt3 = 0;
  bool forced = false;
  const Sel s = sel_replay(c, passes + 1, passes, s_sc, &forced, &h0);
  uint64_t bkey = s.bkey, ktop = s.ktop;
  if (s.state == 2) {
    uint64_t best = 0;
    for (uint32_t j = tid; j < c.nl1; j += kPassThreads) {
      const uint64_t k = node_key(c, j);
      best = k > best ? k : best;
    }
    best = wave_max_u64(best);
    if (lane == 0) s_wk[wave] = best;
    __syncthreads();
    best = 0;
    for (uint32_t w = 0; w < kPassWaves; ++w) best = s_wk[w] > best ? s_wk[w] : best;
    bkey = ktop = best;
  }
  if (PROF) gt1 = __builtin_amdgcn_s_memrealtime();
  if (blockIdx.x == 0) {  // uniform
    const uint32_t T = rs.ntaken, m = c.m;
    bool fin = (uint32_t)(ktop >> 32) == 0u;  // only points at distance 0 are left
    if (!fin && T >= m) {
      // the samples above every key left: all of the rounds whose thresholds
      // were, and those of the later rounds that are
      __shared__ uint32_t s_first, s_above;
      if (tid == 0) {
        s_first = T;
        s_above = 0;
      }
      __syncthreads();
      for (uint32_t j = tid; j < rs.nlog; j += kPassThreads)
        if (gptr(c.log_bmin)[j] <= ktop) atomicMin(&s_first, gptr(c.log_start)[j]);
      __syncthreads();
      const uint32_t w0 = s_first;
      uint32_t n = 0;
      for (uint32_t j = w0 + tid; j < T; j += kPassThreads)
        n += (((uint64_t)gptr(c.smp_d)[j] << 32) | gptr(c.smp_lo)[j]) > ktop ? 1u : 0u;
      n = rdlane(wave_incl_scan(n), 63);
      if (lane == 0) atomicAdd(&s_above, n);
      __syncthreads();
      fin = w0 + s_above >= m;
    }
    if (tid == 0) {
      rs.bkey = bkey;
      rs.ktop = ktop;
      // rounds that take samples one after another, and the one after them
      const bool early = rs.seq != 0u || T < c.seq_samples;
      rs.seq = may_seq && T < c.seq_samples ? 1u : 0u;
      // the first rounds start from windows over the whole key range and are
      // forced as a rule, and few of a list are sampled in the early ones;
      // later forced rounds ask for refinement passes
      rs.forced += forced && rs.rounds >= 2 && (!early || s.total < 64u) ? 1u : 0u;
      // next round: bins of 1/512 to 1/1024 of this round's key span, over 3
      // spans (a window that ends above the next threshold leaves the list
      // short; most leaves with a key in it are read anyway, for a sample
      // reaches them); where the list came out short, over four to eight
      // times the whole window down to the threshold.  8M clustered points:
      // 1.75 spans 292 rounds, 17.8 ms; 2: 261, 16.5; 3: 247, 16.1; 4: 246,
      // 16.2 (1M cube 2.57, 2.55, 2.62, 2.68; with kListGrow 8 for 4, 3 spans
      // 2.56 and 16.0).
      const bool grow = 2 * s.total < rs.cap;
      const uint64_t span = (grow || T < c.seq_samples ? rs.kref0 : ktop) - bkey + 1;
      const uint32_t bins = T < c.seq_samples ? 11u : 10u;
      uint32_t nx = bit_length(span);
      nx = nx > bins ? nx - bins : 0u;
      nx = nx < kMaxShift ? nx : kMaxShift;
      rs.s0_next = nx;
      rs.nb_next = grow || T < c.seq_samples ? kHistBins : min((uint32_t)(span >> nx) * 3 + 1, kHistBins);
      if (fin) {
        *gptr(c.iter) = min(T, m);
        rs.fin = 1;
      }
    }
    if (fin) return;
  }
  // Nodes in chunks of kGatherNodes; lane l of a wave holds leaf l % 4 of the
  // wave's four leaves of node l / 4 of the chunk, so one read brings in all
  // its leaf records.  The points of the first kGatherHold hot leaves stay in
  // registers, the others are read again for writing; the workgroup takes one
  // range of the list per chunk (one global atomic).
  static_assert(kGatherNodes * kLeavesPerWave == 64, "one leaf record per lane");
  __shared__ uint32_t s_cnt, s_base;
  for (uint32_t c0 = blockIdx.x; c0 < c.nl1; c0 += kGatherNodes * gridDim.x) {
    if (c0 != blockIdx.x) read_leaf(c0);
    const bool hot = lcnt != 0 && lkey >= bkey;  // an empty or absent leaf has key 0
    if (PROF) {
      pin_vgpr(lst, lcnt, (uint32_t)hot);
      if (!gt2) gt2 = __builtin_amdgcn_s_memrealtime();
    }
    if (tid == 0) s_cnt = 0;
    uint64_t rest = __ballot(hot);
    if (PROF) {
      const uint64_t hp = __ballot(hot);
      const uint32_t pts = rdlane(wave_incl_scan(hot ? lcnt : 0u), 63);
      if (lane == 0 && hp) {
        atomicAdd((unsigned long long *)gptr(c.prof) + kCtGaLeaves,
                  (unsigned long long)__popcll(hp));
        atomicAdd((unsigned long long *)gptr(c.prof) + kCtGaPoints, (unsigned long long)pts);
      }
    }
    float4 hp[kGatherHold];
    uint2 hr[kGatherHold];
    uint32_t hn[kGatherHold];
    uint64_t htk[kGatherHold];
    // the held leaves' points: every lane loads, without a branch, so that
    // the loads are in flight together; a lane past the leaf's points, or of
    // a wave with fewer hot leaves, reads slot 0 and its values go unused
    // (hn[u] = 0 when there is no leaf)
#pragma unroll
    for (uint32_t u = 0; u < kGatherHold; ++u) {
      const bool have = rest != 0;
      const uint32_t j = have ? (uint32_t)__builtin_ctzll(rest) : 0u;
      rest &= rest - 1;
      const uint32_t st = rdlane(lst, j), cnt = have ? rdlane(lcnt, j) : 0u;
      hn[u] = cnt;
      const uint32_t idx = lane < cnt ? st + lane : 0u;
      hp[u] = gptr(c.P4)[idx];
      hr[u] = gptr(c.RO)[idx];
    }
    uint32_t mine = 0;
#pragma unroll
    for (uint32_t u = 0; u < kGatherHold; ++u) {
      htk[u] = __ballot(lane < hn[u] &&
                        (((uint64_t)__float_as_uint(hp[u].w) << 32) | ~hr[u].x) >= bkey);
      mine += (uint32_t)__popcll(htk[u]);
    }
    const uint64_t later = rest;  // hot leaves beyond the first kGatherHold: counted now,
    while (rest) {                // read again to be written
      const uint32_t j = (uint32_t)__builtin_ctzll(rest);
      rest &= rest - 1;
      const uint32_t st = rdlane(lst, j), cnt = rdlane(lcnt, j);
      bool take = false;
      if (lane < cnt) {
        const float d = ((const NSFPS_GLOBAL float *)gptr(c.P4 + st + lane))[3];
        take = (((uint64_t)__float_as_uint(d) << 32) | ~gptr(c.R)[st + lane]) >= bkey;
      }
      mine += (uint32_t)__popcll(__ballot(take));
    }
    __syncthreads();  // s_cnt is zero
    uint32_t base = 0;
    if (lane == 0 && mine) base = atomicAdd(&s_cnt, mine);
    __syncthreads();
    if (tid == 0) s_base = s_cnt ? atomicAdd(&rs.nl[par], s_cnt) : 0u;
    __syncthreads();
    base = s_base + rdlane(base, 0);
    if (PROF && !gt3) gt3 = __builtin_amdgcn_s_memrealtime();
    // the list's pointers in vector registers: a pointer loaded again from
    // the arguments after a store would first wait for the store
    NSFPS_GLOBAL float4 *const LP = vgpr_ptr(gptr(c.list_p));
    NSFPS_GLOBAL uint2 *const LR = vgpr_ptr(gptr(c.list_r));
    NSFPS_GLOBAL uint32_t *const LF = vgpr_ptr(gptr(c.list_f));
    // arguments by value: a reference into hp / hr would make those arrays
    // memory (the compiler then keeps them in LDS)
    const auto put = [&](float4 p, uint2 ro, uint64_t m) {
      if ((m >> lane) & 1u) {
        const uint32_t i = base + lanes_below(m);
        if (i < kListCap) {
          LP[i] = p;
          LR[i] = ro;
          LF[i] = 0u;  // not in conflict, until the accept pass finds it is
        } else {
          rs.err = 1;
        }
      }
      base += (uint32_t)__popcll(m);
    };
#pragma unroll
    for (uint32_t u = 0; u < kGatherHold; ++u) put(hp[u], hr[u], htk[u]);
    rest = later;
    while (rest) {
      const uint32_t j = (uint32_t)__builtin_ctzll(rest);
      rest &= rest - 1;
      const uint32_t st = rdlane(lst, j), cnt = rdlane(lcnt, j);
      float4 p = make_float4(0.f, 0.f, 0.f, 0.f);
      uint2 ro = make_uint2(0u, 0u);
      if (lane < cnt) {
        p = gptr(c.P4)[st + lane];
        ro = gptr(c.RO)[st + lane];
      }
      const bool take = lane < cnt && (((uint64_t)__float_as_uint(p.w) << 32) | ~ro.x) >= bkey;
      put(p, ro, __ballot(take));
    }
    __syncthreads();  // s_base is read before the next chunk's claim
  }
  if (PROF && tid == 0 && blockIdx.x == 0) {
    unsigned long long *pw = (unsigned long long *)gptr(c.prof);
    atomicAdd(pw + kGaWinKeys, (unsigned long long)s.win);
    atomicAdd(pw + kGaListed, (unsigned long long)s.total);
    atomicMax(pw + kGaWinMax, (unsigned long long)s.win);
  }
  if (PROF && tid == 0 && gt3) {  // the first chunk's clocks; the writes: every chunk's rest
    const uint64_t t = __builtin_amdgcn_s_memrealtime();
    unsigned long long *pw = (unsigned long long *)gptr(c.prof);
    atomicAdd(pw + kGaTSel, (unsigned long long)(gt1 - gt0));
    atomicAdd(pw + kGaTLeaf, (unsigned long long)(gt2 - gt1));
    atomicAdd(pw + kGaTClaim, (unsigned long long)(gt3 - gt2));
    atomicAdd(pw + kGaTWrite, (unsigned long long)(t - gt3));
    atomicAdd(pw + kGaGroups, 1ull);
  }
}

// ------------------------------------------------------------- accept pass

// Settles the list.  Two entries conflict when their sqdist is below the
// larger of their distances: only then can either lower the other.  An entry
// that conflicts with no entry of a larger key is a sample with the key it
// has:
//   - every point of a larger key is in the list, and those not settled yet
//     are too far to lower it;
//   - every sample that precedes it and was near enough has been applied by
//     the update passes since.
// It may be applied to all points at once: a point of a larger key that it
// could lower would have been in conflict with it.  The largest key never has
// a conflict above it, so every round settles at least one entry; entries
// that stay come again in the next round's list.  The samples' order is the
// order of their keys (k_order).
//
// All pairs of the list: a wave's lanes hold two entries each and meet a
// chunk of others, read through the scalar cache (uniform addresses), at 10
// vector instructions a pair.  At 4,096 entries (16.7 M pairs) that is 4.3 us
// of the chip's issue; 1,024 entries are bound by the kernel's latency.  A
// few workgroups beside these find the entries' cubes for the update pass.
constexpr uint32_t kAcceptThreads = 256;
constexpr uint32_t kAcceptWaves = kAcceptThreads / 64;
constexpr uint32_t kAcceptX = 128;  // entries held by a wave
constexpr uint32_t kAcceptChunk = 16;  // others they meet
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
#if defined(__HIP_DEVICE_COMPILE__)
#define NSFPS_CONSTANT __attribute__((address_space(4)))
#else
#define NSFPS_CONSTANT
#endif

// The first seq_samples of a cloud, and the rest of the list that reaches
// them, are taken one after another instead, as the reference does: early
// layers hold few samples, so a list is worth several rounds of them.  One
// workgroup, four entries a thread, one barrier a sample: each wave publishes
// its largest key, every wave takes the largest of those, and the entries that
// the sample's cube holds are lowered; it ends when no listed key is left at
// or above the threshold.  These samples come in order, so a call that ends
// among them needs no sort.  Bound by the chain of one sample: some 200
// instructions, two LDS reads and the barrier, about 0.8 us (1.35 with the
// cube's half-widths worked out on every lane alike, 1.05 with keys compared
// as integer pairs).  Lists and windows are the first rounds' there: 1,024
// entries, bins of 1/1024 to 1/2048 of the span below the last threshold.
constexpr uint32_t kSettleSlots = kSeqList / kAcceptThreads;
static_assert(kSettleSlots * kAcceptThreads == kSeqList, "whole slots");

// Keys as doubles: their high words are finite floats' bits, below the
// exponent of infinities, so they order as the integers do, and one
// instruction takes a maximum (subnormal doubles are kept).
__device__ __forceinline__ double max_key(double a, double b) {
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
template <int CTRL>
__device__ __forceinline__ double max_key_dpp(double a) {
  const uint64_t k = (uint64_t)__double_as_longlong(a);
  const uint64_t o = ((uint64_t)dpp_mov<CTRL>((uint32_t)(k >> 32)) << 32) | dpp_mov<CTRL>((uint32_t)k);
  return max_key(a, __longlong_as_double((long long)o));
}
__device__ __forceinline__ uint64_t wave_max_key(double a) {
  a = max_key_dpp<kDppQuad1032>(a);
  a = max_key_dpp<kDppQuad2301>(a);
  a = max_key_dpp<kDppHalfMirror>(a);
  a = max_key_dpp<kDppMirror>(a);
  const uint64_t k = (uint64_t)__double_as_longlong(a);
  const uint32_t hi = (uint32_t)(k >> 32), lo = (uint32_t)k;
  uint64_t best = ((uint64_t)rdlane(hi, 0) << 32) | rdlane(lo, 0);
#pragma unroll
  for (uint32_t r = 16; r < 64; r += 16) {
    const uint64_t v = ((uint64_t)rdlane(hi, r) << 32) | rdlane(lo, r);
    best = v > best ? v : best;
  }
  return best;
}

template <bool ALIAS>
__device__ __forceinline__ void settle(const CloudDev &c, uint32_t par, uint32_t nl) {
  struct Cand {
    uint64_t key;
    uint32_t row, cell;  // input row, cell (pack11)
    float x, y, z;
    uint32_t entry;  // of the list
  };
  __shared__ Cand s_cand[2][kAcceptWaves];
  // the range at hand: reads of it from memory would wait for the sample's stores
  __shared__ RangeDev s_r;
  NSFPS_GLOBAL RunState &rs = *gptr(c.rs);
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  if (tid < sizeof(RangeDev) / 4)
    reinterpret_cast<uint32_t *>(&s_r)[tid] = reinterpret_cast<const uint32_t *>(&c.r)[tid];
  // lane 8 a + k compares the distance with threshold k of axis a (half_axis)
  static_assert(3 * kCubeThr <= 64, "a lane per threshold");
  const float thr = lane < 3 * kCubeThr ? (&c.r.cube_thr[0][0])[lane] : INFINITY;
  // a sample's words, one a lane: distance, ~rank, row, and the row as a result
  NSFPS_GLOBAL uint32_t *const SW = vgpr_ptr(gptr(
      lane == 0 ? c.smp_d : lane == 1 ? c.smp_lo : lane == 2 ? c.smp_row : reinterpret_cast<uint32_t *>(c.out)));
  NSFPS_GLOBAL uint2 *const LC = vgpr_ptr(gptr(c.list_c));
  const uint32_t T = rs.ntaken, end = c.m;
  const uint64_t bkey = rs.bkey;
  float x[kSettleSlots], y[kSettleSlots], z[kSettleSlots];
  uint32_t row[kSettleSlots], cell[kSettleSlots];
  uint64_t key[kSettleSlots];
#pragma unroll
  for (uint32_t s = 0; s < kSettleSlots; ++s) {
    const uint32_t i = s * kAcceptThreads + tid;
    const float4 p = gptr(c.list_p)[i];
    const uint2 r = gptr(c.list_r)[i];
    x[s] = p.x;
    y[s] = p.y;
    z[s] = p.z;
    key[s] = i < nl ? make_key(p.w, r.x) : 0ull;
    row[s] = r.y;
    cell[s] = i < nl ? pack11(pack_cell(cell_axis(c.r, 0, p.x), cell_axis(c.r, 1, p.y),
                                        cell_axis(c.r, 2, p.z)))
                     : 0u;
  }
  uint32_t cnt = 0, taken = 0;
  uint64_t top;
  __syncthreads();
  const uint32_t b0 = uniform(s_r.blocks[0]), b1 = uniform(s_r.blocks[1]), b2 = uniform(s_r.blocks[2]);
  while (true) {
    double best = __longlong_as_double((long long)key[0]);
#pragma unroll
    for (uint32_t s = 1; s < kSettleSlots; ++s)
      best = max_key(best, __longlong_as_double((long long)key[s]));
    const uint64_t mine = wave_max_key(best);
    Cand *const cd = s_cand[cnt & 1u];
#pragma unroll
    for (uint32_t s = 0; s < kSettleSlots; ++s)
      if (key[s] == mine)  // keys are unique, but for the absent ones' 0
        cd[wave] = Cand{mine, row[s], cell[s], x[s], y[s], z[s], s * kAcceptThreads + tid};
    __syncthreads();
    uint32_t w = 0;
    top = cd[0].key;
#pragma unroll
    for (uint32_t v = 1; v < kAcceptWaves; ++v) {
      const uint64_t k = cd[v].key;
      w = k > top ? v : w;
      top = k > top ? k : top;
    }
    top = uni(top);
    if (top < bkey || (top >> 32) == 0 || T + cnt >= end) break;
    const Cand p = cd[uniform(w)];
    const float px = uni(p.x), py = uni(p.y), pz = uni(p.z), D = key_dist(top);
    const uint32_t c11 = uniform(p.cell), e = uniform(p.entry), at = T + cnt;
    const uint64_t ge = __ballot(D >= thr);
    uint32_t lo_c, hi_c, h = 0, beyond = 0;
#pragma unroll
    for (uint32_t a = 0; a < 3; ++a) {
      const uint32_t k = (uint32_t)__popc((uint32_t)(ge >> (a * kCubeThr)) & ((1u << kCubeThr) - 1));
      h |= k << (10 * a);
      beyond |= k == kCubeThr ? 1u : 0u;
    }
    if (beyond) h = uniform(packed_halves(s_r, D));
    cube_corners((c11 & 1023u) | (((c11 >> 11) & 1023u) << 10) | ((c11 >> 22) << 20), h, b0, b1, b2,
                 lo_c, hi_c);
    const uint2 cube = make_uint2(uniform(pack11(lo_c)), uniform(pack11(hi_c) | kGuards));
    if (tid < 4) SW[at] = lane == 0 ? (uint32_t)(top >> 32) : lane == 1 ? (uint32_t)top : p.row;
    if (tid == e % kAcceptThreads) {
      taken |= 1u << (e / kAcceptThreads);
      LC[e] = cube;
    }
#pragma unroll
    for (uint32_t s = 0; s < kSettleSlots; ++s) {
      const uint32_t dd = __float_as_uint(sqdist(x[s], y[s], z[s], px, py, pz));
      bool in = (dd < (uint32_t)(key[s] >> 32)) &
                (in_box11(cell[s] | kGuards, cell[s], cube.x, cube.y) != 0);
      if (ALIAS && dd < (uint32_t)(key[s] >> 32) && !in) in = bucket_in_cube(s_r, cell[s], cube);
      key[s] = in ? ((uint64_t)dd << 32) | (uint32_t)key[s] : key[s];
    }
    ++cnt;
  }
#pragma unroll
  for (uint32_t s = 0; s < kSettleSlots; ++s)
    if (s * kAcceptThreads + tid < nl)
      gptr(c.list_f)[s * kAcceptThreads + tid] = (taken >> s) & 1u ? 0u : 1u;
  if (tid == 0) {
    // every sample's key is above top, and every key left at or below kref0
    const uint64_t low = top >= bkey ? top + 1 : bkey, b = low < rs.bmin ? low : rs.bmin;
    const uint32_t i = rs.nlog < c.log_cap ? rs.nlog : c.log_cap - 1;
    rs.bmin = b;
    gptr(c.log_bmin)[i] = b;
    if (rs.nlog < c.log_cap) {
      gptr(c.log_ktop)[i] = rs.ktop;
      gptr(c.log_start)[i] = T;
      rs.nlog += 1;
    }
    rs.ntaken = T + cnt;
    *gptr(c.iter) = T + cnt;
    rs.cap = T + cnt < c.seq_samples ? kSeqList : min(kListMin, c.list_cap);
    rs.kref0 = low - 1;
    if (T + cnt >= c.m) *gptr(c.done) = 1;
  }
}

// SEQ: may take the list's samples one after another (rs.seq); a variant of its
// own, for it needs registers that the layers' rounds leave to more waves (in
// one kernel the 50-round scan was 4 % slower).
template <bool ALIAS, bool SEQ>
__global__ __launch_bounds__(kAcceptThreads) void k_accept(const CloudDev *__restrict__ clouds,
                                                           uint32_t par, uint32_t ncube) {
  const CloudDev &c = clouds[blockIdx.y];
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  NSFPS_GLOBAL RunState &rs = *gptr(c.rs);
  // list_cap / kAcceptX groups of entries, each against every chunk
  const uint32_t xgs = c.list_cap / kAcceptX;
  const bool cubes = blockIdx.x < ncube;
  const uint32_t w = uniform(cubes ? 0u : (blockIdx.x - ncube) * kAcceptWaves + (tid >> 6));
  const uint32_t x0 = (w % xgs) * kAcceptX + lane, q0 = (w / xgs) * kAcceptChunk;
  const uint32_t nl = min(rs.nl[par], kListCap), fin = rs.fin;
  // entries past the list are stale and unused
  float4 X[2];
  uint32_t XR[2];
#pragma unroll
  for (uint32_t t = 0; t < 2; ++t) {
    X[t] = gptr(c.list_p)[x0 + 64 * t];
    XR[t] = gptr(c.list_r)[x0 + 64 * t].x;
  }
  if (fin) {  // found by the gather pass, of this round or an earlier one
    if (blockIdx.x == 0 && tid == 0) *gptr(c.done) = 1;
    return;
  }
  // the histograms this round's selection read are cleared for the next
  // round's update pass
  NSFPS_GLOBAL uint4 *const hz = reinterpret_cast<NSFPS_GLOBAL uint4 *>(hist_set(c));
  for (uint32_t j = blockIdx.x * kAcceptThreads + tid; j < kHists * kHistBins / 4;
       j += gridDim.x * kAcceptThreads)
    hz[j] = make_uint4(0u, 0u, 0u, 0u);
  if (blockIdx.x == 0 && tid == 0) {
    rs.nl[par ^ 1u] = 0;  // the next round's list
    rs.kref0 = rs.ktop;   // keys only decrease
    rs.s0 = rs.s0_next;
    rs.nb = rs.nb_next;
    rs.rounds += 1;
  }
  if (SEQ && rs.seq) {  // written by the gather pass
    if (blockIdx.x == 0) settle<ALIAS>(c, par, min(nl, kSeqList));
    return;
  }
  if (cubes) {
    const uint32_t i = blockIdx.x * kAcceptThreads + tid;
    if (i < nl) {
      const float4 p = gptr(c.list_p)[i];
      gptr(c.list_c)[i] = sample_cube(
          c.r, pack11(pack_cell(cell_axis(c.r, 0, p.x), cell_axis(c.r, 1, p.y), cell_axis(c.r, 2, p.z))),
          p.w);
      // a point at distance 0 is never a sample
      if (p.w == 0.0f) gptr(c.list_f)[i] = 1u;
    }
    return;
  }
  if (x0 - lane >= nl || q0 >= nl) return;
  uint64_t kx[2];
#pragma unroll
  for (uint32_t t = 0; t < 2; ++t)
    kx[t] = x0 + 64 * t < nl ? make_key(X[t].w, XR[t]) : ~0ull;  // absent: nothing lies above it
  const NSFPS_CONSTANT v4f *const LP = (const NSFPS_CONSTANT v4f *)c.list_p + q0;
  const NSFPS_CONSTANT v2u *const LR = (const NSFPS_CONSTANT v2u *)c.list_r + q0;
  const uint32_t nq = min(nl - q0, kAcceptChunk);
  bool blocked[2] = {false, false};
#pragma unroll 8
  for (uint32_t j = 0; j < nq; ++j) {
    const v4f q = LP[j];
    const uint64_t kq = make_key(q.w, LR[j].x);
#pragma unroll
    for (uint32_t t = 0; t < 2; ++t)
      blocked[t] |= (kq > kx[t]) & (sqdist(X[t].x, X[t].y, X[t].z, q.x, q.y, q.z) < q.w);
  }
#pragma unroll
  for (uint32_t t = 0; t < 2; ++t)
    if (blocked[t]) gptr(c.list_f)[x0 + 64 * t] = 1u;
}

// Sorts each round's samples by key, descending (one workgroup a round; a
// round settles at most kListCap): bins of equal width over the round's span,
// then each sample's place among its bin's.  The log's last entry may stand
// for many rounds: its samples are sorted kListCap at a time.
constexpr uint32_t kSortThreads = 512;
__global__ __launch_bounds__(kSortThreads) void k_sort_rounds(const CloudDev *__restrict__ clouds) {
  const CloudDev &c = clouds[blockIdx.y];
  constexpr uint32_t kSlots = kListCap / kSortThreads, kWaves = kSortThreads / 64;
  __shared__ uint2 s_key[kListCap];
  __shared__ __align__(16) uint32_t s_bin[kListCap + 4];
  __shared__ uint16_t s_at[kListCap];
  __shared__ uint32_t s_wn[kWaves];
  __shared__ uint64_t s_mx[2];
  if (!*gptr(c.done)) return;
  const NSFPS_GLOBAL RunState &rs = *gptr(c.rs);
  const uint32_t nlog = rs.nlog, T = min(rs.ntaken, c.n), tid = threadIdx.x;
  if (nlog == 0) return;
  // the last entry's pieces go on as if each had an entry
  const uint32_t last = gptr(c.log_start)[nlog - 1];
  const uint32_t pieces = T > last ? (T - last + kListCap - 1) / kListCap : 1u;
  for (uint32_t r = blockIdx.x; r < nlog - 1 + pieces; r += gridDim.x) {
    const uint32_t b = r < nlog ? gptr(c.log_start)[r] : last + (r - (nlog - 1)) * kListCap;
    const uint32_t e = r + 1 < nlog ? gptr(c.log_start)[r + 1] : min(b + kListCap, T);
    const uint32_t n = e - b;
    if (n < 2 || n > kListCap) continue;  // never above it
    uint2 k[kSlots];
    uint32_t row[kSlots], bin[kSlots], at[kSlots];
    for (uint32_t j = tid; j < kListCap + 4; j += kSortThreads) s_bin[j] = 0;
    if (tid < 2) s_mx[tid] = 0;
    __syncthreads();
    uint64_t mx = 0, mn = 0;
#pragma unroll
    for (uint32_t s = 0; s < kSlots; ++s) {
      const uint32_t i = s * kSortThreads + tid;
      k[s] = make_uint2(0u, 0u);
      if (i < n) {
        k[s] = make_uint2(gptr(c.smp_lo)[b + i], gptr(c.smp_d)[b + i]);
        row[s] = gptr(c.smp_row)[b + i];
        const uint64_t kk = ((uint64_t)k[s].y << 32) | k[s].x;
        mx = kk > mx ? kk : mx;
        mn = ~kk > mn ? ~kk : mn;
        s_key[i] = k[s];
      }
    }
    mx = wave_max_u64(mx);
    mn = wave_max_u64(mn);
    if ((tid & 63u) == 0) {
      atomicMax((unsigned long long *)&s_mx[0], (unsigned long long)mx);
      atomicMax((unsigned long long *)&s_mx[1], (unsigned long long)mn);
    }
    __syncthreads();
    const uint64_t top = s_mx[0], span = top - ~s_mx[1];
    const uint32_t bl = bit_length(span), S = bl > 12u ? bl - 12u : 0u;
#pragma unroll
    for (uint32_t s = 0; s < kSlots; ++s) {
      if (s * kSortThreads + tid < n) {
        bin[s] = (uint32_t)((top - (((uint64_t)k[s].y << 32) | k[s].x)) >> S);
        at[s] = atomicAdd(&s_bin[bin[s]], 1u);
      }
    }
    __syncthreads();
    {
      static_assert(kSlots == 8, "two uint4 of bins a thread");
      uint4 v[2];
      uint32_t sum = 0, tot;
#pragma unroll
      for (uint32_t j = 0; j < 2; ++j) {
        v[j] = reinterpret_cast<const uint4 *>(s_bin)[2 * tid + j];
        sum += v[j].x + v[j].y + v[j].z + v[j].w;
      }
      uint32_t pre = block_excl_scan<kWaves>(sum, s_wn, &tot);
#pragma unroll
      for (uint32_t j = 0; j < 2; ++j) {
        reinterpret_cast<uint4 *>(s_bin)[2 * tid + j] =
            make_uint4(pre, pre + v[j].x, pre + v[j].x + v[j].y, pre + v[j].x + v[j].y + v[j].z);
        pre += v[j].x + v[j].y + v[j].z + v[j].w;
      }
      if (tid == 0) s_bin[kListCap] = tot;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t s = 0; s < kSlots; ++s)
      if (s * kSortThreads + tid < n) s_at[s_bin[bin[s]] + at[s]] = (uint16_t)(s * kSortThreads + tid);
    __syncthreads();
#pragma unroll
    for (uint32_t s = 0; s < kSlots; ++s) {
      if (s * kSortThreads + tid < n) {
        const uint32_t b0 = s_bin[bin[s]], b1 = s_bin[bin[s] + 1];
        const uint64_t kk = ((uint64_t)k[s].y << 32) | k[s].x;
        uint32_t p = b0;
        for (uint32_t j = b0; j < b1; ++j) {
          const uint2 o = s_key[s_at[j]];
          p += (((uint64_t)o.y << 32) | o.x) > kk ? 1u : 0u;
        }
        gptr(c.smp_d)[b + p] = k[s].y;
        gptr(c.smp_lo)[b + p] = k[s].x;
        gptr(c.smp_row)[b + p] = row[s];
      }
    }
    __syncthreads();
  }
}

// The samples' places: sample i's is the number of samples with larger keys.
// Samples of rounds whose smallest threshold so far is above its key all
// precede it, those of rounds whose largest key is below it all follow; in
// the rounds between (sorted by key) binary searches find how many precede
// it.  Bound by the latency of their reads: kOrderLanes lanes per sample take
// a round each (1,000 samples: 18 us with one lane a sample, 5 so).
constexpr uint32_t kOrderThreads = 256;
constexpr uint32_t kOrderLanes = 16;
__global__ __launch_bounds__(kOrderThreads) void k_order(const CloudDev *__restrict__ clouds) {
  const CloudDev &c = clouds[blockIdx.y];
  if (!*gptr(c.done)) return;
  const NSFPS_GLOBAL RunState &rs = *gptr(c.rs);
  constexpr uint32_t kPer = kOrderThreads / kOrderLanes;  // samples of a workgroup
  const uint32_t T = min(rs.ntaken, c.n), nlog = rs.nlog, m = c.m;
  const uint32_t sub = threadIdx.x % kOrderLanes;
  const NSFPS_GLOBAL uint32_t *const sd = gptr(c.smp_d), *const sl = gptr(c.smp_lo);
  for (uint32_t i = blockIdx.x * kPer + threadIdx.x / kOrderLanes; i < T; i += gridDim.x * kPer) {
    const uint64_t k = ((uint64_t)sd[i] << 32) | sl[i];
    uint32_t r = 0;
    if (i) {  // sample 0 (input row 0) has the largest key and is in no round
      uint32_t a0 = 0, a1 = nlog, e0 = 0, e1 = nlog;
      while (a0 < a1) {  // the first round whose smallest threshold so far is <= k
        const uint32_t mid = (a0 + a1) / 2;
        if (gptr(c.log_bmin)[mid] <= k) a1 = mid;
        else a0 = mid + 1;
      }
      while (e0 < e1) {  // the first round whose largest key is < k
        const uint32_t mid = (e0 + e1) / 2;
        if (gptr(c.log_ktop)[mid] < k) e1 = mid;
        else e0 = mid + 1;
      }
      if (sub == 0) r = a0 < nlog ? gptr(c.log_start)[a0] : T;
      for (uint32_t q = a0 + sub; q < e0; q += kOrderLanes) {
        const uint32_t end = q + 1 < nlog ? gptr(c.log_start)[q + 1] : T;
        // one sorted piece, but for a full log's last entry
        for (uint32_t b = gptr(c.log_start)[q]; b < end; b += kListCap) {
          const uint32_t e = min(b + kListCap, end);
          if (i >= b && i < e) {
            r += i - b;
            continue;
          }
          uint32_t lo = b, hi = e;
          while (lo < hi) {
            const uint32_t mid = (lo + hi) / 2;
            const uint32_t d = sd[mid];
            if (d > (uint32_t)(k >> 32) || (d == (uint32_t)(k >> 32) && sl[mid] > (uint32_t)k)) lo = mid + 1;
            else hi = mid;
          }
          r += lo - b;
        }
      }
    }
#pragma unroll
    for (uint32_t off = kOrderLanes / 2; off; off >>= 1) r += __shfl_xor(r, off, kOrderLanes);
    if (sub == 0 && r < m) gptr(c.out)[r] = (int32_t)gptr(c.smp_row)[i];
  }
}

// ------------------------------------------------------------------ setup

// First round: the only pick is input row 0 (the first sample) with a cube
// over the whole grid.
__global__ __launch_bounds__(kPassThreads) void k_runs_init(const CloudDev *__restrict__ clouds,
                                                           uint32_t split) {
  const CloudDev &c = clouds[blockIdx.x];
  const uint32_t tid = threadIdx.x;
  // split: each node's key moves into its first part (the other parts and
  // l1_key zero); otherwise the parts are zero
  for (uint32_t i = tid; i < c.nl1; i += kPassThreads) {
    NSFPS_GLOBAL uint64_t *const pp = gptr(c.l1_part) + (size_t)i * kUpdateSplit;
    const uint64_t k = gptr(c.l1_key)[i];
    for (uint32_t s = 0; s < kUpdateSplit; ++s) pp[s] = split && s == 0 ? k : 0ull;
    if (split) gptr(c.l1_key)[i] = 0;
  }
  if (tid == 0) {
    NSFPS_GLOBAL RunState &rs = *gptr(c.rs);
    rs.kref0 = ~0ull;
    rs.bkey = 0;
    rs.s0 = kMaxShift;
    rs.s0_next = kMaxShift;
    rs.nb = rs.nb_next = kHistBins;
    rs.nl[0] = 0;
    rs.nl[1] = 1;  // read by round 0
    rs.ntaken = 1;
    rs.nlog = 0;
    rs.cap = c.seq_samples > 1 ? kSeqList : min(kListMin, c.list_cap);
    rs.seq = 0;
    rs.bmin = ~0ull;
    rs.ktop = ~0ull;
    rs.rounds = 0;
    rs.err = 0;
    rs.forced = 0;
    const float4 p0 = *gptr(c.root_pos);
    gptr(c.smp_d)[0] = gptr(c.smp_lo)[0] = 0xffffffffu;
    gptr(c.smp_row)[0] = 0;
    gptr(c.out)[0] = 0;
    gptr(c.list_f)[0] = 0;
    gptr(c.list_p)[0] = make_float4(p0.x, p0.y, p0.z, INFINITY);
    gptr(c.list_c)[0] = make_uint2(
        0u, pack11(pack_cell(c.r.blocks[0] - 1, c.r.blocks[1] - 1, c.r.blocks[2] - 1)) | kGuards);
    *gptr(c.iter) = 1;
    *gptr(c.done) = rs.fin = c.m <= 1 ? 1u : 0u;
  }
  for (uint32_t j = tid; j < kHists * kHistBins; j += kPassThreads) gptr(c.hist)[j] = 0;
}

// ---------------------------------------------------------------- launchers

// The variants a call without profiling may launch.
hipError_t preload_runs_kernels() {
  constexpr uint32_t S = kUpdateSplit;
  return func_attributes(
      k_runs_init, k_refine, k_gather<false>, k_accept<false, false>, k_accept<false, true>,
      k_accept<true, true>, k_sort_rounds, k_order,
      k_update<false, false, 1, false>, k_update<false, false, S, false>,
      k_update<false, true, 1, false>, k_update<false, true, S, false>,
      k_update<false, false, 1, true>, k_update<false, false, S, true>);
}

hipError_t launch_runs_init(const CloudDev *d_clouds, uint32_t nclouds, uint32_t split,
                            hipStream_t st) {
  k_runs_init<<<nclouds, kPassThreads, 0, st>>>(d_clouds, split);
  return hipGetLastError();
}

// Round `round` of one variant: update (and one workgroup recording the last
// round's samples), gather and accept passes.
template <bool PROF, bool ALIAS, uint32_t SPLIT, bool MIXED>
void launch_round(const CloudDev *d_clouds, uint32_t nclouds, dim3 grid, dim3 sparse,
                  uint32_t passes, uint32_t list_cap, uint32_t round, bool seq, hipStream_t st) {
  k_update<PROF, ALIAS, SPLIT, MIXED>
      <<<dim3(grid.x * SPLIT + 1, grid.y), kPassThreads, 0, st>>>(d_clouds, round);
  for (uint32_t p = 1; p <= passes; ++p)
    k_refine<<<sparse, kPassThreads, 0, st>>>(d_clouds, p, passes);
  k_gather<PROF><<<sparse, kPassThreads, 0, st>>>(d_clouds, passes, round & 1u, seq ? 1u : 0u);
  const uint32_t ncube = (list_cap + kAcceptThreads - 1) / kAcceptThreads;
  const uint32_t xgs = list_cap / kAcceptX;
  const dim3 blocks(ncube + xgs * (list_cap / kAcceptChunk) / kAcceptWaves, nclouds);
  if (seq)
    k_accept<ALIAS, true><<<blocks, kAcceptThreads, 0, st>>>(d_clouds, round & 1u, ncube);
  else
    k_accept<false, false><<<blocks, kAcceptThreads, 0, st>>>(d_clouds, round & 1u, ncube);
}

hipError_t launch_order(const CloudDev *d_clouds, uint32_t nclouds, uint32_t m, hipStream_t st) {
  // some more samples than m are settled
  const uint32_t want = (uint32_t)(((uint64_t)m + m / 8) * kOrderLanes / kOrderThreads) + 2;
  k_sort_rounds<<<dim3(m < 64u ? m : nclouds > 1 ? 64u : 256u, nclouds), kSortThreads, 0, st>>>(d_clouds);
  k_order<<<dim3(want < 8192u ? want : 8192u, nclouds), kOrderThreads, 0, st>>>(d_clouds);
  return hipGetLastError();
}

hipError_t launch_rounds(const CloudDev *d_clouds, uint32_t nclouds, uint32_t max_nl1,
                         uint32_t rounds, uint32_t passes, bool profile, bool alias,
                         bool split, bool mixed, uint32_t list_cap, uint32_t first,
                         uint32_t seq_rounds, hipStream_t st) {
  if (alias && mixed) return hipErrorInvalidValue;  // leaves of several buckets: one cell each
  if (list_cap < kListShort || list_cap > kListCap || (list_cap & (list_cap - 1)))
    return hipErrorInvalidValue;
  const dim3 grid(max_nl1, nclouds);
  const uint32_t share = kSparseLaunch / nclouds < 2 ? 2u : kSparseLaunch / nclouds;
  const uint32_t groups = share < kSparseGroups ? share : kSparseGroups;
  const dim3 sparse(max_nl1 < groups ? max_nl1 : groups, nclouds);
  using Launch = void (*)(const CloudDev *, uint32_t, dim3, dim3, uint32_t, uint32_t, uint32_t,
                          bool, hipStream_t);
  constexpr uint32_t S = kUpdateSplit;
  // [profile][cells: one per leaf, shared buckets, several per leaf][split]
  static constexpr Launch kRound[2][3][2] = {
      {{launch_round<false, false, 1, false>, launch_round<false, false, S, false>},
       {launch_round<false, true, 1, false>, launch_round<false, true, S, false>},
       {launch_round<false, false, 1, true>, launch_round<false, false, S, true>}},
      {{launch_round<true, false, 1, false>, launch_round<true, false, S, false>},
       {launch_round<true, true, 1, false>, launch_round<true, true, S, false>},
       {launch_round<true, false, 1, true>, launch_round<true, false, S, true>}}};
  const Launch one = kRound[profile][alias ? 1 : mixed ? 2 : 0][split];
  for (uint32_t r = 0; r < rounds; ++r)
    one(d_clouds, nclouds, grid, sparse, passes, list_cap, first + r, first + r < seq_rounds, st);
  return hipGetLastError();
}

}  // namespace nsfps
