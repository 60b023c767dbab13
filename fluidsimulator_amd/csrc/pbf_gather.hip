// Neighbor lists and gather passes of the particles outside the LDS tiles.
//
// Every sum of a pass runs over a particle's neighbors in the reference's
// order (27 cells in (dz, dy, dx) order, each by ascending id), because float
// additions do not commute with rounding.  Only the additions are ordered:
// the terms are independent.  So a group of lanes computes the terms of one
// particle's neighbors side by side, hands them over through LDS, and one
// lane per accumulator (rho, the three gradient sums and the sum of squares
// in lambda; the three components elsewhere) adds them in list order.  A
// neighbor then costs the chain one addition instead of a whole term, and no
// lane waits for another particle's longer list.
//
//   runs         maximal runs of consecutive slots of one cell that hold one
//                position and one velocity (bit for bit, after gravity):
//                their lists hold the same values in the same order, so the
//                first slot (the head) stands for all and writes every
//                slot's outputs.  Without runs (gather modes 1 and 3) every
//                slot is a head.  Recorded substeps and diagnostics store
//                the list of every slot of a run.
//   list heads   heads of cells of fewer than kDenseCell particles, with at
//                most row_cap neighbors: their neighbors' slots are stored
//                in a row; kListLanes lanes work on one head.
//   dense units  up to kUnitHeads heads of one cell of kDenseCell particles or more
//                (their 27 cells are the same), or one head with more
//                neighbors than a row holds: no list.  A wavefront walks the
//                runs of the 27 cells, retesting the list predicate on p^0 (the
//                same predicate in the same order visits exactly the list).  A
//                run's neighbors all give one term, added once per member.
//
// Rows lie in the tile list buffer: a slot outside the tiles leaves its part
// of it unused.

#include <algorithm>
#include <type_traits>

#include "exact_sum.h"
#include "pbf_ctx.h"
#include "pbf_device.h"

namespace fluidhip {

namespace {

constexpr int kWave = 64;
constexpr int kBlock = 256;     // workgroup of every kernel here
constexpr int kWaves = kBlock / kWave;
constexpr int kListLanes = 8;   // lanes per list head in the passes
constexpr int kNbrLanes = 32;   // lanes per list head in the neighbor build
constexpr int kExpand = 256;    // candidates a list head's LDS buffer holds
static_assert(kTileList / 2 <= kExpand, "a row must fit the LDS buffer");

__device__ __forceinline__ bool fatal(const unsigned* flags) {
  return (*flags & kFlagFatal) != 0u;
}

__device__ __forceinline__ int lane_id() { return static_cast<int>(threadIdx.x) & (kWave - 1); }

// The value of lane j (uniform).
__device__ __forceinline__ float lane_of(float v, int j) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), j));
}

// Orders this wavefront's LDS accesses: what its lanes stored before is what
// its lanes load after.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Keep loads of these (uniform, or per lane) from being moved below the next branch.
__device__ __forceinline__ void loaded(int a) { asm volatile("" ::"s"(a)); }
__device__ __forceinline__ void loaded(const int4& v) {
  asm volatile("" ::"v"(v.x), "v"(v.y), "v"(v.z), "v"(v.w));
}

// Inclusive prefix sum over groups of kW lanes.
template <int kW>
__device__ __forceinline__ int incl_scan(int v) {
  const int g = lane_id() & (kW - 1);
#pragma unroll
  for (int o = 1; o < kW; o <<= 1) {
    const int u = __shfl_up(v, o, kW);
    if (g >= o) v += u;
  }
  return v;
}

__device__ __forceinline__ bool same_bits3(const float3& a, const float3& b) {
  return ((__float_as_uint(a.x) ^ __float_as_uint(b.x)) | (__float_as_uint(a.y) ^ __float_as_uint(b.y)) |
          (__float_as_uint(a.z) ^ __float_as_uint(b.z))) == 0u;
}

// ------------------------------------------------------------ heads

// Bits of a slot's class: a run head, a list head, a dense cell's head, a
// cell's first slot.
constexpr int kHead = 1, kList = 2, kDense = 4, kCell = 8;
// Heads of a dense unit, at most, and the heads of dense cells a batch has for
// each head of a unit.  A unit's wavefront shares every ordered addition among
// its heads, but units of more heads are fewer and longer.  Measured (ms per
// four substeps of the splashing 262,144-particle dam breaks, 11,700 such heads):
// units of up to 1 / 4 / 8 heads 12.0 / 8.1 / 8.1; one more head a unit for every
// 512 / 2,048 / 4,096 heads 8.8 / 8.1 / 10.6.  Eight heads only where that
// leaves a unit for every wavefront the chip holds at once (4,096; ms per two
// substeps of the piled-up million-particle block, 56,000 such heads: 12.3
// with four, 10.8 with eight).
constexpr int kUnitHeads = 8;
constexpr int kHeadsPerUnitHead = 2048;

// Heads per dense unit (a power of two) for `heads` heads of dense cells.
__device__ __forceinline__ int unit_heads(int heads) {
  const int k = heads / kHeadsPerUnitHead;
  return k >= 2 * kUnitHeads ? kUnitHeads : k >= 4 ? 4 : k >= 2 ? 2 : 1;
}

// The class of slot s (0 for slots that are no head; a tile's heads are
// neither list nor dense heads, the tile kernels compute each of its slots).
__device__ __forceinline__ int slot_class(const StepConsts& c, int s,
                                          const float4* __restrict__ posB,
                                          const float4* __restrict__ velB,
                                          const int* __restrict__ slot_key,
                                          const int* __restrict__ start,
                                          const int* __restrict__ in_tile) {
  // every load is issued before any test
  const int before = max(s - 1, 0);
  const int k = slot_key[s], kb = slot_key[before];
  const float3 x = ld3(posB, s), xb = ld3(posB, before);
  const float3 v = ld3(velB, s), vb = ld3(velB, before);
  const int tile = in_tile ? in_tile[s] : 0;
  const int a = start[k], b = start[k + 1];
  if (c.runs && s > 0 && k == kb && same_bits3(x, xb) && same_bits3(v, vb)) return 0;
  if (tile) return kHead;
  if (b - a < kDenseCell) return kHead | kList;
  return s == a ? kHead | kDense | kCell : kHead | kDense;
}

// The slots of workgroup b of the two kernels below: whole multiples of
// kBlock slots.
__device__ __forceinline__ void head_range(int n, int& b0, int& b1) {
  const int per = (n + static_cast<int>(gridDim.x) * kBlock - 1) /
                  (static_cast<int>(gridDim.x) * kBlock) * kBlock;
  b0 = min(n, static_cast<int>(blockIdx.x) * per);
  b1 = min(n, b0 + per);
}

// Each slot's class (into run_no) and each workgroup's counts of runs, list
// heads and dense cells' heads (partial[0..G), [G..2G), [2G..3G)).
__global__ __launch_bounds__(kBlock) void k_head_count(
    StepConsts c, const float4* __restrict__ posB, const float4* __restrict__ velB,
    const int* __restrict__ slot_key, const int* __restrict__ start,
    const int* __restrict__ in_tile, int* __restrict__ run_no, int* __restrict__ partial,
    const unsigned* __restrict__ flags) {
  __shared__ int sums[3][kWaves];
  if (fatal(flags)) return;
  int b0, b1;
  head_range(c.n, b0, b1);
  int nh = 0, nl = 0, nd = 0;  // uniform over a wavefront
  for (int s0 = b0; s0 < b1; s0 += kBlock) {
    const int s = s0 + static_cast<int>(threadIdx.x);
    int cls = 0;
    if (s < b1) {
      cls = slot_class(c, s, posB, velB, slot_key, start, in_tile);
      run_no[s] = cls;
    }
    nh += __popcll(__ballot(cls & kHead));
    nl += __popcll(__ballot(cls & kList));
    nd += __popcll(__ballot(cls & kDense));
  }
  if (lane_id() == 0) {
    const int w = threadIdx.x / kWave;
    sums[0][w] = nh;
    sums[1][w] = nl;
    sums[2][w] = nd;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    int t = 0;
    for (int w = 0; w < kWaves; ++w) t += sums[threadIdx.x][w];
    partial[threadIdx.x * gridDim.x + blockIdx.x] = t;
  }
}

// From the classes: each slot's run number, the runs' first slots (rep, with
// rep[runs] = n) and the list heads (units[].x, scene in units[].w) in slot
// order, and the dense units in any order (one atomic per kBlock slots);
// info = {runs, list heads, dense units, heads per unit}.  velB.w holds each slot's scene
// here.  Slots outside the tiles start without a stored list.
__global__ __launch_bounds__(kBlock) void k_heads(
    StepConsts c, const int* __restrict__ partial, const float4* __restrict__ velB,
    int* __restrict__ run_no, int* __restrict__ rep, int4* __restrict__ units,
    int2* __restrict__ dense, int* __restrict__ info, const int* __restrict__ in_tile,
    long long* __restrict__ noff, int* __restrict__ nwords, int* __restrict__ ncount,
    const unsigned* __restrict__ flags) {
  __shared__ int red[6][kWaves];
  __shared__ int wsum[kWaves];
  __shared__ int dsum[kWaves];
  __shared__ int dbase;
  if (fatal(flags)) return;
  const int G = gridDim.x;
  const int lane = lane_id(), w = threadIdx.x / kWave;
  // counts of the workgroups before this one, and of all
  int pre[3] = {0, 0, 0}, all[3] = {0, 0, 0};
  for (int j = threadIdx.x; j < G; j += kBlock) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int v = partial[k * G + j];
      all[k] += v;
      pre[k] += j < static_cast<int>(blockIdx.x) ? v : 0;
    }
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    for (int o = kWave / 2; o > 0; o >>= 1) {
      pre[k] += __shfl_xor(pre[k], o);
      all[k] += __shfl_xor(all[k], o);
    }
    if (lane == 0) {
      red[k][w] = pre[k];
      red[3 + k][w] = all[k];
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    pre[k] = all[k] = 0;
    for (int v = 0; v < kWaves; ++v) {
      pre[k] += red[k][v];
      all[k] += red[3 + k][v];
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    info[0] = all[0];
    info[1] = all[1];
    info[3] = unit_heads(all[2]);
    rep[all[0]] = c.n;
  }
  const int unit = unit_heads(all[2]);
  int b0, b1;
  head_range(c.n, b0, b1);
  const unsigned long long below = (1ull << lane) - 1ull;
  for (int s0 = b0; s0 < b1; s0 += kBlock) {
    const int s = s0 + static_cast<int>(threadIdx.x);
    const int cls = s < b1 ? run_no[s] : 0;
    const unsigned long long mh = __ballot(cls & kHead), ml = __ballot(cls & kList);
    // two counts of at most kBlock each in one word
    if (lane == 0) wsum[w] = __popcll(mh) | (__popcll(ml) << 16);
    __syncthreads();
    int mine = 0, total = 0;
    for (int v = 0; v < kWaves; ++v) {
      mine += v < w ? wsum[v] : 0;
      total += wsum[v];
    }
    const int r = pre[0] + (mine & 0xffff) + __popcll(mh & below);
    // a dense unit starts at its cell's first run and at multiples of `unit`
    const bool lead = (cls & kDense) && ((cls & kCell) || (r & (unit - 1)) == 0);
    const unsigned long long md = __ballot(lead);
    if (lane == 0) dsum[w] = __popcll(md);
    __syncthreads();
    int dmine = 0, dtotal = 0;
    for (int v = 0; v < kWaves; ++v) {
      dmine += v < w ? dsum[v] : 0;
      dtotal += dsum[v];
    }
    if (dtotal > 0) {  // uniform over the workgroup
      if (threadIdx.x == 0) dbase = atomicAdd(info + 2, dtotal);
      __syncthreads();
      if (lead)
        dense[dbase + dmine + __popcll(md & below)] =
            make_int2(s, __float_as_int(velB[s].w));
    }
    if (s < b1) {
      const bool head = (cls & kHead) != 0;
      run_no[s] = head ? r : r - 1;
      if (head) rep[r] = s;
      if (cls & kList)
        units[pre[1] + (mine >> 16) + __popcll(ml & below)] =
            make_int4(s, 0, 0, __float_as_int(velB[s].w));
      if (!(in_tile && in_tile[s])) {
        noff[s] = 0;
        nwords[s] = -1;
        ncount[s] = 0;
      }
    }
    pre[0] += total & 0xffff;
    pre[1] += total >> 16;
    __syncthreads();  // wsum, dsum and dbase are reused
  }
}

// Both kernels in one workgroup, for batches of up to kSmallHeads particles
// (two launches of 5 us each become one): thread t holds slots t, t + 1024, ...
__global__ __launch_bounds__(1024) void k_heads_small(
    StepConsts c, const float4* __restrict__ posB, const float4* __restrict__ velB,
    const int* __restrict__ slot_key, const int* __restrict__ start,
    const int* __restrict__ in_tile, int* __restrict__ run_no, int* __restrict__ rep,
    int4* __restrict__ units, int2* __restrict__ dense, int* __restrict__ info,
    long long* __restrict__ noff, int* __restrict__ nwords, int* __restrict__ ncount,
    const unsigned* __restrict__ flags) {
  constexpr int kT = 1024, kW = kT / kWave, kR = kSmallHeads / kT;
  static_assert(kR * kT == kSmallHeads, "whole rounds");
  // (round, wavefront) counts, padded to whole rounds of their scan
  constexpr int kCounts = kR * kW, kScan = (kCounts + kWave - 1) / kWave * kWave;
  __shared__ int runs[kScan], lists[kScan];
  __shared__ int nd_sh, ndense;
  if (fatal(flags)) return;
  const int n = c.n, tid = threadIdx.x, lane = lane_id(), w = tid / kWave;
  const unsigned long long below = (1ull << lane) - 1ull;
  if (tid == 0) nd_sh = ndense = 0;
  if (tid < kScan - kCounts) runs[kCounts + tid] = lists[kCounts + tid] = 0;
  int cls[kR];
#pragma unroll
  for (int r = 0; r < kR; ++r) {
    const int s = r * kT + tid;
    cls[r] = s < n ? slot_class(c, s, posB, velB, slot_key, start, in_tile) : 0;
  }
  __syncthreads();
  int nd = 0;
#pragma unroll
  for (int r = 0; r < kR; ++r) {
    const int h = __popcll(__ballot(cls[r] & kHead)), l = __popcll(__ballot(cls[r] & kList));
    nd += __popcll(__ballot(cls[r] & kDense));
    if (lane == 0) {
      runs[r * kW + w] = h;
      lists[r * kW + w] = l;
    }
  }
  if (lane == 0 && nd) atomicAdd(&nd_sh, nd);
  __syncthreads();
  // exclusive sums over the (round, wavefront) counts, in slot order
  if (w < 2) {
    int* a = w == 0 ? runs : lists;
    int carry = 0;
#pragma unroll
    for (int i = 0; i < kScan; i += kWave) {
      const int v = a[i + lane];
      const int inc = incl_scan<kWave>(v);
      a[i + lane] = carry + inc - v;
      carry += __shfl(inc, kWave - 1);
    }
    if (lane == 0) {
      info[w] = carry;
      if (w == 0) rep[carry] = n;
    }
  }
  __syncthreads();
  const int unit = unit_heads(nd_sh);
#pragma unroll
  for (int r = 0; r < kR; ++r) {
    const int s = r * kT + tid;
    const unsigned long long mh = __ballot(cls[r] & kHead), ml = __ballot(cls[r] & kList);
    const int run = runs[r * kW + w] + __popcll(mh & below);
    if (s < n) {
      const bool head = (cls[r] & kHead) != 0;
      run_no[s] = head ? run : run - 1;
      if (head) rep[run] = s;
      if (cls[r] & (kList | kDense)) {
        const int sc = __float_as_int(velB[s].w);
        if (cls[r] & kList)
          units[lists[r * kW + w] + __popcll(ml & below)] = make_int4(s, 0, 0, sc);
        else if ((cls[r] & kCell) || (run & (unit - 1)) == 0)
          dense[atomicAdd(&ndense, 1)] = make_int2(s, sc);
      }
      if (!(in_tile && in_tile[s])) {
        noff[s] = 0;
        nwords[s] = -1;
        ncount[s] = 0;
      }
    }
  }
  __syncthreads();
  if (tid == 0) {
    info[2] = ndense;
    info[3] = unit;
  }
}

// ------------------------------------------------------------ cells

// The slot range of cell `ci` (0..26, in (dz, dy, dx) order) around the cell
// of slot s of scene sc; bad when it lies outside the table (which has a one-cell margin
// around the bounding box of these same cells: never for a valid slot).
__device__ __forceinline__ bool cell_range(const GatherView& gv, int s, int sc, int ci, int& a,
                                           int& b) {
  a = b = 0;
  const GridDesc g = gv.grid[sc];
  int x, y, z;
  unpack_cell(gv.slot_cell[s], x, y, z);
  const int rx = x - g.ox, ry = y - g.oy, rz = z - g.oz;
  const int ext = 1 << g.bshift;  // cells per brick edge
  if (rx < 1 || ry < 1 || rz < 1 || rx > ext * g.nbx - 2 || ry > ext * g.nby - 2 ||
      rz > ext * g.nbz - 2)
    return false;
  if (ci < 27) {
    const int k = cell_key(rx + ci % 3 - 1, ry + (ci / 3) % 3 - 1, rz + ci / 9 - 1, g);
    a = gv.start[k];
    b = gv.start[k + 1];
  }
  return true;
}

// The non-empty ranges of a walk in order: range j holds entries
// [off[j], off[j + 1]), entry e being index base[j] + e; off[m] = total for
// the last range m and INT_MAX-like bounds are not needed beyond it.
struct Ranges {
  int off[28];
  int base[28];
};

// Lane j < 27 of a group of kW lanes brings range [lo, hi); returns the
// total.  Every lane of the group calls it.
template <int kW>
__device__ __forceinline__ int pack_ranges(Ranges& R, int lo, int hi) {
  const int lane = lane_id();
  const int g = lane & (kW - 1);
  const int cnt = g < 27 ? hi - lo : 0;
  const int inc = incl_scan<kW>(cnt);
  const int total = __shfl(inc, kW - 1, kW);
  unsigned long long m = __ballot(cnt > 0);
  if (kW < kWave) m = (m >> (lane & ~(kW - 1))) & ((1ull << (kW & 63)) - 1ull);
  if (cnt > 0) {
    const int j = __popcll(m & ((1ull << g) - 1ull));
    R.off[j] = inc - cnt;
    R.base[j] = lo - (inc - cnt);
  }
  if (g == 0) R.off[__popcll(m)] = total;
  return total;
}

// A lane's position in the ranges: entries are asked for in ascending order.
struct RangeCursor {
  int j = 0;
  int next;  // off[j + 1]
  int base;
  __device__ __forceinline__ void begin(const Ranges& R) {
    next = R.off[1];
    base = R.base[0];
  }
  // the index of entry e < total
  __device__ __forceinline__ int at(const Ranges& R, int e) {
    while (e >= next) {
      ++j;
      next = R.off[j + 1];
      base = R.base[j];
    }
    return base + e;
  }
};

// The run numbers of the non-empty slot range [a, b) (runs do not span cells).
__device__ __forceinline__ void run_range(const GatherView& gv, int a, int b, int& ra, int& rb) {
  ra = rb = 0;
  if (a < b) {
    ra = gv.run_no[a];
    rb = gv.run_no[b - 1] + 1;
  }
}

// ------------------------------------------------------------ lists

// Encodes a list as run-length words: a word t >= 0 is the single neighbor
// t; a word with the top bit set starts a run of consecutive slots, the next
// word being its length (3 or more, so that a list of as many words as
// neighbors is plain slots).  The words in order give the neighbors in order.
// Used by whole wavefronts with uniform values; `write` marks the lane that
// stores.
struct RunWriter {
  int* out;
  bool write;
  long long words = 0;
  int count = 0;
  int run_start = -1;
  int run_len = 0;
  template <bool kFill>
  __device__ __forceinline__ void flush() {
    if (run_len == 1 || run_len == 2) {  // (two words either way)
      if (kFill && write)
        for (int i = 0; i < run_len; ++i) out[words + i] = run_start + i;
      words += run_len;
    } else if (run_len > 2) {
      if (kFill && write) {
        out[words] = run_start | static_cast<int>(0x80000000u);
        out[words + 1] = run_len;
      }
      words += 2;
    }
    run_len = 0;
  }
  // neighbors a, a+1, ..., b-1
  template <bool kFill>
  __device__ __forceinline__ void add_range(int a, int b) {
    if (a >= b) return;
    count += b - a;
    if (run_len > 0 && a == run_start + run_len) {
      run_len += b - a;
      return;
    }
    flush<kFill>();
    run_start = a;
    run_len = b - a;
  }
};

// Neighbor lists of the list heads (core.cpp:205-247): candidates are the 27
// cells in (dz, dy, dx) order, each by ascending slot (= ascending id);
// neighbors the other candidates with near0.  kNbrLanes lanes per head: lane
// j < 27 looks cell j up, the cells' slots are laid out in LDS, and each lane
// tests every kNbrLanes-th candidate; a ballot keeps the order.  A head with
// more than kExpand candidates walks the 27 cells' runs instead (one test per
// run) and stops once its neighbors outgrow the row: it becomes a dense unit,
// and its own unit is left without neighbors.  units[u] becomes {slot, neighbors
// (-1: dense), slots of the run, scene}.  kFull also stores every list as
// run-length words (the diagnostics read them).
//
// One lane per particle used to walk the 27 cells twice (count, then fill),
// a chain of dependent loads: 127 us per launch for a 19x17x13 block, where
// this takes 6.7, and 617 for the 256-scene ensemble, where this takes 467
// (beside the tile lists; the 27 cell lookups of sparse spray bound it).
template <bool kFull>
__global__ __launch_bounds__(kBlock) void k_neighbors(
    StepConsts c, GatherView gv, int4* __restrict__ units, int2* __restrict__ dense,
    int* __restrict__ info, int4* __restrict__ rows, long long* __restrict__ noff,
    int* __restrict__ nwords, int* __restrict__ ncount, int* __restrict__ nbr, long long nbr_cap,
    unsigned long long* __restrict__ nbr_total, unsigned* __restrict__ flags) {
  constexpr int kHeads = kBlock / kNbrLanes;  // heads per workgroup and round
  __shared__ __align__(16) int buf_sh[kHeads][kExpand];
  __shared__ Ranges rng_sh[kHeads];
  __shared__ int cnt_sh[kHeads];
  __shared__ long long base_sh;
  __shared__ int abort_sh;
  const int grp = static_cast<int>(threadIdx.x) / kNbrLanes;
  // asked for at once, as in the passes
  const int4 ahead = units[min(c.n - 1, static_cast<int>(blockIdx.x) * kHeads + grp)];
  const int L = info[1];
  const bool failed = fatal(flags);
  loaded(L);
  loaded(ahead);
  if (kFull) {
    // Other workgroups may raise the neighbor flag at any time: read it once
    // per workgroup so that the barriers below stay uniform.
    if (threadIdx.x == 0) abort_sh = failed ? 1 : 0;
    __syncthreads();
    if (abort_sh) return;
  } else if (failed) {
    return;
  }
  const int g = static_cast<int>(threadIdx.x) & (kNbrLanes - 1);
  const int half = lane_id() & ~(kNbrLanes - 1);
  const unsigned below = (1u << g) - 1u;
  int* buf = buf_sh[grp];
  for (int u0 = blockIdx.x * kHeads; u0 < L; u0 += gridDim.x * kHeads) {
    const int u = u0 + grp;
    const bool on = u < L;
    int4 unit = make_int4(0, 0, 0, 0);
    if (u0 == static_cast<int>(blockIdx.x) * kHeads) {
      if (on) unit = ahead;
    } else if (on) {
      unit = units[u];
    }
    const int s = unit.x;
    const float3 me = ld3(gv.p0, s);
    int a = 0, b = 0;
    bool ok = on;
    if (on && !cell_range(gv, s, unit.w, g, a, b)) {
      ok = false;
      if (g == 0) atomicOr(flags, kFlagRange);
    }
    const int cnt27 = b - a;
    const int inc = incl_scan<kNbrLanes>(cnt27);
    const int E = ok ? __shfl(inc, kNbrLanes - 1, kNbrLanes) : 0;
    const bool wide = E > kExpand;
    int cnt = 0;
    // this group's ballot
    auto votes = [&](bool v) { return static_cast<unsigned>(__ballot(v) >> half); };
    {
      // candidate slots, in order
      const int off = inc - cnt27;
      if (!wide)
        for (int j = 0; j < cnt27; ++j) buf[off + j] = a + j;
      wave_sync();
      const int lim = wide ? 0 : E;
      // kR rounds of candidate loads in flight before any test (as many as the
      // wavefront's heads have candidates for, up to four); the neighbors
      // move to the front of the buffer (never past a candidate that is still
      // to be read)
      auto rounds = [&](auto kr) {
        constexpr int kR = decltype(kr)::value;
        for (int e0 = 0; __any(e0 < lim); e0 += kR * kNbrLanes) {
          int t[kR];
          float3 q[kR];
#pragma unroll
          for (int r = 0; r < kR; ++r) {
            const int e = e0 + r * kNbrLanes + g;
            t[r] = e < lim ? buf[e] : s;
          }
#pragma unroll
          for (int r = 0; r < kR; ++r) q[r] = ld3(gv.p0, t[r]);
          wave_sync();
#pragma unroll
          for (int r = 0; r < kR; ++r) {
            const bool in = t[r] != s && near0(me, q[r], c);
            const unsigned m = votes(in);
            if (in) buf[cnt + __popc(m & below)] = t[r];
            cnt += __popc(m);
          }
          wave_sync();
        }
      };
      if (!__any(lim > kNbrLanes))
        rounds(std::integral_constant<int, 1>{});
      else if (!__any(lim > 2 * kNbrLanes))
        rounds(std::integral_constant<int, 2>{});
      else
        rounds(std::integral_constant<int, 4>{});
    }
    if (__any(wide)) {
      // the runs of the 27 cells, one per lane
      int ra = 0, rb = 0;
      if (wide && g < 27) run_range(gv, a, b, ra, rb);
      Ranges& R = rng_sh[grp];
      const int total = pack_ranges<kNbrLanes>(R, ra, rb);
      wave_sync();
      RangeCursor cur;
      if (total > 0) cur.begin(R);
      bool going = wide;
      for (int e0 = 0; __any(going && e0 < total); e0 += kNbrLanes) {
        const int e = e0 + g;
        const bool v = going && e < total;
        int t = s, k = 0;
        if (v) {
          const int r = cur.at(R, e);
          t = gv.rep[r];
          k = gv.rep[r + 1] - t;
        }
        const bool in = v && near0(me, ld3(gv.p0, t), c);
        const bool own = in && s >= t && s < t + k;  // every slot but s itself
        const int put = in ? k - (own ? 1 : 0) : 0;
        const int pi = incl_scan<kNbrLanes>(put);
        const int sum = __shfl(pi, kNbrLanes - 1, kNbrLanes);
        if (going && cnt + sum <= gv.row_cap) {
          int at = cnt + pi - put;
          for (int j = 0; j < (put > 0 ? k : 0); ++j)
            if (t + j != s) buf[at++] = t + j;
        }
        if (going) cnt += sum;
        if (cnt > gv.row_cap) going = false;  // too long for a row
      }
      wave_sync();
    }
    const bool row = ok && cnt <= gv.row_cap;
    // the row, 16 bytes a store
    if (row)
      for (int k = g; k < (cnt + 3) / 4; k += kNbrLanes)
        rows[static_cast<size_t>(k) * c.n + s] = reinterpret_cast<const int4*>(buf)[k];
    long long off = 0;
    int words = 0;
    bool stored = false;
    if (kFull) {
      // the run-length words of the list, counted or stored at `at`
      auto encode = [&](int* at) {
        int sum = 0;
        for (int k0 = 0; __any(row && k0 < cnt); k0 += kNbrLanes) {
          const int k = k0 + g;
          const bool head = row && k < cnt && (k == 0 || buf[k] != buf[k - 1] + 1);
          int len = 0;
          if (head)
            for (len = 1; k + len < cnt && buf[k + len] == buf[k] + len;) ++len;
          const int w = head ? min(len, 2) : 0;
          const int wi = incl_scan<kNbrLanes>(w);
          if (at && head) {
            int* out = at + sum + wi - w;
            if (len <= 2) {
              for (int i = 0; i < len; ++i) out[i] = buf[k + i];
            } else {
              out[0] = buf[k] | static_cast<int>(0x80000000u);
              out[1] = len;
            }
          }
          sum += __shfl(wi, kNbrLanes - 1, kNbrLanes);
        }
        return sum;
      };
      words = encode(nullptr);
      if (g == 0) cnt_sh[grp] = words;
      __syncthreads();
      int pre = 0, total = 0;
      for (int v = 0; v < kHeads; ++v) {
        pre += v < grp ? cnt_sh[v] : 0;
        total += cnt_sh[v];
      }
      if (threadIdx.x == 0)
        base_sh = static_cast<long long>(
            atomicAdd(nbr_total, static_cast<unsigned long long>(total)));
      __syncthreads();
      off = base_sh + pre;
      stored = row && off + words <= nbr_cap;
      if (row && !stored && g == 0) atomicOr(flags, kFlagNeighbors);
      (void)encode(stored ? nbr + off : nullptr);
    }
    if (ok && g == 0) {
      const int r = gv.run_no[s];
      units[u] = make_int4(s, row ? cnt : -1, gv.rep[r + 1] - s, unit.w);
      if (!row) dense[atomicAdd(info + 2, 1)] = make_int2(s, unit.w | kSingle);
      ncount[s] = row ? cnt : 0;
      noff[s] = stored ? off : 0;
      nwords[s] = stored ? words : (row ? kRowList : kLongList);
    } else if (on && !ok && g == 0) {
      units[u].y = -1;
    }
    if (kFull) __syncthreads();  // cnt_sh and base_sh are reused
    wave_sync();                 // ... and the buffer
  }
}

// The rows of a recorded substep's list heads as plain words, one list for every
// slot of the head's run (the run's slots but the list's own are one stretch of
// it): a workgroup takes consecutive units, whose lists it
// allocates with one atomic (atomics on one address take about 10 ns each: one
// for every 8 heads made the neighbor kernel take 107 us at 65,536 particles;
// without them it takes 27, and this one 24).
__global__ __launch_bounds__(kBlock) void k_store_rows(
    StepConsts c, GatherView gv, long long* __restrict__ noff, int* __restrict__ nwords,
    int* __restrict__ ncount, int* __restrict__ nbr, long long nbr_cap,
    unsigned long long* __restrict__ nbr_total, unsigned* __restrict__ flags) {
  constexpr int kLanes = 8, kUnits = kBlock / kLanes;
  __shared__ long long wsum[kWaves];
  __shared__ int round[kWaves];
  __shared__ long long base_sh;
  __shared__ int abort_sh;
  if (threadIdx.x == 0) abort_sh = fatal(flags) ? 1 : 0;
  __syncthreads();
  if (abort_sh) return;
  const int L = gv.info[1];
  const int per = (L + static_cast<int>(gridDim.x) - 1) / static_cast<int>(gridDim.x);
  const int u0 = blockIdx.x * per, u1 = min(L, u0 + per);
  if (u0 >= u1) return;  // uniform
  long long sum = 0;
  for (int u = u0 + static_cast<int>(threadIdx.x); u < u1; u += kBlock) {
    const int4 unit = gv.units[u];
    sum += static_cast<long long>(max(unit.y, 0)) * unit.z;
  }
  for (int o = kWave / 2; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
  if (lane_id() == 0) wsum[threadIdx.x / kWave] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    long long total = 0;
    for (int w = 0; w < kWaves; ++w) total += wsum[w];
    const long long at =
        static_cast<long long>(atomicAdd(nbr_total, static_cast<unsigned long long>(total)));
    base_sh = at + total <= nbr_cap ? at : -1;
    if (base_sh < 0) atomicOr(flags, kFlagNeighbors);
  }
  __syncthreads();
  long long at = base_sh;
  if (at < 0) return;
  const int* rows = reinterpret_cast<const int*>(gv.rows);
  const int g = static_cast<int>(threadIdx.x) / kLanes, q = lane_id() & (kLanes - 1);
  for (int b = u0; b < u1; b += kUnits) {
    const int u = b + g;
    const int4 unit = u < u1 ? gv.units[u] : make_int4(0, -1, 0, 0);
    const int s = unit.x, cnt = max(unit.y, 0), len = unit.z;
    const int mine = cnt * len;  // (a row's entries times a sparse cell's slots)
    // the lists before this unit's: within the wavefront (its groups' first
    // lanes), then the wavefronts before
    int inc = mine;
    for (int o = kLanes; o < kWave; o <<= 1) {
      const int v = __shfl_up(inc, o);
      if (lane_id() >= o) inc += v;
    }
    __syncthreads();  // round is reused
    if (lane_id() == kWave - 1) round[threadIdx.x / kWave] = inc;
    __syncthreads();
    long long off = at + inc - mine;
    for (int w = 0; w < kWaves; ++w) {
      off += w < static_cast<int>(threadIdx.x) / kWave ? round[w] : 0;
      at += round[w];
    }
    auto row = [&](int k) { return rows[(static_cast<size_t>(k >> 2) * c.n + s) * 4 + (k & 3)]; };
    if (!__any(len > 1)) {  // no run among the wavefront's heads
      for (int k = q; k < cnt; k += kLanes) nbr[off + k] = row(k);
      if (q == 0 && unit.y >= 0) {
        noff[s] = off;
        nwords[s] = cnt;
      }
      continue;
    }
    // the run's other slots: entries [own, own + len - 1) of the row
    int own = cnt;
    if (len > 1)
      for (int k = q; k < cnt; k += kLanes)
        if (row(k) == s + 1) own = k;
    for (int o = kLanes / 2; o > 0; o >>= 1) own = min(own, __shfl_xor(own, o));
    for (int k = q; k < cnt; k += kLanes) {
      const int v = row(k), i = k - own;
      const bool in_run = i >= 0 && i < len - 1;
      for (int j = 0; j < len; ++j) nbr[off + j * cnt + k] = in_run ? s + i + (i >= j ? 1 : 0) : v;
    }
    if (unit.y >= 0)
      for (int j = q; j < len; j += kLanes) {
        noff[s + j] = off + j * cnt;
        nwords[s + j] = cnt;
        ncount[s + j] = cnt;
      }
  }
}

// A dense unit: `heads` consecutive runs from run r0 on, the first at slot s
// (`unit`: the heads of a unit, at most).
struct DenseUnit {
  int s, sc, r0, heads;
  bool single;
};

__device__ __forceinline__ DenseUnit dense_unit(const GatherView& gv, int u, int unit) {
  DenseUnit d;
  const int2 w = gv.dense[u];
  d.s = __builtin_amdgcn_readfirstlane(w.x);
  const int sc = __builtin_amdgcn_readfirstlane(w.y);
  d.single = sc < 0;
  d.sc = sc & ~kSingle;
  d.r0 = __builtin_amdgcn_readfirstlane(gv.run_no[d.s]);
  d.heads = 1;
  if (!d.single) {
    const int end = gv.start[gv.slot_key[d.s] + 1];  // of the cell
    const int left = __builtin_amdgcn_readfirstlane(gv.run_no[end - 1]) + 1 - d.r0;
    d.heads = min(left, unit - (d.r0 & (unit - 1)));
  }
  return d;
}

// ------------------------------------------------------------ dense walk

// Walks the runs of the 27 cells whose entries R holds, in list order, one run
// per lane.  body(e0, r, k, p, q): the lane's entry e0 + lane is run r of k
// slots (0 past the end, where the last entry repeats), p its p^0, q the
// load() of its first slot.  The next two steps' loads are issued before a
// step is processed.  Whole wavefronts; `total` is the entries of R.
template <typename Load, typename Body>
__device__ __forceinline__ void walk_runs(const GatherView& gv, const Ranges& R, int total,
                                          Load&& load, Body&& body) {
  if (total <= 0) return;
  using Q = decltype(load(0));
  const int lane = lane_id();
  RangeCursor cur;
  cur.begin(R);
  auto entry = [&](int e, int& r, int& t, int& k) {
    r = cur.at(R, min(e, total - 1));
    t = gv.rep[r];
    k = e < total ? gv.rep[r + 1] - t : 0;
  };
  int r0, t0, k0, r1, t1, k1;
  entry(lane, r0, t0, k0);
  entry(lane + kWave, r1, t1, k1);
  float3 p = ld3(gv.p0, t0);
  Q q = load(t0);
  for (int e0 = 0; e0 < total; e0 += kWave) {
    const float3 pn = ld3(gv.p0, t1);
    const Q qn = load(t1);
    int r2, t2, k2;
    entry(e0 + 2 * kWave + lane, r2, t2, k2);
    body(e0, r0, k0, p, q);
    p = pn;
    q = qn;
    r0 = r1;
    k0 = k1;
    r1 = r2;
    t1 = t2;
    k1 = k2;
  }
}

// The entries of the walk around slot s of scene sc into R; returns their
// total (0 when the slot's cell lies outside the table).
__device__ __forceinline__ int dense_ranges(const GatherView& gv, Ranges& R, int s, int sc) {
  int a, b, ra, rb;
  cell_range(gv, s, sc, lane_id(), a, b);
  run_range(gv, a, b, ra, rb);
  const int total = pack_ranges<kWave>(R, ra, rb);
  wave_sync();
  return __builtin_amdgcn_readfirstlane(total);
}

// ------------------------------------------------------------ lists of dense units

// Builds the list of slot s, at me, in w: the runs of the 27 cells (entries of R)
// 64 at a time; a run's slots are neighbors together.
template <bool kFill>
__device__ __forceinline__ void list_walk(const StepConsts& c, const GatherView& gv,
                                          const Ranges& R, int total, int s, const float3& me,
                                          RunWriter& w) {
  walk_runs(gv, R, total, [](int t) { return t; },
            [&](int, int, int k, const float3& p, int t) {
              const int to = t + k;
              unsigned long long m = __ballot(k > 0 && near0(me, p, c));
              // entries whose slots follow the entry's before (lane 0's comes with w)
              const unsigned long long follow = __ballot(t == __shfl_up(to, 1)) & ~1ull;
              while (m != 0ull) {
                const int j = __builtin_ctzll(m);
                const int len = 1 + __builtin_ctzll(~((m & follow) >> j >> 1));
                const int t0 = __builtin_amdgcn_readlane(t, j);
                const int t1 = __builtin_amdgcn_readlane(to, j + len - 1);
                if (t0 <= s && s < t1) {  // every slot but s itself
                  w.template add_range<kFill>(t0, s);
                  w.template add_range<kFill>(s + 1, t1);
                } else {
                  w.template add_range<kFill>(t0, t1);
                }
                m = (j + len >= kWave) ? 0ull : (m & (~0ull << (j + len)));
              }
            });
  w.template flush<kFill>();
}

// Counts, allocates (one atomic) and fills the list of slot s of scene sc, by a
// whole wavefront; false when it does not fit.
__device__ __forceinline__ bool store_list(const StepConsts& c, const GatherView& gv, Ranges& R,
                                           int s, int sc, long long* __restrict__ noff,
                                           int* __restrict__ nwords, int* __restrict__ ncount,
                                           int* __restrict__ nbr, long long nbr_cap,
                                           unsigned long long* __restrict__ nbr_total) {
  const int lane = lane_id();
  wave_sync();  // R is reused
  const int total = dense_ranges(gv, R, s, sc);
  const float3 me = ld3(gv.p0, s);
  RunWriter w{nullptr, false};
  list_walk<false>(c, gv, R, total, s, me, w);
  unsigned long long at = 0;
  if (lane == 0) at = atomicAdd(nbr_total, static_cast<unsigned long long>(w.words));
  const long long off = static_cast<long long>(__shfl(at, 0));
  if (off + w.words > nbr_cap) return false;
  RunWriter f{nbr + off, lane == 0};
  list_walk<true>(c, gv, R, total, s, me, f);
  if (lane == 0) {
    noff[s] = off;
    nwords[s] = static_cast<int>(w.words);
    ncount[s] = w.count;
  }
  return true;
}

// On request: the lists of the heads too long for a row.  No flag is raised when
// they do not fit (*nbr_total says what they need).
__global__ __launch_bounds__(kBlock) void k_long_lists(
    StepConsts c, GatherView gv, long long* __restrict__ noff, int* __restrict__ nwords,
    int* __restrict__ ncount, int* __restrict__ nbr, long long nbr_cap,
    unsigned long long* __restrict__ nbr_total, const unsigned* __restrict__ flags) {
  __shared__ Ranges rng[kWaves];
  if (fatal(flags)) return;
  const int D = gv.info[2];
  const int nw = static_cast<int>(gridDim.x) * kWaves;
  for (int u = blockIdx.x * kWaves + threadIdx.x / kWave; u < D; u += nw) {
    const DenseUnit d = dense_unit(gv, u, gv.info[3]);
    if (d.single)
      (void)store_list(c, gv, rng[threadIdx.x / kWave], d.s, d.sc, noff, nwords, ncount, nbr,
                       nbr_cap, nbr_total);
  }
}

// After the list heads' lists are stored: the lists of all other slots (nwords <
// 0), those of dense units and of runs.  Wavefront w of W takes slots w, w + W,
// ...: the slots of a pile, whose lists are the longest, lie side by side.
// (velB.w: scenes.)  Bound by the loads and serial bits of two walks per list.
// With one wavefront per unit, walking slots instead of runs, and every slot a
// head, the recorded substep of the million-particle block after 100 substeps took
// 377 ms, and takes 10 (diagnostics 442 and 11); after 40 substeps of the
// 32,768-particle dam break this kernel 137 us, and takes 124.
__global__ __launch_bounds__(kBlock) void k_dense_lists(
    StepConsts c, GatherView gv, const float4* __restrict__ velB, long long* __restrict__ noff,
    int* __restrict__ nwords, int* __restrict__ ncount, int* __restrict__ nbr, long long nbr_cap,
    unsigned long long* __restrict__ nbr_total, unsigned* __restrict__ flags) {
  __shared__ Ranges rng[kWaves];
  if (fatal(flags) || (gv.info[2] == 0 && gv.info[0] == c.n)) return;
  const int lane = lane_id();
  const long long W = static_cast<long long>(gridDim.x) * kWaves;
  for (long long s0 = blockIdx.x * kWaves + threadIdx.x / kWave; s0 < c.n; s0 += kWave * W) {
    const long long mine = s0 + lane * W;
    unsigned long long todo = __ballot(mine < c.n && nwords[mine < c.n ? mine : 0] < 0);
    while (todo != 0ull) {
      const int s = __builtin_amdgcn_readfirstlane(
          static_cast<int>(s0 + __builtin_ctzll(todo) * W));
      todo &= todo - 1ull;
      const int sc = __builtin_amdgcn_readfirstlane(__float_as_int(velB[s].w));
      const bool fits = store_list(c, gv, rng[threadIdx.x / kWave], s, sc, noff, nwords, ncount,
                                   nbr, nbr_cap, nbr_total);
      if (!fits && lane == 0) atomicOr(flags, kFlagNeighbors);
    }
  }
}

// Neighbor counts of the dense units' heads (statistics).  Nothing is counted
// after a substep that failed, whose arrays are of two substeps.
__global__ __launch_bounds__(kBlock) void k_count_dense(const StepConsts* __restrict__ last,
                                                        GatherView gv,
                                                        int* __restrict__ ncount,
                                                        const unsigned* __restrict__ flags) {
  __shared__ Ranges rng[kWaves];
  if (fatal(flags) || last->full_lists) return;
  const StepConsts c = *last;
  const int D = gv.info[2];
  Ranges& R = rng[threadIdx.x / kWave];
  const int nw = static_cast<int>(gridDim.x) * kWaves;
  for (int u = blockIdx.x * kWaves + threadIdx.x / kWave; u < D; u += nw) {
    const DenseUnit d = dense_unit(gv, u, gv.info[3]);
    wave_sync();
    const int total = dense_ranges(gv, R, d.s, d.sc);
    for (int h = 0; h < d.heads; ++h) {
      const int s = __builtin_amdgcn_readfirstlane(gv.rep[d.r0 + h]);
      const float3 me = ld3(gv.p0, s);
      int cnt = 0;
      walk_runs(gv, R, total, [&](int) { return 0; },
                [&](int, int r, int k, const float3& p, int) {
                  if (near0(me, p, c)) cnt += max(0, k - (r == d.r0 + h ? 1 : 0));
                });
      for (int o = kWave / 2; o > 0; o >>= 1) cnt += __shfl_xor(cnt, o);
      if (lane_id() == 0) ncount[s] = cnt;
    }
  }
}

// Every slot's count from its run's head (from the tile lists for tile
// slots), and the sum of all (0 after a substep that failed, or that stored every
// list and with it every count).
__global__ __launch_bounds__(kBlock) void k_count_slots(int n, const int* __restrict__ run_no,
                                                        const int* __restrict__ rep,
                                                        const StepConsts* __restrict__ last,
                                                        const int* __restrict__ in_tile,
                                                        const int* __restrict__ tile_cnt,
                                                        int* __restrict__ ncount,
                                                        unsigned long long* __restrict__ total,
                                                        const unsigned* __restrict__ flags) {
  if (fatal(flags) || last->full_lists) return;
  if (!last->tiles) in_tile = nullptr;
  unsigned long long v = 0ull;
  const int stride = static_cast<int>(gridDim.x) * kBlock;
  for (int s = blockIdx.x * kBlock + threadIdx.x; s < n; s += stride) {
    int k;
    if (in_tile && in_tile[s] > 0) {
      k = tile_cnt[s];
      ncount[s] = k;
    } else {
      const int h = rep[run_no[s]];
      k = ncount[h];
      if (h != s) ncount[s] = k;
    }
    v += static_cast<unsigned long long>(k);
  }
  for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o);
  if (lane_id() == 0 && v != 0ull) atomicAdd(total, v);
}

// ------------------------------------------------------------ passes

// LDS of one wavefront of a pass: the list heads' terms (kListLanes heads'
// groups, kAcc rows of 32 terms, padded) and sums, or a dense unit's 64
// entries and terms.
constexpr int kListRow = 36;
constexpr int kMaxAcc = 5;
constexpr int kTermFloats = (kWave / kListLanes) * kMaxAcc * kListRow;
constexpr int kEntryQuads = 2;  // float4s of an entry: the heads that take it, a record
// floats of a dense unit's terms: rows of 2 G terms (G for a single head),
// padded by 4, for kAcc accumulators of 64 / G heads
constexpr int kDenseTerms = std::max(kUnitHeads * kMaxAcc * (2 * kWave / kUnitHeads + 4),
                                     kMaxAcc * (kWave + 4));
constexpr int kPassFloats = std::max(4 * kEntryQuads * kWave + kDenseTerms, kTermFloats);

struct PassLds {
  float4 term[kWaves][kPassFloats / 4];
  float sums[kWaves][kMaxAcc * kWave];
  Ranges rng[kWaves];
};

// A pass:
//   kAcc                 accumulators
//   Self, self(s)        a particle's own state
//   Rec, load(t)         a neighbor's record
//   term(me, q, o)       what q adds to each accumulator.  Terms of +-0 change
//                        no sum (a sum starts at +0 and never becomes -0, as
//                        x + y rounds an exact cancellation to +0), so they
//                        stand for "nothing" too
//   finish(s, sc, len, j, step, me, sum)   the outputs of the particle at slot
//                        s of scene sc, written to slots s + j, s + j + step,
//                        ... of its run of len slots

__device__ __forceinline__ void add4(float& acc, const float4& x) {
  acc += x.x;
  acc += x.y;
  acc += x.z;
  acc += x.w;
}

// List heads: kListLanes lanes each, 32 neighbors at a time.  Bound by the
// latency of unit, row and record loads in a small batch (4,199 particles: 4.7
// us per lambda launch, where one lane per particle walking its own list took
// 49) and by vector instructions in a large one.  A wavefront
// takes up to kWave consecutive heads, kWave / kListLanes at a time, and then
// finishes them with a lane each (the outputs' arithmetic, once per particle,
// would otherwise run once for every kListLanes lanes); few heads are spread
// over the wavefronts instead.
template <typename Pass>
__device__ __forceinline__ void pass_lists(const StepConsts& c, const GatherView& gv,
                                           const Pass& pass, float* lds, float* sums, int first,
                                           int waves, int L, const int4& ahead) {
  constexpr int kA = Pass::kAcc;
  constexpr int kHeads = kWave / kListLanes;
  const int lane = lane_id();
  const int q = lane & (kListLanes - 1);
  const int grp = lane / kListLanes;
  float* T = lds + grp * (kA * kListRow);
  const float4* mine = reinterpret_cast<const float4*>(T + min(q, kA - 1) * kListRow);
  const int* rows = reinterpret_cast<const int*>(gv.rows);
  const int chunk = kHeads * max(1, min(kListLanes, L / (waves * kHeads)));
  for (int base = first * chunk; base < L; base += waves * chunk) {
    for (int h = 0; h < chunk && base + h < L; h += kHeads) {
      const int u = base + h + grp;
      int4 unit = make_int4(0, -1, 0, 0);
      if (chunk == kHeads && base == first * kHeads) {
        if (u < L) unit = ahead;
      } else if (u < L) {
        unit = gv.units[u];
      }
      const int s = unit.x, cnt = unit.y;
      const typename Pass::Self me = pass.self(s);
      int mx = cnt;
      for (int o = kListLanes; o < kWave; o <<= 1) mx = max(mx, __shfl_xor(mx, o));
      mx = __builtin_amdgcn_readfirstlane(mx);
      float acc = 0.0f;
      for (int k0 = 0; k0 < mx; k0 += 32) {
        int t[4];
        typename Pass::Rec v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int k = k0 + r * kListLanes + q;
          t[r] = k < cnt ? rows[(static_cast<size_t>(k >> 2) * c.n + s) * 4 + (k & 3)] : s;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = pass.load(t[r]);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (k0 + r * kListLanes < mx) {
            const int k = r * kListLanes + q;
            float o[kA];
            pass.term(me, v[r], o);
#pragma unroll
            for (int i = 0; i < kA; ++i) T[i * kListRow + k] = k0 + k < cnt ? o[i] : 0.0f;
          }
        }
        wave_sync();
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (k0 + r * kListLanes < mx) {
            const float4 x = mine[2 * r], y = mine[2 * r + 1];
            add4(acc, x);
            add4(acc, y);
          }
        }
        wave_sync();
      }
      if (q < kA) sums[q * kWave + h + grp] = acc;
    }
    wave_sync();
    const int u = base + lane;
    if (lane < chunk && u < L) {
      const int4 unit = gv.units[u];
      if (unit.y >= 0) {
        float sum[kA];
#pragma unroll
        for (int i = 0; i < kA; ++i) sum[i] = sums[i * kWave + lane];
        pass.finish(unit.x, unit.w, unit.z, 0, 1, pass.self(unit.x), sum);
      }
    }
    wave_sync();
  }
}

// Dense units: a wavefront each, 64 runs of candidates (entries) at a time;
// those that are neighbors of one of its heads are packed in LDS.  The lanes
// form G-lane groups, one per head (G = 64 for a single head, 8 for eight); a
// group's lanes compute the packed entries' terms of its head side by side, and
// then one lane per head and accumulator adds them in order.  All heads of the
// unit see one sequence of entries, so an entry's multiplicity is uniform: a
// run of k slots is added k times by all sums at once (an entry that is no
// neighbor of a head adds zeros).
//
// Bound by the vector instructions of the ordered additions and their
// multiplicities (about half) and of the terms, and by the longest units (5,800
// entries in the piled-up million-particle block).  One lane per particle over
// all candidates in turn, the walk this replaces, was bound by the latency of
// its longest wavefronts (0.4 us per candidate): lambda of the splashing
// 32,768-particle dam break took 237 us per launch and takes 28, the
// 262,144-particle dam breaks' 725 and 96, the piled-up million-particle
// block's 2,000 and 292 (beside its tiles).
template <typename Pass>
__device__ __forceinline__ void pass_dense(const StepConsts& c, const GatherView& gv,
                                           const Pass& pass, float* lds, float* sums, Ranges& R,
                                           int block, int nblocks, int D, int unit) {
  constexpr int kA = Pass::kAcc;
  using Rec = typename Pass::Rec;
  constexpr int kRec = sizeof(Rec) / sizeof(float);
  constexpr int kQ = (1 + kRec + 3) / 4;  // the heads that take it, its record
  static_assert(kQ <= kEntryQuads, "an entry must fit");
  static_assert(kMaxAcc * kWave >= 2 * kWave, "an entry's run must fit the sums");
  const int lane = lane_id();
  float4* ent = reinterpret_cast<float4*>(lds);
  float* T = lds + 4 * kEntryQuads * kWave;
  const int waves = nblocks * kWaves;
  const int first = __builtin_amdgcn_readfirstlane(block * kWaves +
                                                   static_cast<int>(threadIdx.x) / kWave);
  const int hp = lane / kA, ha = lane % kA;  // the head and accumulator this lane adds
  for (int u = first; u < D; u += waves) {
    const DenseUnit d = dense_unit(gv, u, unit);
    const int lg = d.heads > 4 ? 3 : d.heads > 2 ? 2 : d.heads > 1 ? 1 : 0;
    const int G = kWave >> lg;
    const int p = lane >> (6 - lg), g = lane & (G - 1);
    const int step = lg == 0 ? kWave : 2 * G;  // entries per round
    const int row = step + 4;
    wave_sync();
    const int total = dense_ranges(gv, R, d.s, d.sc);
    const int own = d.r0 + min(p, d.heads - 1);
    const int s = gv.rep[own];
    const int len = gv.rep[own + 1] - s;
    const float3 me0 = ld3(gv.p0, s);
    const typename Pass::Self me = pass.self(s);
    const float4* mine =
        reinterpret_cast<const float4*>(T + (min(hp, (1 << lg) - 1) * kA + ha) * row);
    float* put = T + p * kA * row + g;
    int2* runs = reinterpret_cast<int2*>(sums);
    float acc = 0.0f;
    walk_runs(
        gv, R, total, [&](int t) { return pass.load(t); },
        [&](int, int run, int k, const float3& p0, const Rec& rec) {
          // the heads that take this lane's entry (bit h: head h), and the
          // entries that some head takes, packed to the front
          unsigned takes = 0u;
          for (int h = 0; h < d.heads; ++h) {
            const int from = h << (6 - lg);
            const float3 ph = make_float3(lane_of(me0.x, from), lane_of(me0.y, from),
                                          lane_of(me0.z, from));
            if (near0(ph, p0, c) && k > (run == d.r0 + h ? 1 : 0)) takes |= 1u << h;
          }
          const unsigned long long kept = __ballot(takes != 0u);
          if (kept == 0ull) return;
          const int m = __popcll(kept);
          if (takes != 0u) {
            const int at = __popcll(kept & ((1ull << lane) - 1ull));
            float f[4 * kQ] = {};
            f[0] = __uint_as_float(takes);
            __builtin_memcpy(f + 1, &rec, sizeof(Rec));
#pragma unroll
            for (int i = 0; i < kQ; ++i)
              ent[i * kWave + at] =
                  make_float4(f[4 * i], f[4 * i + 1], f[4 * i + 2], f[4 * i + 3]);
            runs[at] = make_int2(run, k);
          }
          wave_sync();
          const int2 mine_run = runs[lane];
          const int times = lane < m ? mine_run.y : 0;
          const unsigned long long many = __ballot(times > 1);
          for (int j = 0; j < m; j += step) {
            // entries j + g and, but for a single head, j + G + g
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              if (h == 1 && lg == 0) break;
              const int at = j + h * G + g;
              float f[4 * kQ];
#pragma unroll
              for (int i = 0; i < kQ; ++i) {
                const float4 x = ent[i * kWave + at];
                f[4 * i] = x.x;
                f[4 * i + 1] = x.y;
                f[4 * i + 2] = x.z;
                f[4 * i + 3] = x.w;
              }
              const bool near = at < m && ((__float_as_uint(f[0]) >> p) & 1u) != 0u;
              Rec v;
              __builtin_memcpy(&v, f + 1, sizeof(Rec));
              float o[kA];
              pass.term(me, v, o);
#pragma unroll
              for (int i = 0; i < kA; ++i) put[i * row + h * G] = near ? o[i] : 0.0f;
            }
            wave_sync();
            const int end = min(step, m - j);
            for (int i = 0; i < end; i += 8) {
              const float4 x = mine[i >> 2], y = mine[(i >> 2) + 1];
              const unsigned some = static_cast<unsigned>(many >> (j + i)) & 255u;
              if (some == 0u) {
                add4(acc, x);
                add4(acc, y);
                continue;
              }
              const float z[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
              for (int b = 0; b < 8; ++b) {
                if (((some >> b) & 1u) == 0u) {
                  acc += z[b];
                } else if (__any(z[b] != 0.0f)) {
                  // one addition for each of the run's slots, one less for
                  // the head that the run is
                  const int head = __builtin_amdgcn_readlane(mine_run.x, j + i + b) - d.r0;
                  acc = add_k(acc, z[b], __builtin_amdgcn_readlane(times, j + i + b) - 1);
                  acc += hp == head ? 0.0f : z[b];
                }
              }
            }
            wave_sync();
          }
        });
    wave_sync();
    sums[lane] = acc;
    wave_sync();
    float sum[kA];
#pragma unroll
    for (int i = 0; i < kA; ++i) sum[i] = sums[p * kA + i];
    if (p < d.heads) pass.finish(s, d.sc, len, g, G, me, sum);
  }
}

// The first gv.dense_blocks workgroups take the dense units (the longest
// work, dispatched first), the others the list heads.  In a small batch a pass
// is a chain of loads that miss (each about 0.5 us: the producer ran on other
// XCDs), so the fatal flag, the counts and the list heads a wavefront will
// take if it takes one round are asked for at once (the heads' array has an entry
// for every particle).  One after the other before: lambda of 4,199 particles
// 5.0 -> 4.7 us per launch, of 7,680 5.85 -> 5.3, delta 6.2 -> 5.8 and 7.3 -> 6.6;
// of 262,144, bound by instructions, 29.2 either way.
template <typename Pass>
__device__ __forceinline__ void gather(const StepConsts& c, const GatherView& gv,
                                       const Pass& pass, PassLds& lds, const unsigned* flags) {
  const int w = threadIdx.x / kWave;
  float* term = reinterpret_cast<float*>(lds.term[w]);
  const int b = static_cast<int>(blockIdx.x) - gv.dense_blocks;
  if (b < 0) {
    const int D = gv.info[2], unit = gv.info[3];
    const bool failed = fatal(flags);
    loaded(D);
    loaded(unit);
    if (failed) return;
    pass_dense(c, gv, pass, term, lds.sums[w], lds.rng[w], blockIdx.x, gv.dense_blocks, D, unit);
  } else {
    const int first = b * kWaves + w;
    const int4 ahead = gv.units[min(c.n - 1, first * (kWave / kListLanes) + lane_id() / kListLanes)];
    const int L = gv.info[1];
    const bool failed = fatal(flags);
    loaded(L);
    loaded(ahead);
    if (failed) return;
    pass_lists(c, gv, pass, term, lds.sums[w], first,
               (static_cast<int>(gridDim.x) - gv.dense_blocks) * kWaves, L, ahead);
  }
}

// lambda (core.cpp:281-329): rho, the gradient sum, the sum of squares.
// Writes lambda into P[s].w; with `sq` (a recorded substep) also the gradient
// sum S (xyz) and the denominator sum Q (w), lambda = -C / (Q + eps).
struct LambdaPass {
  static constexpr int kAcc = 5;
  using Self = float3;
  using Rec = float3;
  const StepConsts& c;
  float4* __restrict__ P;
  float* __restrict__ rho;  // null unless this is the last iteration
  float4* __restrict__ sq;
  __device__ __forceinline__ Self self(int s) const { return ld3(P, s); }
  __device__ __forceinline__ Rec load(int t) const { return ld3(P, t); }
  __device__ __forceinline__ void term(const Self& p, const Rec& q, float (&o)[kAcc]) const {
    const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
    const float r2 = dx * dx + dy * dy + dz * dz;
    const float ngs = -c.grad_scale;
    const bool grad = r2 < c.h2;
    const float f = pair_spiky(r2, c);  // used for grad only
    const float gx = f * dx, gy = f * dy, gz = f * dz;
    const float jx = ngs * gx, jy = ngs * gy, jz = ngs * gz;
    o[0] = poly6(r2, c);
    o[1] = grad ? gx : 0.0f;
    o[2] = grad ? gy : 0.0f;
    o[3] = grad ? gz : 0.0f;
    o[4] = grad ? jx * jx + jy * jy + jz * jz : 0.0f;
  }
  __device__ __forceinline__ void finish(int s, int, int len, int j, int step, const Self&,
                                         const float (&sum)[kAcc]) const {
    float r = sum[0];
    r += c.w0;
    r *= c.mass;
    const float C = r * c.inv_density - 1.0f;
    const float gix = c.grad_scale * sum[1], giy = c.grad_scale * sum[2],
                giz = c.grad_scale * sum[3];
    const float sg2 = sum[4] + (gix * gix + giy * giy + giz * giz);
    const float lam = -C / (sg2 + c.eps);
    for (; j < len; j += step) {
      reinterpret_cast<float*>(P + s + j)[3] = lam;
      if (rho) rho[s + j] = r;
      if (sq) sq[s + j] = make_float4(sum[1], sum[2], sum[3], sg2);
    }
  }
};

__global__ __launch_bounds__(kBlock) void k_lambda(StepConsts c, GatherView gv,
                                                   float4* __restrict__ P,
                                                   float* __restrict__ rho,
                                                   float4* __restrict__ sq,
                                                   const unsigned* __restrict__ flags) {
  __shared__ PassLds lds;
  gather(c, gv, LambdaPass{c, P, rho, sq}, lds, flags);
}

// What the commit of the last iteration reads and writes (core.cpp:414-421).
struct Commit {
  const ScenePlanes* __restrict__ sp;
  const float4* __restrict__ posB;
  float4* __restrict__ posA;
  float4* __restrict__ vout;
  const float* __restrict__ rho;   // null: zero iterations
  unsigned* __restrict__ rmask;    // a recorded substep's restitution decisions
};

// Commits slots s + j, s + j + step, ... of a run of len slots at (nx, ny,
// nz): each slot keeps its own id.
template <bool kRest>
__device__ __forceinline__ void commit_run(const StepConsts& c, const Commit& k, int sc, int s,
                                           int len, int j, int step, float nx, float ny,
                                           float nz) {
  if (j >= len) return;
  const float4 x = k.posB[s];
  float vx = (nx - x.x) / c.dt;  // core.cpp:415-417
  float vy = (ny - x.y) / c.dt;
  float vz = (nz - x.z) / c.dt;
  unsigned rm = 0;
  if (kRest) rm = restitute(vx, vy, vz, nx, ny, nz, k.sp[sc]);
  const float r = k.rho ? k.rho[s] : 0.0f;
  for (; j < len; j += step) {
    k.posA[s + j] = make_float4(nx, ny, nz, reinterpret_cast<const float*>(k.posB + s + j)[3]);
    k.vout[s + j] = make_float4(vx, vy, vz, r);
    if (kRest && k.rmask) k.rmask[s + j] = rm;
  }
}

// delta with plane projection and apply (core.cpp:334-407).  kLast also
// commits, kRest fuses plane restitution (core.cpp:573-612).  A recorded
// substep stores the planes that pushed (pmask).
template <bool kLast, bool kRest, int kCorr>
struct DeltaPass {
  static constexpr int kAcc = 3;
  using Self = float4;
  using Rec = float4;
  const StepConsts& c;
  const float4* __restrict__ P;
  float4* __restrict__ Pnext;
  Commit k;
  unsigned* __restrict__ pmask;
  __device__ __forceinline__ Self self(int s) const { return P[s]; }
  __device__ __forceinline__ Rec load(int t) const { return P[t]; }
  __device__ __forceinline__ void term(const Self& p, const Rec& q, float (&o)[kAcc]) const {
    const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
    const float r2 = dx * dx + dy * dy + dz * dz;
    const bool in = r2 < c.h2;
    const float sf = pair_lambda<kCorr>(p.w, q.w, r2, c) * pair_spiky(r2, c);
    o[0] = in ? sf * dx : 0.0f;
    o[1] = in ? sf * dy : 0.0f;
    o[2] = in ? sf * dz : 0.0f;
  }
  __device__ __forceinline__ void finish(int s, int sc, int len, int j, int step, const Self& p,
                                         const float (&sum)[kAcc]) const {
    float ddx = sum[0] * c.inv_density, ddy = sum[1] * c.inv_density,
          ddz = sum[2] * c.inv_density;
    const ScenePlanes& plane = k.sp[sc];
    unsigned pushed = 0;
    if (plane.n_planes > 0) {
      float qx = p.x + ddx, qy = p.y + ddy, qz = p.z + ddz;
      pushed = project_planes(qx, qy, qz, plane);
      ddx = qx - p.x;
      ddy = qy - p.y;
      ddz = qz - p.z;
    }
    const float nx = p.x + ddx, ny = p.y + ddy, nz = p.z + ddz;  // core.cpp:404-406
    if (pmask)
      for (int i = j; i < len; i += step) pmask[s + i] = pushed;
    if (!kLast) {
      for (int i = j; i < len; i += step) Pnext[s + i] = make_float4(nx, ny, nz, 0.0f);
      return;
    }
    commit_run<kRest>(c, k, sc, s, len, j, step, nx, ny, nz);
  }
};

template <bool kLast, bool kRest, int kCorr>
__global__ __launch_bounds__(kBlock) void k_delta(StepConsts c, GatherView gv,
                                                  const float4* __restrict__ P,
                                                  float4* __restrict__ Pnext, Commit k,
                                                  unsigned* __restrict__ pmask,
                                                  const unsigned* __restrict__ flags) {
  __shared__ PassLds lds;
  gather(c, gv, DeltaPass<kLast, kRest, kCorr>{c, P, Pnext, k, pmask}, lds, flags);
}

// The commit of a substep without iterations: every slot on its own.
template <bool kRest>
__global__ __launch_bounds__(kBlock) void k_commit(StepConsts c, const float4* __restrict__ P,
                                                   const int* __restrict__ seg, Commit k,
                                                   const unsigned* __restrict__ flags) {
  const int s = blockIdx.x * kBlock + threadIdx.x;
  if (fatal(flags) || s >= c.n) return;
  const float3 p = ld3(P, s);
  commit_run<kRest>(c, k, scene_of(s, seg, c.n_scenes), s, 1, 0, 1, p.x, p.y, p.z);
}

// A particle's position and velocity, and a neighbor's with m / rho (0 when
// rho <= 0).
struct PosVel {
  float3 x;
  float3 v;
};
struct PosVelM {
  float3 x;
  float3 v;
  float m;
};

// XSPH (core.cpp:430-465); vin.w carries rho of the last lambda pass.
template <bool kRest>
struct XsphPass {
  static constexpr int kAcc = 3;
  using Self = PosVel;
  using Rec = PosVelM;
  const StepConsts& c;
  const float4* __restrict__ pos;
  const float4* __restrict__ vin;
  float4* __restrict__ vout;
  const ScenePlanes* __restrict__ sp;
  unsigned* __restrict__ rmask;
  __device__ __forceinline__ Self self(int s) const { return Self{ld3(pos, s), ld3(vin, s)}; }
  __device__ __forceinline__ Rec load(int t) const {
    const float4 v = vin[t];
    return Rec{ld3(pos, t), make_float3(v.x, v.y, v.z), v.w};
  }
  __device__ __forceinline__ void term(const Self& p, const Rec& q, float (&o)[kAcc]) const {
    const float dx = p.x.x - q.x.x, dy = p.x.y - q.x.y, dz = p.x.z - q.x.z;
    const float r2 = dx * dx + dy * dy + dz * dz;
    const bool in = r2 < c.h2;
    const float W = tile_poly6(r2, c);
    const float m = (q.m > 0.0f) ? (c.mass / q.m) : 0.0f;
    o[0] = in ? (q.v.x - p.v.x) * W * m : 0.0f;
    o[1] = in ? (q.v.y - p.v.y) * W * m : 0.0f;
    o[2] = in ? (q.v.z - p.v.z) * W * m : 0.0f;
  }
  __device__ __forceinline__ void finish(int s, int sc, int len, int j, int step, const Self& p,
                                         const float (&sum)[kAcc]) const {
    if (j >= len) return;
    float vx = p.v.x + c.visc_c * sum[0];
    float vy = p.v.y + c.visc_c * sum[1];
    float vz = p.v.z + c.visc_c * sum[2];
    unsigned rm = 0;
    if (kRest)
      rm = restitute(vx, vy, vz, p.x.x, p.x.y, p.x.z, sp[sc]);
    for (; j < len; j += step) {
      vout[s + j] = make_float4(vx, vy, vz, 0.0f);
      if (kRest && rmask) rmask[s + j] = rm;
    }
  }
};

template <bool kRest>
__global__ __launch_bounds__(kBlock) void k_xsph(StepConsts c, GatherView gv,
                                                 const float4* __restrict__ pos,
                                                 const float4* __restrict__ vin,
                                                 float4* __restrict__ vout,
                                                 const ScenePlanes* __restrict__ sp,
                                                 unsigned* __restrict__ rmask,
                                                 const unsigned* __restrict__ flags) {
  __shared__ PassLds lds;
  gather(c, gv, XsphPass<kRest>{c, pos, vin, vout, sp, rmask}, lds, flags);
}

// vorticity: omega and |omega| (core.cpp:472-508)
struct OmegaPass {
  static constexpr int kAcc = 3;
  using Self = PosVel;
  using Rec = PosVel;
  const StepConsts& c;
  const float4* __restrict__ pos;
  const float4* __restrict__ vel;
  float4* __restrict__ omega;
  __device__ __forceinline__ Self self(int s) const { return load(s); }
  __device__ __forceinline__ Rec load(int t) const { return Rec{ld3(pos, t), ld3(vel, t)}; }
  __device__ __forceinline__ void term(const Self& p, const Rec& q, float (&o)[kAcc]) const {
    const float dx = p.x.x - q.x.x, dy = p.x.y - q.x.y, dz = p.x.z - q.x.z;
    const float r2 = dx * dx + dy * dy + dz * dz;
    const bool in = r2 < c.h2;
    const float f = pair_spiky(r2, c);
    const float gx = f * dx, gy = f * dy, gz = f * dz;
    const float dvx = q.v.x - p.v.x, dvy = q.v.y - p.v.y, dvz = q.v.z - p.v.z;
    o[0] = in ? dvy * gz - dvz * gy : 0.0f;
    o[1] = in ? dvz * gx - dvx * gz : 0.0f;
    o[2] = in ? dvx * gy - dvy * gx : 0.0f;
  }
  __device__ __forceinline__ void finish(int s, int, int len, int j, int step, const Self&,
                                         const float (&sum)[kAcc]) const {
    const float w = sqrtf(sum[0] * sum[0] + sum[1] * sum[1] + sum[2] * sum[2]);
    for (; j < len; j += step) omega[s + j] = make_float4(sum[0], sum[1], sum[2], w);
  }
};

__global__ __launch_bounds__(kBlock) void k_vort_omega(StepConsts c, GatherView gv,
                                                       const float4* __restrict__ pos,
                                                       const float4* __restrict__ vel,
                                                       float4* __restrict__ omega,
                                                       const unsigned* __restrict__ flags) {
  __shared__ PassLds lds;
  gather(c, gv, OmegaPass{c, pos, vel, omega}, lds, flags);
}

// vorticity: eta, confinement force, velocity update (core.cpp:512-570), in
// place on vel (no neighbor reads vel here).  w of a record is |omega|.
template <bool kRest>
struct EtaPass {
  static constexpr int kAcc = 3;
  using Self = float4;
  using Rec = float4;
  const StepConsts& c;
  const float4* __restrict__ pos;
  const float4* __restrict__ omega;
  float4* __restrict__ vel;
  const ScenePlanes* __restrict__ sp;
  __device__ __forceinline__ Self self(int s) const { return load(s); }
  __device__ __forceinline__ Rec load(int t) const {
    const float3 x = ld3(pos, t);
    return make_float4(x.x, x.y, x.z, reinterpret_cast<const float*>(omega + t)[3]);
  }
  __device__ __forceinline__ void term(const Self& p, const Rec& q, float (&o)[kAcc]) const {
    const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
    const float r2 = dx * dx + dy * dy + dz * dz;
    const bool in = r2 < c.h2;
    const float f = pair_spiky(r2, c);
    const float gx = f * dx, gy = f * dy, gz = f * dz;
    const float co = q.w - p.w;
    o[0] = in ? co * gx : 0.0f;
    o[1] = in ? co * gy : 0.0f;
    o[2] = in ? co * gz : 0.0f;
  }
  __device__ __forceinline__ void finish(int s, int sc, int len, int j, int step, const Self& p,
                                         const float (&sum)[kAcc]) const {
    if (j >= len) return;
    const float ex = sum[0], ey = sum[1], ez = sum[2];
    const float ln = sqrtf(ex * ex + ey * ey + ez * ez);
    float nx = 0.0f, ny = 0.0f, nz = 0.0f;
    if (ln > c.vort_norm_eps) {
      const float inv = 1.0f / ln;
      nx = ex * inv;
      ny = ey * inv;
      nz = ez * inv;
    }
    const float3 om = ld3(omega, s);
    const float fx = c.vort_eps * (ny * om.z - nz * om.y);
    const float fy = c.vort_eps * (nz * om.x - nx * om.z);
    const float fz = c.vort_eps * (nx * om.y - ny * om.x);
    // every slot of the run holds one velocity; each is updated from its own
    for (; j < len; j += step) {
      const float4 v = vel[s + j];
      float vx = v.x + c.dt * fx;
      float vy = v.y + c.dt * fy;
      float vz = v.z + c.dt * fz;
      if (kRest) restitute(vx, vy, vz, p.x, p.y, p.z, sp[sc]);
      vel[s + j] = make_float4(vx, vy, vz, 0.0f);
    }
  }
};

template <bool kRest>
__global__ __launch_bounds__(kBlock) void k_vort_apply(StepConsts c, GatherView gv,
                                                       const float4* __restrict__ pos,
                                                       const float4* __restrict__ omega,
                                                       float4* __restrict__ vel,
                                                       const ScenePlanes* __restrict__ sp,
                                                       const unsigned* __restrict__ flags) {
  __shared__ PassLds lds;
  gather(c, gv, EtaPass<kRest>{c, pos, omega, vel, sp}, lds, flags);
}

__global__ void k_reset_total(unsigned long long* total) {
  if (threadIdx.x == 0) *total = 0ull;
}

inline int blocks_for(long long n, int bs) { return static_cast<int>((n + bs - 1) / bs); }

// Workgroups of the passes: enough wavefronts for every head of a small
// batch at once, a fixed grid that loops over the heads of a large one.
constexpr int kDenseGrid = 1024;
constexpr int kListGrid = 2048;
// A unit takes up to a hundred times as long as another: beyond the workgroups
// the chip holds at once (kDenseGrid) the dispatcher hands the next units to
// whichever CU is free.  Only a large batch has that many units, and workgroups
// without one cost each pass 0.3 us a thousand.  Lambda of the piled-up
// million-particle block with 1,024 / 2,048 / 4,096 / 8,192 workgroups: 440 / 365 /
// 344 / 345 us per launch; of the 256-scene ensemble 101 / 102 / 103 / 104.
// (A counter that the wavefronts of a workgroup share: 355 with 1,024, but 262,144
// splashing particles 96 -> 99.)
int dense_blocks(const Ctx& c) {
  return std::min(std::max(kDenseGrid, std::min(4 * kDenseGrid, c.n / 256)),
                  blocks_for(c.n, kWaves));
}
int list_blocks(const Ctx& c) {
  return std::min(kListGrid, blocks_for(c.n, kBlock / kListLanes));
}

}  // namespace

GatherView gather_view(const Ctx& c, const float4* p0) {
  return GatherView{c.info,   c.units, c.dense, c.run_no, c.rep_list,
                    reinterpret_cast<const int4*>(c.tile_list), row_capacity(c),
                    c.slot_cell, c.slot_key, c.grid, c.start, p0, dense_blocks(c)};
}

hipError_t enqueue_heads(Ctx& c, const StepConsts& k) {
  const int G = std::min(c.scan_blocks, blocks_for(c.n, 4 * kBlock));
  const int* tile = k.tiles ? c.in_tile : nullptr;
  if (c.n <= kSmallHeads) {
    k_heads_small<<<1, 1024, 0, c.stream>>>(k, c.posB, c.velB, c.slot_key, c.start, tile,
                                            c.run_no, c.rep_list, c.units, c.dense, c.info,
                                            c.noff, c.nwords, c.ncount, c.flags);
    return hipGetLastError();
  }
  k_head_count<<<G, kBlock, 0, c.stream>>>(k, c.posB, c.velB, c.slot_key, c.start, tile, c.run_no,
                                           c.scan_partial, c.flags);
  k_heads<<<G, kBlock, 0, c.stream>>>(k, c.scan_partial, c.velB, c.run_no, c.rep_list, c.units,
                                      c.dense, c.info, tile, c.noff, c.nwords, c.ncount,
                                      c.flags);
  return hipGetLastError();
}

hipError_t enqueue_neighbors(Ctx& c, const StepConsts& k, const GatherView& gv) {
  const int nb = std::min(4096, blocks_for(c.n, kBlock / kNbrLanes));
  int4* rows = reinterpret_cast<int4*>(c.tile_list);
  if (k.full_lists == 1)
    k_neighbors<true><<<nb, kBlock, 0, c.stream>>>(k, gv, c.units, c.dense, c.info, rows, c.noff,
                                                   c.nwords, c.ncount, c.nbr, c.nbr_cap,
                                                   c.nbr_total, c.flags);
  else
    k_neighbors<false><<<nb, kBlock, 0, c.stream>>>(k, gv, c.units, c.dense, c.info, rows, c.noff,
                                                    c.nwords, c.ncount, c.nbr, c.nbr_cap,
                                                    c.nbr_total, c.flags);
  if (!k.full_lists) return hipGetLastError();
  if (k.full_lists == 2)
    k_store_rows<<<std::min(kDenseGrid, blocks_for(c.n, 32)), kBlock, 0, c.stream>>>(
        k, gv, c.noff, c.nwords, c.ncount, c.nbr, c.nbr_cap, c.nbr_total, c.flags);
  k_dense_lists<<<std::min(kDenseGrid, blocks_for(c.n, kWaves)), kBlock, 0, c.stream>>>(
      k, gv, c.velB, c.noff, c.nwords, c.ncount, c.nbr, c.nbr_cap, c.nbr_total, c.flags);
  return hipGetLastError();
}

hipError_t enqueue_long_lists(Ctx& c, const StepConsts& k) {
  if (c.n == 0) return hipSuccess;
  k_reset_total<<<1, 64, 0, c.stream>>>(c.nbr_total);
  k_long_lists<<<std::min(kDenseGrid, blocks_for(c.n, kWaves)), kBlock, 0, c.stream>>>(
      k, gather_view(c, c.pred[0]), c.noff, c.nwords, c.ncount, c.nbr, c.nbr_cap, c.nbr_total,
      c.flags);
  return hipGetLastError();
}

hipError_t enqueue_count_pairs(Ctx& c) {
  k_reset_total<<<1, 64, 0, c.stream>>>(c.pair_total);
  if (c.n == 0) return hipGetLastError();
  k_count_dense<<<std::min(kDenseGrid, blocks_for(c.n, kWaves)), kBlock, 0, c.stream>>>(
      c.last, gather_view(c, c.pred[0]), c.ncount, c.flags);
  k_count_slots<<<std::min(1024, blocks_for(c.n, kBlock)), kBlock, 0, c.stream>>>(
      c.n, c.run_no, c.rep_list, c.last, c.in_tile, c.tile_cnt, c.ncount,
      c.pair_total, c.flags);
  return hipGetLastError();
}

hipError_t enqueue_lambda(Ctx& c, const StepConsts& k, const GatherView& gv, float4* P, bool last,
                          float4* sq) {
  const int nb = gv.dense_blocks + list_blocks(c);
  k_lambda<<<nb, kBlock, 0, c.stream>>>(k, gv, P, last ? c.rho : nullptr, sq, c.flags);
  return hipGetLastError();
}

hipError_t enqueue_delta(Ctx& c, const StepConsts& k, const GatherView& gv, const float4* P,
                         float4* Pn, bool last, bool rest, float4* vout, unsigned* pm,
                         unsigned* rm) {
  const int nb = gv.dense_blocks + list_blocks(c);
  const Commit cm{c.planes, c.posB, c.posA, vout, c.rho, rm};
  with_corr(k, [&](auto corr) {
    constexpr int kCorr = decltype(corr)::value;
    if (!last)
      k_delta<false, false, kCorr><<<nb, kBlock, 0, c.stream>>>(k, gv, P, Pn, cm, pm, c.flags);
    else if (rest)
      k_delta<true, true, kCorr><<<nb, kBlock, 0, c.stream>>>(k, gv, P, Pn, cm, pm, c.flags);
    else
      k_delta<true, false, kCorr><<<nb, kBlock, 0, c.stream>>>(k, gv, P, Pn, cm, pm, c.flags);
  });
  return hipGetLastError();
}

hipError_t enqueue_commit(Ctx& c, const StepConsts& k, const float4* P, bool rest, float4* vout) {
  const Commit cm{c.planes, c.posB, c.posA, vout, nullptr, nullptr};
  if (rest)
    k_commit<true><<<blocks_for(c.n, kBlock), kBlock, 0, c.stream>>>(k, P, c.seg, cm, c.flags);
  else
    k_commit<false><<<blocks_for(c.n, kBlock), kBlock, 0, c.stream>>>(k, P, c.seg, cm, c.flags);
  return hipGetLastError();
}

hipError_t enqueue_xsph(Ctx& c, const StepConsts& k, const GatherView& gv, bool rest,
                        unsigned* rm) {
  const int nb = gv.dense_blocks + list_blocks(c);
  if (rest)
    k_xsph<true><<<nb, kBlock, 0, c.stream>>>(k, gv, c.posA, c.velB, c.velA, c.planes, rm,
                                              c.flags);
  else
    k_xsph<false><<<nb, kBlock, 0, c.stream>>>(k, gv, c.posA, c.velB, c.velA, c.planes, nullptr,
                                               c.flags);
  return hipGetLastError();
}

hipError_t enqueue_vort_omega(Ctx& c, const StepConsts& k, const GatherView& gv) {
  k_vort_omega<<<gv.dense_blocks + list_blocks(c), kBlock, 0, c.stream>>>(k, gv, c.posA, c.velA,
                                                                          c.omega, c.flags);
  return hipGetLastError();
}

hipError_t enqueue_vort_apply(Ctx& c, const StepConsts& k, const GatherView& gv, bool rest) {
  const int nb = gv.dense_blocks + list_blocks(c);
  if (rest)
    k_vort_apply<true><<<nb, kBlock, 0, c.stream>>>(k, gv, c.posA, c.omega, c.velA, c.planes,
                                                    c.flags);
  else
    k_vort_apply<false><<<nb, kBlock, 0, c.stream>>>(k, gv, c.posA, c.omega, c.velA, c.planes,
                                                     c.flags);
  return hipGetLastError();
}

}  // namespace fluidhip
