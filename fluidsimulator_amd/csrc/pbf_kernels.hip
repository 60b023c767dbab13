// gfx950 kernels of one PBF substep and the plan that queues them.
//
// Functional spec: the reference CPU step `fluid::step`
// (core/src/core.cpp:119-615).  Everything here is written for CDNA4:
// 64-lane wavefronts, float4 AoS state resident in HBM, a dense per-scene
// cell table of e x e x e-cell bricks (Z-order inside a brick), a stable LSD
// radix sort of the cell keys into the reference's (cell, id) order, and
// run-length-encoded neighbor lists allocated per workgroup.
//
// Phase order of one substep (one launch each unless noted; every launch
// covers all scenes of a batch):
//   predict_bbox  v' = v + g dt, pred0 = x + v' dt, cell = floor(pred0/h),
//                 per-tile bounding boxes of cells        (core.cpp:150-161)
//   grid_setup    per-scene table origin/extent, key offsets, counters
//   sort          cell keys in original-id order, then 8-bit LSD radix passes
//                 (digit histogram, its scan, stable ballot-ranked scatter;
//                 small batches in one workgroup): sorting stably by key
//                 leaves each cell's particles in ascending id, the
//                 reference's order (core.cpp:164-203)
//   reorder       gather each particle's state into its slot, recompute
//                 pred0; cell starts from the sorted keys
//   tiles         with 4-cell bricks: the bricks that run through LDS (the
//                 particles of their good cells) and their neighbor lists
//                 (pbf_tiles.hip; on the side stream in large batches)
//   runs          runs of identical consecutive particles and their first
//                 slots, the heads that the other passes compute (tile slots
//                 are left out); this and what follows: pbf_gather.hip
//   neighbors     27 cells in (dz, dy, dx) order, each by ascending id,
//                 j != i and r^2 < h^2 on pred0       (core.cpp:205-247)
//   lambda/delta  x solver_iterations, Jacobi double buffer (core.cpp:277-408);
//                 the last delta also commits x and v  (core.cpp:410-421)
//   xsph          (core.cpp:423-466)
//   vorticity     omega, then eta + confinement        (core.cpp:468-571)
//   plane restitution/friction fused into whichever kernel ends the chain
//                                                      (core.cpp:573-612)
// Each gather pass also runs its tile kernel.

#include <algorithm>
#include <climits>

#include "pbf_ctx.h"
#include "pbf_device.h"

namespace fluidhip {

namespace {

constexpr int kWave = 64;

// Kernels launched after the grid setup stop as soon as an earlier phase has
// raised a fatal flag; the committed state is then left untouched.
__device__ __forceinline__ bool fatal(const unsigned* flags) {
  return (*flags & kFlagFatal) != 0u;
}

template <typename T>
__device__ __forceinline__ T wave_min(T v) {
  for (int o = kWave / 2; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, kWave));
  return v;
}
template <typename T>
__device__ __forceinline__ T wave_max(T v) {
  for (int o = kWave / 2; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, kWave));
  return v;
}

// Inclusive prefix sum over the wavefront.
__device__ __forceinline__ int wave_incl_scan(int v) {
  const int lane = threadIdx.x & (kWave - 1);
  for (int o = 1; o < kWave; o <<= 1) {
    const int u = __shfl_up(v, o, kWave);
    if (lane >= o) v += u;
  }
  return v;
}

// Exclusive prefix sum over the workgroup; *total receives the sum.
// `lds` needs blockDim.x / 64 ints.
__device__ __forceinline__ int block_excl_scan(int v, int* lds, int* total) {
  const int lane = threadIdx.x & (kWave - 1);
  const int w = threadIdx.x / kWave;
  const int nw = blockDim.x / kWave;
  const int inc = wave_incl_scan(v);
  if (lane == kWave - 1) lds[w] = inc;
  __syncthreads();
  if (threadIdx.x == 0) {
    int run = 0;
    for (int i = 0; i < nw; ++i) {
      const int t = lds[i];
      lds[i] = run;
      run += t;
    }
    lds[nw] = run;
  }
  __syncthreads();
  const int r = lds[w] + inc - v;
  *total = lds[nw];
  __syncthreads();
  return r;
}

// ---------------------------------------------------------------- transfers

__global__ void k_upload(int n, const float* __restrict__ pos, const float* __restrict__ vel,
                         float4* __restrict__ posA, float4* __restrict__ velA) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const size_t N = static_cast<size_t>(n);
  posA[i] = make_float4(pos[i], pos[N + i], pos[2 * N + i], __int_as_float(i));
  velA[i] = make_float4(vel[i], vel[N + i], vel[2 * N + i], 0.0f);
}

__global__ void k_download(int n, const float4* __restrict__ posA, const float4* __restrict__ velA,
                           float* __restrict__ pos, float* __restrict__ vel) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const float4 p = posA[s];
  const float4 v = velA[s];
  const size_t id = static_cast<size_t>(__float_as_int(p.w));
  const size_t N = static_cast<size_t>(n);
  pos[id] = p.x;
  pos[N + id] = p.y;
  pos[2 * N + id] = p.z;
  vel[id] = v.x;
  vel[N + id] = v.y;
  vel[2 * N + id] = v.z;
}

__global__ void k_reset_flags(unsigned* flags, int* steps_started, int* info) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    *flags = 0u;
    *steps_started = 0;
    info[4] = 0;  // workgroups of k_predict_setup that have finished
  }
}

__global__ void k_init_bbox(int n_scenes, int* bbox) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n_scenes) return;
  bbox[6 * s + 0] = INT_MAX;
  bbox[6 * s + 1] = INT_MAX;
  bbox[6 * s + 2] = INT_MAX;
  bbox[6 * s + 3] = INT_MIN;
  bbox[6 * s + 4] = INT_MIN;
  bbox[6 * s + 5] = INT_MIN;
}

// ---------------------------------------------------------------- grid build

// Calls fn(leader, mine) once per distinct key among the lanes with
// want == true: `leader` is the lowest such lane holding the key and `mine`
// marks the lanes that share it.  Wavefront-uniform control flow; every
// lane must be present.
template <typename Fn>
__device__ __forceinline__ void for_each_key_group(bool want, int key, Fn&& fn) {
  bool pend = want;
  while (true) {
    const unsigned long long m = __ballot(pend);
    if (m == 0ull) break;
    const int leader = __builtin_ctzll(m);
    const int kl = __builtin_amdgcn_readlane(key, leader);
    const bool mine = pend && key == kl;
    fn(leader, mine);
    pend = pend && !mine;
  }
}

// Waits until the calling wavefront's earlier atomics are done at agent scope.
// The barrier of a workgroup waits for none of them.
__device__ __forceinline__ void release_agent() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
}

// kCounted: the caller counts the workgroup as finished after a barrier, and
// whoever counts it reads the boxes and the flags (k_predict_setup).  A tile of
// one scene has its box stored by the thread that counts, but the boxes of a
// tile that straddles scenes, and the range flag, are atomics of any wavefront:
// each releases its own.
template <bool kCounted>
__device__ __forceinline__ void predict_bbox(
    const StepConsts& c, const float4* __restrict__ pos, const float4* __restrict__ vel,
    const ScenePlanes* __restrict__ sp, const int* __restrict__ seg,
    uint64_t* __restrict__ cellc, int* __restrict__ bbox, int* __restrict__ tile_bbox,
    unsigned* __restrict__ flags) {
  __shared__ int red[6][1024 / kWave];
  const int tile = tile_index(c.xcd_remap);
  const int base = tile * blockDim.x;
  const int i = base + threadIdx.x;
  const bool active = i < c.n;
  int mn0 = INT_MAX, mn1 = INT_MAX, mn2 = INT_MAX;
  int mx0 = INT_MIN, mx1 = INT_MIN, mx2 = INT_MIN;
  bool bad = false;
  int sc = 0;
  if (active) {
    sc = scene_of(i, seg, c.n_scenes);
    const ScenePlanes& s = sp[sc];
    const float3 x = ld3(pos, i);
    const float3 v = ld3(vel, i);
    const float vx = v.x + s.gx * c.dt;  // core.cpp:155-157
    const float vy = v.y + s.gy * c.dt;
    const float vz = v.z + s.gz * c.dt;
    const float px = x.x + vx * c.dt;    // core.cpp:158-160
    const float py = x.y + vy * c.dt;
    const float pz = x.z + vz * c.dt;
    const int cx = floor_cell(px, c.inv_h, bad);
    const int cy = floor_cell(py, c.inv_h, bad);
    const int cz = floor_cell(pz, c.inv_h, bad);
    cellc[i] = pack_cell(cx, cy, cz);
    mn0 = mx0 = cx;
    mn1 = mx1 = cy;
    mn2 = mx2 = cz;
  }
  if (bad) {
    atomicOr(flags, kFlagRange);
    if (kCounted) release_agent();
  }
  const int last = min(base + static_cast<int>(blockDim.x), c.n) - 1;
  if (base > last) return;  // whole block past the end (uniform)
  const int s_first = scene_of(base, seg, c.n_scenes);
  const int s_last = scene_of(last, seg, c.n_scenes);
  if (s_first == s_last) {
    // one scene: reduce the workgroup, then one set of atomics
    mn0 = wave_min(mn0), mn1 = wave_min(mn1), mn2 = wave_min(mn2);
    mx0 = wave_max(mx0), mx1 = wave_max(mx1), mx2 = wave_max(mx2);
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    if (lane == 0) {
      red[0][w] = mn0, red[1][w] = mn1, red[2][w] = mn2;
      red[3][w] = mx0, red[4][w] = mx1, red[5][w] = mx2;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      const int nw = blockDim.x / kWave;
      for (int k = 1; k < nw; ++k) {
        mn0 = min(mn0, red[0][k]), mn1 = min(mn1, red[1][k]), mn2 = min(mn2, red[2][k]);
        mx0 = max(mx0, red[3][k]), mx1 = max(mx1, red[4][k]), mx2 = max(mx2, red[5][k]);
      }
      // one plain store per tile; grid_setup reduces the tiles of a scene
      int* b = tile_bbox + 6 * tile;
      b[0] = mn0, b[1] = mn1, b[2] = mn2, b[3] = mx0, b[4] = mx1, b[5] = mx2;
    }
  } else {
    // a tile that straddles scenes: each wavefront reduces the lanes of each
    // of its scenes and takes one set of atomics per scene (in a batch of
    // small scenes many tiles straddle, and per-particle atomics on one
    // scene's six words serialize)
    const int lane = threadIdx.x & (kWave - 1);
    for_each_key_group(active, sc, [&](int leader, bool mine) {
      const int a0 = wave_min(mine ? mn0 : INT_MAX), a1 = wave_min(mine ? mn1 : INT_MAX),
                a2 = wave_min(mine ? mn2 : INT_MAX);
      const int b0 = wave_max(mine ? mx0 : INT_MIN), b1 = wave_max(mine ? mx1 : INT_MIN),
                b2 = wave_max(mine ? mx2 : INT_MIN);
      if (lane == leader) {
        int* b = bbox + 6 * sc;
        atomicMin(b + 0, a0), atomicMin(b + 1, a1), atomicMin(b + 2, a2);
        atomicMax(b + 3, b0), atomicMax(b + 4, b1), atomicMax(b + 5, b2);
      }
    });
    if (kCounted) release_agent();
    if (threadIdx.x == 0) {
      int* b = tile_bbox + 6 * tile;
      b[0] = b[1] = b[2] = INT_MAX;
      b[3] = b[4] = b[5] = INT_MIN;
    }
  }
}

// What the grid setup reads and writes besides the boxes.
struct GridSetup {
  int n_scenes;
  const int* __restrict__ seg;
  int tile_size;
  GridDesc* __restrict__ grid;
  int* __restrict__ total_cells;
  long long cell_cap;
  int bshift;
  unsigned long long* __restrict__ nbr_total;
  unsigned long long* __restrict__ need_cells;
  int* __restrict__ steps_started;
  int* __restrict__ tile_count;  // null without tiles
  int* __restrict__ info;
  StepConsts* __restrict__ last;  // the constants of the last good substep
};

constexpr int kGridSetupThreads = 1024;
constexpr int kLocalBoxes = 64;  // scenes whose boxes are folded in LDS

// One workgroup: per-scene table extents and key offsets; resets the per-step
// counters (kFew: no more scenes than threads).
template <bool kFew>
__device__ __forceinline__ void grid_setup(const StepConsts& c, const GridSetup& gs,
                                           const int* tile_bbox, int* bbox, unsigned* flags) {
  const int n_scenes = gs.n_scenes, tile_size = gs.tile_size, bshift = gs.bshift;
  const long long cell_cap = gs.cell_cap;
  const int* __restrict__ seg = gs.seg;
  GridDesc* __restrict__ grid = gs.grid;
  __shared__ long long sh[kGridSetupThreads / kWave];
  __shared__ int box[6 * kLocalBoxes];
  // After a failed substep the counters keep what the host needs to size
  // the retry; only the bounding boxes are reset.
  const bool was_fatal = (*flags & kFlagFatal) != 0u;
  // Fold each scene's tile partials into its box (which already holds the
  // atomics of tiles that straddle two scenes): `per` wavefronts per scene,
  // each folding every per-th stretch of 64 tiles; with one wavefront or a few
  // per scene, through LDS.
  const int lane = threadIdx.x & (kWave - 1);
  const int nw = static_cast<int>(blockDim.x) / kWave;
  const int w = static_cast<int>(threadIdx.x) / kWave;
  const bool local = n_scenes <= kLocalBoxes;
  if (local)
    for (int i = threadIdx.x; i < 6 * n_scenes; i += blockDim.x) box[i] = bbox[i];
  __syncthreads();
  {
    const int per = n_scenes >= nw ? 1 : nw / n_scenes;
    for (int sc = w / per; sc < n_scenes; sc += nw / per) {
      const int a = seg[sc], b = seg[sc + 1];
      int v[6] = {INT_MAX, INT_MAX, INT_MAX, INT_MIN, INT_MIN, INT_MIN};
      if (b > a) {
        for (int t = a / tile_size + (w % per) * kWave + lane; t <= (b - 1) / tile_size;
             t += per * kWave) {
          const int* p = tile_bbox + 6 * t;
          v[0] = min(v[0], p[0]), v[1] = min(v[1], p[1]), v[2] = min(v[2], p[2]);
          v[3] = max(v[3], p[3]), v[4] = max(v[4], p[4]), v[5] = max(v[5], p[5]);
        }
      }
      for (int k = 0; k < 3; ++k) v[k] = wave_min(v[k]);
      for (int k = 3; k < 6; ++k) v[k] = wave_max(v[k]);
      if (lane == 0) {
        int* bb = (local ? box : bbox) + 6 * sc;
        for (int k = 0; k < 3; ++k) atomicMin(bb + k, v[k]);
        for (int k = 3; k < 6; ++k) atomicMax(bb + k, v[k]);
      }
    }
  }
  __syncthreads();
  // Scene s's extents and the cells of its table.
  auto extents = [&](int s, GridDesc& g) -> long long {
    if (s >= n_scenes) return 0;
    const int* from = (local ? box : bbox) + 6 * s;
    const long long lx = from[0], ly = from[1], lz = from[2];
    const long long hx = from[3], hy = from[4], hz = from[5];
    g.bshift = bshift;
    if (lx > hx || ly > hy || lz > hz) return 0;
    // (cells of a margin of one on each side, in whole bricks)
    const int up = (1 << bshift) + 2;
    const long long bx = (hx - lx + up) >> bshift, by = (hy - ly + up) >> bshift,
                    bz = (hz - lz + up) >> bshift;
    g.ox = static_cast<int>(lx - 1);
    g.oy = static_cast<int>(ly - 1);
    g.oz = static_cast<int>(lz - 1);
    g.nbx = static_cast<int>(bx);
    g.nby = static_cast<int>(by);
    g.nbz = static_cast<int>(bz);
    // (a table this large never fits, and neither the product nor the sum over
    // scenes that lie in the whole coordinate range fits 64 bits)
    const long long many = 1ll << 40;
    const long long layer = bx * by < many ? bx * by : many;
    const long long bricks = layer * bz < many ? layer * bz : many;
    return bricks << (3 * bshift);
  };
  // Exclusive prefix of one value per thread; `all` receives the sum.
  auto prefix = [&](long long v, long long& all) {
    long long inc = v;
    for (int o = 1; o < kWave; o <<= 1) {
      const long long u = __shfl_up(inc, o, kWave);
      if (lane >= o) inc += u;
    }
    if (lane == kWave - 1) sh[w] = inc;
    __syncthreads();
    long long before = 0;
    all = 0;
    for (int u = 0; u < nw; ++u) {
      before += u < w ? sh[u] : 0;
      all += sh[u];
    }
    __syncthreads();  // sh is reused
    return inc - v + before;
  };
  // A substep that fails leaves the grid of the last good one, which belongs to
  // the other arrays of that substep: the scenes' cells in all are known before
  // any scene's grid is written.
  const bool few = kFew || n_scenes <= static_cast<int>(blockDim.x);
  long long total = 0, carry = 0;
  if (!few)
    for (int b0 = 0; b0 < n_scenes; b0 += blockDim.x) {
      GridDesc g{};
      long long all;
      (void)prefix(extents(b0 + threadIdx.x, g), all);
      total += all;
    }
  for (int b0 = 0; b0 < (kFew ? 1 : n_scenes); b0 += blockDim.x) {
    const int s = b0 + threadIdx.x;
    GridDesc g{};
    const long long nc = extents(s, g);
    long long all;
    const long long excl = prefix(nc, all) + carry;
    if (few) total = all;
    if (s < n_scenes) {
      if (total <= cell_cap && !was_fatal) {
        g.cell_off = static_cast<int>(excl);
        g.ncells = static_cast<int>(nc);
        grid[s] = g;
      }
      int* bb = bbox + 6 * s;
      bb[0] = INT_MAX, bb[1] = INT_MAX, bb[2] = INT_MAX;
      bb[3] = INT_MIN, bb[4] = INT_MIN, bb[5] = INT_MIN;
    }
    carry += all;
  }
  if (threadIdx.x == 0 && !was_fatal) {
    if (total <= cell_cap) {
      // word by word: as a struct it goes through scratch memory, which costs
      // every wavefront of the launch
      static_assert(sizeof(StepConsts) % sizeof(int) == 0, "whole words");
      const int* from = reinterpret_cast<const int*>(&c);
      int* to = reinterpret_cast<int*>(gs.last);
#pragma unroll
      for (size_t i = 0; i < sizeof(StepConsts) / sizeof(int); ++i) to[i] = from[i];
      *gs.nbr_total = 0ull;
      gs.info[2] = 0;  // dense units
      if (gs.tile_count) {
        gs.tile_count[0] = 0;  // tiles
        gs.tile_count[1] = 0;  // candidate bricks
      }
      *gs.total_cells = static_cast<int>(total);
      atomicAdd(gs.steps_started, 1);
    } else {
      atomicOr(flags, kFlagCells);
      *gs.total_cells = 0;
      *gs.need_cells = static_cast<unsigned long long>(total);
    }
  }
}

__global__ __launch_bounds__(1024) void k_predict_bbox(
    StepConsts c, const float4* __restrict__ pos, const float4* __restrict__ vel,
    const ScenePlanes* __restrict__ sp, const int* __restrict__ seg,
    uint64_t* __restrict__ cellc, int* __restrict__ bbox, int* __restrict__ tile_bbox,
    unsigned* __restrict__ flags) {
  predict_bbox<false>(c, pos, vel, sp, seg, cellc, bbox, tile_bbox, flags);
}

__global__ __launch_bounds__(kGridSetupThreads) void k_grid_setup(StepConsts c, GridSetup gs,
                                                                  const int* tile_bbox, int* bbox,
                                                                  unsigned* flags) {
  grid_setup<false>(c, gs, tile_bbox, bbox, flags);
}

// Both in one launch: the workgroup that finishes last (a device counter,
// which it clears again) sets the grid up from all workgroups' boxes.
__global__ __launch_bounds__(1024) void k_predict_setup(
    StepConsts c, GridSetup gs, const float4* __restrict__ pos, const float4* __restrict__ vel,
    const ScenePlanes* __restrict__ sp, uint64_t* __restrict__ cellc, int* bbox, int* tile_bbox,
    int* finished, unsigned* flags) {
  __shared__ int last_sh;
  predict_bbox<true>(c, pos, vel, sp, gs.seg, cellc, bbox, tile_bbox, flags);
  __syncthreads();
  if (threadIdx.x == 0) {
    __threadfence();  // this thread's box before its workgroup's count
    last_sh = atomicAdd(finished, 1) == static_cast<int>(gridDim.x) - 1;
    __threadfence();  // every workgroup's box after the last count
  }
  __syncthreads();
  if (!last_sh) return;
  if (threadIdx.x == 0) *finished = 0;
  grid_setup<true>(c, gs, tile_bbox, bbox, flags);
}

// The cell key of slot p of the previous substep's order.
__device__ __forceinline__ int slot_cell_key(const StepConsts& c, int p,
                                             const uint64_t* __restrict__ cellc,
                                             const int* __restrict__ seg,
                                             const GridDesc* __restrict__ grid) {
  const GridDesc g = grid[scene_of(p, seg, c.n_scenes)];
  int x, y, z;
  unpack_cell(cellc[p], x, y, z);
  return cell_key(x - g.ox, y - g.oy, z - g.oz, g);
}

// ---- exclusive scan (fixed grid)

// In two launches: k_scan_reduce writes each workgroup's range sum to
// partial, k_scan_down scans.
__global__ __launch_bounds__(256) void k_scan_reduce(const int* __restrict__ in, int len,
                                                     int* __restrict__ partial,
                                                     const unsigned* __restrict__ flags) {
  __shared__ int lds[8];
  if (fatal(flags)) return;
  const int G = gridDim.x;
  const int chunk = (len + G - 1) / G;
  const int b0 = blockIdx.x * chunk;
  const int b1 = min(len, b0 + chunk);
  int acc = 0;
  for (int i = b0 + threadIdx.x; i < b1; i += blockDim.x) acc += in[i];
  int total;
  block_excl_scan(acc, lds, &total);
  if (threadIdx.x == 0) partial[blockIdx.x] = total;
}

// out[i] = exclusive prefix.  Each workgroup first sums the partials of the
// workgroups before it, then scans its own range, each thread taking four
// consecutive elements per block scan.
__global__ __launch_bounds__(256) void k_scan_down(const int* __restrict__ in, int len,
                                                   const int* __restrict__ partial,
                                                   int* __restrict__ out,
                                                   const unsigned* __restrict__ flags) {
  __shared__ int lds[8];
  if (fatal(flags)) return;
  const int G = gridDim.x;
  const int chunk = (len + G - 1) / G;
  const int b0 = blockIdx.x * chunk;
  const int b1 = min(len, b0 + chunk);
  int run, p = 0;
  for (int j = threadIdx.x; j < static_cast<int>(blockIdx.x); j += blockDim.x) p += partial[j];
  block_excl_scan(p, lds, &run);
  constexpr int kPer = 4;
  for (int t0 = b0; t0 < b1; t0 += kPer * static_cast<int>(blockDim.x)) {
    const int i0 = t0 + kPer * static_cast<int>(threadIdx.x);
    int v[kPer];
    int sum = 0;
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
      v[q] = (i0 + q < b1) ? in[i0 + q] : 0;
      sum += v[q];
    }
    int total;
    int e = run + block_excl_scan(sum, lds, &total);
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
      if (i0 + q < b1) out[i0 + q] = e;
      e += v[q];
    }
    run += total;
  }
}

// ---- stable radix sort of the slots by (cell key, original id)
//
// The keys are written in original-id order, so a stable sort by key alone
// leaves the particles of each cell in ascending id: the reference's order.
// Each pass sorts 8 bits: a per-workgroup digit histogram, the device scan
// of the histogram in digit-major order, and a stable scatter.

// Keys and values in original-id order: k[id] = cell key, v[id] = slot.
__global__ __launch_bounds__(256) void k_sort_keys(StepConsts c, const float4* __restrict__ pos,
                                                   const uint64_t* __restrict__ cellc,
                                                   const int* __restrict__ seg,
                                                   const GridDesc* __restrict__ grid,
                                                   int* __restrict__ kout, int* __restrict__ vout,
                                                   unsigned* __restrict__ flags) {
  if (fatal(flags)) return;
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= c.n) return;
  const int id = __float_as_int(reinterpret_cast<const float*>(pos + p)[3]);
  if (id < 0 || id >= c.n) {  // ids are 0..n-1; refuse rather than write outside
    atomicOr(flags, kFlagRange);
    return;
  }
  kout[id] = slot_cell_key(c, p, cellc, seg, grid);
  vout[id] = p;
}

// Every key lies below the substep's table size, so a pass whose digits
// start at or above its bit length has only digit 0: the stable pass keeps
// the order, its histogram is not needed and its scatter is a copy.
__device__ __forceinline__ bool pass_is_identity(const int* total_cells, int shift) {
  return static_cast<long long>(*total_cells) <= (1ll << shift);
}

// Items of each workgroup (kRadixTile of them) per digit: hist[d * G + b] for
// the scan, or with `rows` hist[b * 256 + d] for the scatter's own sums.
__global__ __launch_bounds__(256) void k_radix_hist(int n, const int* __restrict__ kin, int shift,
                                                    int* __restrict__ hist, int rows,
                                                    const int* __restrict__ total_cells,
                                                    const unsigned* __restrict__ flags) {
  __shared__ int h[256];
  if (fatal(flags) || pass_is_identity(total_cells, shift)) return;
  h[threadIdx.x] = 0;
  __syncthreads();
  const int b0 = blockIdx.x * kRadixTile;
  const int b1 = min(n, b0 + kRadixTile);
  for (int i = b0 + static_cast<int>(threadIdx.x); i < b1; i += 256)
    atomicAdd(&h[(kin[i] >> shift) & 255], 1);
  __syncthreads();
  hist[rows ? blockIdx.x * 256 + threadIdx.x : threadIdx.x * gridDim.x + blockIdx.x] =
      h[threadIdx.x];
}

// The lanes among `ok` whose digit equals this lane's.
__device__ __forceinline__ unsigned long long digit_peers(int d, bool ok) {
  unsigned long long peers = __ballot(ok);
#pragma unroll
  for (int bit = 0; bit < 8; ++bit) {
    const bool x = (d >> bit) & 1;
    const unsigned long long bb = __ballot(x);
    peers &= x ? bb : ~bb;
  }
  return ok ? peers : 0ull;
}

// Stable scatter of one pass: the workgroup's items in index order, 256 per
// round; an item goes to its digit's offset for this workgroup, plus the
// items of that digit in earlier rounds, earlier wavefronts and lower lanes.
// The offsets come from the scanned histogram, or with `hist` (up to
// kRowScatter workgroups) each workgroup sums the histogram's rows itself.
__global__ __launch_bounds__(256) void k_radix_scatter(int n, const int* __restrict__ kin,
                                                       const int* __restrict__ vin,
                                                       int* __restrict__ kout,
                                                       int* __restrict__ vout, int shift,
                                                       const int* __restrict__ off,
                                                       const int* __restrict__ hist,
                                                       const int* __restrict__ total_cells,
                                                       const unsigned* __restrict__ flags) {
  __shared__ int run[256];      // per digit: where the next item of this workgroup goes
  __shared__ int wcnt[4][256];  // per wavefront of the round: items per digit
  __shared__ int scan_lds[8];
  if (fatal(flags)) return;
  const int tid = threadIdx.x;
  if (pass_is_identity(total_cells, shift)) {
    const int b1 = min(n, static_cast<int>(blockIdx.x) * kRadixTile + kRadixTile);
    for (int i = blockIdx.x * kRadixTile + tid; i < b1; i += 256) {
      kout[i] = kin[i];
      vout[i] = vin[i];
    }
    return;
  }
  const int lane = tid & (kWave - 1);
  const int w = tid >> 6;
  if (hist) {
    int before = 0, total = 0;
#pragma unroll 8
    for (int b = 0; b < static_cast<int>(gridDim.x); ++b) {
      const int v = hist[b * 256 + tid];
      total += v;
      before += b < static_cast<int>(blockIdx.x) ? v : 0;
    }
    int all;
    run[tid] = block_excl_scan(total, scan_lds, &all) + before;
  } else {
    run[tid] = off[tid * gridDim.x + blockIdx.x];
  }
  const int b0 = blockIdx.x * kRadixTile;
  for (int r = 0; r < kRadixTile / 256; ++r) {
    const int i = b0 + r * 256 + tid;
    const bool ok = i < n;
    const int kk = ok ? kin[i] : 0;
    const int d = (kk >> shift) & 255;
    const unsigned long long peers = digit_peers(d, ok);
    const int below = __popcll(peers & ((1ull << lane) - 1ull));
    for (int v = 0; v < 4; ++v) wcnt[v][tid] = 0;
    __syncthreads();
    if (ok && below == 0) wcnt[w][d] = __popcll(peers);
    __syncthreads();
    if (ok) {
      int pos = run[d] + below;
      for (int v = 0; v < w; ++v) pos += wcnt[v][d];
      if (pos < n) {  // always, as the histogram counted these same items
        kout[pos] = kk;
        vout[pos] = vin[i];
      }
    }
    __syncthreads();
    run[tid] += wcnt[0][tid] + wcnt[1][tid] + wcnt[2][tid] + wcnt[3][tid];
    // the next round's zeroing of wcnt[.][tid] follows this read in the same thread
  }
}

// The whole sort of a batch of up to kRankSort particles in one launch: the slot
// of a particle is the number of particles with a lower key, or the same key and
// a lower id.  Every workgroup lays the keys of all particles out in LDS by id
// and counts for kRankIds consecutive ids; lane l and l + 32 of its wavefronts
// count for the same id over different blocks of 32 keys.  Ids below the
// workgroup's count with key <= its key, ids above with key <, so each pair is
// one comparison and one addition with carry.
//
// Bound by launch and load latency in the smallest batches and by the keys, which
// every workgroup computes, and the comparisons in the largest: 1,728 / 4,199 /
// 7,680 particles take 6.3 / 9.6 / 16.4 us; a radix sort in one workgroup, which
// this replaces, 10.4 / 16.7 / 27.5.  Beyond kRankSort the work grows with the
// square: k_sort_keys and the radix passes (us per 8 substeps, this against
// them: 9,216 particles 1,295 / 1,303, 13,824 1,460 / 1,420, 16,250 1,558 / 1,423).
constexpr int kRankIds = 32;
constexpr int kRankSort = 8192;
__global__ __launch_bounds__(1024) void k_rank_sort(
    StepConsts c, const float4* __restrict__ pos, const uint64_t* __restrict__ cellc,
    const int* __restrict__ seg, const GridDesc* __restrict__ grid, int* __restrict__ kout,
    int* __restrict__ vout, unsigned* __restrict__ flags) {
  constexpr int kT = 1024, kHalves = kT / kRankIds;
  __shared__ __align__(16) unsigned key[kRankSort];
  __shared__ int slot[kRankIds];
  __shared__ int rank[kRankIds];
  // (the flag may be raised by other workgroups at any time: no barrier depends on it)
  const bool failed = fatal(flags);
  const int n = c.n, tid = threadIdx.x;
  const int i0 = blockIdx.x * kRankIds;
  const int blocks = (n + kRankIds - 1) / kRankIds;
  if (tid < kRankIds) {
    rank[tid] = 0;
    slot[tid] = -1;
    if (n + tid < blocks * kRankIds) key[n + tid] = INT_MAX;  // below no key
  }
  __syncthreads();
#pragma unroll 4
  for (int p = tid; p < n; p += kT) {
    const int id = __float_as_int(reinterpret_cast<const float*>(pos + p)[3]);
    if (id < 0 || id >= n) {  // ids are 0..n-1; refuse rather than write outside
      atomicOr(flags, kFlagRange);
      continue;
    }
    key[id] = static_cast<unsigned>(slot_cell_key(c, p, cellc, seg, grid));
    if (id - i0 >= 0 && id - i0 < kRankIds) slot[id - i0] = p;
  }
  __syncthreads();
  const int i = tid & (kRankIds - 1);
  const unsigned mine = key[i0 + i];
  int count[2] = {0, 0};
  for (int b = tid / kRankIds; b < blocks; b += kHalves) {
    const uint4* q = reinterpret_cast<const uint4*>(key + b * kRankIds);
    if (b != static_cast<int>(blockIdx.x)) {
      const unsigned lim = mine + (b < static_cast<int>(blockIdx.x) ? 1u : 0u);
#pragma unroll
      for (int j = 0; j < kRankIds / 4; ++j) {
        const uint4 k = q[j];
        count[0] += k.x < lim ? 1 : 0;
        count[1] += k.y < lim ? 1 : 0;
        count[0] += k.z < lim ? 1 : 0;
        count[1] += k.w < lim ? 1 : 0;
      }
    } else {
      const unsigned* k = key + b * kRankIds;
#pragma unroll 1
      for (int j = 0; j < kRankIds; ++j) count[0] += k[j] < mine + (j < i ? 1u : 0u) ? 1 : 0;
    }
  }
  atomicAdd(&rank[i], count[0] + count[1]);
  __syncthreads();
  if (tid < kRankIds && i0 + tid < n && !failed) {
    const int r = rank[tid];  // below n: the particle itself is not counted
    kout[r] = static_cast<int>(mine);
    vout[r] = slot[tid];
  }
}

// First index in the sorted sk[0, n) whose key is not below `target`: a
// wavefront probes 64 places at a time.
__device__ __forceinline__ int lower_bound64(const int* __restrict__ sk, int n, int target) {
  const int lane = threadIdx.x & (kWave - 1);
  int lo = 0, hi = n;
  while (lo < hi) {
    const int step = (hi - lo + kWave - 1) / kWave;
    const int i = lo + lane * step;
    const int less = __popcll(__ballot(i < hi && sk[i] < target));
    if (less == 0) return lo;
    hi = min(hi, lo + less * step);
    lo += (less - 1) * step + 1;
  }
  return lo;
}

// Cells a workgroup of k_table fills at a time: kTableCells of a sparse table,
// kTableDense of one with fewer than kTableSparse cells per particle (whose
// ranges hold more keys to read).
constexpr int kTableCells = 4096, kTableDense = 512, kTableSparse = 8;

// Gathers the particle of slot dest of the (cell, id) order (sv: the sorted
// previous slots, sk: their cell keys) and recomputes pred there.
__device__ __forceinline__ void reorder_slot(
    const StepConsts& c, int dest, const int* __restrict__ sk, const int* __restrict__ sv,
    const int* __restrict__ seg, const ScenePlanes* __restrict__ sp,
    const float4* __restrict__ posA, const float4* __restrict__ velA, float4* __restrict__ posB,
    float4* __restrict__ velB, float4* __restrict__ pred, const uint64_t* __restrict__ cellc,
    uint64_t* __restrict__ slot_cell, int* __restrict__ slot_key,
    unsigned* __restrict__ flags) {
  if (dest >= c.n) return;
  const int p = sv[dest];
  if (p < 0 || p >= c.n) {  // never for a complete sort; refuse rather than read outside
    atomicOr(flags, kFlagRange);
    return;
  }
  const int scn = scene_of(dest, seg, c.n_scenes);
  const ScenePlanes& s = sp[scn];
  const float4 x = posA[p];
  const float4 v = velA[p];
  const float vx = v.x + s.gx * c.dt;
  const float vy = v.y + s.gy * c.dt;
  const float vz = v.z + s.gz * c.dt;
  posB[dest] = x;
  velB[dest] = make_float4(vx, vy, vz, __int_as_float(scn));  // read by the heads' kernels
  pred[dest] = make_float4(x.x + vx * c.dt, x.y + vy * c.dt, x.z + vz * c.dt, 0.0f);
  slot_cell[dest] = cellc[p];
  slot_key[dest] = sk[dest];
}

// Writes start[c0 .. c0 + m), m <= 256 kPer, from the sorted keys: two searches
// give the cells' slots, whose runs' heads set their cells' starts in LDS, and a
// suffix minimum gives an empty cell the next cell's start.
template <int kPer>
__device__ __forceinline__ void table_range(int n, const int* __restrict__ sk, int c0, int m,
                                            int total, int* first, int* range, int* wmin,
                                            int* __restrict__ start) {
  const int tid = threadIdx.x, lane = tid & (kWave - 1), w = tid / kWave;
  if (w < 2) {
    // (the last cells' end: every key lies below the table's size)
    const int at = w == 1 && c0 + m == total ? n : lower_bound64(sk, n, c0 + w * m);
    if (lane == 0) range[w] = at;
  }
#pragma unroll
  for (int i = 0; i < kPer; ++i) first[i * 256 + tid] = INT_MAX;
  __syncthreads();
  const int lo = range[0], hi = range[1];
  for (int i0 = lo; i0 < hi;) {
    int k[4], before[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int i = min(i0 + q * 256 + tid, hi - 1);
      k[q] = sk[i];
      before[q] = sk[max(i - 1, 0)];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int i = i0 + q * 256 + tid;
      if (i < hi && (i == lo || before[q] != k[q])) first[k[q] - c0] = i;
    }
    i0 += 1024;
    // a pile of particles in one cell: on to the next cell's first
    if (i0 + 8192 < hi) {
      const int pile = sk[i0 - 1];
      if (sk[i0 + 8192] == pile) {
        __syncthreads();
        if (w == 0) {
          const int at = lower_bound64(sk, n, pile + 1);
          if (lane == 0) range[1] = at;
        }
        __syncthreads();
        i0 = range[1];
      }
    }
  }
  __syncthreads();
  int v[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) v[i] = first[tid * kPer + i];
#pragma unroll
  for (int i = kPer - 2; i >= 0; --i) v[i] = min(v[i], v[i + 1]);
  // the least start in the cells of the threads after this one, else hi
  int suf = v[0];
  for (int o = 1; o < kWave; o <<= 1) {
    const int u = __shfl_down(suf, o, kWave);
    if (lane + o < kWave) suf = min(suf, u);
  }
  if (lane == 0) wmin[w] = suf;
  int after = __shfl_down(suf, 1, kWave);
  if (lane == kWave - 1) after = INT_MAX;
  __syncthreads();
  for (int u = w + 1; u < 4; ++u) after = min(after, wmin[u]);
  after = min(after, hi);
  int* out = start + c0 + tid * kPer;
#pragma unroll
  for (int i = 0; i < kPer; ++i)
    if (tid * kPer + i < m) out[i] = min(v[i], after);
  if (tid == 0 && c0 + m == total) start[total] = n;
  __syncthreads();  // LDS is reused
}

// The first `reorder_blocks` workgroups gather the particles into their slots;
// the others write the cell table, start[k] = first slot of cell k, straight
// from the sorted keys.  The table is written once; its histogram, scanned and
// cleared in three launches before, moved four times as much: 270 us for the
// 256-scene ensemble's table of 44 M cells, whose cells and particles take 170
// together here (the particles alone 80).
__global__ __launch_bounds__(256) void k_table(
    StepConsts c, const int* __restrict__ sk, const int* __restrict__ sv,
    const int* __restrict__ seg, const ScenePlanes* __restrict__ sp,
    const float4* __restrict__ posA, const float4* __restrict__ velA, float4* __restrict__ posB,
    float4* __restrict__ velB, float4* __restrict__ pred, const uint64_t* __restrict__ cellc,
    uint64_t* __restrict__ slot_cell, int* __restrict__ slot_key, int reorder_blocks,
    const int* __restrict__ total_cells, int* __restrict__ start,
    unsigned* __restrict__ flags) {
  __shared__ int first[kTableCells];
  __shared__ int range[2];
  __shared__ int wmin[4];
  if (fatal(flags)) return;
  if (static_cast<int>(blockIdx.x) < reorder_blocks) {
    reorder_slot(c, blockIdx.x * 256 + threadIdx.x, sk, sv, seg, sp, posA, velA, posB, velB,
                 pred, cellc, slot_cell, slot_key, flags);
    return;
  }
  const int total = *total_cells;
  const int blocks = static_cast<int>(gridDim.x) - reorder_blocks;
  const bool sparse = total / kTableSparse > c.n;
  const int cells = sparse ? kTableCells : kTableDense;
  for (long long c0 = static_cast<long long>(static_cast<int>(blockIdx.x) - reorder_blocks) * cells;
       c0 < total; c0 += static_cast<long long>(blocks) * cells) {
    const int at = static_cast<int>(c0), m = min(cells, total - at);
    if (sparse)
      table_range<kTableCells / 256>(c.n, sk, at, m, total, first, range, wmin, start);
    else
      table_range<kTableDense / 256>(c.n, sk, at, m, total, first, range, wmin, start);
  }
}

// ---------------------------------------------------------------- launching

struct Launcher {
  Ctx& c;
  template <typename F>
  hipError_t operator()(const char* name, F&& f) {
    return on(c.stream, name, f);
  }
  // events on stream `st` (a tile kernel on the side stream: its pass's own
  // events on the main stream span the fork to the join)
  template <typename F>
  hipError_t on(hipStream_t st, const char* name, F&& f) {
    if (c.prof.on) {
      hipEvent_t a, b;
      if (c.prof.pool.size() >= 2) {
        a = c.prof.pool.back();
        c.prof.pool.pop_back();
        b = c.prof.pool.back();
        c.prof.pool.pop_back();
      } else {
        hipError_t e = hipEventCreate(&a);
        if (e != hipSuccess) return e;
        e = hipEventCreate(&b);
        if (e != hipSuccess) return e;
      }
      (void)hipEventRecord(a, st);
      f();
      (void)hipEventRecord(b, st);
      c.prof.pending.push_back({name, a, b, c.prof.step});
    } else {
      f();
    }
    return hipGetLastError();
  }
};

inline int blocks_for(long long n, int bs) { return static_cast<int>((n + bs - 1) / bs); }

}  // namespace

hipError_t enqueue_reset_flags(Ctx& c) {
  k_reset_flags<<<1, 64, 0, c.stream>>>(c.flags, c.steps_started, c.info);
  return hipGetLastError();
}

hipError_t enqueue_init_grid(Ctx& c) {
  k_init_bbox<<<blocks_for(c.n_scenes, 256), 256, 0, c.stream>>>(c.n_scenes, c.bbox);
  return hipGetLastError();
}

hipError_t enqueue_upload(Ctx& c, const float* d_pos, const float* d_vel) {
  if (c.n == 0) return hipSuccess;
  k_upload<<<blocks_for(c.n, 256), 256, 0, c.stream>>>(c.n, d_pos, d_vel, c.posA, c.velA);
  return hipGetLastError();
}

hipError_t enqueue_download(Ctx& c, float* d_pos, float* d_vel) {
  if (c.n == 0) return hipSuccess;
  k_download<<<blocks_for(c.n, 256), 256, 0, c.stream>>>(c.n, c.posA, c.velA, d_pos, d_vel);
  return hipGetLastError();
}

// Batches of up to this many particles fuse the prediction and the grid setup.
constexpr int kFusedSetup = 1 << 15;
// Workgroups of the radix sort up to which each sums the digit counts of the
// others itself (a chain of 64 loads a digit, about what two launches take).
constexpr int kRowScatter = 64;
// Workgroups of k_table that write the cell table.
constexpr int kTableGrid = 2048;

hipError_t enqueue_substep(Ctx& c, const SubstepRec* rec) {
  if (c.n == 0) return hipSuccess;
  if (rec && c.iterations < 1) return hipErrorInvalidValue;
  // iterate k of the constraint loop: p^0 stays in its own array for the
  // whole substep and later iterates alternate between two others, or the
  // recording's own array per iterate
  auto PK = [&](int k) { return rec ? rec->P[k] : iterate_buffer(c, k); };
  Launcher L{c};
  StepConsts k = c.consts;
  // a recorded substep keeps every particle's own list (the adjoint reads them)
  if (rec) k.full_lists = 2;
  // sparse bricks through the LDS-tiled passes: their slots are no heads of
  // the other passes
  const bool tiles = k.tiles != 0 && c.tile_list != nullptr;
  if (!tiles) k.tiles = 0;
  const TileArgs ta{c.slot_cell, c.tile_count, static_cast<int>(c.tile_cap), c.tile_rec,
                    c.tile_seg,  c.tile_src,   c.tile_list, c.tile_list_cap, c.tile_cnt};
  const GatherView gv = gather_view(c, PK(0));
  const int bs = c.block;
  const int nb = blocks_for(c.n, bs);
  hipStream_t st = c.stream;
  hipError_t e;

#define FH_TRY(x)                      \
  do {                                 \
    e = (x);                           \
    if (e != hipSuccess) return e;     \
  } while (0)

  const GridSetup gs{c.n_scenes,    c.seg,        bs,           c.grid,
                     c.total_cells, c.cell_cap,   c.brick_shift, c.nbr_total,
                     c.need_cells,  c.steps_started, tiles ? c.tile_count : nullptr, c.info,
                     c.last};
  // A small batch's launches take about 4 us each, whatever they do: one less.
  // (In a large one the workgroups' fences cost more, and many scenes' boxes
  // are folded by 1,024 threads.)
  const bool fused_setup = c.n <= kFusedSetup && c.n_scenes <= 16;
  if (fused_setup) {
    FH_TRY(L("predict_bbox", [&] {
      k_predict_setup<<<nb, bs, 0, st>>>(k, gs, c.posA, c.velA, c.planes, c.cellc, c.bbox,
                                         c.tile_bbox, c.info + 4, c.flags);
    }));
  } else {
    FH_TRY(L("predict_bbox", [&] {
      k_predict_bbox<<<nb, bs, 0, st>>>(k, c.posA, c.velA, c.planes, c.seg, c.cellc, c.bbox,
                                        c.tile_bbox, c.flags);
    }));
    FH_TRY(L("grid_setup", [&] {
      k_grid_setup<<<1, kGridSetupThreads, 0, st>>>(k, gs, c.tile_bbox, c.bbox, c.flags);
    }));
  }
  // keys lie below the cell table's capacity: 8 bits per pass
  int key_bits = 1;
  while (key_bits < 31 && (1ll << key_bits) < c.cell_cap) ++key_bits;
  const int passes = (key_bits + 7) / 8;
  int sorted = passes & 1;  // which buffers end up sorted
  FH_TRY(L("sort", [&] {
    if (c.n <= kRankSort) {
      sorted = 0;
      k_rank_sort<<<blocks_for(c.n, kRankIds), 1024, 0, st>>>(
          k, c.posA, c.cellc, c.seg, c.grid, c.sort_k[0], c.sort_v[0], c.flags);
      return;
    }
    k_sort_keys<<<blocks_for(c.n, 256), 256, 0, st>>>(k, c.posA, c.cellc, c.seg, c.grid,
                                                      c.sort_k[0], c.sort_v[0], c.flags);
    const bool rows = c.radix_blocks <= kRowScatter;
    const int len = 256 * c.radix_blocks;
    for (int q = 0; q < passes; ++q) {
      const int i = q & 1, o = i ^ 1;
      k_radix_hist<<<c.radix_blocks, 256, 0, st>>>(c.n, c.sort_k[i], 8 * q, c.radix_hist,
                                                   rows ? 1 : 0, c.total_cells, c.flags);
      if (!rows) {
        k_scan_reduce<<<c.scan_blocks, 256, 0, st>>>(c.radix_hist, len, c.scan_partial, c.flags);
        k_scan_down<<<c.scan_blocks, 256, 0, st>>>(c.radix_hist, len, c.scan_partial,
                                                   c.radix_off, c.flags);
      }
      k_radix_scatter<<<c.radix_blocks, 256, 0, st>>>(
          c.n, c.sort_k[i], c.sort_v[i], c.sort_k[o], c.sort_v[o], 8 * q, c.radix_off,
          rows ? c.radix_hist : nullptr, c.total_cells, c.flags);
    }
  }));
  FH_TRY(L("reorder", [&] {
    const int rb = blocks_for(c.n, 256);
    const int tb = static_cast<int>(
        std::min<long long>(kTableGrid, (c.cell_cap + kTableDense - 1) / kTableDense));
    k_table<<<rb + tb, 256, 0, st>>>(k, c.sort_k[sorted], c.sort_v[sorted], c.seg, c.planes,
                                     c.posA, c.velA, c.posB, c.velB, PK(0), c.cellc, c.slot_cell,
                                     c.slot_key, rb, c.total_cells, c.start, c.flags);
  }));
  // Each pass's tile kernel runs on the side stream beside the heads' kernel
  // on the main stream: they write disjoint slots (a run lies in one cell,
  // which is a tile's as a whole or not at all, and tile slots are no list or
  // dense heads) and read only what earlier passes finished.  fork() makes
  // the side stream wait for the main stream's work so far, join() the main
  // stream for the side stream's.  Both are edges of a captured graph too.
  // An event record and a cross-stream wait leave the device idle for tens
  // of microseconds (about 30 us per fork measured at 65,536 particles), so
  // small batches, whose tile kernels take about as long, stay on one stream.
  const bool forked = tiles && c.side != nullptr && c.n >= kForkMinParticles;
  hipStream_t tst = forked ? c.side : st;
  hipError_t fj = hipSuccess;
  auto fork = [&] {
    if (!forked || fj != hipSuccess) return;
    fj = hipEventRecord(c.ev_fork, st);
    if (fj == hipSuccess) fj = hipStreamWaitEvent(c.side, c.ev_fork, 0);
  };
  auto join = [&] {
    if (!forked || fj != hipSuccess) return;
    fj = hipEventRecord(c.ev_join, c.side);
    if (fj == hipSuccess) fj = hipStreamWaitEvent(st, c.ev_join, 0);
  };
  // The tile lists come before the heads when a tile can go back to them (a
  // particle with more neighbors than its list holds).  A large batch's lists
  // hold every possible neighbor, so its tiles are final after classify: the
  // heads are listed first (their short kernels would wait for CUs behind the
  // tile list build), then the tile lists are built on the side stream while
  // the main stream builds the heads' lists (which write no tile slot).
  const bool early_heads = forked && c.tile_list_cap >= kTileMaxCand - 1;
  auto tile_lists = [&](hipStream_t s) {
    (void)L.on(s, "tile_neighbors", [&] {
      (void)enqueue_tile_neighbors(c, k, ta, PK(0), rec != nullptr, s);
    });
  };
  if (tiles)
    FH_TRY(L("tiles", [&] {
      (void)enqueue_tile_classify(c, k);
      if (!early_heads) tile_lists(st);
    }));
  FH_TRY(L("runs", [&] { (void)enqueue_heads(c, k); }));
  FH_TRY(L("neighbors", [&] {
    if (early_heads) {
      fork();
      tile_lists(tst);
    }
    (void)enqueue_neighbors(c, k, gv);
    if (early_heads) join();
  }));
  FH_TRY(fj);

  // velocity buffer that the commit writes: XSPH needs a second buffer to
  // stay Jacobi, so the commit goes to velB and XSPH back to velA.
  float4* v1 = c.xsph ? c.velB : c.velA;
  const bool rest_in_delta = c.restitution_any && !c.xsph && !c.vort;
  // One pass: its tile kernel forked off beside its kernel over the heads.
  auto pass = [&](const char* name, const char* tile_name, auto&& tile, auto&& heads) {
    const hipError_t pe = L(name, [&] {
      if (tiles) {
        fork();
        (void)L.on(tst, tile_name, [&] { (void)tile(); });
      }
      (void)heads();
      if (tiles) join();
    });
    return pe != hipSuccess ? pe : fj;
  };
  const int I = c.iterations;
  for (int it = 0; it < I; ++it) {
    const bool last = (it + 1 == I);
    float4* P = PK(it);
    float4* Pn = last ? nullptr : PK(it + 1);
    float4* sq = rec ? rec->SQ[it] : nullptr;
    unsigned* pm = rec ? rec->M[it] : nullptr;
    unsigned* rm = rec && last && rest_in_delta ? rec->RM : nullptr;
    const bool rest = last && rest_in_delta;
    FH_TRY(pass(
        "lambda", "tile_lambda",
        [&] { return enqueue_tile_lambda(c, k, ta, P, last ? 1 : 0, sq, tst); },
        [&] { return enqueue_lambda(c, k, gv, P, last, sq); }));
    FH_TRY(pass(
        "delta", "tile_delta",
        [&] { return enqueue_tile_delta(c, k, ta, P, Pn, last, rest, v1, pm, rm, tst); },
        [&] { return enqueue_delta(c, k, gv, P, Pn, last, rest, v1, pm, rm); }));
  }
  if (I == 0)
    FH_TRY(L("delta", [&] { (void)enqueue_commit(c, k, PK(0), rest_in_delta, v1); }));
  if (c.xsph) {
    const bool rest = c.restitution_any && !c.vort;
    unsigned* rm = rest && rec ? rec->RM : nullptr;
    FH_TRY(pass(
        "xsph", "tile_xsph", [&] { return enqueue_tile_xsph(c, k, ta, rest, rm, tst); },
        [&] { return enqueue_xsph(c, k, gv, rest, rm); }));
  }
  if (c.vort) {
    FH_TRY(pass(
        "vorticity_omega", "tile_vorticity_omega",
        [&] { return enqueue_tile_vort_omega(c, k, ta, tst); },
        [&] { return enqueue_vort_omega(c, k, gv); }));
    FH_TRY(pass(
        "vorticity_apply", "tile_vorticity_apply",
        [&] { return enqueue_tile_vort_apply(c, k, ta, c.restitution_any, tst); },
        [&] { return enqueue_vort_apply(c, k, gv, c.restitution_any); }));
  }
#undef FH_TRY
  return hipSuccess;
}

}  // namespace fluidhip
