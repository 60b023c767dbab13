// Device-side data structures and helpers of the gfx950 PBF step.
//
// Arithmetic in this file follows the reference CPU step
// (core/src/core.cpp:35-71, :119-615) operation for operation; the whole
// library is compiled with -ffp-contract=off and IEEE division/sqrt, so each
// expression rounds exactly as the reference's does.
#pragma once

#include <hip/hip_runtime.h>
#include <limits.h>
#include <stdint.h>

#include <type_traits>

namespace fluidhip {

constexpr int kMaxPlanes = 8;
constexpr int kCoordLimit = 1 << 20;

// Device error flags (sticky until the host clears them).
constexpr unsigned kFlagRange = 1u;     // non-finite / out-of-range position
constexpr unsigned kFlagCells = 2u;     // cell table capacity exceeded
constexpr unsigned kFlagNeighbors = 4u; // neighbor list capacity exceeded
constexpr unsigned kFlagFatal = kFlagRange | kFlagCells | kFlagNeighbors;

// Loop-invariant constants of one substep, computed on the host with the
// same float expressions the reference evaluates inside its loops.
// Items per workgroup of the radix sort that orders slots by (cell, id).
// A scatter workgroup ranks its items in serial rounds of 256, so small
// tiles (more workgroups per CU) hide more of each round's latency: 1024
// took the 65,536-particle sort from 86 to 54-62 us and the 1,048,576-particle
// one from 148 to 135 us against 4096 (2048: 71 and 133 us).
constexpr int kRadixTile = 1024;

// The heads of batches of up to this many particles are listed by one workgroup
// instead of in two launches: its rounds over 1,024 slots each are in series.
// Measured, one / two launches, us per 8 substeps of a block just released and
// after 24 substeps, with a workgroup for 8,192: 1,728 particles 724 / 755 and
// 714 / 743; 4,199: 852 / 864 and 919 / 932; 4,896: 895 / 898 and 940 / 942;
// 5,760: 961 / 961 and 1,069 / 1,062; 6,800: 947 / 935 and 998 / 983; 8,000:
// 1,142 / 1,117 and 1,167 / 1,141.
constexpr int kSmallHeads = 5120;

struct StepConsts {
  int n;            // particles, all scenes
  int n_scenes;
  float dt;
  float h;
  float inv_h;      // 1.0f / h            (core.cpp:29)
  float h2;         // h * h               (core.cpp:140)
  float min_r2;     // (0.01f*h)^2         (core.cpp:141-142)
  float f_min;      // spiky(sqrt(min_r2)): the factor of every clamped pair
  float w_coeff;    // 315 / (64 pi h^9)   (core.cpp:44)
  float w0;         // poly6(0, h)         (core.cpp:319)
  float s_coeff;    // -45 / (pi h^6)      (core.cpp:55)
  float inv_density;
  float mass;
  float grad_scale; // m * (1/rho0)        (core.cpp:273)
  float eps;
  int scorr_on;     // enable_scorr && k != 0 && inv_wdq > 0
  float scorr_inv_wdq;
  float scorr_neg_k;  // -k
  int scorr_n;
  float visc_c;
  float vort_eps;
  float vort_norm_eps;
  int xcd_remap;
  int runs;         // 1: a run of identical consecutive slots is computed once
  int full_lists;   // 1: every particle's list is stored (diagnostics), 2: as
                    //    plain slots where it fits a row (the adjoint's)
  int iterations;   // of the constraint loop
  int tiles;        // 1: sparse 4x4x4-cell bricks run the LDS-tiled passes
  int exact_terms;  // 1: pair terms need no range tests (tile_spiky)
};

struct ScenePlanes {
  float gx, gy, gz;
  int n_planes;
  int restitution_on;  // e > 0 || f > 0 for some plane (core.cpp:573)
  int pad[3];
  float4 planes[kMaxPlanes];  // (nx, ny, nz, d)
  float rest_of[kMaxPlanes];  // restitution e of each plane (the scene's
                              // plane_restitution unless given per plane)
  float fric_of[kMaxPlanes];  // friction f of each plane
};

// Per-scene grid descriptor, rebuilt every substep from the predicted
// positions' bounding box.
struct GridDesc {
  int ox, oy, oz;     // cell coordinate of table origin (bbox min - 1)
  int nbx, nby, nbz;  // bricks per axis
  int cell_off;       // first key of this scene
  int ncells;         // nbx*nby*nbz bricks of 2^(3 bshift) cells
  int bshift;         // log2 of the cells per brick edge (0..3)
};

__device__ __forceinline__ float poly6(float r2, const StepConsts& c) {
  // core.cpp:35-46 with the coefficient hoisted (same float value).
  if (r2 > c.h2) return 0.0f;
  const float diff = c.h2 - r2;
  const float diff3 = diff * diff * diff;
  return c.w_coeff * diff3;
}

// The correctly rounded square root (IEEE sqrt, as sqrtf under
// -fhip-fp32-correctly-rounded-divide-sqrt).  For finite x >= 2^-96 the root
// g = x y from the hardware's reciprocal root y is corrected once by its
// residual x - g^2 (one fused operation, exact up to its rounding) times y / 2:
// a Newton step that leaves an error far below the distance of a square root of
// a float from the midpoint of two floats, so rounding it gives sqrtf's bits
// (checked on every such float); other x go through sqrtf itself.  Five
// instructions, where testing the hardware root's two neighbors takes nine; the
// gather passes take one root per neighbor (with the range tests gone too, lambda
// of 262,144 particles without tiles went from 31.1 to 29.1 us).
__device__ __forceinline__ float sqrt_core(float x) {
  // the correction alone: finite x >= 2^-96 only
  const float y = __builtin_amdgcn_rsqf(x);
  const float g = x * y;
  return fmaf(fmaf(-g, g, x), 0.5f * y, g);
}

__device__ __forceinline__ float sqrt_rn(float x) {
  if (x >= 0x1p-96f && x <= 0x1.fffffep+127f) return sqrt_core(x);
  return sqrtf(x);
}

__device__ __forceinline__ float spiky(float r, const StepConsts& c) {
  // core.cpp:48-57 with the coefficient hoisted.
  if (r > c.h) return 0.0f;
  const float diff = c.h - r;
  return c.s_coeff * diff * diff;
}

__device__ __forceinline__ float pow_ratio(float ratio, int n) {
  // core.cpp:59-71.  n outside {2,3,4} goes through powf, whose last bit
  // may differ from the host libm's.
  if (n == 2) return ratio * ratio;
  if (n == 3) return ratio * ratio * ratio;
  if (n == 4) {
    const float r2 = ratio * ratio;
    return r2 * r2;
  }
  return powf(ratio, static_cast<float>(n));
}

// Pair terms of a pair with r2 < h2 (other pairs' values are not used).  With
// c.exact_terms (min_r2 >= 2^-96 and sqrt(max(pred(h2), min_r2)) <= h, checked
// on the host) the clamped argument of the square root is a finite float >=
// 2^-96, where sqrt_core is the correctly rounded square root, and r <= h,
// where spiky's r > h test is false: tile_poly6 and tile_spiky return what
// poly6 and pair_spiky return (core.cpp:35-57 and the clamp of core.cpp:303),
// bit for bit, without their range tests.
__device__ __forceinline__ float tile_poly6(float r2, const StepConsts& c) {
  const float diff = c.h2 - r2;
  const float diff3 = diff * diff * diff;
  return c.w_coeff * diff3;
}

__device__ __forceinline__ float tile_spiky(float r2, const StepConsts& c) {
  // r2 < min_r2 ? min_r2 : r2 for 0 <= r2 < h2 and min_r2 > 0, where the
  // bit patterns order as the floats do (one integer max)
  const float r = sqrt_core(__int_as_float(max(__float_as_int(r2), __float_as_int(c.min_r2))));
  const float diff = c.h - r;
  return c.s_coeff * diff * diff;
}

// li + lj and the tensile correction -k (W / W(dq))^n (core.cpp:334-407).  The
// exponent's kind is a template parameter (corr_kind) so that a walk's terms
// hold no branches: off, one of 2, 3, 4 (selected factors; a factor of 1 is
// exact), or any other, through powf.
constexpr int kCorrOff = 0, kCorrFew = 1, kCorrPow = 2;
inline int corr_kind(const StepConsts& c) {
  if (!c.scorr_on) return kCorrOff;
  return c.scorr_n >= 2 && c.scorr_n <= 4 ? kCorrFew : kCorrPow;
}

// Calls f with the constant of the exponent's kind.
template <typename F>
inline void with_corr(const StepConsts& c, F&& f) {
  if (corr_kind(c) == kCorrOff)
    f(std::integral_constant<int, kCorrOff>{});
  else if (corr_kind(c) == kCorrFew)
    f(std::integral_constant<int, kCorrFew>{});
  else
    f(std::integral_constant<int, kCorrPow>{});
}

template <int kCorr>
__device__ __forceinline__ float pair_lambda(float li, float lj, float r2, const StepConsts& c) {
  float sv = li + lj;
  if (kCorr == kCorrOff) return sv;
  const float ratio = tile_poly6(r2, c) * c.scorr_inv_wdq;
  const float sq = ratio * ratio;
  const float more = c.scorr_n == 3 ? ratio : c.scorr_n == 4 ? sq : 1.0f;
  sv += c.scorr_neg_k * (kCorr == kCorrFew ? sq * more : pow_ratio(ratio, c.scorr_n));
  return sv;
}

// Spiky factor of a pair at squared distance r2 < h2: pairs closer than
// min_r share one factor (core.cpp:303-304 clamps r there).
__device__ __forceinline__ float pair_spiky(float r2, const StepConsts& c) {
  if (c.exact_terms) return tile_spiky(r2, c);
  if (r2 < c.min_r2) return c.f_min;
  return spiky(sqrt_rn(r2), c);
}

// The neighbor predicate: candidate q is a neighbor of a particle at p when
// |p - q|^2 < h^2, both at their predicted positions p^0 (core.cpp:140-142
// and 222-245).  Lists are built with it, and walks without a list retest
// it, so all must use this one expression.
__device__ __forceinline__ bool near0(const float3& p, const float3& q, const StepConsts& c) {
  const float ex = p.x - q.x;
  const float ey = p.y - q.y;
  const float ez = p.z - q.z;
  return ex * ex + ey * ey + ez * ez < c.h2;
}

// Particles of cells of at least this many walk the 27 cells in every pass
// instead of storing a list.
constexpr int kDenseCell = 32;

// A dense unit of one head only (in the scene's sign bit).
constexpr int kSingle = INT_MIN;

// nwords of a slot without words: none stored, neighbors in the slot's row,
// or too many for a row.
constexpr int kRowList = -2, kLongList = -3;

// Z-order of a cell inside its brick of up to 8 cells an edge: the low bits
// of x, y, z interleaved as x0 y0 z0 x1 y1 z1 x2 y2 z2.
__device__ __forceinline__ int morton_in_brick(int x, int y, int z) {
  int m = 0;
#pragma unroll
  for (int b = 0; b < 3; ++b)
    m |= (((x >> b) & 1) << (3 * b)) | (((y >> b) & 1) << (3 * b + 1)) |
         (((z >> b) & 1) << (3 * b + 2));
  return m;
}

// Key of the cell at table-relative coordinates (rx, ry, rz) >= 0: bricks
// in x-fastest order, cells in Z-order inside a brick.  The key only sets
// where a cell's particles sit in the sorted arrays; every sum visits cells
// in (dz, dy, dx) order and particles by id, so the brick edge never
// changes a result.
__device__ __forceinline__ int cell_key(int rx, int ry, int rz, const GridDesc& g) {
  const int s = g.bshift;
  const int m = (1 << s) - 1;
  const int b = ((rz >> s) * g.nby + (ry >> s)) * g.nbx + (rx >> s);
  return g.cell_off + (b << (3 * s)) + morton_in_brick(rx & m, ry & m, rz & m);
}

__device__ __forceinline__ int floor_cell(float v, float inv_h, bool& bad) {
  // static_cast<int>(std::floor(v * inv)) — core.cpp:28-34
  const float s = v * inv_h;
  if (!(fabsf(s) < static_cast<float>(kCoordLimit))) {
    bad = true;
    return 0;
  }
  return static_cast<int>(floorf(s));
}

__device__ __forceinline__ uint64_t pack_cell(int x, int y, int z) {
  const uint64_t m = (1ull << 21) - 1ull;
  return ((uint64_t(x + kCoordLimit) & m) << 42) | ((uint64_t(y + kCoordLimit) & m) << 21) |
         (uint64_t(z + kCoordLimit) & m);
}

__device__ __forceinline__ void unpack_cell(uint64_t k, int& x, int& y, int& z) {
  const uint64_t m = (1ull << 21) - 1ull;
  x = int((k >> 42) & m) - kCoordLimit;
  y = int((k >> 21) & m) - kCoordLimit;
  z = int(k & m) - kCoordLimit;
}

// Scene of a slot: scenes are contiguous, fixed-size slot segments.
__device__ __forceinline__ int scene_of(int slot, const int* __restrict__ seg, int n_scenes) {
  if (n_scenes == 1) return 0;
  int lo = 0, hi = n_scenes - 1;  // seg has n_scenes+1 entries
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (seg[mid] <= slot)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

// Workgroup -> particle tile, so that each XCD (dispatched round-robin)
// streams a contiguous range of the sorted arrays through its own L2.
__device__ __forceinline__ int tile_index(int remap) {
  const int bid = blockIdx.x;
  if (!remap) return bid;
  const int nb = gridDim.x;
  const int q = nb >> 3, r = nb & 7;
  const int xcd = bid & 7, local = bid >> 3;
  return xcd * q + (xcd < r ? xcd : r) + local;
}

__device__ __forceinline__ float3 ld3(const float4* p, int i) {
  const float* f = reinterpret_cast<const float*>(p + i);
  return make_float3(f[0], f[1], f[2]);
}

// Sequential push-out along each plane normal (core.cpp:372-389).  Returns
// the planes that pushed (bit p), which fixes the Jacobian of the
// projection: I - n n^T per pushing plane, applied in plane order.
__device__ __forceinline__ unsigned project_planes(float& qx, float& qy, float& qz,
                                                   const ScenePlanes& sp) {
  unsigned mask = 0;
  for (int p = 0; p < sp.n_planes; ++p) {
    const float4 pl = sp.planes[p];
    const float sd = pl.x * qx + pl.y * qy + pl.z * qz - pl.w;
    const float pen = -sd;
    if (pen > 0.0f) {
      qx += pl.x * pen;
      qy += pl.y * pen;
      qz += pl.z * pen;
      mask |= 1u << p;
    }
  }
  return mask;
}

// Plane restitution and friction (core.cpp:573-612), with each plane's own
// e and f (equal to the scene's globals unless set per plane).  Returns the planes in
// contact (bit p) and, among those, the ones the velocity approached
// (bit 8 + p): with them the map is linear, v -> (1-f) v + (a - (1-f)) (n.v) n
// with a = -e when approaching and 1 otherwise.
__device__ __forceinline__ unsigned restitute(float& vx, float& vy, float& vz, float px, float py,
                                              float pz, const ScenePlanes& sp) {
  if (!sp.restitution_on) return 0;
  unsigned mask = 0;
  for (int p = 0; p < sp.n_planes; ++p) {
    const float4 pl = sp.planes[p];
    const float sd = pl.x * px + pl.y * py + pl.z * pz - pl.w;
    if (sd <= 0.0f) {
      const float vn = pl.x * vx + pl.y * vy + pl.z * vz;
      float vn_new = vn;
      mask |= 1u << p;
      if (vn < 0.0f) {
        vn_new = -sp.rest_of[p] * vn;
        mask |= 1u << (8 + p);
      }
      const float tx = vx - vn * pl.x;
      const float ty = vy - vn * pl.y;
      const float tz = vz - vn * pl.z;
      const float scale = 1.0f - sp.fric_of[p];
      vx = tx * scale + vn_new * pl.x;
      vy = ty * scale + vn_new * pl.y;
      vz = tz * scale + vn_new * pl.z;
    }
  }
  return mask;
}

// Neighbor lists in slot space: a word t >= 0 is the single neighbor t; a word
// with the top bit set starts a run of consecutive slots (t & 0x7fffffff) .. +
// next word - 1, three or more of them.  A list of as many words as neighbors
// holds single neighbors only.
struct NbrView {
  const long long* __restrict__ off;
  const int* __restrict__ nw;
  const int* __restrict__ list;
  const int* __restrict__ count;
};

}  // namespace fluidhip
