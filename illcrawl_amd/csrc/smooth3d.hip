// Volumetric smoothing on gfx950: the 3-D grid reconstruction of dm::grid
// (dm_reconstruction_backend_grid.cl:26-52 running spg_run_reconstruction,
// smoothing_particle_grid.cl:31-127, without SPG_PROJECTION).  Every
// evaluation point (x, y, z) sums w * quartic_polynomial3d(|x_p - x|, h)
// (smoothing_kernel.cl:27-37) over the particles of the cells in its search
// box.
//
// Candidates come from the level index of the grid, not from the reference
// cells: particles binned by h into levels (level L holds h <= max_h 2^(L-23)),
// each level sorted by a fine cell key (z, y, x) whose cell size is 0.7 of the
// level's h.  The reference's cells are coarse (64 particles each on average,
// far more in clustered regions), and a tile inside a cell would stream all
// of them; a level row holds only the particles near the tile.
// The result is the reference's, since the search box test is made on each
// particle's reference cell.
//
// One workgroup of 4 waves owns a tile of T x T points (16 or 8) of the point
// array seen as an image (e.g. a volumetric slice).  It
//   1. loads its points and, in reference mode, each point's search box as
//      the reference computes it (radius = min(max_h[cell] + cell_radius,
//      max_h) from the unclamped 64-bit key of the point's cell, index box of
//      x -/+ radius on each axis);
//   2. reduces the tile's 3-D bounding box, its extent along the normal of its
//      plane, and the union and intersection of the search boxes;
//   3. per level, takes the fine cells within the level's max h of the tile
//      box: one key range per (y, z) row of them (per z plane, or one range,
//      when the rows are too many), a row's cells trimmed to what the level's
//      max h can reach of the box and of the plane, found by binary search in
//      the level's sorted keys.
// The waves then stream the ranges' particles, 64 at a time in turn.  Each
// wave
//   4. culls each particle against the tile box (support sphere vs box) and
//      the tile's plane and, in reference mode, drops it when its reference
//      cell is in no point's search box; the survivors go by ballot to the
//      wave's own LDS lists:
//        cover  - every point may use it and its support holds the whole
//                 tile: its term w (1 - r^2/h^2)^2 is a polynomial over the
//                 tile, quadratic in (1, u, |u|^2) with u relative to the tile
//                 centre; the lane adds its 15 coefficients (FP64), and each
//                 point evaluates the sum once;
//        full   - every point may use it;
//        masked - reference mode, its cell may be inside some points' search
//                 box and outside others';
//   5. evaluates full lists from LDS for every point of the tile, FP32 over 32
//      particles, then into FP64 accumulators.
// At the end the waves' sums are added, in wave order.
//
#include <hip/hip_runtime.h>

#include <algorithm>

#include "cellmax.hpp"
#include "common.hpp"
#include "kernels.hpp"
#include "wave.hpp"

namespace ilc {

namespace {

constexpr int kWaves3 = 4;
// a wave evaluates a list when it reaches kFlush3 entries; a batch of 64
// lands on at most kFlush3 - 1.  full and masked share an array from its two
// ends, each with room to pad to a multiple of 4.
constexpr int kFlush3 = 32;
constexpr int kCap3 = kFlush3 - 1 + 64 + 1;
constexpr int kPool3 = 2 * (kFlush3 - 1) + 64 + 6;
static_assert(kCap3 % 4 == 0 && kPool3 % 4 == 0, "whole groups of 4 entries");
constexpr uint32_t kRowCap3 = 64;  // key rows per level and tile before coarser ranges

// grid3d_get_cell_indices of p + r on one axis, FP32, no FMA
__device__ inline int32_t cell_of(float p, float r, float mn, float cs) {
#pragma clang fp contract(off)
  const float a = p + r;
  const float d = a - mn;
  return floor_to_int(d / cs);
}

__device__ inline uint32_t prefix_count(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(mask >> 32),
                                   __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(mask), 0u));
}
__device__ inline int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// orders this wave's LDS accesses
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <bool REF>
struct lists3 {
  float4 S[kPool3];  // full from the front, masked from the back: (x, y, z, 1/h^2)
  float w[kPool3];   // coef
  alignas(16) int2 M[REF ? kCap3 : 1];  // masked: reference cell (cx | cy << 16, cz)
  uint32_t C[128];   // cover: index
};

template <int T, bool REF>
struct smem3 {
  static constexpr int NP = T * T;
  union {
    lists3<REF> L[kWaves3];
    double sum[kWaves3][NP];  // at the end of the tile
  };
  double poly[kWaves3][16];  // the cover form's coefficients
  float4 pt[NP];
  // the points' search boxes: (x0 | xw << 16, y0 | yw << 16, z0, zw)
  uint4 box[REF ? NP : 1];
  uint32_t row_b[kBlock];
  uint32_t row_off[kBlock];
  uint32_t scan_ws[4];
  uint32_t hits[4];
  float redf[kWaves3][8];
  float minr[kWaves3];
  int redi[kWaves3][13];
  int covered;
  // the tile's key rows per level: fine box, row mode, first row, start
  int lv_f0[kLevels3][3];
  int lv_f1[kLevels3][3];
  int lv_mode[kLevels3];
  float lv_r[kLevels3];  // the level's max h
  uint32_t lv_row0[kLevels3 + 1];
  uint32_t lv_s[kLevels3 + 1];
  uint32_t lv_p[kLevels3 + 1];  // plane directory offsets
};

// level of a particle: the smallest L with h <= max_h 2^(L - 23) (by the
// exponent of max_h / h; a level may also hold smaller h: the gather
// searches it with its largest possible h)
__device__ inline int level_of(float h, float max_h, int lmin) {
  const float r = max_h / h;
  const int e = int((__float_as_uint(r) >> 23) & 0xffu) - 127;
  return min(max(kLevels3 - 1 - e, lmin), kLevels3 - 1);
}

// fine cell coordinate, clamped to [0, fmax]; monotone in x
__device__ inline uint32_t fine_of(float x, float mn, float cs, uint32_t fmax) {
#pragma clang fp contract(off)
  const float f = floorf((x - mn) / cs);
  if (!(f >= 0.0f)) return 0u;
  if (f >= float(fmax)) return fmax;
  return uint32_t(f);
}

__device__ inline unsigned long long fine_key(const level_key& b, int l, uint32_t fx, uint32_t fy,
                                              uint32_t fz) {
  using u64 = unsigned long long;
  return (u64(l - b.lmin) << b.shift[3]) | (u64(fz) << b.shift[2]) | (u64(fy) << b.shift[1]) |
         u64(fx);
}

// first index in [a, b) whose key is >= k (keys sorted ascending)
__device__ inline uint32_t lower_bound_u64(const unsigned long long* __restrict__ key, uint32_t a,
                                           uint32_t b, unsigned long long k) {
  while (a < b) {
    const uint32_t m = (a + b) >> 1;
    if (key[m] < k)
      a = m + 1;
    else
      b = m;
  }
  return a;
}

// the same for a k expected close after a: steps of 1, 2, 4, ... from a
// bracket it, then a binary search inside the bracket (a row of fine cells
// holds few particles, so this takes a few dependent loads, not log2 n)
__device__ inline uint32_t gallop_lower_bound_u64(const unsigned long long* __restrict__ key,
                                                  uint32_t a, uint32_t b, unsigned long long k) {
  uint32_t lo = a, step = 1;
  while (lo < b && key[lo] < k) {
    a = lo + 1;
    lo = (b - lo > step) ? lo + step : b;
    step <<= 1;
  }
  return lower_bound_u64(key, a, lo, k);
}

__device__ inline uint32_t block_scan_excl(uint32_t v, uint32_t* total, uint32_t* ws) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t incl = v;
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(incl, o, 64);
    if (lane >= o) incl += y;
  }
  if (lane == 63) ws[wave] = incl;
  __syncthreads();
  uint32_t off = 0, tot = 0;
  for (int w = 0; w < 4; ++w) {
    if (w < wave) off += ws[w];
    tot += ws[w];
  }
  __syncthreads();
  *total = tot;
  return off + incl - v;
}

// Bound by issue slots and, with 5 or 6 waves a SIMD, by waiting for them: a VALU
// instruction issues in 81% of the busy cycles (SQ_ACTIVE_INST_VALU over
// SQ_BUSY_CU_CYCLES).  A tile's fixed work is a quarter of its instructions, the
// candidates' culling half (8 slices of 2048^2 through 16M particles: about 80
// pairs kept and 80 covered of 2000 candidates a 16x16 tile).  Against one point a
// lane at 7 waves, one list a workgroup, every row streamed whole and no cover
// form: a 250 x 180 slice through 60k 205 -> 50 us, 4 slices of 1024^2 through 1M
// 0.70 -> 0.55 ms, through 4M of one h 6.9 -> 4.2; 8 slices of 2048^2 through 16M 3.34
// -> 3.40 (exact search 2.85 -> 2.79), and with the h of a neighbour search
// 2.53 -> 3.01: as many instructions (1.46e9 against 1.50e9), issued in 81%
// instead of 99% of the cycles.  5 waves a SIMD keep the registers of 4 points a
// lane, 6 without search boxes (8 slices 2.98 ms at 5, 2.79 at 6, 3.13 at 7); with
// them 6 waves spill (3.5 ms against 3.0).
template <int T, bool REF, bool COUNT>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(T == 16 && !REF ? 6 : 5, 8))) void k_smooth3d(
    grid_view g, level_view lv, point_view p, uint32_t tiles_x, double* __restrict__ acc,
    unsigned long long* __restrict__ cnt) {
  static_assert(!(REF && COUNT), "evaluations are counted with the exact search");
  constexpr int NP = T * T, PPT = NP / 64;
  static_assert(NP <= kBlock && kBlock == 64 * kWaves3, "one point per thread at most");
  __shared__ smem3<T, REF> sm;
  const int t = threadIdx.x;
  const int lane = t & 63, wave = t >> 6;
  const uint32_t tx = blockIdx.x % tiles_x, ty = blockIdx.x / tiles_x;

  // ---- thread t: point t, its search box (reference mode)
  float4 q = make_float4(0.f, 0.f, 0.f, 0.f);
  // a point with an infinite or NaN coordinate is out of every particle's
  // reach: it has no part in the tile's box, plane and search boxes, which
  // would lose the other points their particles
  bool pv = false, on = false;
  int lo[3] = {0, 0, 0}, hi[3] = {-1, -1, -1};
  float minr = INFINITY;  // the search radius (the smallest of the tile's is wanted)
  if (t < NP) {
    const uint32_t px = tx * T + uint32_t(t % T), py = ty * T + uint32_t(t / T);
    const uint32_t pid = py * p.lnx + px;
    pv = px < p.lnx && py < p.lny && pid < p.n;
    if (pv) q = p.pts[pid];
    on = pv && isfinite(q.x) && isfinite(q.y) && isfinite(q.z);
    sm.pt[t] = make_float4(q.x, q.y, q.z, on ? 1.0f : 0.0f);
  }
  const float qc[3] = {q.x, q.y, q.z};
  if (REF && on) {
    int32_t c[3];
    for (int a = 0; a < 3; ++a) c[a] = cell_of(qc[a], 0.0f, g.minc[a], g.cs[a]);
    const uint64_t nx = uint64_t(int64_t(g.nc[0])), ny = uint64_t(int64_t(g.nc[1]));
    const uint64_t key = uint64_t(int64_t(c[0])) + uint64_t(int64_t(c[1])) * nx +
                         uint64_t(int64_t(c[2])) * nx * ny;
    float R = g.max_h;
    if (key < uint64_t(g.ncells)) {
#pragma clang fp contract(off)
      R = fminf(__uint_as_float(g.maxh_bits[key]) + g.cell_radius, g.max_h);
    }
    for (int a = 0; a < 3; ++a) {
      lo[a] = cell_of(qc[a], -R, g.minc[a], g.cs[a]);
      hi[a] = cell_of(qc[a], R, g.minc[a], g.cs[a]);
    }
    minr = R;
  }
  if constexpr (REF) {
    if (t < NP) {
      // the box clamped to the cells a list entry can carry (0..65535 in x,
      // y), as first cell and width; an empty one fails every cell (a grid
      // has no cell (65535, 65535))
      uint4 b = make_uint4(0xffffu, 0xffffu, 0u, 0u);
      const int x0 = max(lo[0], 0), x1 = min(hi[0], 65535);
      const int y0 = max(lo[1], 0), y1 = min(hi[1], 65535);
      const int z0 = max(lo[2], 0), z1 = min(hi[2], INT32_MAX - 1);
      if (on && x0 <= x1 && y0 <= y1 && z0 <= z1)
        b = make_uint4(uint32_t(x0) | uint32_t(x1 - x0) << 16,
                       uint32_t(y0) | uint32_t(y1 - y0) << 16, uint32_t(z0), uint32_t(z1 - z0));
      sm.box[t] = b;
    }
  }
  if (t == 0) sm.covered = 0;
  if (lane < 16) sm.poly[wave][lane] = 0.0;

  // ---- tile reductions: bounding box; union and intersection of the boxes
  {
    const bool some = wave * 64 < NP;
    for (int a = 0; a < 3; ++a) {
      const float f0 = some ? wave_minf(on ? qc[a] : INFINITY) : INFINITY;
      const float f1 = some ? wave_maxf(on ? qc[a] : -INFINITY) : -INFINITY;
      if (lane == 0) {
        sm.redf[wave][a] = f0;
        sm.redf[wave][3 + a] = f1;
      }
      if constexpr (REF) {
        const int i0 = some ? wave_mini(on ? lo[a] : INT32_MAX) : INT32_MAX;  // union
        const int i1 = some ? wave_maxi(on ? hi[a] : INT32_MIN) : INT32_MIN;
        const int i2 = some ? wave_maxi(on ? lo[a] : INT32_MIN) : INT32_MIN;  // intersection
        const int i3 = some ? wave_mini(on ? hi[a] : INT32_MAX) : INT32_MAX;
        if (lane == 0) {
          sm.redi[wave][a] = i0;
          sm.redi[wave][3 + a] = i1;
          sm.redi[wave][6 + a] = i2;
          sm.redi[wave][9 + a] = i3;
        }
      }
    }
    if constexpr (REF) {
      const float r = some ? wave_minf(minr) : INFINITY;
      if (lane == 0) sm.minr[wave] = r;
    }
    const uint64_t any = __ballot(on);
    if (lane == 0) sm.redi[wave][12] = any ? 1 : 0;
  }
  __syncthreads();
  float bmin[3], bmax[3];
  int ulo[3], uhi[3], ilo[3], ihi[3];
  int any = 0;
  for (int w = 0; w < kWaves3; ++w) any |= sm.redi[w][12];
  for (int a = 0; a < 3; ++a) {
    bmin[a] = INFINITY;
    bmax[a] = -INFINITY;
    ulo[a] = ihi[a] = INT32_MAX;
    uhi[a] = ilo[a] = INT32_MIN;
    for (int w = 0; w < kWaves3; ++w) {
      bmin[a] = fminf(bmin[a], sm.redf[w][a]);
      bmax[a] = fmaxf(bmax[a], sm.redf[w][3 + a]);
      if constexpr (REF) {
        ulo[a] = min(ulo[a], sm.redi[w][a]);
        uhi[a] = max(uhi[a], sm.redi[w][3 + a]);
        ilo[a] = max(ilo[a], sm.redi[w][6 + a]);
        ihi[a] = min(ihi[a], sm.redi[w][9 + a]);
      }
    }
    // the boxes are the workgroup's: scalar registers, not vector ones
    bmin[a] = __int_as_float(uniform(__float_as_int(bmin[a])));
    bmax[a] = __int_as_float(uniform(__float_as_int(bmax[a])));
    ulo[a] = uniform(ulo[a]);
    uhi[a] = uniform(uhi[a]);
    ilo[a] = uniform(ilo[a]);
    ihi[a] = uniform(ihi[a]);
  }
  if (!uniform(any)) return;
  float tc[3], hd2 = 0.0f;  // centre and squared half-diagonal
  for (int a = 0; a < 3; ++a) {
    tc[a] = 0.5f * (bmin[a] + bmax[a]);
    const float hd = 0.5f * (bmax[a] - bmin[a]);
    hd2 = fmaf(hd, hd, hd2);
  }
  const float hd = sqrtf(hd2);
  // the size of the coordinates, for rounding margins
  const float at =
      fmaxf(fmaxf(fabsf(g.minc[0]), fabsf(g.minc[1])), fabsf(g.minc[2])) +
      fmaxf(fmaxf(fabsf(tc[0]), fabsf(tc[1])), fabsf(tc[2]));

  // A particle whose h is below every point's search radius R is in the box of
  // every point that its support covers, since the cell arithmetic is
  // monotone (|x - x_p| < h <= R - margin on every axis; the margin covers the
  // rounding of x_p -/+ R and of the support test): no box test, and its cell
  // is not read.
  float unmask_ih2 = INFINITY;
  if constexpr (REF) {
    float r = INFINITY;
    for (int w = 0; w < kWaves3; ++w) r = fminf(r, sm.minr[w]);
    r = __int_as_float(uniform(__float_as_int(r)));
    float pmax = 0.0f;
    for (int a = 0; a < 3; ++a) pmax = fmaxf(pmax, fmaxf(fabsf(bmin[a]), fabsf(bmax[a])));
    const float rs = 0.99999f * r - 1e-6f * (pmax + r);
    if (rs > 0.0f && rs < INFINITY) unmask_ih2 = 1.0f / (rs * rs);
  }

  // ---- the tile's plane: the normal of three of its corners (0 without
  // one), and the points' extent along it.  Any points are allowed, so the
  // extent is reduced over them all.
  float n[3] = {0.f, 0.f, 0.f};
  {
    const float4 a = sm.pt[0], b = sm.pt[T - 1], c = sm.pt[NP - T];
    const float u[3] = {b.x - a.x, b.y - a.y, b.z - a.z}, v[3] = {c.x - a.x, c.y - a.y, c.z - a.z};
    const float m[3] = {u[1] * v[2] - u[2] * v[1], u[2] * v[0] - u[0] * v[2],
                        u[0] * v[1] - u[1] * v[0]};
    const float l2 = m[0] * m[0] + m[1] * m[1] + m[2] * m[2];
    if (a.w != 0.0f && b.w != 0.0f && c.w != 0.0f && l2 > 1e-30f && l2 < 1e30f) {
      const float il = 1.0f / sqrtf(l2);
      for (int k = 0; k < 3; ++k) n[k] = m[k] * il;
    }
    for (int k = 0; k < 3; ++k) n[k] = __int_as_float(uniform(__float_as_int(n[k])));
    const float d = n[0] * (q.x - tc[0]) + n[1] * (q.y - tc[1]) + n[2] * (q.z - tc[2]);
    const float d0 = wave_minf(on ? d : INFINITY), d1 = wave_maxf(on ? d : -INFINITY);
    if (lane == 0) {
      sm.redf[wave][6] = d0;
      sm.redf[wave][7] = d1;
    }
  }

  double a64[PPT];
#pragma unroll
  for (int k = 0; k < PPT; ++k) a64[k] = 0.0;
  auto& L = sm.L[wave];
  int ns = 0, nm = 0, nc = 0;
  // full entries: pairs of the wave's list and every point
  auto eval_full = [&]() {
    const int cnt_ = uniform(ns), n4 = (cnt_ + 3) & ~3;
    if (lane < n4 - cnt_) {
      L.S[cnt_ + lane] = make_float4(0.f, 0.f, 0.f, 0.f);
      L.w[cnt_ + lane] = 0.0f;
    }
    wave_sync();
    float ex[PPT], ey[PPT], ez[PPT];
#pragma unroll
    for (int k = 0; k < PPT; ++k) {
      const float4 e = sm.pt[lane + 64 * k];
      ex[k] = e.x;
      ey[k] = e.y;
      ez[k] = e.z;
    }
    for (int j0 = 0; j0 < n4; j0 += 32) {
      const int jn = min(32, n4 - j0);
      float a[PPT];
#pragma unroll
      for (int k = 0; k < PPT; ++k) a[k] = 0.0f;
      for (int j = 0; j < jn; j += 4) {
        const float4 w4 = *reinterpret_cast<const float4*>(&L.w[j0 + j]);
        const float ww[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float4 e = L.S[j0 + j + u];
#pragma unroll
          for (int k = 0; k < PPT; ++k) {
            const float dx = e.x - ex[k], dy = e.y - ey[k], dz = e.z - ez[k];
            const float r2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
            const float s = fmaxf(fmaf(-r2, e.w, 1.0f), 0.0f);
            if constexpr (COUNT)
              a[k] += (s > 0.0f && ww[u] != 0.0f) ? 1.0f : 0.0f;
            else
              a[k] = fmaf(ww[u], s * s, a[k]);
          }
        }
      }
#pragma unroll
      for (int k = 0; k < PPT; ++k) a64[k] += double(a[k]);
    }
    wave_sync();
    ns = 0;
  };
  // masked entries: each point tests the entry's cell against its own box, as
  // unsigned(c - c0) <= width per axis
  auto eval_masked = [&]() {
    if constexpr (REF) {
      const int cnt_ = uniform(nm);
      wave_sync();
      float ex[PPT], ey[PPT], ez[PPT];
      uint4 bx[PPT];
#pragma unroll
      for (int k = 0; k < PPT; ++k) {
        const float4 e = sm.pt[lane + 64 * k];
        ex[k] = e.x;
        ey[k] = e.y;
        ez[k] = e.z;
        bx[k] = sm.box[lane + 64 * k];
      }
      for (int j0 = 0; j0 < cnt_; j0 += 32) {
        const int jn = min(32, cnt_ - j0);
        float a[PPT];
#pragma unroll
        for (int k = 0; k < PPT; ++k) a[k] = 0.0f;
        for (int j = 0; j < jn; ++j) {
          const float4 e = L.S[kPool3 - 1 - (j0 + j)];
          const float w = L.w[kPool3 - 1 - (j0 + j)];
          const int2 c = L.M[j0 + j];
          const uint32_t cx = uint32_t(uniform(c.x)) & 0xffffu, cy = uint32_t(uniform(c.x)) >> 16;
          const uint32_t cz = uint32_t(uniform(c.y));
#pragma unroll
          for (int k = 0; k < PPT; ++k) {
            const bool in = cx - (bx[k].x & 0xffffu) <= bx[k].x >> 16 &&
                            cy - (bx[k].y & 0xffffu) <= bx[k].y >> 16 && cz - bx[k].z <= bx[k].w;
            const float dx = e.x - ex[k], dy = e.y - ey[k], dz = e.z - ez[k];
            const float r2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
            const float s = fmaxf(fmaf(-r2, e.w, 1.0f), 0.0f);
            a[k] = fmaf(in ? w : 0.0f, s * s, a[k]);
          }
        }
#pragma unroll
        for (int k = 0; k < PPT; ++k) a64[k] += double(a[k]);
      }
      wave_sync();
    }
    nm = 0;
  };
  // cover entries, one per lane: with v = (1, u, |u|^2), u relative to the
  // tile centre, s = f . v, f = (1 - |x|^2/h^2, 2 x/h^2, -1/h^2), and w s^2 =
  // sum w f_i f_j v_i v_j.  The 15 products (in FP64: their FP32 rounding would
  // show where s is small) are summed over the wave, each step halving the
  // sums a lane holds: lane l ends with number l / 4.
  auto eval_cover = [&]() {
    if constexpr (!COUNT) {
      const int m = min(uniform(nc), 64);
      wave_sync();
      double x[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) x[k] = 0.0;
      if (lane < m) {
        const uint32_t si = L.C[nc - m + lane];
        const float4 e = lv.pos[si];
        const double w = double(lv.w[si]), ih2 = double(e.w);
        const double ux = double(e.x) - double(tc[0]), uy = double(e.y) - double(tc[1]),
                     uz = double(e.z) - double(tc[2]);
        const double f[5] = {1.0 - (ux * ux + uy * uy + uz * uz) * ih2, 2.0 * ih2 * ux,
                             2.0 * ih2 * uy, 2.0 * ih2 * uz, -ih2};
        int k = 0;
#pragma unroll
        for (int i = 0; i < 5; ++i) {
          const double wf = w * f[i];
#pragma unroll
          for (int j = i; j < 5; ++j, ++k) x[k] = wf * f[j];
        }
      }
#pragma unroll
      for (int half = 8, o = 32; half >= 1; half >>= 1, o >>= 1) {
        const bool up = (lane & o) != 0;
#pragma unroll
        for (int k = 0; k < half; ++k) {
          const double mine = up ? x[half + k] : x[k], theirs = up ? x[k] : x[half + k];
          x[k] = mine + __shfl_xor(theirs, o, 64);
        }
      }
      x[0] += __shfl_xor(x[0], 2, 64);
      x[0] += __shfl_xor(x[0], 1, 64);
      if ((lane & 3) == 0) sm.poly[wave][lane >> 2] += x[0];
      if (lane == 0) sm.covered = 1;
      wave_sync();
      nc -= m;
    }
  };

  const float sup2 = 1.00002f;  // support 1 h, slack for rounding

  // ---- the tile's key rows, level by level
  if (wave == 0) {
    uint32_t rows = 0;
    if (lane < kLevels3) {
      const int l = lane;
      int f0[3] = {0, 0, 0}, f1[3] = {-1, -1, -1};
      int mode = 0;
      float R = 0.0f;
      if (lv.meta[l + 1] != lv.meta[l]) {
        // every particle whose support reaches a point of the tile lies within
        // the level's largest h of the tile box; the margin covers rounding
        R = ldexpf(g.max_h, l - (kLevels3 - 1));
        const float c = lv.cs[l];
        for (int a = 0; a < 3; ++a) {
          const float m = R + 1e-5f * (fabsf(bmin[a]) + fabsf(bmax[a]) + R + fabsf(g.minc[a]));
          f0[a] = int(fine_of(bmin[a] - m, g.minc[a], c, lv.bits.fmax[a]));
          f1[a] = int(fine_of(bmax[a] + m, g.minc[a], c, lv.bits.fmax[a]));
        }
        const uint32_t ny = uint32_t(f1[1] - f0[1] + 1), nz = uint32_t(f1[2] - f0[2] + 1);
        if (ny <= kRowCap3 && nz <= kRowCap3 && ny * nz <= kRowCap3) {
          mode = 0;
          rows = ny * nz;
        } else if (nz <= kRowCap3) {
          mode = 1;  // one range per z plane over rows f0y..f1y
          rows = nz;
        } else {
          mode = 2;  // one range over the whole box
          rows = 1;
        }
      }
      for (int a = 0; a < 3; ++a) {
        sm.lv_f0[l][a] = f0[a];
        sm.lv_f1[l][a] = f1[a];
      }
      sm.lv_mode[l] = mode;
      sm.lv_r[l] = R;
      sm.lv_s[l] = lv.meta[l];
      sm.lv_p[l] = lv.poff[l];
      if (l == kLevels3 - 1) {
        sm.lv_s[kLevels3] = lv.meta[kLevels3];
        sm.lv_p[kLevels3] = lv.poff[kLevels3];
      }
    }
    uint32_t incl = rows;
    for (int o = 1; o < 32; o <<= 1) {
      const uint32_t y = __shfl_up(incl, o, 64);
      if (lane >= o) incl += y;
    }
    if (lane < kLevels3) sm.lv_row0[lane + 1] = incl;
    if (lane == 0) sm.lv_row0[0] = 0;
  }
  __syncthreads();
  const uint32_t nrows = uint32_t(uniform(int(sm.lv_row0[kLevels3])));
  float dlo = INFINITY, dhi = -INFINITY;
  for (int w = 0; w < kWaves3; ++w) {
    dlo = fminf(dlo, sm.redf[w][6]);
    dhi = fmaxf(dhi, sm.redf[w][7]);
  }
  dlo = __int_as_float(uniform(__float_as_int(dlo)));
  dhi = __int_as_float(uniform(__float_as_int(dhi)));

  for (uint32_t rbase = 0; rbase < nrows; rbase += kBlock) {
    const uint32_t r = rbase + uint32_t(t);
    uint32_t rb = 0, rn = 0;
    if (r < nrows) {
      int l = 0;
      for (int step = 16; step > 0; step >>= 1)  // the last level with row0 <= r
        if (l + step <= kLevels3 - 1 && sm.lv_row0[l + step] <= r) l += step;
      const uint32_t k = r - sm.lv_row0[l];
      const int mode = sm.lv_mode[l];
      const int* f0 = sm.lv_f0[l];
      const int* f1 = sm.lv_f1[l];
      int x0 = f0[0], x1 = f1[0], y0 = f0[1], y1 = f1[1], z0 = f0[2], z1 = f1[2];
      if (mode == 0) {
        const uint32_t ny = uint32_t(f1[1] - f0[1] + 1);
        y0 = y1 = f0[1] + int(k % ny);
        z0 = z1 = f0[2] + int(k / ny);
        // the row's cells that the level's largest h can reach: of the tile
        // box, and of the points' extent along the plane's normal.  A fine
        // cell's particles lie inside it up to a few ulps of the
        // coordinates; the outermost cells also hold what was clamped.
        if (y0 > 0 && y0 < int(lv.bits.fmax[1]) && z0 > 0 && z0 < int(lv.bits.fmax[2])) {
          const float c = lv.cs[l];
          const float mg = 1e-3f * c + 5e-7f * at + 1e-5f * hd;
          const float R = sm.lv_r[l] * 1.00002f + mg;
          const float ylo = fmaf(float(y0), c, g.minc[1]) - mg, yhi = ylo + c + 2.0f * mg;
          const float zlo = fmaf(float(z0), c, g.minc[2]) - mg, zhi = zlo + c + 2.0f * mg;
          const float dy = fmaxf(fmaxf(ylo - bmax[1], bmin[1] - yhi), 0.0f);
          const float dz = fmaxf(fmaxf(zlo - bmax[2], bmin[2] - zhi), 0.0f);
          const float rem = fmaf(-dz, dz, fmaf(-dy, dy, R * R));
          float xa = 0.0f, xb = -1.0f;  // the reachable range relative to the tile centre
          if (rem >= 0.0f) {
            const float rx = sqrtf(rem) + mg;
            xa = bmin[0] - tc[0] - rx;
            xb = bmax[0] - tc[0] + rx;
            // dlo - R <= n . (x - tc) <= dhi + R over the row's y and z
            const float hy = 0.5f * (yhi - ylo), hz = 0.5f * (zhi - zlo);
            const float s0 = n[1] * (ylo + hy - tc[1]) + n[2] * (zlo + hz - tc[2]);
            const float sl = fabsf(n[1]) * hy + fabsf(n[2]) * hz + mg;
            const float u0 = dlo - R - s0 - sl, u1 = dhi + R - s0 + sl;
            if (fabsf(n[0]) > 1e-3f) {
              const float i0 = u0 / n[0], i1 = u1 / n[0];
              xa = fmaxf(xa, fminf(i0, i1) - mg);
              xb = fminf(xb, fmaxf(i0, i1) + mg);
            } else {
              const float sx = fabsf(n[0]) * fmaxf(fabsf(xa), fabsf(xb));
              if (u0 > sx || u1 < -sx) xb = xa - 1.0f;
            }
          }
          if (xa <= xb) {
            x0 = max(x0, int(fine_of(tc[0] + xa - mg, g.minc[0], c, lv.bits.fmax[0])));
            x1 = min(x1, int(fine_of(tc[0] + xb + mg, g.minc[0], c, lv.bits.fmax[0])));
          } else {
            x1 = x0 - 1;
          }
        }
      } else if (mode == 1) {
        z0 = z1 = f0[2] + int(k);
      }
      if (x0 <= x1) {
        const auto klo = fine_key(lv.bits, l, uint32_t(x0), uint32_t(y0), uint32_t(z0));
        const auto khi = fine_key(lv.bits, l, uint32_t(x1), uint32_t(y1), uint32_t(z1));
        // the keys of planes z0 .. z1 from the plane directory (a plane
        // beyond the level's last holds no particle)
        const uint32_t planes = sm.lv_p[l + 1] - sm.lv_p[l] - 1;
        const uint32_t za = min(uint32_t(z0), planes - 1), zb = min(uint32_t(z1), planes - 1);
        const uint32_t s_ = lv.pdir[sm.lv_p[l] + za];
        const uint32_t e_ = lv.pdir[sm.lv_p[l] + zb + 1];
        const uint32_t a_ = lower_bound_u64(lv.key, s_, e_, klo);
        rb = a_;
        rn = gallop_lower_bound_u64(lv.key, a_, e_, khi + 1ull) - a_;
      }
    }
    // the rows that hold particles, packed (most of them are trimmed away)
    const uint64_t some = __ballot(rn != 0u);
    if (lane == 0) sm.hits[wave] = uint32_t(__popcll(some));
    uint32_t tot;
    const uint32_t roff = block_scan_excl(rn, &tot, sm.scan_ws);
    uint32_t hit = prefix_count(some), hits = 0;
    for (int w = 0; w < kWaves3; ++w) {
      if (w < wave) hit += sm.hits[w];
      hits += sm.hits[w];
    }
    if (rn) {
      sm.row_b[hit] = rb - roff;
      sm.row_off[hit] = roff;
    }
    __syncthreads();
    tot = uint32_t(uniform(int(tot)));
    hits = uint32_t(uniform(int(hits)));
    const uint32_t top = hits > 1u ? 1u << (31 - __clz(int(hits - 1u))) : 0u;
    // the rows' particles, 64 at a time, dealt to the waves in turn; after
    // the last of them the wave's lists are evaluated whatever their size
    const bool last = rbase + kBlock >= nrows;
    for (uint32_t v0 = uint32_t(wave) * 64u;; v0 += kBlock) {
      const bool done = v0 >= tot;
      if (done && !last) break;
      const uint32_t v = v0 + uint32_t(lane);
      bool keep = false, full = false, cover = false;
      float4 e = make_float4(0.f, 0.f, 0.f, 0.f);
      float w = 0.0f;
      int2 cinf = make_int2(0, 0);
      uint32_t sidx = 0;
      if (v < tot) {
        // the last row whose offset is <= v
        uint32_t l = 0;
        for (uint32_t step = top; step > 0; step >>= 1) {
          const uint32_t k = l + step;
          if (k < hits && sm.row_off[k] <= v) l = k;
        }
        sidx = sm.row_b[l] + v;
        e = lv.pos[sidx];  // (x, y, z, 1/h^2)
        const float pc[3] = {e.x, e.y, e.z};
        float d2 = 0.0f, nd = 0.0f;
        for (int a = 0; a < 3; ++a) {
          const float d = fmaxf(fmaxf(bmin[a] - pc[a], pc[a] - bmax[a]), 0.0f);
          d2 = fmaf(d, d, d2);
          nd = fmaf(n[a], pc[a] - tc[a], nd);
        }
        // the support sphere against the box and against the points' extent
        // along the normal
        const float gap = fmaxf(fmaxf(dlo - nd, nd - dhi), 0.0f) * 0.99999f - 1e-5f * hd;
        keep = d2 * e.w < sup2 && (gap <= 0.0f || gap * gap * e.w < sup2);
        if (keep) {
          w = lv.w[sidx];
          keep = w != 0.0f;
        }
        full = keep;
        if (REF && keep && e.w < unmask_ih2) {
          // the reference sums a particle only when its cell is in the
          // point's search box: none (drop), every (full) or some (masked)
          cinf = lv.cell[sidx];
          const int cc[3] = {cinf.x & 0xffff, int(uint32_t(cinf.x) >> 16), cinf.y};
          bool inu = true, ini = true;
          for (int a = 0; a < 3; ++a) {
            inu = inu && cc[a] >= ulo[a] && cc[a] <= uhi[a];
            ini = ini && cc[a] >= ilo[a] && cc[a] <= ihi[a];
          }
          keep = inu;
          full = inu && ini;
        }
        if constexpr (!COUNT) {
          if (full) {
            float m2 = 0.0f;  // to the box's farthest corner
            for (int a = 0; a < 3; ++a) {
              const float m = fmaxf(pc[a] - bmin[a], bmax[a] - pc[a]);
              m2 = fmaf(m, m, m2);
            }
            cover = m2 * e.w < 0.9999f;
          }
        }
      }
      const uint64_t bc = COUNT ? 0ull : __ballot(cover);
      const uint64_t bs = __ballot(full && !cover);
      const uint64_t bm = __ballot(keep && !full);
      if constexpr (!COUNT)
        if (cover) L.C[nc + int(prefix_count(bc))] = sidx;
      if (full && !cover) {
        const int pos = ns + int(prefix_count(bs));
        L.S[pos] = e;
        L.w[pos] = w;
      }
      if (REF && keep && !full) {
        const int pos = nm + int(prefix_count(bm));
        L.S[kPool3 - 1 - pos] = e;
        L.w[kPool3 - 1 - pos] = w;
        L.M[pos] = cinf;
      }
      if constexpr (!COUNT) nc += __popcll(bc);
      ns += __popcll(bs);
      nm += __popcll(bm);
      const int lim = done ? 1 : kFlush3;
      if constexpr (!COUNT)
        if (nc >= (done ? 1 : 64)) eval_cover();
      if (ns >= lim) eval_full();
      if (nm >= lim) eval_masked();
      if (done) break;
    }
    __syncthreads();  // the row table is rewritten by the next chunk
  }

  // ---- the waves' sums, in wave order
  __syncthreads();
#pragma unroll
  for (int k = 0; k < PPT; ++k) sm.sum[wave][lane + 64 * k] = a64[k];
  __syncthreads();
  if (!pv) return;
  const uint32_t pid = (ty * T + uint32_t(t / T)) * p.lnx + tx * T + uint32_t(t % T);
  double v = sm.sum[0][t];
  for (int w = 1; w < kWaves3; ++w) v += sm.sum[w][t];
  if constexpr (COUNT) {
    cnt[pid] += static_cast<unsigned long long>(v);
  } else {
    if (sm.covered && on) {
      const double x = double(q.x) - double(tc[0]), y = double(q.y) - double(tc[1]),
                   z = double(q.z) - double(tc[2]);
      const double b[5] = {1.0, x, y, z, x * x + y * y + z * z};
      int k = 0;
#pragma unroll
      for (int i = 0; i < 5; ++i)
#pragma unroll
        for (int j = i; j < 5; ++j, ++k) {
          double c = sm.poly[0][k];
          for (int w = 1; w < kWaves3; ++w) c += sm.poly[w][k];
          v = fma(c * (i == j ? 1.0 : 2.0), b[i] * b[j], v);
        }
    }
    acc[pid] += v;
  }
}

// ---- level index build, from the particles in input order

// grid3d_get_cell_indices of a particle (particle_grid.cl) as the grid build
// computes it; false when the particle lies outside the grid
__device__ inline bool cell_index_3d(const float4& q, const grid_params& g, int32_t idx[3]) {
#pragma clang fp contract(off)
  const float c[3] = {q.x, q.y, q.z};
  bool ok = true;
  for (int a = 0; a < 3; ++a) {
    const float d = c[a] - g.minc[a];
    idx[a] = floor_to_int(d / g.cs[a]);
    ok = ok && idx[a] >= 0 && idx[a] < g.nc[a];
  }
  return ok;
}

__device__ inline unsigned long long particle_key(const float4& q, float h, float max_h,
                                                  const grid_params& g, const level_view& lv,
                                                  const float* scs) {
  const int l = level_of(h, max_h, lv.bits.lmin);
  const float cs = scs[l];
  return fine_key(lv.bits, l, fine_of(q.x, g.minc[0], cs, lv.bits.fmax[0]),
                  fine_of(q.y, g.minc[1], cs, lv.bits.fmax[1]),
                  fine_of(q.z, g.minc[2], cs, lv.bits.fmax[2]));
}

// particles i0 .. i1 - 1: the reference cell's max h, the particle's fine key
// (low and high words; the low one alone in hi when the key has no more than 32
// bits), and a 32-byte record (x, y, z, h | w, cell xy, cell z, 0) in input
// order, so that the sorted gather reads one line per particle instead of one
// from p4 and one from h.  Bound by memory (60 bytes a particle): 16M particles
// 471 us, 867 with the levels counted here on a few common words and the
// maxima read past the caches.
__global__ __launch_bounds__(kBlock) void k_vol_keys(const float4* __restrict__ p4,
                                                      const float* __restrict__ hsml, uint32_t i0,
                                                      uint32_t i1, grid_params g, float max_h,
                                                      level_view lv, float4* __restrict__ rec,
                                                      uint32_t* __restrict__ lo,
                                                      uint32_t* __restrict__ hi,
                                                      uint32_t* __restrict__ maxh_bits,
                                                      uint32_t* __restrict__ err) {
  __shared__ float scs[kLevels3];
  __shared__ float4 srec[2 * kBlock];
  __shared__ unsigned long long slots[kMaxSlots];
  const int t = threadIdx.x;
  if (t == 0) {
#pragma unroll
    for (int l = 0; l < kLevels3; ++l) scs[l] = lv.cs[l];
  }
  __syncthreads();
  const uint32_t nx = uint32_t(g.nc[0]), nxy = nx * uint32_t(g.nc[1]);
  const uint32_t base = i0 + blockIdx.x * kBlock, i = base + uint32_t(t);
  bool ok = false;
  uint32_t cell = 0, hb = 0;
  if (i < i1) {
    const float4 q = p4[i];
    const float h = hsml[i];
    int32_t c[3];
    ok = cell_index_3d(q, g, c);
    if (ok) {
      cell = uint32_t(c[0]) + uint32_t(c[1]) * nx + uint32_t(c[2]) * nxy;
      hb = __float_as_uint(h);
    } else {
      atomicAdd(err, 1u);
      c[0] = c[1] = c[2] = 0;
    }
    srec[2 * t] = make_float4(q.x, q.y, q.z, h);
    srec[2 * t + 1] = make_float4(q.w, __uint_as_float(uint32_t(c[0]) | (uint32_t(c[1]) << 16)),
                                  __uint_as_float(uint32_t(c[2])), 0.0f);
    const auto k = particle_key(q, h, max_h, g, lv, scs);
    if (lv.bits.bits > 32) {
      lo[i] = uint32_t(k);
      hi[i] = uint32_t(k >> 32);
    } else {
      hi[i] = uint32_t(k);
    }
  }
  block_raise_max(maxh_bits, cell, hb, ok, slots);  // has a barrier
  // the block's records are contiguous: whole 16-byte words per lane
  const uint32_t m2 = 2u * min(uint32_t(kBlock), i1 - base);
  for (uint32_t k = uint32_t(t); k < m2; k += kBlock) rec[2 * uint64_t(base) + k] = srec[k];
}

// lower_bound_u64 in few rounds of 15 independent loads: a search has nothing
// else to wait for (60k particles: 20 us a launch with dependent loads, 8 now)
__device__ inline uint32_t wide_lower_bound_u64(const unsigned long long* __restrict__ key,
                                                uint32_t a, uint32_t b, unsigned long long k) {
  while (b - a >= 16u) {
    const uint32_t step = (b - a) >> 4;  // a + 15 step < b
    uint32_t below = 0;
#pragma unroll
    for (uint32_t j = 1; j <= 15; ++j) below += key[a + j * step] < k ? 1u : 0u;
    if (below < 15u) b = a + (below + 1) * step;
    if (below) a += below * step + 1;
  }
  uint32_t below = 0;
#pragma unroll
  for (uint32_t j = 0; j < 15; ++j)
    if (a + j < b) below += key[a + j] < k ? 1u : 0u;
  return a + below;
}

// pdir[poff[L] + z]: first index of level L whose fine z is >= z; the last
// entry of a level is its end
__global__ __launch_bounds__(kBlock) void k_lv_planes(level_view lv, uint32_t* __restrict__ pdir) {
  __shared__ uint32_t sp[kLevels3 + 1], ss[kLevels3 + 1];
  if (threadIdx.x == 0) {
#pragma unroll
    for (int l = 0; l <= kLevels3; ++l) {
      sp[l] = lv.poff[l];
      ss[l] = lv.meta[l];
    }
  }
  __syncthreads();
  const uint32_t e = blockIdx.x * kBlock + threadIdx.x;
  if (e >= sp[kLevels3]) return;
  int l = 0;
  while (sp[l + 1] <= e) ++l;  // e < sp[kLevels3] ends the walk
  const uint32_t z = e - sp[l];
  const uint32_t last = sp[l + 1] - sp[l] - 1;
  pdir[e] = z == last ? ss[l + 1]
                      : wide_lower_bound_u64(lv.key, ss[l], ss[l + 1],
                                             fine_key(lv.bits, l, 0u, 0u,
                                                      min(z, lv.bits.fmax[2])));
}

// the level-ordered arrays: key, (x, y, z, 1/h^2), coef = w norm / h^3 and
// the reference cell; and the levels' starts, where the level changes
__global__ __launch_bounds__(kBlock) void k_vol_soa(const float4* __restrict__ rec, uint32_t n,
                                                     grid_params g, float max_h, float norm,
                                                     level_view lv,
                                                     const uint32_t* __restrict__ order,
                                                     unsigned long long* __restrict__ key,
                                                     float4* __restrict__ pos,
                                                     float* __restrict__ w,
                                                     int2* __restrict__ cell,
                                                     uint32_t* __restrict__ start) {
  __shared__ float scs[kLevels3];
  const int t = threadIdx.x;
  if (t == 0) {
#pragma unroll
    for (int l = 0; l < kLevels3; ++l) scs[l] = lv.cs[l];
  }
  __syncthreads();
  const uint32_t j = blockIdx.x * kBlock + uint32_t(t);
  if (j >= n) return;
  const uint32_t i = order[j];
  // the particle before the wave's first one
  float h0 = 0.0f;
  if ((t & 63) == 0 && j > 0) h0 = rec[2 * uint64_t(order[j - 1])].w;
  const float4 r0 = rec[2 * uint64_t(i)];
  const float4 r1 = rec[2 * uint64_t(i) + 1];
  const float4 q = make_float4(r0.x, r0.y, r0.z, r1.x);
  const float h = r0.w;
  const auto k = particle_key(q, h, max_h, g, lv, scs);
  key[j] = k;
  const int l = lv.bits.lmin + int(k >> lv.bits.shift[3]);
  int before = __shfl_up(l, 1, 64);
  if ((t & 63) == 0) before = j > 0 ? level_of(h0, max_h, lv.bits.lmin) : -1;
  for (int m = before + 1; m <= l; ++m) start[m] = j;
  if (j == n - 1)
    for (int m = l + 1; m <= kLevels3; ++m) start[m] = n;
  const float ih2 = 1.0f / (h * h);
  pos[j] = make_float4(q.x, q.y, q.z, ih2);
  w[j] = q.w * (norm * (ih2 / h));
  cell[j] = make_int2(int(__float_as_uint(r1.y)), int(__float_as_uint(r1.z)));
}

}  // namespace

void launch_volumetric_index(const float4* p4, const float* h, uint32_t n, const grid_params& g,
                             float max_h, float norm, const level_view& lv,
                             unsigned long long* key, float4* pos, float* w, int2* cell,
                             uint32_t* meta, uint32_t* pdir, uint32_t* maxh_bits, uint32_t* err,
                             uint32_t* tmp, uint32_t* radix_temp, hipStream_t s) {
  // the sort by the level key: its low word, if it has two, then its high
  uint32_t* hi_out = tmp + 8 * uint64_t(n);
  uint32_t* idx = hi_out + n;
  const int bits = std::max(lv.bits.bits, 1);
  const radix_chain c = plan_radix_chain(hi_out, idx, n, bits > 32 ? 32 : 0,
                                         bits > 32 ? bits - 32 : bits, radix_temp);
  launch_zero({radix_chain_zero(c), {meta, kLvMetaWords}, {maxh_bits, g.ncells()}, {err, 1}}, s);
  if (n) {
    float4* rec = reinterpret_cast<float4*>(tmp);
    const dim3 grid{(n + kBlock - 1) / kBlock}, block{kBlock};
    for_ranges(n, [&](uint32_t i0, uint32_t i1) {
      hipLaunchKernelGGL(k_vol_keys, dim3((i1 - i0 + kBlock - 1) / kBlock), block, 0, s, p4, h, i0,
                         i1, g, max_h, lv, rec, c.a[c.in], c.b[c.in], maxh_bits, err);
      ILC_HIP(hipGetLastError());
    });
    launch_radix_chain(c, true, false, s);
    hipLaunchKernelGGL(k_vol_soa, grid, block, 0, s, rec, n, g, max_h, norm, lv, idx, key, pos, w,
                       cell, meta);
    ILC_HIP(hipGetLastError());
  }
  // the directory searches the sorted keys (lv.key is key, lv.meta is meta)
  const uint32_t nd = lv.poff[kLevels3];
  ILC_REQUIRE(lv.key == key && lv.meta == meta && lv.pdir == pdir, "level index buffers");
  if (nd) {
    hipLaunchKernelGGL(k_lv_planes, dim3((nd + kBlock - 1) / kBlock), dim3(kBlock), 0, s, lv, pdir);
    ILC_HIP(hipGetLastError());
  }
}

// 8 x 8 tiles below this many points.  A larger tile streams its candidates
// for four times the points, but a launch needs tiles enough for the chip and
// a tile wide against h streams what few of its points use.  8 x 8 against
// 16 x 16 tiles (ms, index build included): 60k particles 0.28/0.34 with 40k
// points, 0.29/0.31 with 160k, 0.43/0.32 with 640k; 1M particles 0.82/0.93
// with 320k points, 1.12/0.91 with 1.3M; 16M particles 3.01/3.76 with 640k,
// 3.51/3.29 with 2.6M.
constexpr uint32_t kPointsFor16 = 1u << 19;

void launch_smooth3d(const grid_view& g, const level_view& lv, const point_view& p, int op,
                     double* acc, hipStream_t s, unsigned long long* cnt) {
  if (!p.n) return;
  ILC_REQUIRE(lv.key != nullptr, "the grid is not a volumetric grid");
  ILC_REQUIRE(op == OP_REFERENCE || op == OP_EXACT || op == OP_COUNT, "bad op %d", op);
  ILC_REQUIRE(op == OP_COUNT ? cnt != nullptr : acc != nullptr, "null output");
  const uint32_t side = p.n < kPointsFor16 ? 8 : 16;
  const uint32_t tiles_x = (p.lnx + side - 1) / side;
  const uint64_t tiles = uint64_t(tiles_x) * ((p.lny + side - 1) / side);
  ILC_REQUIRE(tiles < (uint64_t(1) << 31), "too many tiles");
  const dim3 grid{static_cast<uint32_t>(tiles)}, block{kBlock};
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, block, 0, s, g, lv, p, tiles_x, acc, cnt);
  };
  if (op == OP_REFERENCE)
    side == 8 ? go(k_smooth3d<8, true, false>) : go(k_smooth3d<16, true, false>);
  else if (op == OP_EXACT)
    side == 8 ? go(k_smooth3d<8, false, false>) : go(k_smooth3d<16, false, false>);
  else
    side == 8 ? go(k_smooth3d<8, false, true>) : go(k_smooth3d<16, false, true>);
  ILC_HIP(hipGetLastError());
}

}  // namespace ilc
