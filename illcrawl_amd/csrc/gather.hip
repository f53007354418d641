// Per-point projected-kernel gather on gfx950.
//
// Replaces projective_smoothing_grid -> spg_run_reconstruction
// (projective_smoothing_backend_grid.cl:30-56, smoothing_particle_grid.cl:31-127).
//
// One 256-thread workgroup (4 waves of 64) owns a tile of T x T points (16 or
// 8) of the point array seen as an image.  The workgroup
//   1. loads its points and, in reference mode, each point's search box
//      exactly as the reference computes it (cell of the point, radius =
//      min(max_h[cell] + cell_radius, max_h), index box of p -/+ radius, from
//      the unclamped 64-bit key of the reference);
//   2. reduces the tile's bounding box and the union / intersection of the
//      points' index boxes;
//   3. visits the candidate cells 256 at a time, skips every cell whose max h
//      cannot reach the tile, and builds an offset table of the others'
//      particles.  A cell holds its particles by descending h, so a binary
//      search on h finds the prefix that can reach the tile and the rest is
//      never read.
// The waves then stream the chunk's particles, 64 at a time in turn
// (coalesced 16-byte loads).  Each wave
//   4. culls each particle against the tile (support disk vs tile box) and
//      compacts the survivors into its own LDS lists with ballots:
//        far    - (16x16 tiles) the tile lies well inside its support: summed
//                 at 64 nodes and interpolated, see is_far;
//        big    - every point may use it and its support is at least twice
//                 the tile's half-diagonal: stored, like far, as the
//                 coefficients of its kernel argument expanded about the
//                 tile centre;
//        small  - every point may use it, stored by position;
//        masked - reference mode, its cell may be inside some points' index
//                 box and outside others': stored by position and cell;
//   5. when a list is full, evaluates it from LDS (broadcast reads) for every
//      point of the tile (far: every node), FP32 over 32 particles, then into
//      FP64 accumulators.
// At the end of the tile the waves' sums are added, in wave order, and the
// far field is interpolated.
//
// Kernel arithmetic.  With c = coef^0.4, the quartic term coef*s^2.5,
// s = 1 - r^2/h^2, equals (c*s)^2.5, and c*s is affine in the point's
// coordinates u (relative to the tile centre t) and |u|^2:
//   c*s = c(1 - |x-t|^2/h^2) + (2c/h^2)(x-t).u - (c/h^2)|u|^2,
// three FMAs per point for big particles (their expansion stays well
// conditioned: |x-t| <= 1.5 h), then max, sqrt, mul, fma.  Small and masked
// particles use c*s = c - (c/h^2) r^2 directly.
//
// The cell-distance cull of the reference (smoothing_particle_grid.cl:95-100)
// never removes a particle whose support covers the point (a cell's centre
// is within the cell half-diagonal of every particle in it), so it is not
// repeated; particles outside their support contribute exactly 0 in the
// reference and are culled here.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"
#include "pixel.hpp"
#include "wave.hpp"

namespace ilc {

namespace {

// a tile of a sparse grid leaves the row streaming for the cell enumeration
// above this many particles per candidate cell
constexpr uint32_t kDenseRows = 2;
constexpr int kCubicTable = 4096;

// grid3d_get_cell_indices of p + r on one axis, FP32, no FMA.
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
__device__ inline float uniformf(float v) { return __int_as_float(uniform(__float_as_int(v))); }

// Exclusive scan over the NB threads of the workgroup; *total = sum.
// Contains two workgroup barriers.
template <int NB>
__device__ inline uint32_t block_scan_excl(uint32_t v, uint32_t* total, uint32_t* ws) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t incl = wave_scan(v);
  if (lane == 63) ws[wave] = incl;
  __syncthreads();
  uint32_t off = 0, tot = 0;
  for (int w = 0; w < NB / 64; ++w) {
    if (w < wave) off += ws[w];
    tot += ws[w];
  }
  __syncthreads();
  *total = tot;
  return off + incl - v;
}

// (c s)^2.5 for a scaled kernel argument cs = c*s, clamped at the support.
__device__ inline float pow25(float cs) {
  cs = fmaxf(cs, 0.0f);
  return (cs * cs) * __builtin_amdgcn_sqrtf(cs);
}

// The same for an argument known to be positive.
__device__ inline float pow25_pos(float cs) { return (cs * cs) * __builtin_amdgcn_sqrtf(cs); }

// The projected quartic clipped along the line of sight.  The 3-D kernel
// along a line at projected distance r from the particle is proportional to
// (a^2 - z^2)^2 on |z| < a = h s^(1/2), s = 1 - r^2/h^2; its integral over
// the depth range [z0, z1] relative to the particle is the full column's
// times (15/16) (G(u1) - G(u0)), G(u) = u - 2u^3/3 + u^5/5, u = z / a clamped
// to [-1, 1].  With v = c s (the argument of pow25) and t = (z / h) c^(1/2),
// u = t / v^(1/2).  tc: (t0, t1) of the range's two ends.
__device__ inline float clip_pow(float v, float2 tc) {
  v = fmaxf(v, 0.0f);
  const float sv = __builtin_amdgcn_sqrtf(v);
  const float iv = v > 0.0f ? __builtin_amdgcn_rcpf(sv) : 0.0f;
  const float u0 = __builtin_amdgcn_fmed3f(tc.x * iv, -1.0f, 1.0f);
  const float u1 = __builtin_amdgcn_fmed3f(tc.y * iv, -1.0f, 1.0f);
  const float q0 = u0 * u0, q1 = u1 * u1;
  const float g0 = u0 * fmaf(q0, fmaf(q0, 0.2f, -2.0f / 3.0f), 1.0f);
  const float g1 = u1 * fmaf(q1, fmaf(q1, 0.2f, -2.0f / 3.0f), 1.0f);
  return ((v * v) * sv) * ((g1 - g0) * 0.9375f);
}

// Tabulated projected cubic spline on u = r^2/h^2 in [0, 4), linear.
__device__ inline float cubic_shape(float u, const float* tab) {
  const float x = fminf(u * (float(kCubicTable - 1) / 4.0f), float(kCubicTable - 1));
  const int i = min(int(x), kCubicTable - 2);
  const float f = x - float(i);
  const float a = tab[i], b = tab[i + 1];
  return fmaf(f, b - a, a);
}

// Adjoint inputs and outputs.
struct adjoint_io {
  const float* grad;  // dL/d(point value), one per point
  float scale;        // points' value = scale * accumulator
  float norm;         // kernel normalisation K (W = K shape / h^2)
  const float* ftab;  // cubic: F(u) and dF/du on u = r^2/h^2 in [0, 4] (kCubicTable nodes)
  const float* dtab;
  float* gw;          // per sorted particle: dL/dw, dL/dh, dL/dx, dL/dy (atomic adds)
  float* gh;
  float* gx;
  float* gy;
};

// ---- the far field of a tile
//
// Over a tile well inside a particle's support the quartic's s^2.5 is smooth,
// and the sum of all such particles is evaluated at 8 x 8 Chebyshev nodes of
// the tile box instead of at its points, then interpolated once per point (in
// FP64): a particle costs one wave 64 evaluations instead of the tile's 256.
constexpr int kNodes = 8;
// nodes cos((2 i + 1) pi / 16), and the Lagrange weights 1 / prod_{j != i}
// (x_i - x_j) = (-1)^i 16 sin((2 i + 1) pi / 16)
__device__ constexpr double kNodeX[kNodes] = {
    0.98078528040323044913,  0.83146961230254523708,  0.55557023301960222474,
    0.19509032201612826785,  -0.19509032201612826785, -0.55557023301960222474,
    -0.83146961230254523708, -0.98078528040323044913};
__device__ constexpr double kNodeW[kNodes] = {
    16 * 0.19509032201612826785,  -16 * 0.55557023301960222474, 16 * 0.83146961230254523708,
    -16 * 0.98078528040323044913, 16 * 0.98078528040323044913,  -16 * 0.83146961230254523708,
    16 * 0.55557023301960222474,  -16 * 0.19509032201612826785};

// the Lagrange basis of the nodes at u
__device__ inline void node_basis(double u, double* b) {
  double pre = 1.0;
#pragma unroll
  for (int i = 0; i < kNodes; ++i) {
    b[i] = pre * kNodeW[i];
    pre *= u - kNodeX[i];
  }
  double suf = 1.0;
#pragma unroll
  for (int i = kNodes - 1; i >= 0; --i) {
    b[i] *= suf;
    suf *= u - kNodeX[i];
  }
}

// A particle at r from the tile centre is far when a <= (0.4 + 0.22 r / h) (h - r),
// a = sqrt(2) times the tile's larger half-side (the half-diagonal of a square
// one): the interpolation then errs by at most 4e-8 of the particle's value at the
// tile centre and 3.3e-7 of its value at the point itself (the largest over all
// tile shapes, directions and r / h up to 0.999; s^2.5 is singular at the
// support's edge only, h - r and h + r away), below the FP32 rounding of the
// direct form.  The half-diagonal would not do in strip tiles (an image's last
// row or column of tiles), whose nodes lie wider for it: 5.6e-7 and 6.3e-6.  The
// adjoint's s^1.5 meets 4.1e-8 and 1.2e-7 with a slope of 0.16 (its nodes'
// gradients are FP32: up to 2e-7 of the value at the centre more).  Up to 0.999 h, so
// that every argument is positive by far more than its rounding (s >= 7e-4): the
// nodes need no clamp at 0, one of the 6 issue slots of a pair (3 FMAs, clamp,
// square, multiply-add; the square root runs beside them).  Without it, and
// with the tile's reductions on DPP: 32 views of 16M particles 49.6 -> 48.6 ms.
// ih2 = 1 / h^2, r2 = r^2, a2 = a^2.
__device__ inline bool is_far(float r2, float ih2, float a2, float slope = 0.22f) {
  const float x = __builtin_amdgcn_sqrtf(r2 * ih2);  // r / h
  const float lim = fmaf(x, slope, 0.4f) * (1.0f - x);
  return x < 0.999f && a2 * ih2 <= lim * lim;
}

// ---- tiles of the sums (every op but the adjoint)
//
// A workgroup of 4 waves owns a tile of T x T points, and every wave works on
// all of them (T * T / 64 per lane) with its own share of the candidates and
// its own LDS lists: between the workgroup's cell chunks a wave never waits
// for the others, and a list entry read from LDS serves T * T / 64 points per
// lane.  The waves' sums are added once, at the end of the tile.  (With the
// points dealt to the waves and shared lists, every 256 candidates cost two
// workgroup barriers, and a tile of 64 points had one wave: one wave per tile
// takes 1.25 ms for a 512^2 view of 1M particles, four 0.80, eight 0.79, at
// 8x8 points; 6 frames of 160x120 1.12, 0.71, 0.73.)
//
// QUAD: in a 16x16 tile every wave works on one 8x8 quarter, one point a lane,
// with all of the tile's candidates.  Nothing is added up at the end, a lane
// needs 64 registers (8 waves a SIMD, not 5), and a particle smaller than the
// tile costs only the quarters that it reaches; but a candidate is culled four
// times, and wide particles have no nodes.  Taken where quarter_tiles says.
constexpr int kSumW = 4;

// A wave's lists.  It evaluates one when it reaches FLUSH entries; a batch of 64
// candidates lands on a list of at most FLUSH - 1.
template <bool REF, int KERNEL, bool CLIP, bool COUNT, bool QUAD>
struct wave_lists {
  static constexpr int FLUSH = QUAD ? 16 : 32;
  // one list, and two lists sharing an array from its two ends, with room to
  // pad either to a multiple of 4 entries
  static constexpr int CAP = FLUSH - 1 + 64 + 1;
  static constexpr int POOL = 2 * (FLUSH - 1) + 64 + 6;
  static_assert(CAP % 4 == 0 && POOL % 4 == 0, "whole groups of 4 entries");
  static constexpr bool QUARTIC = KERNEL == 0 && !COUNT;
  alignas(16) float4 X[QUARTIC ? POOL : 1];  // expansion form: far from the front, big from the back
  float4 S[REF ? POOL : CAP];  // position form: small from the front, masked from the back
  alignas(16) int M[REF ? CAP : 1];  // masked: packed cell (cx | cy << 16)
  // line-of-sight clip: per entry, the depth range relative to the particle
  // in units of h, times c^(1/2) (see clip_pow)
  float2 Xz[CLIP ? POOL : 1];
  float2 Sz[CLIP ? CAP : 1];
};

// The workgroup's chunk of candidate cells (or of rows of them).
struct cell_table {
  uint32_t b[64 * kSumW];    // first particle
  uint32_t off[64 * kSumW];  // exclusive sum of the particles
  int info[64 * kSumW];      // cells: packed cell cx | cy << 16 (unsigned); rows: base key
  int y[64 * kSumW];         // cells: 1 when in every point's search box; rows: the row's cy
  uint32_t scan_ws[kSumW];
};

// Streams the candidate particles of the cell box [cx0, cx1] x [cy0, cy1] x
// [cz0, cz1] for the tile box (tbx0, tby0, tbx1, tby1): calls batch(have,
// sorted index, packed cell, in_all(cell), done) on the waves, up to 64
// candidates at a time, and once per wave at the end with done set and no
// candidate.  The candidates are dealt to the waves in turn, or every wave takes
// all of them (DEAL_ALL).  Every thread of the workgroup takes part.
enum deal_kind { DEAL_64, DEAL_EVEN, DEAL_ALL };
template <bool REF, deal_kind DEAL, class InAll, class Batch>
__device__ __attribute__((always_inline)) inline void stream_candidates(
    const grid_view& g, int cx0, int cx1, int cy0, int cy1, int cz0, int cz1, float tbx0,
    float tby0, float tbx1, float tby1, float support, InAll&& in_all, cell_table& ct,
    Batch&& batch) {
  // ---- candidates.  The particles of the cells cx0..cx1 of one row (y, z)
  // are contiguous in the sorted order, so the box's particles form nrows *
  // nlays ranges.  Dense grids visit the box's cells NB at a time (x
  // fastest) and skip the cells whose max h cannot reach the tile; sparse
  // grids (well under one particle per cell, e.g. the depth-cut lists of a
  // slab) stream the row ranges and cull per particle.  Both give the same
  // candidates in the same order (rows, cells by x, particles in sorted
  // order).  A sparse grid can still be dense where the tile is (a halo
  // inside a slab): when the first chunk of rows holds more than
  // kDenseRows particles per cell of the box, the tile switches to the cell
  // enumeration, whose max-h skip and prefix search read far fewer.
  constexpr int NB = 64 * kSumW;
  const int t = threadIdx.x;
  const int lane = t & 63, wave = t >> 6;
  const int ncols = cx1 >= cx0 ? cx1 - cx0 + 1 : 0;
  const int nrows = cy1 >= cy0 ? cy1 - cy0 + 1 : 0;
  const int nlays = cz1 >= cz0 ? cz1 - cz0 + 1 : 0;
  // the box lies inside the grid, whose cells have 32-bit keys: 32-bit
  // counts and indices (one layer, as in reference mode, skips a division)
  const uint32_t ncand = uint32_t(ncols) * uint32_t(nrows) * uint32_t(nlays);
  const uint32_t nrowz = ncols > 0 ? uint32_t(nrows) * uint32_t(nlays) : 0u;
  const uint32_t nxny = uint32_t(g.nc[0]) * uint32_t(g.nc[1]);
  const float sup_h2 = support * support * 1.00002f;
  bool rows_mode = g.sparse != 0 && ncand > uint32_t(NB);
  const bool one_layer = nlays == 1;
  uint64_t nitems = rows_mode ? nrowz : ncand;
  for (uint64_t c0 = 0; c0 < nitems; c0 += NB) {
    const bool in_box = c0 + uint64_t(t) < nitems;
    const uint32_t ci = uint32_t(c0) + uint32_t(t);
    uint32_t cb = 0, cn = 0;
    int ccx = 0, ccy = 0, cfull = 0;
    if (rows_mode) {
      if (in_box) {
        const uint32_t lay = one_layer ? 0u : ci / uint32_t(nrows);
        ccy = cy0 + int(ci - lay * uint32_t(nrows));
        const uint32_t kb = uint32_t(ccy) * uint32_t(g.nc[0]) + uint32_t(cz0 + int(lay)) * nxny;
        cb = g.start[kb + uint32_t(cx0)];
        cn = g.start[kb + uint32_t(cx1) + 1] - cb;
        ccx = int(kb);  // stored as the row's base key
      }
    } else if (in_box) {
      const uint32_t rest = ci / uint32_t(ncols);
      const int col_c = int(ci - rest * uint32_t(ncols));
      const uint32_t lay = one_layer ? 0u : rest / uint32_t(nrows);
      ccx = cx0 + col_c;
      ccy = cy0 + int(rest - lay * uint32_t(nrows));
      const int ccz = cz0 + int(lay);
      const uint32_t key = uint32_t(ccx) + uint32_t(ccy) * uint32_t(g.nc[0]) + uint32_t(ccz) * nxny;
      cb = g.start[key];
      const uint32_t ce = g.start[key + 1];
      if (ce > cb) {
        const float mh = __uint_as_float(g.maxh_bits[key]);
        const float lo_x = g.minc[0] + float(ccx) * g.cs[0];
        const float lo_y = g.minc[1] + float(ccy) * g.cs[1];
        // a particle's cell comes from fl((x - min) / w): its coordinate can
        // sit a few ulps of |x| + |min| outside the cell's float edges
        const float mgx = 1e-4f * g.cs[0] + 4e-7f * (fabsf(g.minc[0]) + fabsf(lo_x) + g.cs[0]);
        const float mgy = 1e-4f * g.cs[1] + 4e-7f * (fabsf(g.minc[1]) + fabsf(lo_y) + g.cs[1]);
        const float dx = fmaxf(fmaxf((lo_x - mgx) - tbx1, tbx0 - (lo_x + g.cs[0] + mgx)), 0.0f);
        const float dy = fmaxf(fmaxf((lo_y - mgy) - tby1, tby0 - (lo_y + g.cs[1] + mgy)), 0.0f);
        const float d2c = dx * dx + dy * dy;
        if (d2c < mh * mh * sup_h2) {
          // the cell's particles come by descending h (to the top 16 bits of
          // its pattern): only a prefix can reach the tile.  With h rounded
          // up to its 16-bit bucket the test is monotone along the cell.
          uint32_t lo = 0, hi = ce - cb;
          while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            const float hu = __uint_as_float(__float_as_uint(g.hs[cb + mid]) | 0xffffu);
            if (d2c < hu * hu * sup_h2)
              lo = mid + 1;
            else
              hi = mid;
          }
          cn = lo;
        }
        if constexpr (REF)
          cfull = in_all(ccx, ccy) ? 1 : 0;
      }
    }
    uint32_t tot;
    const uint32_t coff = block_scan_excl<NB>(cn, &tot, ct.scan_ws);
    tot = uint32_t(uniform(int(tot)));
    if (rows_mode && c0 == 0 && uint64_t(tot) > uint64_t(kDenseRows) * ncand) {
      // nothing of this chunk is in LDS yet: start over with the cells
      rows_mode = false;
      nitems = ncand;
      c0 = uint64_t(0) - uint64_t(NB);
      continue;
    }
    ct.b[t] = cb;
    ct.off[t] = coff;
    if (rows_mode) {
      ct.info[t] = ccx;
      ct.y[t] = ccy;
    } else {
      ct.info[t] = int(uint32_t(ccx) | (uint32_t(ccy) << 16));
      ct.y[t] = cfull;
    }
    __syncthreads();
    // the chunk's particles, 64 at a time, dealt to the waves in turn; after
    // the last of them the wave's lists are evaluated whatever their size
    // (here and not behind the loop: one copy of the evaluation code).
    // DEAL_EVEN: a chunk of less than 64 for each wave is dealt evenly, for the sums
    // of 16x16 tiles: a candidate is work for the whole wave, and in sparse
    // tiles (100 candidates) two waves had all the pairs and two had none (16
    // slabs of 4096^2 through 32M particles, gather 13.6 -> 12.1 ms; a cubic
    // 2048^2 view of 1M 13.5 -> 12.7).  With one pair a lane and candidate (8x8
    // tiles) the half-empty culls cost as much (24 views of 200^2 of 1M 3.9 ->
    // 4.06); in the adjoint a candidate is a lane's.
    const bool last_chunk = c0 + NB >= nitems;
    const uint32_t deal =
        DEAL == DEAL_EVEN && tot < uint32_t(NB) ? max(1u, (tot + kSumW - 1) / kSumW) : 64u;
    constexpr uint32_t TURNS = DEAL == DEAL_ALL ? 1 : kSumW;
    for (uint32_t v0 = uint32_t(wave) % TURNS * deal;; v0 += deal * TURNS) {
      const bool done = v0 >= tot;
      if (done && !last_chunk) break;
      const uint32_t v = v0 + uint32_t(lane);
      bool have = false;
      uint32_t sidx = 0;
      int cinf = 0, cf = 0;
      if (v < tot && uint32_t(lane) < deal) {
        // last cell whose offset is <= v (it has a nonzero count)
        int lo = 0;
#pragma unroll
        for (int step = NB / 2; step > 0; step >>= 1)
          if (ct.off[lo + step] <= v) lo += step;
        sidx = ct.b[lo] + (v - ct.off[lo]);
        if constexpr (REF) {
          cinf = ct.info[lo];
          cf = ct.y[lo];
          if (rows_mode) {
            // the particle's cell from its key and the row's base key
            const int px_c = int(g.key[sidx] - uint32_t(cinf));
            const int py_c = cf;
            cinf = int(uint32_t(px_c) | (uint32_t(py_c) << 16));
            cf = in_all(px_c, py_c) ? 1 : 0;
          }
        }
        have = true;
      }
      batch(have, sidx, cinf, cf != 0, done);
      if (done) break;
    }
    __syncthreads();  // the cell table is rewritten by the next chunk
  }
}

template <int T, bool REF, int KERNEL, bool CLIP, bool COUNT, bool QUAD>
struct tile_smem {
  static constexpr int W = kSumW, NB = 64 * W;
  union {
    wave_lists<REF, KERNEL, CLIP, COUNT, QUAD> L[W];
    struct {                      // at the end of the tile: the waves' sums
      double sum[QUAD ? 1 : W][QUAD ? 1 : T * T];
      double node[KERNEL == 0 && !CLIP && !COUNT && !QUAD && T * T > 64 ? W : 1][64];
    };
  };
  int far_used;
  float2 pt[QUAD ? 1 : T * T];          // the tile's points
  uint2 box[REF && !QUAD ? T * T : 1];  // their search boxes: (x0 | xw << 16, y0 | yw << 16)
  float tab[KERNEL == 2 ? kCubicTable : 1];
  cell_table cells;
  float redf[W][5];
  int redi[W][11];
};

// orders this wave's LDS accesses: its lists are written by some lanes and
// read by others
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One tile (tx, ty) of the point image: everything between the point loads
// and the accumulator update.  All threads of the workgroup call it with the
// same arguments.
template <int T, int OP, int KERNEL, bool QUAD>
__device__ __attribute__((always_inline)) inline void sum_tile(
    const grid_view& g, const point_view& p, uint32_t tx, uint32_t ty, double* __restrict__ acc_out,
    unsigned long long* __restrict__ counts, float support,
    tile_smem<T, OP == OP_REFERENCE, KERNEL, OP == OP_CLIP, OP == OP_COUNT, QUAD>& sm,
    float* __restrict__ img_out = nullptr, float img_scale = 1.0f, int fused = 0) {
  constexpr int W = kSumW, NB = 64 * W, NP = T * T, PPT = QUAD ? 1 : NP / 64;
  constexpr bool REF = OP == OP_REFERENCE;
  constexpr bool COUNT = OP == OP_COUNT;
  constexpr bool CLIP = OP == OP_CLIP;
  constexpr bool QUARTIC = KERNEL == 0 && !COUNT;
  // with one point per lane the nodes would save nothing
  constexpr bool FAR = QUARTIC && !CLIP && PPT > 1;
  static_assert(!CLIP || KERNEL == 0, "the line-of-sight clip is the quartic's");
  static_assert(NP % 64 == 0, "whole points per lane");
  static_assert(!QUAD || (T == 16 && W == 4), "a wave for each 8x8 quarter");
  using lists = wave_lists<REF, KERNEL, CLIP, COUNT, QUAD>;
  constexpr int POOL = lists::POOL, FLUSH = lists::FLUSH;

  const int t = threadIdx.x;
  const int lane = t & 63, wave = t >> 6;

  // point pt's column and row in the tile
  auto col_of = [](int pt) { return QUAD ? (pt >> 6 & 1) * 8 + (pt & 7) : pt % T; };
  auto row_of = [](int pt) { return QUAD ? (pt >> 7) * 8 + (pt >> 3 & 7) : pt / T; };
  // QUAD: the lane's point and its search box
  float2 my_pt = make_float2(0.f, 0.f);
  uint2 my_box = make_uint2(0xffffu, 0xffffu);

  // ---- the tile's points (thread t: points t, t + NB, ...), their search
  // boxes, and the tile reductions
  float bminx = INFINITY, bminy = INFINITY, bmaxx = -INFINITY, bmaxy = -INFINITY;
  int ulx = INT32_MAX, uly = INT32_MAX, uhx = INT32_MIN, uhy = INT32_MIN;
  int ilx = INT32_MIN, ily = INT32_MIN, ihx = INT32_MAX, ihy = INT32_MAX;
  int anyz = 0, allz = 1, anyv = 0;
  float minr = INFINITY;  // reference mode: the smallest search radius of the points
#pragma unroll 1
  for (int pt = t; pt < NP; pt += NB) {
    const uint32_t px = tx * T + uint32_t(col_of(pt)), py = ty * T + uint32_t(row_of(pt));
    const uint32_t pid = py * p.lnx + px;
    const bool pv = px < p.lnx && py < p.lny && pid < p.n;
    float4 q = make_float4(0.f, 0.f, 0.f, 0.f);
    if (pv) q = p.gen ? pixel_point(p.pg, px, py) : p.pts[pid];
    uint2 box = make_uint2(0xffffu, 0xffffu);  // no such cell in a grid of < 2^32
    if (pv) {
      anyv = 1;
      bminx = fminf(bminx, q.x);
      bmaxx = fmaxf(bmaxx, q.x);
      bminy = fminf(bminy, q.y);
      bmaxy = fmaxf(bmaxy, q.y);
      if constexpr (REF) {
        // search radius of spg_run_reconstruction (smoothing_particle_grid.cl:54-75)
        const int32_t c0 = cell_of(q.x, 0.0f, g.minc[0], g.cs[0]);
        const int32_t c1 = cell_of(q.y, 0.0f, g.minc[1], g.cs[1]);
        const int32_t c2 = cell_of(q.z, 0.0f, g.minc[2], g.cs[2]);
        const uint64_t nx = uint64_t(int64_t(g.nc[0])), ny = uint64_t(int64_t(g.nc[1]));
        const uint64_t key = uint64_t(int64_t(c0)) + uint64_t(int64_t(c1)) * nx +
                             uint64_t(int64_t(c2)) * nx * ny;
        float R = g.max_h;
        if (key < uint64_t(g.ncells)) {
#pragma clang fp contract(off)
          R = fminf(__uint_as_float(g.maxh_bits[key]) + g.cell_radius, g.max_h);
        }
        minr = fminf(minr, R);
        const int lox = cell_of(q.x, -R, g.minc[0], g.cs[0]);
        const int hix = cell_of(q.x, R, g.minc[0], g.cs[0]);
        const int loy = cell_of(q.y, -R, g.minc[1], g.cs[1]);
        const int hiy = cell_of(q.y, R, g.minc[1], g.cs[1]);
        const int32_t loz = cell_of(q.z, -R, g.minc[2], g.cs[2]);
        const int32_t hiz = cell_of(q.z, R, g.minc[2], g.cs[2]);
        const bool zin = loz <= g.kz0 && g.kz0 <= hiz;
        ilx = max(ilx, lox);
        ihx = min(ihx, hix);
        ily = max(ily, loy);
        ihy = min(ihy, hiy);
        allz &= int(zin);
        if (zin) {
          anyz = 1;
          ulx = min(ulx, lox);
          uhx = max(uhx, hix);
          uly = min(uly, loy);
          uhy = max(uhy, hiy);
          // the box clamped to the cells a list entry can have (0..65535 per
          // axis), as first cell and width
          const int x0 = max(lox, 0), x1 = min(hix, 65535);
          const int y0 = max(loy, 0), y1 = min(hiy, 65535);
          if (x0 <= x1 && y0 <= y1)
            box = make_uint2(uint32_t(x0) | uint32_t(x1 - x0) << 16,
                             uint32_t(y0) | uint32_t(y1 - y0) << 16);
        }
      }
    }
    if constexpr (QUAD) {
      my_pt = make_float2(q.x, q.y);
      my_box = box;
    } else {
      sm.pt[pt] = make_float2(q.x, q.y);
      if constexpr (REF) sm.box[pt] = box;
    }
  }
  // QUAD: the box of the wave's points
  float wbx0, wby0, wbx1, wby1;
  {
    const float v0 = wave_minf(bminx), v1 = wave_minf(bminy), v2 = wave_maxf(bmaxx), v3 = wave_maxf(bmaxy);
    wbx0 = v0;
    wby0 = v1;
    wbx1 = v2;
    wby1 = v3;
    int iv[11] = {0};
    float v4 = INFINITY;
    if constexpr (REF) {
      v4 = wave_minf(minr);
      iv[0] = wave_mini(ulx);
      iv[1] = wave_mini(uly);
      iv[2] = wave_maxi(uhx);
      iv[3] = wave_maxi(uhy);
      iv[4] = wave_maxi(ilx);
      iv[5] = wave_maxi(ily);
      iv[6] = wave_mini(ihx);
      iv[7] = wave_mini(ihy);
      iv[8] = __ballot(anyz) != 0;
      iv[9] = __ballot(!allz) == 0;
    }
    iv[10] = __ballot(anyv) != 0;
    if (lane == 0) {
      sm.redf[wave][0] = v0;
      sm.redf[wave][1] = v1;
      sm.redf[wave][2] = v2;
      sm.redf[wave][3] = v3;
      sm.redf[wave][4] = v4;
      for (int j = 0; j < 11; ++j) sm.redi[wave][j] = iv[j];
    }
  }
  __syncthreads();
  float tbx0 = INFINITY, tby0 = INFINITY, tbx1 = -INFINITY, tby1 = -INFINITY, r_minr = INFINITY;
  int r_ulx = INT32_MAX, r_uly = INT32_MAX, r_uhx = INT32_MIN, r_uhy = INT32_MIN;
  int r_ilx = INT32_MIN, r_ily = INT32_MIN, r_ihx = INT32_MAX, r_ihy = INT32_MAX;
  int r_anyz = 0, r_allz = 1, any_valid = 0;
  for (int w = 0; w < W; ++w) {
    tbx0 = fminf(tbx0, sm.redf[w][0]);
    tby0 = fminf(tby0, sm.redf[w][1]);
    tbx1 = fmaxf(tbx1, sm.redf[w][2]);
    tby1 = fmaxf(tby1, sm.redf[w][3]);
    r_minr = fminf(r_minr, sm.redf[w][4]);
    r_ulx = min(r_ulx, sm.redi[w][0]);
    r_uly = min(r_uly, sm.redi[w][1]);
    r_uhx = max(r_uhx, sm.redi[w][2]);
    r_uhy = max(r_uhy, sm.redi[w][3]);
    r_ilx = max(r_ilx, sm.redi[w][4]);
    r_ily = max(r_ily, sm.redi[w][5]);
    r_ihx = min(r_ihx, sm.redi[w][6]);
    r_ihy = min(r_ihy, sm.redi[w][7]);
    r_anyz |= sm.redi[w][8];
    r_allz &= sm.redi[w][9];
    any_valid |= sm.redi[w][10];
  }
  tbx0 = uniformf(tbx0);
  tby0 = uniformf(tby0);
  tbx1 = uniformf(tbx1);
  tby1 = uniformf(tby1);
  r_ilx = uniform(r_ilx);
  r_ily = uniform(r_ily);
  r_ihx = uniform(r_ihx);
  r_ihy = uniform(r_ihy);
  if (!uniform(any_valid)) {
    __syncthreads();  // the reductions are read; the caller may start the next tile
    return;
  }

  // the box that the wave's lists serve, the tile's or its quarter's (of no
  // point: infinite, and nothing is kept)
  if constexpr (!QUAD) {
    wbx0 = tbx0;
    wby0 = tby0;
    wbx1 = tbx1;
    wby1 = tby1;
  }
  // its centre: the origin of the expansion form
  const float tcx = 0.5f * (wbx0 + wbx1), tcy = 0.5f * (wby0 + wby1);
  // a particle is "big" when h >= 2 * half-diagonal
  const float hd_x = 0.5f * (wbx1 - wbx0), hd_y = 0.5f * (wby1 - wby0);
  const float hd2 = fmaf(hd_y, hd_y, hd_x * hd_x);
  const float big_r2 = 4.0f * hd2 * 1.0001f + 1e-30f;
  const float far_a2 = 2.0f * fmaxf(hd_x * hd_x, hd_y * hd_y);  // see is_far

  // ---- candidate cell box
  int cx0, cx1, cy0, cy1, cz0, cz1;
  if constexpr (REF) {
    if (!uniform(r_anyz) || g.kz0 < 0 || g.kz0 >= g.nc[2]) {
      cx0 = 1;
      cx1 = 0;
    } else {
      cx0 = max(r_ulx, 0);
      cx1 = min(r_uhx, g.nc[0] - 1);
    }
    cy0 = max(r_uly, 0);
    cy1 = min(r_uhy, g.nc[1] - 1);
    cz0 = cz1 = g.kz0;
  } else {
    // one extra cell on each side absorbs rounding in p -/+ reach
    const float reach = support * g.max_h;
    cx0 = max(max(cell_of(tbx0, -reach, g.minc[0], g.cs[0]), INT32_MIN + 1) - 1, 0);
    cx1 = min(min(cell_of(tbx1, reach, g.minc[0], g.cs[0]), INT32_MAX - 1) + 1, g.nc[0] - 1);
    cy0 = max(max(cell_of(tby0, -reach, g.minc[1], g.cs[1]), INT32_MIN + 1) - 1, 0);
    cy1 = min(min(cell_of(tby1, reach, g.minc[1], g.cs[1]), INT32_MAX - 1) + 1, g.nc[1] - 1);
    cz0 = 0;
    cz1 = g.nc[2] - 1;
  }
  cx0 = uniform(cx0);
  cx1 = uniform(cx1);
  cy0 = uniform(cy0);
  cy1 = uniform(cy1);
  cz0 = uniform(cz0);
  cz1 = uniform(cz1);
  const bool allz_u = uniform(r_allz) != 0;
  // A particle whose h is below every point's search radius R is in the box of
  // every point its support covers: with |x - x_p| < h the particle's cell is
  // at or above the box's first cell, floor((fl(x_p - R) - min) / w), since
  // the cell arithmetic is monotone and fl(x_p - R) <= x once R - h exceeds
  // half an ulp of x_p - R (the same on the other side and in y); at the other
  // points it adds 0 either way.  The margin (1e-6 of the coordinates, 1e-5
  // of R) also covers the rounding of the support test.  A dense cell's small
  // particles thus need no box test: a slab's lists were 94% masked, since R
  // takes the largest h of the cell over all depths (16 slabs of 2048^2, 32M
  // cells: 21.9 -> 14.5 ms a render; a 256^2 crawler block of 600k rows: 6.0 ->
  // 3.7 ms).
  float unmask_ih2 = INFINITY;
  if constexpr (REF) {
    r_minr = uniformf(r_minr);
    const float pmax = fmaxf(fmaxf(fabsf(tbx0), fabsf(tbx1)), fmaxf(fabsf(tby0), fabsf(tby1)));
    const float rs = 0.99999f * r_minr - 1e-6f * (pmax + r_minr);
    if (allz_u && rs > 0.0f && rs < INFINITY) unmask_ih2 = 1.0f / (rs * rs);
  }
  const float cull2 = COUNT ? support * support * 1.0001f : support * support;

  double a64[PPT];
  uint32_t cnt_acc[COUNT ? PPT : 1];
#pragma unroll
  for (int k = 0; k < PPT; ++k) a64[k] = 0.0;
  if constexpr (COUNT)
    for (int k = 0; k < PPT; ++k) cnt_acc[k] = 0;

  auto& L = sm.L[wave];
  // list sizes (wave-uniform)
  int nf = 0, nb = 0, ns = 0, nm = 0;
  // the far field: the sum at this lane's node, and whether the wave used it
  double node64 = 0.0;
  int far_used = 0;
  if constexpr (FAR)
    if (t == 0) sm.far_used = 0;

  // ---- evaluation of the wave's lists for every point of the tile (lane l:
  // points l, l + 64, ...).  Each pads its list to a multiple of 4 with
  // entries that add nothing.
  auto eval_big = [&]() {
    if constexpr (QUARTIC) {
      const int n = uniform(nb), n4 = (n + 3) & ~3;
      if (lane < n4 - n) L.X[POOL - 1 - (n + lane)] = make_float4(0.f, 0.f, 0.f, 0.f);
      if constexpr (CLIP)
        if (lane < n4 - n) L.Xz[POOL - 1 - (n + lane)] = make_float2(0.f, 0.f);
      wave_sync();
      float lx[PPT], ly[PPT], l2[PPT];
#pragma unroll
      for (int k = 0; k < PPT; ++k) {
        const float2 e = QUAD ? my_pt : sm.pt[lane + 64 * k];
        lx[k] = e.x - tcx;
        ly[k] = e.y - tcy;
        l2[k] = fmaf(ly[k], ly[k], lx[k] * lx[k]);
      }
      for (int j0 = 0; j0 < n4; j0 += 32) {
        const int jn = min(32, n4 - j0);
        float a[PPT];
#pragma unroll
        for (int k = 0; k < PPT; ++k) a[k] = 0.0f;
        for (int j = 0; j < jn; j += 4) {
          float4 q[4];
          float2 z[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            q[u] = L.X[POOL - 1 - (j0 + j + u)];
            if constexpr (CLIP) z[u] = L.Xz[POOL - 1 - (j0 + j + u)];
          }
#pragma unroll
          for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int k = 0; k < PPT; ++k) {
              const float v = fmaf(q[u].y, lx[k], fmaf(q[u].z, ly[k], fmaf(q[u].w, l2[k], q[u].x)));
              if constexpr (CLIP)
                a[k] += clip_pow(v, z[u]);
              else
                a[k] += pow25(v);
            }
        }
#pragma unroll
        for (int k = 0; k < PPT; ++k) a64[k] += double(a[k]);
      }
      wave_sync();
    }
    nb = 0;
  };
  // far entries at the nodes (lane l: node l % 8, l / 8)
  auto eval_far = [&]() {
    if constexpr (FAR) {
      const int n = uniform(nf), n4 = (n + 3) & ~3;
      if (lane < n4 - n) L.X[n + lane] = make_float4(0.f, 0.f, 0.f, 0.f);
      wave_sync();
      float fx = 0.f, fy = 0.f;
#pragma unroll
      for (int i = 0; i < kNodes; ++i) {
        if ((lane & 7) == i) fx = float(kNodeX[i]);
        if ((lane >> 3) == i) fy = float(kNodeX[i]);
      }
      const float lx = hd_x * fx, ly = hd_y * fy;
      const float l2 = fmaf(ly, ly, lx * lx);
      for (int j0 = 0; j0 < n4; j0 += 32) {
        const int jn = min(32, n4 - j0);
        float a[4] = {0.f, 0.f, 0.f, 0.f};
        for (int j = 0; j < jn; j += 4) {
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const float4 q = L.X[j0 + j + u];
            a[u] += pow25_pos(fmaf(q.y, lx, fmaf(q.z, ly, fmaf(q.w, l2, q.x))));
          }
        }
        node64 += double((a[0] + a[1]) + (a[2] + a[3]));
      }
      wave_sync();
      far_used = 1;
    }
    nf = 0;
  };
  auto eval_small = [&]() {
    const int n = uniform(ns), n4 = (n + 3) & ~3;
    if (lane < n4 - n) L.S[n + lane] = make_float4(0.f, 0.f, 0.f, 0.f);
    if constexpr (CLIP)
      if (lane < n4 - n) L.Sz[n + lane] = make_float2(0.f, 0.f);
    wave_sync();
    float ex[PPT], ey[PPT];
#pragma unroll
    for (int k = 0; k < PPT; ++k) {
      const float2 e = QUAD ? my_pt : sm.pt[lane + 64 * k];
      ex[k] = e.x;
      ey[k] = e.y;
    }
    if constexpr (COUNT) {
#pragma clang fp contract(off)
      for (int j = 0; j < n; ++j) {
        const float4 q = L.S[j];
        const double hs = double(support) * double(q.z);
        const double hs2 = hs * hs;
#pragma unroll
        for (int k = 0; k < PPT; ++k) {
          const double dx = double(q.x) - double(ex[k]);
          const double dy = double(q.y) - double(ey[k]);
          const double r2 = dx * dx + dy * dy;
          cnt_acc[k] += (r2 < hs2) ? 1u : 0u;
        }
      }
    } else {
      for (int j0 = 0; j0 < n4; j0 += 32) {
        const int jn = min(32, n4 - j0);
        float a[PPT];
#pragma unroll
        for (int k = 0; k < PPT; ++k) a[k] = 0.0f;
        for (int j = 0; j < jn; j += 4) {
          float4 q[4];
          float2 z[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            q[u] = L.S[j0 + j + u];
            if constexpr (CLIP) z[u] = L.Sz[j0 + j + u];
          }
#pragma unroll
          for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int k = 0; k < PPT; ++k) {
              const float dx = q[u].x - ex[k], dy = q[u].y - ey[k];
              const float r2 = fmaf(dy, dy, dx * dx);
              if constexpr (KERNEL == 2)
                a[k] = fmaf(q[u].z, cubic_shape(r2 * q[u].w, sm.tab), a[k]);
              else if constexpr (CLIP)
                a[k] += clip_pow(fmaf(-r2, q[u].z, q[u].w), z[u]);
              else
                a[k] += pow25(fmaf(-r2, q[u].z, q[u].w));
            }
        }
#pragma unroll
        for (int k = 0; k < PPT; ++k) a64[k] += double(a[k]);
      }
    }
    wave_sync();
    ns = 0;
  };
  // masked entries: each point tests the entry's cell against its own search
  // box, as unsigned(cx - x0) <= width (and the same for y)
  auto eval_masked = [&]() {
    if constexpr (REF) {
      const int n = uniform(nm), n4 = (n + 3) & ~3;
      if (lane < n4 - n) {
        L.S[POOL - 1 - (n + lane)] = make_float4(0.f, 0.f, 0.f, 0.f);
        L.M[n + lane] = 0;
      }
      wave_sync();
      float ex[PPT], ey[PPT];
      uint2 bx[PPT];
#pragma unroll
      for (int k = 0; k < PPT; ++k) {
        const float2 e = QUAD ? my_pt : sm.pt[lane + 64 * k];
        ex[k] = e.x;
        ey[k] = e.y;
        bx[k] = QUAD ? my_box : sm.box[lane + 64 * k];
      }
      for (int j0 = 0; j0 < n4; j0 += 32) {
        const int jn = min(32, n4 - j0);
        float a[PPT];
#pragma unroll
        for (int k = 0; k < PPT; ++k) a[k] = 0.0f;
        for (int j = 0; j < jn; j += 4) {
          const int4 c4 = *reinterpret_cast<const int4*>(&L.M[j0 + j]);
          const int cc[4] = {uniform(c4.x), uniform(c4.y), uniform(c4.z), uniform(c4.w)};
          float4 q[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) q[u] = L.S[POOL - 1 - (j0 + j + u)];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const uint32_t cx = uint32_t(cc[u]) & 0xffffu, cy = uint32_t(cc[u]) >> 16;
#pragma unroll
            for (int k = 0; k < PPT; ++k) {
              const bool in = cx - (bx[k].x & 0xffffu) <= bx[k].x >> 16 &&
                              cy - (bx[k].y & 0xffffu) <= bx[k].y >> 16;
              const float dx = q[u].x - ex[k], dy = q[u].y - ey[k];
              const float r2 = fmaf(dy, dy, dx * dx);
              a[k] = fmaf(in ? 1.0f : 0.0f, pow25(fmaf(-r2, q[u].z, q[u].w)), a[k]);
            }
          }
        }
#pragma unroll
        for (int k = 0; k < PPT; ++k) a64[k] += double(a[k]);
      }
      wave_sync();
    }
    nm = 0;
  };

  stream_candidates<REF, QUAD ? DEAL_ALL : (PPT > 1 ? DEAL_EVEN : DEAL_64)>(
      g, cx0, cx1, cy0, cy1, cz0, cz1, tbx0, tby0, tbx1, tby1, support,
      [&](int cx, int cy) {
        return allz_u && cy >= r_ily && cy <= r_ihy && cx >= r_ilx && cx <= r_ihx;
      },
      sm.cells, [&](bool have, uint32_t sidx, int cinf, bool cf, bool done) {
        float4 e = make_float4(0.f, 0.f, 0.f, 0.f);
        bool keep = false, full = false, big = false, far = false;
        float2 tcl = make_float2(0.0f, 0.0f);
        if (have) {
          // (x, y, coef, 1/h^2); the quartic's z is c = coef^0.4
          const float4 q = g.part[sidx];
          if (q.z != 0.0f) {
            const float dx = fmaxf(fmaxf(wbx0 - q.x, q.x - wbx1), 0.0f);
            const float dy = fmaxf(fmaxf(wby0 - q.y, q.y - wby1), 0.0f);
            const float d2 = fmaf(dy, dy, dx * dx);
            keep = d2 * q.w < cull2;
          }
          if constexpr (CLIP) {
            // the depth range relative to the particle, in units of h: its
            // support must overlap it
            const float2 zc = g.clip[sidx];
            keep = keep && zc.x < 1.0f && zc.y > -1.0f;
            const float rc = __builtin_amdgcn_sqrtf(q.z);
            tcl = make_float2(zc.x * rc, zc.y * rc);
          }
          full = keep && (!REF || cf || q.w >= unmask_ih2);
          if (keep) {
            if constexpr (COUNT) {
              e = make_float4(q.x, q.y, g.hs[sidx], 0.0f);
            } else if constexpr (KERNEL == 2) {
              e = q;
            } else {
              const float c = q.z;        // coef^0.4
              const float ci2 = c * q.w;  // c / h^2
              big = full && big_r2 * q.w <= 1.0f;
              if (big) {
                const float xr = q.x - tcx, yr = q.y - tcy;
                const float d2r = fmaf(yr, yr, xr * xr);
                e = make_float4(c * fmaf(-q.w, d2r, 1.0f), 2.0f * ci2 * xr, 2.0f * ci2 * yr, -ci2);
                if constexpr (FAR) far = is_far(d2r, q.w, far_a2);
              } else {
                e = make_float4(q.x, q.y, ci2, c);
              }
            }
          }
        }
        const uint64_t bf = FAR ? __ballot(far) : 0ull;
        const uint64_t bb = __ballot(big && !far);
        const uint64_t bs = __ballot(full && !big);
        const uint64_t bm = __ballot(keep && !full);
        if constexpr (FAR)
          if (far) L.X[nf + int(prefix_count(bf))] = e;
        if constexpr (QUARTIC) {
          if (big && !far) {
            const int pos = POOL - 1 - (nb + int(prefix_count(bb)));
            L.X[pos] = e;
            if constexpr (CLIP) L.Xz[pos] = tcl;
          }
        }
        if (full && !big) {
          const int pos = ns + int(prefix_count(bs));
          L.S[pos] = e;
          if constexpr (CLIP) L.Sz[pos] = tcl;
        }
        if constexpr (REF) {
          if (keep && !full) {
            const int pos = nm + int(prefix_count(bm));
            L.S[POOL - 1 - pos] = e;
            L.M[pos] = cinf;
          }
        }
        if constexpr (FAR) nf += __popcll(bf);
        nb += __popcll(bb);
        ns += __popcll(bs);
        nm += __popcll(bm);
        const int lim = done ? 1 : FLUSH;
        if constexpr (FAR) {
          if (done && !far_used && nf > 0) {
            // too few far entries to pay for the tile's interpolation
            const int n = uniform(nf);
            const float4 x = lane < n ? L.X[lane] : make_float4(0.f, 0.f, 0.f, 0.f);
            wave_sync();
            if (lane < n) L.X[POOL - 1 - (nb + lane)] = x;
            nb += n;
            nf = 0;
          }
          if (nf >= lim) eval_far();
        }
        if (nb >= lim) eval_big();
        if (ns >= lim) eval_small();
        if (nm >= lim) eval_masked();
      });
  if constexpr (FAR)
    if (far_used && lane == 0) sm.far_used = 1;

  if constexpr (QUAD) {
    const uint32_t px = tx * T + uint32_t(col_of(t)), py = ty * T + uint32_t(row_of(t));
    const uint32_t pid = py * p.lnx + px;
    if (!(px < p.lnx && py < p.lny && pid < p.n)) return;
    if (fused) {
      acc_out[pid] = a64[0];
      img_out[pid] = static_cast<float>(a64[0] * static_cast<double>(img_scale));
    } else {
      acc_out[pid] += a64[0];
    }
    return;
  }

  // ---- the waves' sums, in wave order
  __syncthreads();
#pragma unroll
  for (int k = 0; k < PPT; ++k) {
    double v = a64[k];
    if constexpr (COUNT) v = double(cnt_acc[k]);
    sm.sum[wave][lane + 64 * k] = v;
  }
  bool interp = false;
  if constexpr (FAR) {
    interp = sm.far_used != 0;
    sm.node[wave][lane] = node64;
  }
  __syncthreads();
  if constexpr (FAR && W > 1) {
    if (interp) {
      if (t < 64) {
        double n = sm.node[0][t];
        for (int w = 1; w < W; ++w) n += sm.node[w][t];
        sm.node[0][t] = n;
      }
      __syncthreads();
    }
  }
#pragma unroll 1
  for (int pt = t; pt < NP; pt += NB) {
    const uint32_t px = tx * T + uint32_t(col_of(pt)), py = ty * T + uint32_t(row_of(pt));
    const uint32_t pid = py * p.lnx + px;
    if (!(px < p.lnx && py < p.lny && pid < p.n)) continue;
    double v = sm.sum[0][pt];
    for (int w = 1; w < W; ++w) v += sm.sum[w][pt];
    if constexpr (FAR) {
      // the far field at the point (a NaN coordinate is in no support)
      const float2 e = sm.pt[pt];
      if (interp && e.x == e.x && e.y == e.y) {
        double bx[kNodes], by[kNodes];
        node_basis(hd_x > 0.0f ? double(e.x - tcx) / double(hd_x) : 0.0, bx);
        node_basis(hd_y > 0.0f ? double(e.y - tcy) / double(hd_y) : 0.0, by);
        double f = 0.0;
#pragma unroll
        for (int iy = 0; iy < kNodes; ++iy) {
          double r = 0.0;
#pragma unroll
          for (int ix = 0; ix < kNodes; ++ix) r = fma(bx[ix], sm.node[0][8 * iy + ix], r);
          f = fma(by[iy], r, f);
        }
        v += f;
      }
    }
    if constexpr (COUNT) {
      if (counts) counts[pid] += static_cast<unsigned long long>(v);
    } else if (fused) {
      // the only visit of this point in the launch: no read of the
      // accumulator, and the image as the retrieval computes it
      acc_out[pid] = v;
      img_out[pid] = static_cast<float>(v * static_cast<double>(img_scale));
    } else {
      acc_out[pid] += v;
    }
  }
}

// Waves per SIMD asked of the compiler for whole tiles: at 5 (96 VGPRs; 12 spilled
// in the reference-mode batch when this was measured, 3 now) 32 views of a 16M
// snapshot take 50.0 ms, at 4 (no spills) 53.5, at 3 60.2.  The LDS allows 5
// workgroups per CU.  Quarters take 8 (64 VGPRs, 3 spilled).
constexpr int kSumWaves = 5;

template <int T, int OP, int KERNEL>
__global__ __launch_bounds__(64 * kSumW) __attribute__((amdgpu_waves_per_eu(kSumWaves, 8))) void k_gather(
    grid_view g, point_view p, uint32_t tiles_x, uint32_t ntiles, double* __restrict__ acc_out,
    unsigned long long* __restrict__ counts, const float* __restrict__ cubic_table, float support) {
  __shared__ tile_smem<T, OP == OP_REFERENCE, KERNEL, OP == OP_CLIP, OP == OP_COUNT, false> sm;
  if constexpr (KERNEL == 2) {
    for (int i = threadIdx.x; i < kCubicTable; i += 64 * kSumW) sm.tab[i] = cubic_table[i];
  }
  // XCD-contiguous tile order: workgroups are dealt round-robin to the 8
  // XCDs, so give XCD x the x-th eighth of the tiles (shared L2 reuse of the
  // neighbouring tiles' particle spans).
  const uint32_t bid = blockIdx.x;
  const uint32_t per = ntiles / 8u;
  const uint32_t tile = bid < per * 8u ? (bid % 8u) * per + bid / 8u : bid;
  const uint32_t tx = tile % tiles_x, ty = tile / tiles_x;
  sum_tile<T, OP, KERNEL, false>(g, p, tx, ty, acc_out, counts, support, sm);
}

// Persistent gather over (view, tile) items.  Workgroups are dealt to the 8
// XCDs round-robin by id, and each XCD has its own L2: queue q holds the q-th
// eighth of every view's tiles (contiguous rows), so the tiles one XCD works
// on at a time are neighbours that read the same particle spans.  A
// workgroup drains its XCD's queue, then helps with the others; every queue
// counter only grows, so every workgroup leaves once all queues are empty.
template <int T, int OP, int KERNEL, bool QUAD>
__global__ __launch_bounds__(64 * kSumW) __attribute__((amdgpu_waves_per_eu(QUAD ? 8 : kSumWaves, 8))) void k_gather_batch(
    const view_desc* __restrict__ views, const uint2* __restrict__ items, queue_segs segs,
    uint32_t* __restrict__ counters, const float* __restrict__ cubic_table, float support) {
  __shared__ tile_smem<T, OP == OP_REFERENCE, KERNEL, OP == OP_CLIP, OP == OP_COUNT, QUAD> sm;
  __shared__ uint32_t next;
  if constexpr (KERNEL == 2) {
    for (int i = threadIdx.x; i < kCubicTable; i += 64 * kSumW) sm.tab[i] = cubic_table[i];
  }
  const uint32_t home = blockIdx.x % uint32_t(kQueues);
  for (uint32_t k = 0; k < uint32_t(kQueues); ++k) {
    const uint32_t q = (home + k) % uint32_t(kQueues);
    const uint32_t qb = segs.seg[q], qe = segs.seg[q + 1];
    for (;;) {
      __syncthreads();
      if (threadIdx.x == 0) next = atomicAdd(counters + q * kQueueStride, 1u);
      __syncthreads();
      const uint32_t got = uint32_t(uniform(int(next)));
      if (got >= qe - qb) break;
      const uint2 it = items[qb + got];
      const uint32_t vi = uint32_t(uniform(int(it.x))), ti = uint32_t(uniform(int(it.y)));
      const view_desc& vd = views[vi];
      const uint32_t tiles_x = vd.tiles_x;
      sum_tile<T, OP, KERNEL, QUAD>(vd.g, vd.p, ti % tiles_x, ti / tiles_x, vd.acc, nullptr, support,
                                 sm, vd.img, vd.scale, vd.fused);
    }
  }
}

// ---- the adjoint of the exact-mode gather
//
// A workgroup owns a tile of T x T points with their gradients; its waves
// stream the candidates as the gather does.  A wave lists the kept particles'
// indices, and with 64 of them gives each lane one: the lane visits the 8x8
// point blocks that some listed particle's support reaches and sums over
// their points moments of g = dL/dvalue * s^1.5 (s = 1 - r^2/h^2); the
// weights are recomputed, not stored.  One atomic add per gradient component,
// particle and tile:
//   dL/dw = K/h^2        sum g s
//   dL/dh = w K/h^3      sum g (7 r^2/h^2 - 2)
//   dL/dx = -5 w K/h^4   sum g (x - x_point)     (same for y)
// In 16x16 tiles the far particles (is_far) take the transpose of the
// gather's interpolation: the tile's gradients are first summed onto the 64
// nodes, and the particle visits the nodes instead of the 256 points.
// VALU-bound (16 operations a pair).  Against shared lists of 32x32 tiles,
// one particle per thread: 4M particles on 1024^2 points 10.8 -> 4.1 ms, 20k on
// 96^2 (9 workgroups before, 144 now) 1.34 -> 0.06 ms; every component's error
// against 64 bits is at or below what it was.
constexpr int kAdjCap = 2 * 63 + 64;  // two index lists from the two ends of one array

template <int T, int KERNEL>
struct adjoint_smem {
  static constexpr int NP = T * T;
  float4 pt[NP];  // tile points (x, y, dL/dvalue, -), 8x8 block after 8x8 block
  float4 box[NP / 64];  // the blocks' boxes of points with a gradient (x0, y0, x1, y1)
  int wild[NP / 64];    // whether a block's gradients are infinite or NaN somewhere
  alignas(16) float node[KERNEL == 0 && NP > 64 ? 64 : 1];  // the gradients at the nodes
  union {
    uint32_t idx[kSumW][kAdjCap];
    struct {  // while the nodes are summed: the points' Lagrange bases
      float bx[KERNEL == 0 && NP > 64 ? NP : 1][kNodes];
      float by[KERNEL == 0 && NP > 64 ? NP : 1][kNodes];
      double part[KERNEL == 0 && NP > 64 ? kSumW : 1][64];
    };
  };
  cell_table cells;
  float tab[KERNEL == 2 ? kCubicTable : 1];
  float dtab[KERNEL == 2 ? kCubicTable : 1];
};

template <int T, int KERNEL>
__global__ __launch_bounds__(64 * kSumW) void k_adjoint(grid_view g, point_view p,
                                                        uint32_t tiles_x, uint32_t ntiles,
                                                        adjoint_io io) {
  constexpr int NB = 64 * kSumW, NP = T * T, NBLK = NP / 64;
  constexpr bool FAR = KERNEL == 0 && NP > 64;
  static_assert(NP <= NB, "one point per thread");
  __shared__ adjoint_smem<T, KERNEL> sm;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const uint32_t bid = blockIdx.x;
  const uint32_t per = ntiles / 8u;
  const uint32_t tile = bid < per * 8u ? (bid % 8u) * per + bid / 8u : bid;
  const uint32_t tx = tile % tiles_x, ty = tile / tiles_x;
  if constexpr (KERNEL == 2) {
    for (int i = t; i < kCubicTable; i += NB) {
      sm.tab[i] = io.ftab[i];
      sm.dtab[i] = io.dtab[i];
    }
  }
  const float support = KERNEL == 2 ? 2.0f : 1.0f;

  // ---- thread t: point t of the blocks' order; the blocks' boxes of the
  // points with a gradient, and the tile box over them
  float px = 0.f, py = 0.f, pg = 0.f;
  if (t < NP) {
    const int blk = t >> 6, in = t & 63;
    const uint32_t ix = tx * T + uint32_t((blk % (T / 8)) * 8 + (in & 7));
    const uint32_t iy = ty * T + uint32_t((blk / (T / 8)) * 8 + (in >> 3));
    const uint32_t pid = iy * p.lnx + ix;
    if (ix < p.lnx && iy < p.lny && pid < p.n) {
      const float4 q = p.gen ? pixel_point(p.pg, ix, iy) : p.pts[pid];
      // a point with an infinite or NaN coordinate is in no support (its
      // moments would be 0 times that)
      if (isfinite(q.x) && isfinite(q.y)) {
        px = q.x;
        py = q.y;
        pg = io.grad[pid] * io.scale;
      }
    }
    sm.pt[t] = make_float4(px, py, pg, 0.0f);
  }
  {
    const bool on = pg != 0.0f;
    const float x0 = wave_minf(on ? px : INFINITY), y0 = wave_minf(on ? py : INFINITY);
    const float x1 = wave_maxf(on ? px : -INFINITY), y1 = wave_maxf(on ? py : -INFINITY);
    const bool wild = __ballot(!isfinite(pg)) != 0;
    if (lane == 0 && wave < NBLK) {
      sm.box[wave] = make_float4(x0, y0, x1, y1);
      sm.wild[wave] = wild;
    }
  }
  __syncthreads();
  float tbx0 = INFINITY, tby0 = INFINITY, tbx1 = -INFINITY, tby1 = -INFINITY;
  int wild = 0;
  for (int b = 0; b < NBLK; ++b) {
    wild |= sm.wild[b];
    const float4 x = sm.box[b];
    tbx0 = fminf(tbx0, x.x);
    tby0 = fminf(tby0, x.y);
    tbx1 = fmaxf(tbx1, x.z);
    tby1 = fmaxf(tby1, x.w);
  }
  tbx0 = uniformf(tbx0);
  tby0 = uniformf(tby0);
  tbx1 = uniformf(tbx1);
  tby1 = uniformf(tby1);
  if (!(tbx0 <= tbx1)) return;  // no gradient in the tile
  const float tcx = 0.5f * (tbx0 + tbx1), tcy = 0.5f * (tby0 + tby1);
  const float hd_x = 0.5f * (tbx1 - tbx0), hd_y = 0.5f * (tby1 - tby0);
  const float far_a2 = 2.0f * fmaxf(hd_x * hd_x, hd_y * hd_y);  // see is_far

  // ---- the gradients at the nodes (when any particle is wide enough; an
  // infinite one would meet weights of either sign there)
  const bool nodes = FAR && !uniform(wild) && g.max_h * g.max_h * 0.16f >= far_a2;
  if constexpr (FAR) {
    if (nodes) {
      double b[kNodes];
      node_basis(pg != 0.0f && hd_x > 0.0f ? double(px - tcx) / double(hd_x) : 0.0, b);
#pragma unroll
      for (int i = 0; i < kNodes; ++i) sm.bx[t][i] = float(b[i] * double(pg));
      node_basis(pg != 0.0f && hd_y > 0.0f ? double(py - tcy) / double(hd_y) : 0.0, b);
#pragma unroll
      for (int i = 0; i < kNodes; ++i) sm.by[t][i] = float(b[i]);
      __syncthreads();
      double sum = 0.0;
      for (int k = 64 * wave; k < 64 * wave + 64; ++k)
        sum += double(sm.bx[k][lane & 7]) * double(sm.by[k][lane >> 3]);
      sm.part[wave][lane] = sum;
      __syncthreads();
      if (t < 64) {
        double n = 0.0;
        for (int w = 0; w < kSumW; ++w) n += sm.part[w][t];
        sm.node[t] = float(n);
      }
    }
  }
  __syncthreads();

  // ---- candidate cell box (one extra cell on each side absorbs rounding)
  const float reach = support * g.max_h;
  const int cx0 = uniform(max(max(cell_of(tbx0, -reach, g.minc[0], g.cs[0]), INT32_MIN + 1) - 1, 0));
  const int cx1 = uniform(
      min(min(cell_of(tbx1, reach, g.minc[0], g.cs[0]), INT32_MAX - 1) + 1, g.nc[0] - 1));
  const int cy0 = uniform(max(max(cell_of(tby0, -reach, g.minc[1], g.cs[1]), INT32_MIN + 1) - 1, 0));
  const int cy1 = uniform(
      min(min(cell_of(tby1, reach, g.minc[1], g.cs[1]), INT32_MAX - 1) + 1, g.nc[1] - 1));
  const float cull2 = support * support;

  uint32_t* const idx = sm.idx[wave];
  int nf = 0, nn = 0;  // far from the front, near from the back

  // the moments of the particle's lane into the gradients
  auto add = [&](uint32_t si, const float4& q, float coef, float a0, float a1, float a2,
                 float a3, float a4) {
    if constexpr (KERNEL == 2) {
      // value = w K F(u) / h^2: d/dh = -2 w K / h^3 (F + u F'),
      // d/dx = 2 w K / h^4 F' (x - x_point)
      const float c2 = 2.0f * coef * q.w;
      atomicAdd(io.gw + si, io.norm * q.w * a0);
      atomicAdd(io.gh + si, -2.0f * coef * __builtin_amdgcn_sqrtf(q.w) * (a0 + a1));
      atomicAdd(io.gx + si, c2 * a3);
      atomicAdd(io.gy + si, c2 * a4);
    } else {
      const float c5 = -5.0f * coef * q.w;  // -5 w K / h^4
      atomicAdd(io.gw + si, io.norm * q.w * a0);
      atomicAdd(io.gh + si, coef * __builtin_amdgcn_sqrtf(q.w) * fmaf(7.0f * q.w, a2, -2.0f * a1));
      atomicAdd(io.gx + si, c5 * a3);
      atomicAdd(io.gy + si, c5 * a4);
    }
  };
  auto near_batch = [&]() {
    const int n = min(uniform(nn), 64);
    const bool act = lane < n;
    const uint32_t si = act ? idx[kAdjCap - nn + lane] : 0u;  // the list's last 64
    float4 q = make_float4(0.f, 0.f, 1.f, 0.f);
    if (act) q = g.part[si];
    float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f, a4 = 0.f;
    for (int blk = 0; blk < NBLK; ++blk) {
      const float4 bx = sm.box[blk];
      const float bdx = fmaxf(fmaxf(bx.x - q.x, q.x - bx.z), 0.0f);
      const float bdy = fmaxf(fmaxf(bx.y - q.y, q.y - bx.w), 0.0f);
      if (!__ballot(act && bx.x <= bx.z && fmaf(bdy, bdy, bdx * bdx) * q.w < cull2)) continue;
#pragma unroll 8
      for (int k = 0; k < 64; ++k) {
        const float4 pt = sm.pt[64 * blk + k];
        const float dx = q.x - pt.x, dy = q.y - pt.y;
        const float r2 = fmaf(dy, dy, dx * dx);
        if constexpr (KERNEL == 2) {
          // F and dF/du at u = r^2/h^2, linear in the tables (0 beyond u = 4)
          const float uu = r2 * q.w;
          const float xx = fminf(uu * (float(kCubicTable - 1) / 4.0f), float(kCubicTable - 1));
          const int ti = min(int(xx), kCubicTable - 2);
          const float tf = xx - float(ti);
          const float F = fmaf(tf, sm.tab[ti + 1] - sm.tab[ti], sm.tab[ti]);
          const float D = fmaf(tf, sm.dtab[ti + 1] - sm.dtab[ti], sm.dtab[ti]);
          const float gd = pt.z * D;
          a0 = fmaf(pt.z, F, a0);
          a1 = fmaf(gd, uu, a1);
          a3 = fmaf(gd, dx, a3);
          a4 = fmaf(gd, dy, a4);
        } else {
          const float sv = fmaxf(fmaf(-r2, q.w, 1.0f), 0.0f);
          const float gq = pt.z * (sv * __builtin_amdgcn_sqrtf(sv));
          a0 = fmaf(gq, sv, a0);
          a1 += gq;
          a2 = fmaf(gq, r2, a2);
          a3 = fmaf(gq, dx, a3);
          a4 = fmaf(gq, dy, a4);
        }
      }
    }
    if (act) add(si, q, KERNEL == 2 ? q.z : pow25_pos(q.z), a0, a1, a2, a3, a4);
    nn -= n;
  };
  auto far_batch = [&]() {
    if constexpr (FAR) {
      const int n = min(uniform(nf), 64);
      const bool act = lane < n;
      const uint32_t si = act ? idx[nf - n + lane] : 0u;
      float4 q = make_float4(0.f, 0.f, 1.f, 0.f);
      if (act) q = g.part[si];
      const float xr = q.x - tcx, yr = q.y - tcy;
      float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f, a4 = 0.f;
#pragma unroll 1
      for (int iy = 0; iy < kNodes; ++iy) {
        float ny = 0.f;
#pragma unroll
        for (int i = 0; i < kNodes; ++i)
          if (iy == i) ny = float(kNodeX[i]);
        const float dy = fmaf(-hd_y, ny, yr);
        const float dy2 = dy * dy;
#pragma unroll
        for (int ix = 0; ix < kNodes; ++ix) {
          const float gn = sm.node[8 * iy + ix];
          const float dx = fmaf(-hd_x, float(kNodeX[ix]), xr);
          const float r2 = fmaf(dx, dx, dy2);
          const float sv = fmaxf(fmaf(-r2, q.w, 1.0f), 0.0f);
          const float gq = gn * (sv * __builtin_amdgcn_sqrtf(sv));
          a0 = fmaf(gq, sv, a0);
          a1 += gq;
          a2 = fmaf(gq, r2, a2);
          a3 = fmaf(gq, dx, a3);
          a4 = fmaf(gq, dy, a4);
        }
      }
      if (act) add(si, q, pow25_pos(q.z), a0, a1, a2, a3, a4);
      nf -= n;
    }
  };

  stream_candidates<false, DEAL_64>(
      g, cx0, cx1, cy0, cy1, 0, g.nc[2] - 1, tbx0, tby0, tbx1, tby1, support,
      [](int, int) { return true; }, sm.cells,
      [&](bool have, uint32_t sidx, int, bool, bool done) {
        bool keep = false, far = false;
        if (have) {
          const float4 q = g.part[sidx];
          const float dx = fmaxf(fmaxf(tbx0 - q.x, q.x - tbx1), 0.0f);
          const float dy = fmaxf(fmaxf(tby0 - q.y, q.y - tby1), 0.0f);
          keep = fmaf(dy, dy, dx * dx) * q.w < cull2;
          if constexpr (FAR) {
            const float xr = q.x - tcx, yr = q.y - tcy;
            far = keep && nodes && is_far(fmaf(yr, yr, xr * xr), q.w, far_a2, 0.16f);
          }
        }
        const uint64_t bf = FAR ? __ballot(far) : 0ull;
        const uint64_t bn = __ballot(keep && !far);
        if (far) idx[nf + int(prefix_count(bf))] = sidx;
        if (keep && !far) idx[kAdjCap - 1 - (nn + int(prefix_count(bn)))] = sidx;
        nf += __popcll(bf);
        nn += __popcll(bn);
        const int lim = done ? 1 : 64;
        wave_sync();
        if constexpr (FAR)
          while (nf >= lim) far_batch();
        while (nn >= lim) near_batch();
        wave_sync();
      });
}

// gradients in sorted order -> input order
__global__ __launch_bounds__(kBlock) void k_unpermute4(const uint32_t* __restrict__ perm, uint32_t n,
                                                        const float* __restrict__ a,
                                                        const float* __restrict__ b,
                                                        const float* __restrict__ c,
                                                        const float* __restrict__ d, float* oa,
                                                        float* ob, float* oc, float* od) {
  const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
  if (s >= n) return;
  const uint32_t i = perm[s];
  oa[i] = a[s];
  ob[i] = b[s];
  oc[i] = c[s];
  od[i] = d[s];
}

template <int T, int OP, int KERNEL, bool QUAD>
struct plain_launcher {
  static int run(const grid_view& g, const point_view& p, double* acc,
                 unsigned long long* counts, const float* tab, float support, hipStream_t s) {
    const uint32_t tiles_x = (p.lnx + T - 1) / T;
    const uint32_t tiles_y = (p.lny + T - 1) / T;
    const uint32_t ntiles = tiles_x * tiles_y;
    if (!ntiles) return 0;
    if constexpr (QUAD || OP == OP_CLIP) {
      fail(ILC_EINVAL, "quarter tiles and the clip are the persistent gather's");
    } else {
      hipLaunchKernelGGL((k_gather<T, OP, KERNEL>), dim3(ntiles), dim3(64 * kSumW), 0, s, g, p,
                         tiles_x, ntiles, acc, counts, tab, support);
    }
    ILC_HIP(hipGetLastError());
    return 0;
  }
};

template <int T, int OP, int KERNEL, bool QUAD>
struct batch_launcher {
  static int run(const view_desc* v, const uint2* it, const queue_segs& segs, uint32_t* c,
                 const float* tab, float sup, int grid, hipStream_t s) {
    hipLaunchKernelGGL((k_gather_batch<T, OP, KERNEL, QUAD>), dim3(grid), dim3(64 * kSumW), 0, s, v,
                       it, segs, c, tab, sup);
    ILC_HIP(hipGetLastError());
    return 0;
  }
};

template <int T, int OP, int KERNEL, bool QUAD>
struct batch_occ {
  static int run() {
    int per_cu = 0;
    ILC_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &per_cu, k_gather_batch<T, OP, KERNEL, QUAD>, 64 * kSumW, 0));
    return per_cu;
  }
};

// dispatch over (tile side, op, kernel, quarters) to F<T, OP, KERNEL, QUAD>::run
template <template <int, int, int, bool> class F, class... A>
int dispatch(const sum_shape& ts, int op, int kernel, A&&... a) {
  auto by_op = [&](auto tt) -> int {
    constexpr int T = decltype(tt)::value;
    if (op == OP_CLIP) {
      if (kernel == ILC_KERNEL_CUBIC) fail(ILC_EINVAL, "the line-of-sight clip needs a quartic kernel");
      // 16x16 tiles by quarters: the clip has no nodes, and with four points a
      // lane the larger pair leaves 5 waves a SIMD (four 1024^2 views of 16M
      // particles 21.2 ms, 14.3 by quarters, 14.7 in 8x8 tiles; 2048^2 ones 70.7,
      // 50.5, 55.4; 32 slabs of 4096^2 through 64M 98.4, 67.2, 84.1)
      return F<T, OP_CLIP, 0, T == 16>::run(a...);
    }
    if (op == OP_REFERENCE) {
      if (kernel == ILC_KERNEL_CUBIC) fail(ILC_EINVAL, "reference mode uses the quartic kernel");
      return F<T, OP_REFERENCE, 0, false>::run(a...);
    }
    if (kernel == ILC_KERNEL_CUBIC) return F<T, OP_EXACT, 2, false>::run(a...);
    return F<T, OP_EXACT, 0, false>::run(a...);
  };
  if (ts.quad) {
    ILC_REQUIRE(ts.side == 16 && kernel != ILC_KERNEL_CUBIC &&
                    (op == OP_REFERENCE || op == OP_EXACT),
                "quarters are of 16x16 tiles of the quartic");
    return op == OP_REFERENCE ? F<16, OP_REFERENCE, 0, true>::run(a...)
                              : F<16, OP_EXACT, 0, true>::run(a...);
  }
  if (ts.side == 16) return by_op(std::integral_constant<int, 16>{});
  if (ts.side == 8) return by_op(std::integral_constant<int, 8>{});
  fail(ILC_EINVAL, "gather: no tile of side %d", ts.side);
}

}  // namespace

// 16x16 tiles list a candidate once per 256 points and sum the far particles
// at 64 nodes; 8x8 tiles give four times the workgroups and waste fewer pairs
// at the supports' edges.  Below kPointsFor16 points the launch cannot fill
// the GPU with 16x16 tiles and the heaviest one sets its time.  One view of
// 1M / 16M / 100k particles, 8x8 against 16x16 tiles: 300^2 points 0.30, 1.0,
// 0.11 against 0.99, 3.8, 0.21 ms; 700^2 0.61, 1.10, 0.31 against 0.75, 1.71,
// 0.24; 1024^2 1.12, 2.0, 0.57 against 0.93, 1.38, 0.31; 2048^2 3.9, 6.7, 2.0
// against 2.1, 2.9, 0.82.  The cubic, which has no nodes: 300^2 1.2, 2.3, 0.51
// against 3.9, 11.4, 1.1; 1024^2 6.6, 9.6, 3.0 against 6.8, 9.4, 2.7; 2048^2 22.6,
// 34.6, 9.8 against 18.8, 27.4, 8.1.  The number of points is the whole launch's:
// many small views of one batch would be faster in 8x8 tiles past the line, too
// (64 of 128^2 through 1M 2.7 against 6.6 ms), which the caller can ask for or
// have timed (ilc_batch_autotune).
constexpr uint64_t kPointsFor16 = 3u << 18;

sum_shape sum_shape_of(const tile_shape& ts, uint64_t npoints) {
  if (ts.nb == 256) {
    if ((ts.tw == 16 && ts.ppt == 1) || (ts.tw == 32 && (ts.ppt == 2 || ts.ppt == 4)) ||
        (ts.tw == 64 && ts.ppt == 4))
      return sum_shape{npoints < kPointsFor16 ? 8 : 16};
  } else if (ts.nb == 64) {
    if (ts.tw == 16 && ts.ppt == 4) return sum_shape{16};
    if (ts.tw == 8 && ts.ppt == 1) return sum_shape{8};
  }
  fail(ILC_EINVAL, "gather: unsupported tile shape tw=%d ppt=%d nb=%d", ts.tw, ts.ppt, ts.nb);
}

// Slab stacks whose tiles are many and hold few rows: both forms are bound by
// issue slots, and the quarters need 4 to 12% fewer and wait less for them.
// Every wave of a quarter tile streams all candidates, so the tile over the
// densest core ends four times as late; it needs enough other tiles to hide
// behind.  The gather's time, quarters against whole tiles, over slabs of 30k to
// 64M cells (1 to 32 halos, 4 to 32 slabs of 1024^2 to 4096^2 points), by the
// tiles per (row in a tile) in thousands: 0.67 to 1.51 below 13, 1.20 on average;
// 0.76 to 1.23 from 14 to 20; 0.84 on average from 25, at most 1.02 (1.06 in one
// launch of 0.16 ms).  32 slabs of 4096^2 through 64M 28.4 -> 23.0 ms, 16 through
// 32M 12.1 -> 9.9.  Views of any orientation close to a snapshot's centre have
// wide supports, whose nodes they need: 1.0 to 1.9.
bool quarter_tiles(uint64_t ntiles, uint64_t rows) {
  return double(ntiles) * double(ntiles) >= 25000.0 * double(rows);
}

// Clipped slab stacks of few tiles for their rows, where the quarters' densest
// tile sets the time: 8x8 tiles.  By the tiles per (row in a tile) in thousands:
// at 0.01 (8 slabs of 512^2 through 16M particles) 9.5 ms against 32.3 by
// quarters, at 0.06 (512^2, 1M) 1.0 against 2.0, at 0.16 (1024^2, 16M) 6.0 against
// 24.5; at 0.44 (512^2, 100k) 0.56 against 0.38, at 0.95 (1024^2, 1M) 3.3 against 1.8.
bool small_clip_tiles(uint64_t ntiles, uint64_t rows) {
  return double(ntiles) * double(ntiles) < 300.0 * double(rows);
}

void tile_grid(const sum_shape& ts, uint32_t lnx, uint32_t lny, uint32_t* tiles_x,
               uint32_t* ntiles) {
  *tiles_x = (lnx + ts.side - 1) / ts.side;
  *ntiles = *tiles_x * ((lny + ts.side - 1) / ts.side);
}

void launch_adjoint(const grid_view& g, const point_view& p, int kernel, const float* grad,
                    float scale, float norm, const float* ftab, const float* dtab, float* gw,
                    float* gh, float* gx, float* gy, hipStream_t s) {
  uint32_t tiles_x = 0, ntiles = 0;
  const sum_shape ts{p.n < kPointsFor16 ? 8 : 16};
  tile_grid(ts, p.lnx, p.lny, &tiles_x, &ntiles);
  if (!ntiles) return;
  adjoint_io io{grad, scale, norm, ftab, dtab, gw, gh, gx, gy};
  const dim3 grid{ntiles}, block{64 * kSumW};
  if (kernel == ILC_KERNEL_CUBIC) {
    if (!ftab || !dtab) fail(ILC_EINVAL, "cubic adjoint without its tables");
    if (ts.side == 8)
      hipLaunchKernelGGL((k_adjoint<8, 2>), grid, block, 0, s, g, p, tiles_x, ntiles, io);
    else
      hipLaunchKernelGGL((k_adjoint<16, 2>), grid, block, 0, s, g, p, tiles_x, ntiles, io);
  } else if (ts.side == 8) {
    hipLaunchKernelGGL((k_adjoint<8, 0>), grid, block, 0, s, g, p, tiles_x, ntiles, io);
  } else {
    hipLaunchKernelGGL((k_adjoint<16, 0>), grid, block, 0, s, g, p, tiles_x, ntiles, io);
  }
  ILC_HIP(hipGetLastError());
}

void launch_unpermute4(const uint32_t* perm, uint32_t n, const float* a, const float* b,
                       const float* c, const float* d, float* oa, float* ob, float* oc, float* od,
                       hipStream_t s) {
  if (!n) return;
  hipLaunchKernelGGL(k_unpermute4, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, perm, n, a,
                     b, c, d, oa, ob, oc, od);
  ILC_HIP(hipGetLastError());
}

int gather_batch_grid(int op, int kernel, const sum_shape& ts) {
  int dev = 0, cus = 0;
  ILC_HIP(hipGetDevice(&dev));
  ILC_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  const int per_cu = dispatch<batch_occ>(ts, op, kernel);
  return std::max(1, per_cu) * cus;
}

void launch_gather_batch(const view_desc* views, const uint2* items, const queue_segs& segs,
                         uint32_t* counters, int op, int kernel, const sum_shape& ts,
                         const float* cubic_table, int grid_blocks, hipStream_t s) {
  if (kernel == ILC_KERNEL_CUBIC && !cubic_table)
    fail(ILC_EINVAL, "cubic gather without its table");
  const float support = kernel == ILC_KERNEL_CUBIC ? 2.0f : 1.0f;
  // whole rounds of kQueues workgroups, so that every XCD gets the same number
  const int grid = std::max(kQueues, grid_blocks / kQueues * kQueues);
  dispatch<batch_launcher>(ts, op, kernel, views, items, segs, counters, cubic_table, support,
                           grid, s);
}

void launch_gather(const grid_view& g, const point_view& p, int op, int kernel,
                   const sum_shape& ts, double* acc, unsigned long long* counts,
                   const float* cubic_table, hipStream_t s) {
  const float support = kernel == ILC_KERNEL_CUBIC ? 2.0f : 1.0f;
  if (op == OP_COUNT) {
    // the count has its own tile shape: its cost is independent of the render's
    plain_launcher<16, OP_COUNT, 0, false>::run(g, p, nullptr, counts, nullptr, support, s);
    return;
  }
  if (kernel == ILC_KERNEL_CUBIC && !cubic_table)
    fail(ILC_EINVAL, "cubic gather without its table");
  dispatch<plain_launcher>(ts, op, kernel, g, p, acc, counts, cubic_table, support, s);
}

}  // namespace ilc
