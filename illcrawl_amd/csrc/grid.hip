// Particle-grid build on gfx950: bounding box, cell keys, stable LSD radix
// sort, cell offsets, per-cell max h, sorted SoA.
//
// Replaces particle_grid / smoothing_particle_grid (particle_grid.cpp:25-340,
// smoothing_particle_grid.cpp:29-54, particle_grid.cl:45-216, util.cl:24-49).
// The reference sorts ulong keys with boost::compute::sort_by_key (stable for
// integral keys) and then derives cell ranges; here a 8-bit-digit LSD radix
// sort on 32-bit keys gives the same permutation (each pass is a stable
// counting sort, ranks computed with wave64 ballots), and the cell ranges
// come from a scan of per-cell counts.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "common.hpp"
#include "cellmax.hpp"
#include "kernels.hpp"
#include "wave.hpp"

namespace ilc {

namespace {

__device__ inline float wave_min(float v) {
  for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ inline float wave_max(float v) {
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}
// orders this wave's LDS accesses (lanes read what others of the wave wrote)
__device__ inline void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// Descending h: the top 16 bits of its float pattern (h > 0, so the pattern
// orders like the value), reversed.
__device__ inline uint32_t h_order_key(float h) { return 0x7fffu - (__float_as_uint(h) >> 16); }
__device__ inline uint32_t wave_sum(uint32_t v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// lanes below the calling lane
__device__ inline uint64_t lanes_below() {
  const uint32_t lane = threadIdx.x & 63u;
  return lane == 0 ? 0ull : (~0ull >> (64u - lane));
}

__global__ void k_fill_u32(uint32_t* p, uint32_t v, uint64_t n) {
  for (uint64_t i = blockIdx.x * uint64_t(blockDim.x) + threadIdx.x; i < n;
       i += uint64_t(gridDim.x) * blockDim.x)
    p[i] = v;
}

struct fill_regions {
  uint32_t* p[4];
  uint64_t n[4];
};

// zeroes up to four arrays
__global__ __launch_bounds__(kBlock) void k_zero(fill_regions r) {
  const uint64_t i0 = blockIdx.x * uint64_t(kBlock) + threadIdx.x;
  const uint64_t step = uint64_t(gridDim.x) * kBlock;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    for (uint64_t i = i0; i < r.n[k]; i += step) r.p[k][i] = 0u;
}

// Per-block min/max of x, y, z, max h, max -h, and a count of invalid particles.
// Non-finite coordinates or w, and h that is not a positive normal float
// whose square stays finite, are invalid.
__global__ __launch_bounds__(kBlock) void k_bbox_partial(const float4* __restrict__ p4,
                                                          const float* __restrict__ h,
                                                          uint64_t n, float* __restrict__ part) {
  float mn[3] = {INFINITY, INFINITY, INFINITY}, mx[3] = {-INFINITY, -INFINITY, -INFINITY};
  float mh = 0.0f, lh = -INFINITY;
  uint32_t nbad = 0;
  for (uint64_t i = blockIdx.x * uint64_t(kBlock) + threadIdx.x; i < n;
       i += uint64_t(gridDim.x) * kBlock) {
    const float4 q = p4[i];
    const float hh = h[i];
    const bool ok = isfinite(q.x) && isfinite(q.y) && isfinite(q.z) && isfinite(q.w) &&
                    hh >= 1.1e-19f && hh <= 1.8e19f;
    if (!ok) {
      ++nbad;
      continue;
    }
    mn[0] = fminf(mn[0], q.x); mx[0] = fmaxf(mx[0], q.x);
    mn[1] = fminf(mn[1], q.y); mx[1] = fmaxf(mx[1], q.y);
    mn[2] = fminf(mn[2], q.z); mx[2] = fmaxf(mx[2], q.z);
    mh = fmaxf(mh, hh);
    lh = fmaxf(lh, -hh);
  }
  __shared__ float red[4][8];
  __shared__ uint32_t redb[4];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  float v[8] = {wave_min(mn[0]), wave_min(mn[1]), wave_min(mn[2]), wave_max(mx[0]),
                wave_max(mx[1]), wave_max(mx[2]), wave_max(mh), wave_max(lh)};
  uint32_t b = wave_sum(nbad);
  if (lane == 0) {
    for (int k = 0; k < 8; ++k) red[wave][k] = v[k];
    redb[wave] = b;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    float r[8];
    for (int k = 0; k < 8; ++k) r[k] = red[0][k];
    uint32_t bb = redb[0];
    for (int w = 1; w < 4; ++w) {
      for (int k = 0; k < 3; ++k) r[k] = fminf(r[k], red[w][k]);
      for (int k = 3; k < 8; ++k) r[k] = fmaxf(r[k], red[w][k]);
      bb += redb[w];
    }
    float* out = part + blockIdx.x * kBboxWords;
    for (int k = 0; k < 8; ++k) out[k] = r[k];
    out[8] = __uint_as_float(bb);
  }
}

__global__ __launch_bounds__(kBlock) void k_bbox_final(const float* __restrict__ part, int nparts,
                                                        bbox_result* __restrict__ out) {
  __shared__ float red[4][8];
  __shared__ uint32_t redb[4];
  float r[8] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY, 0.0f, -INFINITY};
  uint32_t bad = 0;
  for (int i = threadIdx.x; i < nparts; i += kBlock) {
    const float* p = part + i * kBboxWords;
    for (int k = 0; k < 3; ++k) r[k] = fminf(r[k], p[k]);
    for (int k = 3; k < 8; ++k) r[k] = fmaxf(r[k], p[k]);
    bad += __float_as_uint(p[8]);
  }
  for (int k = 0; k < 3; ++k) r[k] = wave_min(r[k]);
  for (int k = 3; k < 8; ++k) r[k] = wave_max(r[k]);
  bad = wave_sum(bad);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (lane == 0) {
    for (int k = 0; k < 8; ++k) red[wave][k] = r[k];
    redb[wave] = bad;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w) {
      for (int k = 0; k < 3; ++k) r[k] = fminf(r[k], red[w][k]);
      for (int k = 3; k < 8; ++k) r[k] = fmaxf(r[k], red[w][k]);
      bad += redb[w];
    }
    for (int k = 0; k < 3; ++k) {
      out->mn[k] = r[k];
      out->mx[k] = r[3 + k];
    }
    out->max_h = r[6];
    out->min_h = -r[7];
    out->bad = bad;
  }
}

// exclusive scan over the workgroup (kBlock threads)
__device__ inline uint32_t block_exclusive_scan(uint32_t v, uint32_t* total) {
  __shared__ uint32_t ws[4];
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

constexpr int kItems = 16;
constexpr int kTile = kBlock * kItems;  // 4096 keys per workgroup

// The active lanes of the wave whose `bits` low bits of d equal this lane's,
// among the valid ones.
__device__ inline uint64_t match_peers(uint32_t d, int bits, bool valid) {
  uint64_t peers = __ballot(valid);
  for (int b = 0; b < bits; ++b) {
    const bool bit = (d >> b) & 1u;
    const uint64_t m = __ballot(bit);
    peers &= bit ? m : ~m;
  }
  return peers;
}
__device__ inline uint64_t digit_peers(uint32_t d, bool valid) { return match_peers(d, 8, valid); }

// Counts digit d at position pos into its tile's counts hist[tile][256]
// (tiles of 1 << tile_log items, tile_bits bits of tile index), one add per
// distinct (tile, digit) of a wave.
__device__ inline void count_digit(uint32_t* __restrict__ hist, uint32_t pos, uint32_t d,
                                   int tile_log, int tile_bits) {
  const uint32_t bin = (pos >> tile_log) << 8 | d;
  const uint64_t peers = match_peers(bin, 8 + tile_bits, true);
  if ((peers & lanes_below()) == 0) atomicAdd(hist + bin, uint32_t(__popcll(peers)));
}

// keys[i] = cell of particle i (grid3d_generate_sort_keys,
// particle_grid.cl:96-112), hkeys[i] = its descending-h key (launch of the
// sort by (cell, descending h)).  Keys outside the grid (the reference writes
// out of bounds there) are counted in *err and clamped.  hist (may be NULL):
// the first digit of hkeys is counted into it.
__global__ __launch_bounds__(kBlock) void k_keys(const float4* __restrict__ p4,
                                                  const float* __restrict__ h, uint32_t n,
                                                  grid_params g, uint32_t* __restrict__ hkeys,
                                                  uint32_t* __restrict__ keys,
                                                  uint32_t* __restrict__ err,
                                                  uint32_t* __restrict__ hist, int tile_log,
                                                  int tile_bits) {
#pragma clang fp contract(off)
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const float4 q = p4[i];
  const float c[3] = {q.x, q.y, q.z};
  int32_t idx[3];
  bool ok = true;
  for (int a = 0; a < 3; ++a) {
    const float d = c[a] - g.minc[a];
    idx[a] = floor_to_int(d / g.cs[a]);
    ok = ok && idx[a] >= 0 && idx[a] < g.nc[a];
  }
  uint32_t key = 0;
  if (ok)
    key = uint32_t(idx[0]) + uint32_t(idx[1]) * uint32_t(g.nc[0]) +
          uint32_t(idx[2]) * uint32_t(g.nc[0]) * uint32_t(g.nc[1]);
  else
    atomicAdd(err, 1u);
  keys[i] = key;
  const uint32_t hk = h_order_key(h[i]);
  hkeys[i] = hk;
  if (hist) count_digit(hist, i, hk & 255u, tile_log, tile_bits);
}

// Per-tile digit counts, one LDS add per distinct digit of a wave (a digit
// with few distinct values would serialise a wave's 64 adds on one word).
// Layout hist[digit][tile], or hist[tile][digit] (tile_major).
template <int ITEMS>
__global__ __launch_bounds__(kBlock) void k_radix_hist(const uint32_t* __restrict__ keys,
                                                        uint32_t n, int shift, uint32_t ntiles,
                                                        uint32_t* __restrict__ hist,
                                                        int tile_major) {
  __shared__ uint32_t hh[256];
  hh[threadIdx.x] = 0;
  const uint32_t base = blockIdx.x * (kBlock * ITEMS);
  uint32_t k[ITEMS];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const uint32_t i = base + r * kBlock + threadIdx.x;
    k[r] = i < n ? keys[i] : 0u;
  }
  __syncthreads();
  const uint64_t below = lanes_below();
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const bool valid = base + r * kBlock + threadIdx.x < n;
    const uint32_t d = (k[r] >> shift) & 255u;
    const uint64_t peers = digit_peers(d, valid);
    if (valid && (peers & below) == 0) atomicAdd(&hh[d], uint32_t(__popcll(peers)));
  }
  __syncthreads();
  if (tile_major)
    hist[blockIdx.x * 256 + threadIdx.x] = hh[threadIdx.x];
  else
    hist[threadIdx.x * ntiles + blockIdx.x] = hh[threadIdx.x];
}

// One stable pass over an 8-bit digit of kin.  A wave ranks its own 64 *
// ITEMS consecutive items (lanes sharing a digit found with 8 ballots, running
// counts of its own in LDS: no barrier per row); the waves' counts then give
// every item its place in the tile ordered by digit, where it goes through
// LDS, so that each digit's items leave as one contiguous run.  (With shared
// counts and three barriers per row of 256 items a pass over 8k items took
// 13.6 us.)
// vin NULL: the values are the input positions.  kout NULL: the keys are not
// needed afterwards.  BP: a second value array moves with the first.
// SMALL: the counts are hist[tile][digit] of every tile, which the workgroup
// adds up itself (no scan launches); else hist holds the scanned counts
// hist[digit][tile].  With 4 items a thread the next pass's digit (of the key,
// or of the second value) is counted into next.hist (NULL: last pass).
struct radix_next {
  uint32_t* hist;
  int shift;
  int of_second;
  int tile_bits;
};
template <int ITEMS, bool BP, bool SMALL>
__global__ __launch_bounds__(kBlock) void k_radix_scatter(
    const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin,
    const uint32_t* __restrict__ bin, uint32_t* __restrict__ kout, uint32_t* __restrict__ vout,
    uint32_t* __restrict__ bout, uint32_t n, int shift, uint32_t ntiles,
    const uint32_t* __restrict__ hist, radix_next next) {
  constexpr int TILE = kBlock * ITEMS;
  constexpr bool COUNTING = ITEMS == 4;
  // the ordered tile, one array at a time (3 arrays of 4096 words at once
  // left 3 workgroups per CU: 170 us instead of 97 for a pass over 16M rows
  // with both values); before that, the sums of the tiles' counts
  __shared__ union {
    alignas(16) uint32_t so[TILE];
    uint32_t sum[SMALL ? 2 : 1][SMALL ? 4 : 1][256];  // each wave's sums, all tiles and those before
  } sm;
  auto& so = sm.so;
  __shared__ uint32_t gofs[256];
  __shared__ uint32_t wc[4][256];
  const uint32_t t = threadIdx.x;
  const int wave = t >> 6, lane = t & 63;
  const uint32_t tile0 = blockIdx.x * TILE;
  const uint32_t w0 = tile0 + uint32_t(wave) * (64 * ITEMS) + uint32_t(lane);
  uint32_t k[ITEMS], v[ITEMS], b[BP ? ITEMS : 1];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const uint32_t i = w0 + r * 64;
    k[r] = i < n ? kin[i] : 0u;
    v[r] = vin ? (i < n ? vin[i] : 0u) : i;
    if constexpr (BP) b[r] = i < n ? bin[i] : 0u;
  }
  // digit t's first position in the output
  uint32_t g0;
  if constexpr (SMALL) {
    // wave w adds up the counts of tiles w, w + 4, ..., four digits per lane
    const uint4* h4 = reinterpret_cast<const uint4*>(hist);
    uint4 all = make_uint4(0, 0, 0, 0), before = make_uint4(0, 0, 0, 0);
#pragma unroll 16
    for (uint32_t j = uint32_t(wave); j < ntiles; j += 4) {
      const uint4 c = h4[j * 64 + uint32_t(lane)];
      all.x += c.x;
      all.y += c.y;
      all.z += c.z;
      all.w += c.w;
      const bool b4 = j < blockIdx.x;
      before.x += b4 ? c.x : 0u;
      before.y += b4 ? c.y : 0u;
      before.z += b4 ? c.z : 0u;
      before.w += b4 ? c.w : 0u;
    }
    reinterpret_cast<uint4*>(sm.sum[0][wave])[lane] = all;
    reinterpret_cast<uint4*>(sm.sum[1][wave])[lane] = before;
    __syncthreads();
    uint32_t a1 = 0, b1 = 0;
    for (int w = 0; w < 4; ++w) {
      a1 += sm.sum[0][w][t];
      b1 += sm.sum[1][w][t];
    }
    uint32_t tot;
    g0 = block_exclusive_scan(a1, &tot) + b1;  // ends with a barrier
  } else {
    g0 = hist[uint64_t(t) * ntiles + blockIdx.x];
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) wc[wave][lane + 64 * j] = 0;
  wave_fence();
  const uint64_t below = lanes_below();
  uint32_t rank[ITEMS];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const bool valid = w0 + r * 64 < n;
    const uint32_t d = (k[r] >> shift) & 255u;
    const uint64_t peers = digit_peers(d, valid);
    const uint32_t old = wc[wave][d];
    rank[r] = old + uint32_t(__popcll(peers & below));
    wave_fence();
    if (valid && (peers & below) == 0) wc[wave][d] = old + uint32_t(__popcll(peers));
    wave_fence();
  }
  __syncthreads();
  {
    uint32_t c[4], cnt = 0;
    for (int w = 0; w < 4; ++w) {
      c[w] = wc[w][t];
      cnt += c[w];
    }
    uint32_t tot;
    uint32_t ls = block_exclusive_scan(cnt, &tot);
    gofs[t] = g0 - ls;
    for (int w = 0; w < 4; ++w) {
      wc[w][t] = ls;
      ls += c[w];
    }
  }
  __syncthreads();
  // place in the ordered tile, then the keys: item i of the tile goes to
  // gofs[digit] + i
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    rank[r] += wc[wave][(k[r] >> shift) & 255u];
    if (w0 + r * 64 < n) so[rank[r]] = k[r];
  }
  __syncthreads();
  const uint32_t nv = min(uint32_t(TILE), n - tile0);
  uint32_t pos[ITEMS];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const uint32_t i = t + r * kBlock;
    if (i < nv) {
      const uint32_t key = so[i];
      pos[r] = gofs[(key >> shift) & 255u] + i;
      if (kout) kout[pos[r]] = key;
      if constexpr (COUNTING)
        if (next.hist && !(BP && next.of_second))
          count_digit(next.hist, pos[r], (key >> next.shift) & 255u, 10, next.tile_bits);
    }
  }
  auto put = [&](const uint32_t* x, uint32_t* __restrict__ out, bool count) {
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r)
      if (w0 + r * 64 < n) so[rank[r]] = x[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
      const uint32_t i = t + r * kBlock;
      if (i < nv) {
        const uint32_t y = so[i];
        out[pos[r]] = y;
        if constexpr (COUNTING)
          if (count) count_digit(next.hist, pos[r], (y >> next.shift) & 255u, 10, next.tile_bits);
      }
    }
  };
  put(v, vout, false);
  if constexpr (BP) put(b, bout, COUNTING && next.hist && next.of_second);
}

// ---- exclusive scan of uint32 (reduce, scan of block sums, apply)


// A workgroup scans one tile of kTile words.  A whole tile of a 16-byte
// aligned array is read as kItems / 4 passes of one 16-byte vector per
// thread over consecutive 4 KB (coalesced); vector j * kBlock + t holds words
// 4 (j * kBlock + t) .. + 3 of the tile.  Other tiles read one word per thread
// and pass, the same way.
constexpr int kVecPasses = kItems / 4;
static_assert(kItems % 4 == 0, "whole vectors per thread");

__device__ inline bool whole_vec_tile(const void* p, uint64_t base, uint64_t n) {
  return base + kTile <= n && (reinterpret_cast<uintptr_t>(p) & 15u) == 0;
}

__global__ __launch_bounds__(kBlock) void k_scan_reduce(const uint32_t* __restrict__ in, uint64_t n,
                                                         uint32_t* __restrict__ sums) {
  const uint64_t b0 = uint64_t(blockIdx.x) * kTile;
  uint32_t s = 0;
  if (whole_vec_tile(in, b0, n)) {
    const uint4* v = reinterpret_cast<const uint4*>(in + b0);
#pragma unroll
    for (int j = 0; j < kVecPasses; ++j) {
      const uint4 q = v[j * kBlock + threadIdx.x];
      s += (q.x + q.y) + (q.z + q.w);
    }
  } else {
    for (int k = 0; k < kItems; ++k) {
      const uint64_t i = b0 + uint64_t(k) * kBlock + threadIdx.x;
      if (i < n) s += in[i];
    }
  }
  s = wave_sum(s);
  __shared__ uint32_t ws[4];
  if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) sums[blockIdx.x] = ws[0] + ws[1] + ws[2] + ws[3];
}

__global__ __launch_bounds__(kBlock) void k_scan_sums(uint32_t* __restrict__ sums, uint32_t nb) {
  uint32_t carry = 0;
  for (uint32_t c0 = 0; c0 < nb; c0 += kBlock * kItems) {
    const uint32_t base = c0 + threadIdx.x * kItems;
    uint32_t v[kItems], s = 0;
    for (int k = 0; k < kItems; ++k) {
      v[k] = base + k < nb ? sums[base + k] : 0u;
      s += v[k];
    }
    uint32_t tot;
    uint32_t off = block_exclusive_scan(s, &tot) + carry;
    for (int k = 0; k < kItems; ++k) {
      if (base + k < nb) sums[base + k] = off;
      off += v[k];
    }
    carry += tot;
    __syncthreads();
  }
}

__global__ __launch_bounds__(kBlock) void k_scan_apply(const uint32_t* __restrict__ in,
                                                        uint32_t* __restrict__ out, uint64_t n,
                                                        const uint32_t* __restrict__ sums) {
  const uint64_t b0 = uint64_t(blockIdx.x) * kTile;
  if (whole_vec_tile(in, b0, n) && (reinterpret_cast<uintptr_t>(out) & 15u) == 0) {
    // the tile's vectors in order, kBlock at a time: a block scan of the
    // vector sums of each pass, carried over the passes
    const uint4* vin = reinterpret_cast<const uint4*>(in + b0);
    uint4* vout = reinterpret_cast<uint4*>(out + b0);
    uint4 q[kVecPasses];
#pragma unroll
    for (int j = 0; j < kVecPasses; ++j) q[j] = vin[j * kBlock + threadIdx.x];
    uint32_t carry = sums[blockIdx.x];
#pragma unroll
    for (int j = 0; j < kVecPasses; ++j) {
      uint32_t tot;
      const uint32_t off = block_exclusive_scan((q[j].x + q[j].y) + (q[j].z + q[j].w), &tot) + carry;
      uint4 o;
      o.x = off;
      o.y = o.x + q[j].x;
      o.z = o.y + q[j].y;
      o.w = o.z + q[j].z;
      vout[j * kBlock + threadIdx.x] = o;
      carry += tot;
    }
    return;
  }
  const uint64_t base = b0 + uint64_t(threadIdx.x) * kItems;
  uint32_t v[kItems], s = 0;
  for (int k = 0; k < kItems; ++k) {
    v[k] = base + k < n ? in[base + k] : 0u;
    s += v[k];
  }
  uint32_t tot;
  uint32_t off = block_exclusive_scan(s, &tot) + sums[blockIdx.x];
  for (int k = 0; k < kItems; ++k) {
    if (base + k < n) out[base + k] = off;
    off += v[k];
  }
}

// A scan of at most 1024 * ITEMS words in one workgroup of 16 waves (one
// launch, not three).
constexpr uint64_t kOneScanMax = 1 << 15;
template <int ITEMS>
__global__ __launch_bounds__(1024) void k_scan_one(const uint32_t* in, uint32_t* out,
                                                    uint32_t n) {
  __shared__ uint32_t ws[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // word r of the thread: 64 lanes side by side, row r of the wave's block
  const uint32_t base = uint32_t(wave) * (64 * ITEMS) + uint32_t(lane);
  uint32_t v[ITEMS];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) v[r] = base + r * 64 < n ? in[base + r * 64] : 0u;
  uint32_t carry = 0;
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    uint32_t incl = v[r];
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(incl, o, 64);
      if (lane >= o) incl += y;
    }
    v[r] = carry + incl - v[r];
    carry += uint32_t(__builtin_amdgcn_readlane(int(incl), 63));
  }
  if (lane == 0) ws[wave] = carry;
  __syncthreads();
  uint32_t off = 0;
  for (int w = 0; w < wave; ++w) off += ws[w];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r)
    if (base + r * 64 < n) out[base + r * 64] = off + v[r];
}

// Sorted SoA: part[s] = (x, y, coef, 1/h^2) of particle perm[s], hs[s] = h.
// coef = w * C / h^2 with C the kernel's normalisation, so that the kernel
// value is coef * shape(r^2 / h^2).  For the projected quartic (shape
// s^2.5, s = 1 - r^2/h^2) the z slot holds c = coef^0.4 instead: the gather
// evaluates coef s^2.5 as (c s)^2.5, and the power belongs to the particle,
// not to each tile that lists it.
// The same pass derives the per-cell particle counts and max h
// (grid3d_determine_cells_begin/_end and grid3d_determine_max_per_cell,
// particle_grid.cl:114-216): keys are sorted, so the particles of a cell form
// one run; each wave reduces its part of every run (count, max h) and one
// lane per run segment adds it with an atomic (a cell spans at most a few
// waves, so there is no contention).  count and maxh_bits start at 0;
// maxh_bits may be null (no max h wanted).
__global__ __launch_bounds__(kBlock) void k_build_soa(const float4* __restrict__ p4,
                                                       const float* __restrict__ h,
                                                       const uint32_t* __restrict__ perm,
                                                       const uint32_t* __restrict__ skeys,
                                                       uint32_t n, float norm, bool pow04,
                                                       float4* __restrict__ part,
                                                       float* __restrict__ hs,
                                                       uint32_t* __restrict__ count,
                                                       uint32_t* __restrict__ maxh_bits,
                                                       const float2* __restrict__ zc_in,
                                                       float2* __restrict__ zc_out) {
  const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
  const bool valid = s < n;
  const uint32_t lane = threadIdx.x & 63u;
  uint32_t key = 0xffffffffu;
  float hh = 0.0f;
  if (valid) {
    const uint32_t i = perm[s];
    const float4 q = p4[i];
    hh = h ? h[i] : q.z;
    key = skeys[s];
    const float ih2 = 1.0f / (hh * hh);
    const float coef = q.w * (norm * ih2);
    part[s] = make_float4(q.x, q.y, pow04 ? powf(coef, 0.4f) : coef, ih2);
    hs[s] = hh;
    if (zc_out) zc_out[s] = zc_in[i];
  }
  // run heads within the wave
  const uint32_t prev = __shfl_up(key, 1, 64);
  const bool head = lane == 0 || prev != key;
  const uint64_t heads = __ballot(head);
  // end (exclusive) of this lane's run inside the wave
  const uint64_t above = lane == 63 ? 0ull : (heads & (~0ull << (lane + 1)));
  const uint32_t run_end = above ? uint32_t(__builtin_ctzll(above)) : 64u;
  // segmented max towards the run head
  float m = hh;
  for (uint32_t o = 1; o < 64; o <<= 1) {
    const float other = __shfl_down(m, o, 64);
    if (lane + o < run_end) m = fmaxf(m, other);
  }
  if (valid && head) {
    atomicAdd(&count[key], run_end - lane);
    if (maxh_bits) atomicMax(&maxh_bits[key], __float_as_uint(m));
  }
}

// Cell key of every input index (by_index[perm[j]] = key[j]), the input of a
// stable sort by cell key that gives the reference's order (stable by input
// index within a cell).
__global__ __launch_bounds__(kBlock) void k_keys_by_index(const uint32_t* __restrict__ key,
                                                          const uint32_t* __restrict__ perm,
                                                          uint32_t n,
                                                          uint32_t* __restrict__ by_index) {
  const uint32_t j = blockIdx.x * kBlock + threadIdx.x;
  if (j < n) by_index[perm[j]] = key[j];
}

// Reference layout of the grid for parity checks.
__global__ __launch_bounds__(kBlock) void k_export_cells(const uint32_t* __restrict__ start,
                                                          const uint32_t* __restrict__ maxh_bits,
                                                          uint32_t ncells, int2* cells2,
                                                          float* maxh) {
  const uint32_t c = blockIdx.x * kBlock + threadIdx.x;
  if (c >= ncells) return;
  const uint32_t b = start[c], e = start[c + 1];
  if (cells2) cells2[c] = e > b ? make_int2(int(b), int(e)) : make_int2(0, 0);
  if (maxh) maxh[c] = __uint_as_float(maxh_bits[c]);
}

inline uint32_t blocks_for(uint64_t n, uint64_t per) {
  return static_cast<uint32_t>((n + per - 1) / per);
}

// Per-cell max h without the sort (a slab group's shared grid: its views
// read only the per-cell max h and the grid parameters) of particles i0 .. i1 - 1:
// each particle's cell as k_keys computes it.  maxh_bits starts at 0;
// particles outside the grid count in err.
__global__ __launch_bounds__(kBlock) void k_cell_maxh(const float4* __restrict__ p4,
                                                      const float* __restrict__ h, uint32_t i0,
                                                      uint32_t i1, grid_params g,
                                                      uint32_t* __restrict__ maxh_bits,
                                                      uint32_t* __restrict__ err) {
#pragma clang fp contract(off)
  __shared__ unsigned long long slots[kMaxSlots];
  const uint32_t i = i0 + blockIdx.x * kBlock + threadIdx.x;
  bool ok = i < i1;
  uint32_t key = 0, hb = 0;
  if (ok) {
    const float4 q = p4[i];
    const float c[3] = {q.x, q.y, q.z};
    int32_t idx[3];
    for (int a = 0; a < 3; ++a) {
      const float d = c[a] - g.minc[a];
      idx[a] = floor_to_int(d / g.cs[a]);
      ok = ok && idx[a] >= 0 && idx[a] < g.nc[a];
    }
    if (ok) {
      key = uint32_t(idx[0]) + uint32_t(idx[1]) * uint32_t(g.nc[0]) +
            uint32_t(idx[2]) * uint32_t(g.nc[0]) * uint32_t(g.nc[1]);
      hb = __float_as_uint(h[i]);
    } else {
      atomicAdd(err, 1u);
    }
  }
  block_raise_max(maxh_bits, key, hb, ok, slots);
}

}  // namespace

void launch_fill_u32(uint32_t* p, uint32_t v, uint64_t n, hipStream_t s) {
  if (!n) return;
  uint32_t nb = blocks_for(n, kBlock);
  if (nb > 65536) nb = 65536;
  hipLaunchKernelGGL(k_fill_u32, dim3(nb), dim3(kBlock), 0, s, p, v, n);
  ILC_HIP(hipGetLastError());
}

void launch_zero(std::initializer_list<std::pair<uint32_t*, uint64_t>> regions, hipStream_t s) {
  fill_regions r{};
  uint64_t most = 0;
  int k = 0;
  for (const auto& x : regions) {
    ILC_REQUIRE(k < 4, "at most four regions");
    if (!x.second) continue;
    r.p[k] = x.first;
    r.n[k++] = x.second;
    most = std::max(most, x.second);
  }
  if (!k) return;
  uint32_t nb = blocks_for(most, kBlock);
  if (nb > 65536) nb = 65536;
  hipLaunchKernelGGL(k_zero, dim3(nb), dim3(kBlock), 0, s, r);
  ILC_HIP(hipGetLastError());
}

void launch_bbox(const float4* p4, const float* h, uint64_t n, float* partial, int nparts,
                 bbox_result* out, hipStream_t s) {
  hipLaunchKernelGGL(k_bbox_partial, dim3(nparts), dim3(kBlock), 0, s, p4, h, n, partial);
  ILC_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_bbox_final, dim3(1), dim3(kBlock), 0, s, partial, nparts, out);
  ILC_HIP(hipGetLastError());
}

void launch_cell_maxh(const float4* p4, const float* h, uint32_t n, const grid_params& g,
                      uint32_t* maxh_bits, uint32_t* err, hipStream_t s) {
  if (!n) return;
  for_ranges(n, [&](uint32_t i0, uint32_t i1) {
    hipLaunchKernelGGL(k_cell_maxh, dim3(blocks_for(i1 - i0, kBlock)), dim3(kBlock), 0, s, p4, h,
                       i0, i1, g, maxh_bits, err);
    ILC_HIP(hipGetLastError());
  });
}

void launch_keys(const float4* p4, const float* h, uint32_t n, const grid_params& g,
                 const radix_chain& c, uint32_t* err, hipStream_t s) {
  if (!n) return;
  hipLaunchKernelGGL(k_keys, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, s, p4, h, n, g,
                     c.a[c.in], c.b[c.in], err, c.counting ? c.hist : nullptr, c.tile_log,
                     c.tile_bits);
  ILC_HIP(hipGetLastError());
}

uint64_t scan_temp_words(uint64_t n) { return blocks_for(n, kTile) + 1; }

void launch_exclusive_scan(const uint32_t* in, uint32_t* out, uint64_t n, uint32_t* temp,
                           hipStream_t s) {
  if (!n) return;
  if (n <= kOneScanMax) {
    if (n <= 8192)
      hipLaunchKernelGGL(k_scan_one<8>, dim3(1), dim3(1024), 0, s, in, out, uint32_t(n));
    else
      hipLaunchKernelGGL(k_scan_one<32>, dim3(1), dim3(1024), 0, s, in, out, uint32_t(n));
    ILC_HIP(hipGetLastError());
    return;
  }
  const uint32_t nb = blocks_for(n, kTile);
  hipLaunchKernelGGL(k_scan_reduce, dim3(nb), dim3(kBlock), 0, s, in, n, temp);
  ILC_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(kBlock), 0, s, temp, nb);
  ILC_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_scan_apply, dim3(nb), dim3(kBlock), 0, s, in, out, n, temp);
  ILC_HIP(hipGetLastError());
}

// Arrays of up to kSmallTiles tiles are sorted without scan launches: every
// workgroup adds up all tiles' counts itself (256 KB at most, from L2).  Up
// to kCountingRows rows (tiles of 1024 items) the passes also count each
// other's digits with global atomics, one launch a pass: 8k rows 25 us a pass
// with count, scan and scatter launches, 7 now.  Above, a million atomics
// cost more than the count launch (1M rows: 33 us a pass against 27).
constexpr uint32_t kSmallTiles = 256;
constexpr uint64_t kCountingRows = 128u << 10;

namespace {
void radix_shape(uint64_t n, radix_chain* c) {
  c->counting = n <= kCountingRows;
  c->tile_log = c->counting ? 10 : 12;
  c->ntiles = static_cast<uint32_t>((n + (uint64_t(1) << c->tile_log) - 1) >> c->tile_log);
  c->small = c->ntiles <= kSmallTiles;
  c->tile_bits = 0;
  while ((1u << c->tile_bits) < c->ntiles && c->tile_bits < 31) ++c->tile_bits;
}
uint64_t radix_hist_words(const radix_chain& c, int passes) {
  if (c.counting) return uint64_t(passes) * c.ntiles * 256;
  return 256 * uint64_t(c.ntiles) + scan_temp_words(256 * uint64_t(c.ntiles));
}
constexpr int kMaxPasses = 8;
}  // namespace

uint64_t radix_chain_words(uint64_t n) {
  radix_chain c{};
  radix_shape(n, &c);
  return 4 * n + radix_hist_words(c, kMaxPasses);
}

radix_chain plan_radix_chain(uint32_t* b_out, uint32_t* v_out, uint64_t n, int bits_a, int bits_b,
                             uint32_t* temp) {
  radix_chain c{};
  c.n = static_cast<uint32_t>(n);
  c.pa = (bits_a + 7) / 8;
  c.pb = (bits_b + 7) / 8;
  ILC_REQUIRE(c.pa + c.pb <= kMaxPasses, "radix chain of %d passes", c.pa + c.pb);
  radix_shape(n, &c);
  c.b[0] = b_out;
  c.v[0] = v_out;
  c.a[0] = temp;
  c.a[1] = temp + n;
  c.b[1] = temp + 2 * n;
  c.v[1] = temp + 3 * n;
  c.hist = temp + 4 * n;
  c.hist_words = radix_hist_words(c, c.pa + c.pb);
  c.in = (c.pa + c.pb) & 1;
  return c;
}

std::pair<uint32_t*, uint64_t> radix_chain_zero(const radix_chain& c) {
  return {c.hist, c.counting ? c.hist_words : 0};
}

void launch_radix_chain(const radix_chain& c, bool iota, bool counted, hipStream_t s) {
  if (!c.n) return;
  const int passes = c.pa + c.pb;
  int cur = c.in;
  const dim3 grid{c.ntiles}, block{kBlock};
  auto key_of = [&](int p, int set) { return p < c.pa ? c.a[set] : c.b[set]; };
  auto shift_of = [&](int p) { return 8 * (p < c.pa ? p : p - c.pa); };
  if (c.counting && !counted && passes) {
    hipLaunchKernelGGL(k_radix_hist<4>, grid, block, 0, s, key_of(0, cur), c.n, 0, c.ntiles,
                       c.hist, 1);
    ILC_HIP(hipGetLastError());
  }
  for (int p = 0; p < passes; ++p) {
    const bool in_a = p < c.pa, last_a = p + 1 == c.pa, last = p + 1 == passes;
    const uint32_t* kin = key_of(p, cur);
    const uint32_t* vin = p == 0 && iota ? nullptr : c.v[cur];
    const uint32_t* bin = in_a ? c.b[cur] : nullptr;
    // the first keys are not read again once their passes are done
    uint32_t* kout = last_a ? nullptr : key_of(p, cur ^ 1);
    uint32_t* vout = c.v[cur ^ 1];
    uint32_t* bout = in_a ? c.b[cur ^ 1] : nullptr;
    const int shift = shift_of(p);
    uint32_t* hist = c.counting ? c.hist + uint64_t(p) * c.ntiles * 256 : c.hist;
    radix_next next{nullptr, 0, 0, c.tile_bits};
    if (c.counting) {
      if (!last) {
        next.hist = c.hist + uint64_t(p + 1) * c.ntiles * 256;
        next.shift = shift_of(p + 1);
        next.of_second = last_a ? 1 : 0;
      }
    } else {
      hipLaunchKernelGGL(k_radix_hist<16>, grid, block, 0, s, kin, c.n, shift, c.ntiles, hist,
                         c.small ? 1 : 0);
      ILC_HIP(hipGetLastError());
    }
    if (!c.small) {
      launch_exclusive_scan(hist, hist, uint64_t(256) * c.ntiles,
                            hist + 256 * uint64_t(c.ntiles), s);
    }
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, block, 0, s, kin, vin, bin, kout, vout, bout, c.n, shift,
                         c.ntiles, hist, next);
    };
    if (!c.small)
      in_a ? go(k_radix_scatter<16, true, false>) : go(k_radix_scatter<16, false, false>);
    else if (c.counting)
      in_a ? go(k_radix_scatter<4, true, true>) : go(k_radix_scatter<4, false, true>);
    else
      in_a ? go(k_radix_scatter<16, true, true>) : go(k_radix_scatter<16, false, true>);
    ILC_HIP(hipGetLastError());
    cur ^= 1;
  }
}

void launch_build_soa(const float4* p4, const float* h, const uint32_t* perm,
                      const uint32_t* skeys, uint32_t n, float norm, bool pow04, float4* part, float* hs,
                      uint32_t* count, uint32_t* maxh_bits, hipStream_t s, const float2* zc_in,
                      float2* zc_out) {
  if (!n) return;
  ILC_REQUIRE((zc_in == nullptr) == (zc_out == nullptr), "clip parameters need both arrays");
  hipLaunchKernelGGL(k_build_soa, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, s, p4, h, perm,
                     skeys, n, norm, pow04, part, hs, count, maxh_bits, zc_in, zc_out);
  ILC_HIP(hipGetLastError());
}

void launch_reference_perm(const uint32_t* key, const uint32_t* perm, uint32_t n, int key_bits,
                           uint32_t* out_perm, uint32_t* by_index, uint32_t* temp, hipStream_t s) {
  if (!n) return;
  const radix_chain c = plan_radix_chain(by_index, out_perm, n, 0, std::max(key_bits, 1), temp);
  launch_zero({radix_chain_zero(c)}, s);
  hipLaunchKernelGGL(k_keys_by_index, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, s, key, perm,
                     n, c.b[c.in]);
  ILC_HIP(hipGetLastError());
  launch_radix_chain(c, true, false, s);
}

void launch_export_cells(const uint32_t* start, const uint32_t* maxh_bits, uint32_t ncells,
                         int32_t* cells2, float* maxh, hipStream_t s) {
  if (!ncells) return;
  hipLaunchKernelGGL(k_export_cells, dim3(blocks_for(ncells, kBlock)), dim3(kBlock), 0, s, start,
                     maxh_bits, ncells, reinterpret_cast<int2*>(cells2), maxh);
  ILC_HIP(hipGetLastError());
}

}  // namespace ilc
