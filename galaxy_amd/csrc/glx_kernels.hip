// Device kernels of the MI355X LBVH gravity step (gfx950, wave64).
//
// Every kernel is segment-aware: it iterates over a table of Tile descriptors
// ({segment, first element, count}) with a grid-stride loop, so one launch covers
// one system or many uneven systems (batched/served forms) alike.
#include "glx_kernels.h"

#include <math.h>

#include <type_traits>

namespace glx {

// ----------------------------------------------------------------------------------
// helpers
// ----------------------------------------------------------------------------------

// Order-preserving map f64 -> u64 (non-NaN inputs): unsigned compare of the
// encodings equals f64 compare, so min/max reduce with integer atomics exactly.
__device__ __forceinline__ unsigned long long ord_enc(double x) {
  unsigned long long b = (unsigned long long)__double_as_longlong(x);
  return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}
__device__ __forceinline__ double ord_dec(unsigned long long k) {
  unsigned long long b = (k >> 63) ? (k & 0x7FFFFFFFFFFFFFFFull) : ~k;
  return __longlong_as_double((long long)b);
}

__device__ __forceinline__ double wave_min(double v) {
  for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o));
  return v;
}
__device__ __forceinline__ double wave_max(double v) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
  return v;
}
// Butterfly over the wave in registers (every lane ends with the same value; all lanes
// active), in the order xor 32, 16, 8, 4, 2, 1: the lane-half and row swaps, then, within a
// row of 16, rotations by 8 and by 4 (the values repeat with period 8 by then, so the
// rotation pairs a lane with the one at xor 4) and quad permutes. Two to three instructions
// a step, where __shfl_xor is an LDS permute and a wait.
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <class Op>
__device__ __forceinline__ float wave_all(float v, Op op) {
  const auto w = __builtin_amdgcn_permlane32_swap(__float_as_int(v), __float_as_int(v), false, false);
  v = op(__int_as_float(w[0]), __int_as_float(w[1]));
  const auto h = __builtin_amdgcn_permlane16_swap(__float_as_int(v), __float_as_int(v), false, false);
  v = op(__int_as_float(h[0]), __int_as_float(h[1]));
  v = op(v, dpp_move<0x128>(v));  // row_ror:8
  v = op(v, dpp_move<0x124>(v));  // row_ror:4
  v = op(v, dpp_move<0x4E>(v));   // quad_perm [2, 3, 0, 1]
  return op(v, dpp_move<0xB1>(v));  // quad_perm [1, 0, 3, 2]
}
__device__ __forceinline__ float wave_minf(float v) {
  return wave_all(v, [](float a, float b) { return fminf(a, b); });
}
__device__ __forceinline__ float wave_maxf(float v) {
  return wave_all(v, [](float a, float b) { return fmaxf(a, b); });
}
__device__ __forceinline__ float wave_sumf(float v) {
  return wave_all(v, [](float a, float b) { return a + b; });
}
__device__ __forceinline__ double wave_sum(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}
__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// Lanes below this one with their bit set in the wave mask m (v_mbcnt_lo/hi: two VALU
// instructions, against an AND and two bit counts on a per-lane mask).
__device__ __forceinline__ uint32_t lanes_below(unsigned long long m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Orders one wave's LDS accesses among its lanes (the hardware keeps a wave's LDS accesses
// in order): no block barrier, so one wave of a block may use it alone.
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// Block-wide exclusive scan of one u32 per thread, any blockDim that is a multiple of
// 64; sh_wave must hold blockDim / 64 entries (one per wave).
template <class T>
__device__ __forceinline__ T block_exclusive_scan(T v, T* sh_wave) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  T inc = v;
  for (int o = 1; o < 64; o <<= 1) {
    const T t = __shfl_up(inc, o);
    if (lane >= o) inc += t;
  }
  if (lane == 63) sh_wave[w] = inc;
  __syncthreads();
  T pre = 0;
  for (int k = 0; k < w; ++k) pre += sh_wave[k];
  __syncthreads();
  return pre + inc - v;
}

// Reduce a per-thread bbox over the block and fold it into the segment's atomic
// accumulators. min/max are exact and order-independent, so the result is
// bit-identical to a serial fold whatever the arrival order.
__device__ void block_commit_bbox(double lo[3], double hi[3], unsigned long long* bbox,
                                  double* sh /* 6 * waves */) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int a = 0; a < 3; ++a) {
    lo[a] = wave_min(lo[a]);
    hi[a] = wave_max(hi[a]);
  }
  if (lane == 0)
    for (int a = 0; a < 3; ++a) {
      sh[w * 6 + a] = lo[a];
      sh[w * 6 + 3 + a] = hi[a];
    }
  __syncthreads();
  if (threadIdx.x < 6) {
    const int a = threadIdx.x;
    double r = sh[a];
    for (int k = 1; k < kBlock / 64; ++k)
      r = (a < 3) ? fmin(r, sh[k * 6 + a]) : fmax(r, sh[k * 6 + a]);
    // a NaN-only tile contributes the neutral element (f64::min/max ignore NaN)
    if (!isnan(r)) {
      if (a < 3)
        atomicMin(&bbox[a], ord_enc(r));
      else
        atomicMax(&bbox[a], ord_enc(r));
    }
  }
  __syncthreads();
}

__device__ __forceinline__ void bbox_neutral(unsigned long long* bbox, int a) {
  bbox[a] = (a < 3) ? 0xFFFFFFFFFFFFFFFFull : 0ull;
}

// solvers/src/lbvh.rs:37-50
__device__ __forceinline__ uint32_t expand10(uint32_t v) {
  uint32_t x = v & 0x3ffu;
  x = (x | (x << 16)) & 0x030000ffu;
  x = (x | (x << 8)) & 0x0300f00fu;
  x = (x | (x << 4)) & 0x030c30c3u;
  x = (x | (x << 2)) & 0x09249249u;
  return x;
}
// the same spread over 21 bits (63-bit codes)
__device__ __forceinline__ uint64_t expand21(uint64_t x) {
  x &= 0x1fffffull;
  x = (x | (x << 32)) & 0x1f00000000ffffull;
  x = (x | (x << 16)) & 0x1f0000ff0000ffull;
  x = (x | (x << 8)) & 0x100f00f00f00f00full;
  x = (x | (x << 4)) & 0x10c30c30c30c30c3ull;
  x = (x | (x << 2)) & 0x1249249249249249ull;
  return x;
}

template <class K>
struct KeyTraits;
template <>
struct KeyTraits<uint32_t> {
  static constexpr int cell_bits = 10;  // solvers/src/lbvh.rs:32
  static constexpr int tie_base = 32;
  __device__ static uint32_t code(uint32_t x, uint32_t y, uint32_t z) {
    return expand10(x) | (expand10(y) << 1) | (expand10(z) << 2);
  }
  __device__ static int clz(uint32_t v) { return __clz((int)v); }
};
template <>
struct KeyTraits<uint64_t> {
  static constexpr int cell_bits = 21;  // the 63-bit refinement of solvers/src/lbvh.rs:29-31
  static constexpr int tie_base = 64;
  __device__ static uint64_t code(uint32_t x, uint32_t y, uint32_t z) {
    return expand21(x) | (expand21(y) << 1) | (expand21(z) << 2);
  }
  __device__ static int clz(uint64_t v) { return __clzll((long long)v); }
};

// solvers/src/lbvh.rs:110-120: the padded root cube of the segment's bbox, in f64
// with the reference's operation order (no contraction). origin = cube centre.
struct Bounds {
  double bmin[3], size, scale, origin[3];
};
__device__ Bounds seg_bounds(const unsigned long long* bbox, int cell_bits) {
#pragma clang fp contract(off)
  Bounds b;
  double lo[3], hi[3], ext[3];
  for (int a = 0; a < 3; ++a) {
    lo[a] = ord_dec(bbox[a]);
    hi[a] = ord_dec(bbox[3 + a]);
  }
  for (int a = 0; a < 3; ++a) {
    b.origin[a] = (lo[a] + hi[a]) * 0.5;
    ext[a] = hi[a] - lo[a];
  }
  const double maxe = fmax(ext[0], fmax(ext[1], ext[2]));
  const double half = fmax(0.5 * maxe, 1e-12) * (1.0 + 1e-9);
  for (int a = 0; a < 3; ++a) b.bmin[a] = b.origin[a] - half;
  b.size = 2.0 * half;
  b.scale = (double)(1u << cell_bits) / b.size;
  return b;
}

// solvers/src/lbvh.rs:56-64: floor, clamp below at 0 (NaN -> 0), saturate at the top cell.
__device__ __forceinline__ uint32_t quant_lane(double v, double top) {
  const double f = fmax(floor(v), 0.0);
  return f >= top ? (uint32_t)top : (uint32_t)f;
}

// A pointer from a SegDesc as a global-memory pointer: its loads and stores become
// global_load / global_store (counted by vmcnt only) instead of flat ones, which also
// hold up every LDS wait.
template <class T>
__device__ __forceinline__ const __attribute__((address_space(1))) T* gbl(const T* p) {
  return (const __attribute__((address_space(1))) T*)p;
}
template <class T>
__device__ __forceinline__ __attribute__((address_space(1))) T* gblw(T* p) {
  return (__attribute__((address_space(1))) T*)p;
}

// MI355X deals the blocks of a launch round-robin over its 8 XCDs (block b runs on XCD
// b % 8), each with its own L2. Walk groups that are neighbours in Morton order read
// nearly the same nodes, so the walks renumber blocks: in every span of 8 * kXcdRun
// blocks, the kXcdRun blocks an XCD receives take kXcdRun consecutive tiles. Neighbours
// then share an L2 while all XCDs still advance through the tiles together (a whole-range
// split per XCD leaves XCDs with unequal work). Launches use a grid that is a multiple of
// the span (xcd_grid); any other grid keeps the hardware order. Runs of 256 walk tiles
// (16,384 sorted bodies; an XCD holds about two runs at a time) measured fastest on the
// 512-system ensemble: walk -7% against runs of 8, -4.5% against 64, +0.6% at 512.
constexpr uint32_t kXcds = 8;
constexpr uint32_t kXcdRun = 256;
constexpr uint32_t kXcdSpan = kXcds * kXcdRun;

template <uint32_t RUN = kXcdRun>
__device__ __forceinline__ uint32_t xcd_block() {
  constexpr uint32_t span = kXcds * RUN;
  const uint32_t g = gridDim.x, b = blockIdx.x;
  if (g % span) return b;
  const uint32_t w = b % span;
  return (b - w) + (w % kXcds) * RUN + w / kXcds;
}

// The build kernels over sort tiles (2048 keys) take runs of 32 tiles per XCD, so that a
// system of up to 65,536 bodies is gathered, sorted and linked on one XCD and its random
// reads (positions by sorted index, codes in the binary searches) and scattered writes
// stay in that XCD's L2.
constexpr uint32_t kXcdBuildRun = 32;

// The per-target walk keeps short runs (64 blocks of kTargets bodies): its cost per target
// varies far more across a system (dense cores against halos), and long runs leave whole
// cores to one XCD (2^18 collision: 8.7 ms at runs of 16 to 128, 9.4 at 512, 13.4 at 4096).
constexpr uint32_t kXcdTargetRun = 64;

// ----------------------------------------------------------------------------------
// 1. bounding box
// ----------------------------------------------------------------------------------

__global__ void __launch_bounds__(kBlock)
k_bbox(const SegDesc* __restrict__ segs, const Tile* __restrict__ tiles, uint32_t ntiles) {
  __shared__ double sh[6 * (kBlock / 64)];
  for (uint32_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const SegDesc& s = segs[tl.seg];
    double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (uint32_t e = threadIdx.x; e < tl.count; e += kBlock) {
      const size_t i = tl.start + e;
      for (int a = 0; a < 3; ++a) {
        const double p = s.x[3 * i + a];
        lo[a] = fmin(lo[a], p);
        hi[a] = fmax(hi[a], p);
      }
    }
    block_commit_bbox(lo, hi, s.bbox, sh);
  }
}

// Opening half-kick with a(x_n), f64 drift (f32 on the all-f32 path), and the bbox of
// the drifted positions
// (core/src/integrator.rs:59-67; gpu/src/gpu_resident.rs:79-159).
__global__ void __launch_bounds__(kBlock)
k_kick_drift_bbox(const SegDesc* __restrict__ segs, const Tile* __restrict__ tiles,
                  uint32_t ntiles) {
#pragma clang fp contract(off)
  __shared__ double sh[6 * (kBlock / 64)];
  for (uint32_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const SegDesc& s = segs[tl.seg];
    const float h = s.half_dt;
    const double dt = s.dt;
    auto* sv = gblw(s.v);
    auto* sx = gblw(s.x);
    const auto* sa = gbl(s.acc);
    double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    if (s.precision == kPrecAbs32) {  // the all-f32 path drifts in f32 (tile-uniform)
      const float dt32 = (float)dt;
      for (uint32_t e = threadIdx.x; e < tl.count; e += kBlock) {
        const size_t i = tl.start + e;
        for (int a = 0; a < 3; ++a) {
          const float v = sv[3 * i + a] + sa[3 * i + a] * h;
          sv[3 * i + a] = v;
          const double x = (double)((float)sx[3 * i + a] + v * dt32);
          sx[3 * i + a] = x;
          lo[a] = fmin(lo[a], x);
          hi[a] = fmax(hi[a], x);
        }
      }
    } else {
      for (uint32_t e = threadIdx.x; e < tl.count; e += kBlock) {
        const size_t i = tl.start + e;
        for (int a = 0; a < 3; ++a) {
          const float v = sv[3 * i + a] + sa[3 * i + a] * h;
          sv[3 * i + a] = v;
          const double x = sx[3 * i + a] + (double)v * dt;
          sx[3 * i + a] = x;
          lo[a] = fmin(lo[a], x);
          hi[a] = fmax(hi[a], x);
        }
      }
    }
    block_commit_bbox(lo, hi, s.bbox, sh);
  }
}

// ----------------------------------------------------------------------------------
// 2. Morton encode (bit-exact with solvers/src/lbvh.rs:105-129; 63-bit variant with
//    2^21 cells per axis)
// ----------------------------------------------------------------------------------

template <class K>
__global__ void __launch_bounds__(kBlock)
k_encode(const SegDesc* __restrict__ segs, const Tile* __restrict__ tiles, uint32_t ntiles,
         uint32_t* __restrict__ lanes_out, int dst) {
#pragma clang fp contract(off)
  using T = KeyTraits<K>;
  const double top = (double)((1u << T::cell_bits) - 1u);
  for (uint32_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const SegDesc& s = segs[tl.seg];
    const Bounds b = seg_bounds(s.bbox, T::cell_bits);
    if (tl.start == 0 && threadIdx.x == 0) {
      s.bounds[0] = b.bmin[0];
      s.bounds[1] = b.bmin[1];
      s.bounds[2] = b.bmin[2];
      s.bounds[3] = b.size;
      s.bounds[4] = b.scale;
      // walk coordinates are relative to the cube centre, or absolute on the all-f32 path
      const bool abs32 = s.precision == kPrecAbs32;
      s.bounds[5] = abs32 ? 0.0 : b.origin[0];
      s.bounds[6] = abs32 ? 0.0 : b.origin[1];
      s.bounds[7] = abs32 ? 0.0 : b.origin[2];
    }
    auto* keys = gblw(static_cast<K*>(s.keys[dst]));  // the sort's first source buffer
    auto* vals = gblw(s.vals[dst]);
    auto* gend = gblw(s.gend);
    const auto* sx = gbl(s.x);
    for (uint32_t e = threadIdx.x; e < tl.count; e += kBlock) {
      const uint32_t i = tl.start + e;
      uint32_t l[3];
      for (int a = 0; a < 3; ++a)
        l[a] = quant_lane((sx[3 * (size_t)i + a] - b.bmin[a]) * b.scale, top);
      if (lanes_out) {
        lanes_out[3 * (size_t)i] = l[0];
        lanes_out[3 * (size_t)i + 1] = l[1];
        lanes_out[3 * (size_t)i + 2] = l[2];
      }
      keys[i] = T::code(l[0], l[1], l[2]);
      vals[i] = i;
      // a fresh build: group starts are marked by the tree build, which runs after the
      // sort (concurrently with the gather, which therefore leaves the marks alone)
      gend[i] = s.n == 1 ? 0u : kEnd;
      if (s.n == 1) s.parent_leaf[0] = kNoParent;
    }
  }
}

// Bounds only (used when keys are supplied by the caller).
__global__ void k_bounds(const SegDesc* __restrict__ segs, uint32_t nseg, int cell_bits) {
  const uint32_t sidx = blockIdx.x * blockDim.x + threadIdx.x;
  if (sidx >= nseg) return;
  const SegDesc& s = segs[sidx];
  const Bounds b = seg_bounds(s.bbox, cell_bits);
  for (int a = 0; a < 3; ++a) {
    s.bounds[a] = b.bmin[a];
    s.bounds[5 + a] = s.precision == kPrecAbs32 ? 0.0 : b.origin[a];
  }
  s.bounds[3] = b.size;
  s.bounds[4] = b.scale;
}

__global__ void __launch_bounds__(kBlock)
k_iota(const SegDesc* __restrict__ segs, const Tile* __restrict__ tiles, uint32_t ntiles,
       int dst) {
  for (uint32_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const SegDesc& s = segs[tl.seg];
    for (uint32_t e = threadIdx.x; e < tl.count; e += kBlock)
      s.vals[dst][tl.start + e] = tl.start + e;
  }
}

// ----------------------------------------------------------------------------------
// 3. stable LSD radix sort, segmented reduce-then-scan (per pass: upsweep, scan,
//    downsweep) with B-bit digits (B = 8, 9 or 10: 2^B bins). Pure integer; reproduces
//    the (code, index) order of solvers/src/lbvh.rs:143-147 because the payload starts
//    as iota and every pass is stable, whatever the digit width.
// ----------------------------------------------------------------------------------

template <class K, int B>
__global__ void __launch_bounds__(kSortThreads)
k_radix_upsweep(const SegDesc* __restrict__ segs, const Tile* __restrict__ tiles, uint32_t ntiles,
                uint32_t* __restrict__ tile_hist, int shift, int src) {
  constexpr int BINS = 1 << B;
  __shared__ uint32_t hist[BINS];
  for (uint32_t t = xcd_block<kXcdBuildRun>(); t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const SegDesc& s = segs[tl.seg];
    const auto* keys = gbl(static_cast<const K*>(s.keys[src]) + tl.start);
    for (int d = threadIdx.x; d < BINS; d += kSortThreads) hist[d] = 0;
    __syncthreads();
    for (uint32_t e = threadIdx.x; e < tl.count; e += kSortThreads)
      atomicAdd(&hist[(uint32_t)(keys[e] >> shift) & (BINS - 1)], 1u);
    __syncthreads();
    for (int d = threadIdx.x; d < BINS; d += kSortThreads)
      tile_hist[(size_t)t * BINS + d] = hist[d];
    __syncthreads();
  }
}

// Thread (digit d, group g) scans a run of a chunk's tiles, in place of their counts. A
// segment of one chunk takes one block and gets its final offsets, digit bases included. The
// tiles of a longer segment get offsets within their chunk, and the chunk its digit sums: at
// most kScanRows rows, which every block of the downsweep adds up; there a block takes
// kScanDigits digits of a chunk, in four runs. Bound by the latency of two or three dependent
// loads. With sums, their scan and their spreading in a launch each, a pass took five launches
// and the sort of 2^20 bodies with 63-bit keys 211 us, of 2,000,003 278 us; in three, 166 and
// 226 us.
constexpr int kScanThreads = 1024, kScanDigits = 256;

template <int B>
__global__ void __launch_bounds__(kScanThreads)
k_radix_scan(const Tile* __restrict__ chunks, uint32_t nchunks, uint32_t* tile_hist,
             uint32_t* __restrict__ chunk_rows) {
  constexpr uint32_t BINS = 1u << B, PARTS = BINS / kScanDigits, BATCH = 16;
  __shared__ uint32_t part[kScanThreads];
  __shared__ uint32_t base[BINS];
  __shared__ uint32_t shw[kScanThreads / 64];
  for (uint32_t b = blockIdx.x; b < nchunks * PARTS; b += gridDim.x) {
    const uint32_t c = b % nchunks, bins0 = b / nchunks * kScanDigits;  // chunks over all XCDs
    const Tile ch = chunks[c];
    const bool whole = ch.pad != 0;
    if (whole && bins0 != 0) continue;
    const uint32_t width = whole ? BINS : (uint32_t)kScanDigits, groups = kScanThreads / width;
    const uint32_t col = threadIdx.x & (width - 1), g = threadIdx.x / width;
    const uint32_t d = bins0 + col;
    const uint32_t per = (ch.count + groups - 1) / groups;
    const uint32_t first = min(ch.count, g * per), last = min(ch.count, first + per);
    uint32_t* row = tile_hist + (size_t)ch.start * BINS + d;
    uint32_t h[BATCH], run = 0;
    for (uint32_t t = first; t < last; t += BATCH) {  // BATCH loads in flight
#pragma unroll
      for (uint32_t q = 0; q < BATCH; ++q) h[q] = t + q < last ? row[(size_t)(t + q) * BINS] : 0u;
#pragma unroll
      for (uint32_t q = 0; q < BATCH; ++q) run += h[q];
    }
    part[threadIdx.x] = run;
    __syncthreads();
    uint32_t tot = 0;
    run = 0;
    for (uint32_t q = 0; q < groups; ++q) {
      const uint32_t v = part[q * width + col];
      tot += v;
      run += q < g ? v : 0u;
    }
    if (whole) {
      const uint32_t v = block_exclusive_scan(g == 0 ? tot : 0u, shw);
      if (g == 0) base[d] = v;
      __syncthreads();
      run += base[d];
    } else if (g == 0) {
      chunk_rows[(size_t)c * BINS + d] = tot;
    }
    for (uint32_t t = first; t < last; t += BATCH) {
      if (per > BATCH)
#pragma unroll
        for (uint32_t q = 0; q < BATCH; ++q) h[q] = t + q < last ? row[(size_t)(t + q) * BINS] : 0u;
#pragma unroll
      for (uint32_t q = 0; q < BATCH; ++q) {
        if (t + q < last) row[(size_t)(t + q) * BINS] = run;
        run += h[q];
      }
    }
    __syncthreads();
  }
}

// Bound by latency (keys, ranking ballots, LDS scatter) up to about 2^20 bodies, above by the
// scattered stores. CHUNKS: some segment of the launch has several scan chunks, and the block
// finds its offsets from their rows. That costs registers and a row per chunk: in launches of
// one-chunk segments only (512 systems, 7.9M bodies, 30-bit keys), the form without takes 57 us
// a pass, this one 68.
template <class K, int B, bool CHUNKS>
__global__ void __launch_bounds__(kSortThreads)
k_radix_downsweep(const SegDesc* __restrict__ segs, const Tile* __restrict__ tiles, uint32_t ntiles,
                  const uint32_t* __restrict__ tile_off, const uint32_t* __restrict__ chunk_rows,
                  int shift, int src) {
  constexpr int BINS = 1 << B;
  constexpr int W = kSortThreads / 64;
  constexpr int PER_WAVE = kSortTile / W;
  constexpr int R = (BINS + kSortThreads - 1) / kSortThreads;  // digits per thread, tile scan
  __shared__ uint32_t wcnt[W][BINS];
  __shared__ uint32_t dstart[BINS];  // the tile's digit starts
  __shared__ uint32_t goff[CHUNKS ? BINS : 1];  // from places in the tile to the segment's
  __shared__ K skey[kSortTile];
  __shared__ uint32_t sval[kSortTile];
  using Sum = std::conditional_t<CHUNKS, uint64_t, uint32_t>;
  __shared__ Sum shw[W];  // block_exclusive_scan's per-wave totals
  static_assert(kSortThreads % 64 == 0 && W * 64 == kSortThreads,
                "one shw entry per wave of the block");
  static_assert(R * kSortThreads >= BINS, "the tile scan covers every digit");
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const unsigned long long lt = (1ull << lane) - 1ull;
  for (uint32_t t = xcd_block<kXcdBuildRun>(); t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const SegDesc& s = segs[tl.seg];
    const auto* keys_in = gbl(static_cast<const K*>(s.keys[src]) + tl.start);
    const auto* vals_in = gbl(s.vals[src] + tl.start);
    auto* keys_out = gblw(static_cast<K*>(s.keys[src ^ 1]));
    auto* vals_out = gblw(s.vals[src ^ 1]);
    const auto* off = gbl(tile_off) + (size_t)t * BINS;
    for (int k = 0; k < W; ++k)
      for (int d = threadIdx.x; d < BINS; d += kSortThreads) wcnt[k][d] = 0;
    K key[kSortItems];
    uint32_t val[kSortItems], dig[kSortItems], rank[kSortItems];
#pragma unroll
    for (int j = 0; j < kSortItems; ++j) {
      const uint32_t e = w * PER_WAVE + j * 64 + lane;  // striped: index order = (j, lane)
      key[j] = e < tl.count ? keys_in[e] : (K)0;
      val[j] = e < tl.count ? vals_in[e] : 0u;
    }
    // thread q owns digits [q R, q R + R): their counts in the segment (all; none of a
    // segment of one chunk, whose offsets are final) and before the tile (pre)
    uint32_t all[R] = {}, pre[R] = {};
    if (CHUNKS && threadIdx.x * R < BINS) {
      const uint32_t nc = s.scan_chunks, mine = (t - s.sort_tile0) / s.scan_len;
      const auto* row = gbl(chunk_rows) + (size_t)s.scan_chunk0 * BINS + threadIdx.x * R;
#pragma unroll
      for (int r = 0; r < R; ++r) pre[r] = off[threadIdx.x * R + r];
      if (nc > 1)
#pragma unroll 8
        for (uint32_t c = 0; c < nc; ++c)
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const uint32_t v = row[(size_t)c * BINS + r];
            all[r] += v;
            pre[r] += c < mine ? v : 0u;
          }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kSortItems; ++j) {
      const bool valid = w * PER_WAVE + j * 64 + lane < tl.count;
      const uint32_t dd = valid ? ((uint32_t)(key[j] >> shift) & (BINS - 1)) : (uint32_t)BINS;
      // lanes holding the same digit (bit B separates the invalid tail)
      unsigned long long peers = ~0ull;
#pragma unroll
      for (int b = 0; b <= B; ++b) {
        const bool bit = (dd >> b) & 1u;
        const unsigned long long bal = __ballot(bit);
        peers &= bit ? bal : ~bal;
      }
      uint32_t r = 0;
      if (valid) {
        const uint32_t before = wcnt[w][dd];
        r = before + (uint32_t)__popcll(peers & lt);
        if ((peers & lt) == 0ull) wcnt[w][dd] = before + (uint32_t)__popcll(peers);
      }
      dig[j] = dd;
      rank[j] = r;
    }
    __syncthreads();
    {
      // per-wave starts, then the digit starts of the tile (and, above, of the segment)
      uint32_t tot[R];
      Sum sum = 0;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int d = threadIdx.x * R + r;
        uint32_t run = 0;
        for (int k = 0; k < W && d < BINS; ++k) {
          const uint32_t c = wcnt[k][d];
          wcnt[k][d] = run;
          run += c;
        }
        tot[r] = run;
        sum += (Sum)(((uint64_t)all[r] << 32) + run);
      }
      Sum first = block_exclusive_scan(sum, shw);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int d = threadIdx.x * R + r;
        if (d < BINS) {
          dstart[d] = (uint32_t)first;
          if (CHUNKS) goff[d] = (uint32_t)((uint64_t)first >> 32) + pre[r] - (uint32_t)first;
        }
        first += (Sum)(((uint64_t)all[r] << 32) + tot[r]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kSortItems; ++j) {
      if (dig[j] < (uint32_t)BINS) {
        const uint32_t p = dstart[dig[j]] + wcnt[w][dig[j]] + rank[j];
        skey[p] = key[j];
        sval[p] = val[j];
      }
    }
    __syncthreads();
    for (uint32_t p = threadIdx.x; p < tl.count; p += kSortThreads) {
      const K k = skey[p];
      const uint32_t d = (uint32_t)(k >> shift) & (BINS - 1);
      const uint32_t dst = CHUNKS ? goff[d] + p : off[d] + (p - dstart[d]);
      keys_out[dst] = k;
      vals_out[dst] = sval[p];
    }
    __syncthreads();
  }
}

// ----------------------------------------------------------------------------------
// 3b. the same sort for launches of few bodies: buckets by sampled splitters, then every
//     bucket sorted in one block's LDS. The digit passes above are bound there by their
//     launches, three a pass (63-bit keys, 2,000 bodies: 24 launches, 109 us; 30-bit keys,
//     16,384 bodies, 10-bit digits: 9 launches, 48 us). Here a system of up to kLocalDirect
//     bodies takes one launch and a larger one four, whatever the key width: 23 us, and 38 us
//     in all; 63-bit keys, 100,003 bodies: 127 -> 69 us. The digits that no two keys of a
//     bucket differ in are left out. Equal keys keep index order: splitters compare (key,
//     index), and every scatter is stable.
// ----------------------------------------------------------------------------------

constexpr int kLocalThreads = 1024, kLocalItems = 6;
constexpr uint32_t kLocalCap = kLocalThreads * kLocalItems;  // bodies of a bucket in LDS
constexpr uint32_t kOversample = 16;  // samples per bucket
constexpr uint32_t kSampleMax = kSplitMax * kOversample;
// A bucket holds kLocalBucket bodies on average; three times that exceeds the cap about once
// in 1e8 (a Poisson count of 48 below 16), and such a bucket is sorted through memory.
static_assert(kLocalBucket * 3 <= kLocalCap && kLocalDirect <= kLocalCap &&
                  kLocalMax <= kSplitMax * kLocalBucket && kSampleMax <= 1024,
              "bucket sizes");

__host__ __device__ static inline uint32_t bucket_count(uint32_t n) {
  return n <= kLocalDirect ? 1u : (n + kLocalBucket - 1) / kLocalBucket;
}
uint32_t local_buckets(uint32_t n) { return bucket_count(n); }

// Splitters of each system above kLocalDirect bodies: kOversample samples a bucket, one from
// each of as many index strata, sorted by (key, index); every kOversample-th splits.
template <class K>
__global__ void __launch_bounds__(1024)
k_split(const SegDesc* __restrict__ segs, uint32_t nseg, int src, SplitTable st) {
  __shared__ K key[kSampleMax];
  __shared__ uint32_t idx[kSampleMax];
  for (uint32_t sidx = blockIdx.x; sidx < nseg; sidx += gridDim.x) {
    const SegDesc& s = segs[sidx];
    const uint32_t n = s.n;
    if (n <= kLocalDirect) continue;
    const uint32_t nb = bucket_count(n), ns = nb * kOversample, t = threadIdx.x;
    uint32_t size = 64;
    while (size < ns) size *= 2;
    if (t < size) {
      K v = ~(K)0;
      uint32_t i = 0xFFFFFFFFu;
      if (t < ns) {
        const uint32_t a = (uint32_t)((uint64_t)n * t / ns), b = (uint32_t)((uint64_t)n * (t + 1) / ns);
        uint32_t h = t * 2654435761u + 0x9E3779B9u;  // a place in the stratum, not periodic
        h ^= h >> 15;
        h *= 0x85EBCA6Bu;
        i = a + (h >> 8) % (b - a);
        v = gbl(static_cast<const K*>(s.keys[src]))[i];
      }
      key[t] = v;
      idx[t] = i;
    }
    __syncthreads();
    for (uint32_t k = 2; k <= size; k *= 2)  // bitonic sort
      for (uint32_t j = k / 2; j > 0; j /= 2) {
        const uint32_t q = t ^ j;
        if (t < size && q > t) {
          const K a = key[t], b = key[q];
          const uint32_t ia = idx[t], ib = idx[q];
          const bool greater = a > b || (a == b && ia > ib);
          if (greater == ((t & k) == 0u)) {
            key[t] = b;
            key[q] = a;
            idx[t] = ib;
            idx[q] = ia;
          }
        }
        // pairs up to 32 apart lie in one wave, as do the next step's if it stays below 64
        if (j > 32 || (j == 1 && k >= 64)) __syncthreads();
        else wave_lds_order();
      }
    __syncthreads();
    if (t < kSplitMax) {  // splitter t opens bucket t + 1; the rest are never reached
      const bool real = t + 1 < nb;
      st.key[(size_t)sidx * kSplitMax + t] =
          real ? (uint64_t)key[(t + 1) * kOversample] : ~0ull;
      st.idx[(size_t)sidx * kSplitMax + t] = real ? idx[(t + 1) * kOversample] : 0xFFFFFFFFu;
    }
    __syncthreads();
  }
}

// Splitters of a system in LDS, and the bucket of (key, index): the splitters not above it.
struct Splitters {
  uint64_t key[kSplitMax];
  uint32_t idx[kSplitMax];
};
__device__ __forceinline__ uint32_t bucket_of(const Splitters& sp, uint64_t key, uint32_t i) {
  uint32_t b = 0;
#pragma unroll
  for (uint32_t step = kSplitMax / 2; step > 0; step /= 2) {
    const uint64_t k = sp.key[b + step - 1];
    const uint32_t j = sp.idx[b + step - 1];
    if (k < key || (k == key && j <= i)) b += step;
  }
  return b;
}

// Bodies per bucket of each tile of the systems that are split (row tile of hist).
template <class K>
__global__ void __launch_bounds__(kSortThreads)
k_bucket_count(const SegDesc* __restrict__ segs, const Tile* __restrict__ tiles, uint32_t ntiles,
               uint32_t* __restrict__ hist, int src, SplitTable st) {
  __shared__ Splitters sp;
  __shared__ uint32_t cnt[kSplitMax];
  for (uint32_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const SegDesc& s = segs[tl.seg];
    if (s.n <= kLocalDirect) continue;
    if (threadIdx.x < kSplitMax) {
      sp.key[threadIdx.x] = st.key[(size_t)tl.seg * kSplitMax + threadIdx.x];
      sp.idx[threadIdx.x] = st.idx[(size_t)tl.seg * kSplitMax + threadIdx.x];
      cnt[threadIdx.x] = 0u;
    }
    __syncthreads();
    const auto* keys = gbl(static_cast<const K*>(s.keys[src]));
    for (uint32_t e = threadIdx.x; e < tl.count; e += kSortThreads)
      atomicAdd(&cnt[bucket_of(sp, keys[tl.start + e], tl.start + e)], 1u);
    __syncthreads();
    if (threadIdx.x < kSplitMax) hist[(size_t)t * kSplitMax + threadIdx.x] = cnt[threadIdx.x];
    __syncthreads();
  }
}

// Stable scatter of each tile into its system's buckets (buffer src to the other). A tile's
// block adds the tiles' counts itself: at most kLocalMax / kSortTile rows of kSplitMax.
// The first tile's block publishes where the buckets start.
template <class K>
__global__ void __launch_bounds__(kSortThreads)
k_bucket_scatter(const SegDesc* __restrict__ segs, const Tile* __restrict__ tiles, uint32_t ntiles,
                 const uint32_t* __restrict__ hist, int src, SplitTable st) {
  constexpr int W = kSortThreads / 64, PER_WAVE = kSortTile / W;
  static_assert(kSplitMax == 64, "one wave scans the buckets; six ballots rank them");
  __shared__ Splitters sp;
  __shared__ uint32_t all[W][kSplitMax], bef[W][kSplitMax];  // counts of all, of earlier tiles
  __shared__ uint32_t wcnt[W][kSplitMax], dst0[kSplitMax];
  const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
  for (uint32_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const SegDesc& s = segs[tl.seg];
    if (s.n <= kLocalDirect) continue;
    if (w == 0) {
      sp.key[lane] = st.key[(size_t)tl.seg * kSplitMax + lane];
      sp.idx[lane] = st.idx[(size_t)tl.seg * kSplitMax + lane];
    }
    wcnt[w][lane] = 0u;
    uint32_t a = 0, b = 0;
#pragma unroll 4
    for (uint32_t q = s.sort_tile0 + w; q < s.sort_tile0 + s.sort_tiles; q += W) {
      const uint32_t c = hist[(size_t)q * kSplitMax + lane];
      a += c;
      b += q < t ? c : 0u;
    }
    all[w][lane] = a;
    bef[w][lane] = b;
    __syncthreads();
    const auto* keys_in = gbl(static_cast<const K*>(s.keys[src]));
    const auto* vals_in = gbl(s.vals[src]);
    auto* keys_out = gblw(static_cast<K*>(s.keys[src ^ 1]));
    auto* vals_out = gblw(s.vals[src ^ 1]);
    K key[kSortItems];
    uint32_t val[kSortItems], dig[kSortItems], rank[kSortItems];
#pragma unroll
    for (int j = 0; j < kSortItems; ++j) {
      const uint32_t e = w * PER_WAVE + j * 64 + lane;  // striped: index order = (j, lane)
      const bool valid = e < tl.count;
      key[j] = valid ? keys_in[tl.start + e] : (K)0;
      val[j] = valid ? vals_in[tl.start + e] : 0u;
      const uint32_t d = valid ? bucket_of(sp, key[j], tl.start + e) : 64u;
      unsigned long long peers = ~0ull;
#pragma unroll
      for (int q = 0; q <= 6; ++q) {
        const unsigned long long bal = __ballot((d >> q) & 1u);
        peers &= (d >> q) & 1u ? bal : ~bal;
      }
      const uint32_t below = lanes_below(peers);
      uint32_t r = 0;
      if (valid) {
        const uint32_t before = wcnt[w][d];
        r = before + below;
        if (below == 0u) wcnt[w][d] = before + (uint32_t)__popcll(peers);
      }
      dig[j] = d;
      rank[j] = r;
    }
    __syncthreads();
    if (w == 0) {  // bucket starts, then each wave's first place per bucket
      uint32_t tot = 0, pre = 0;
      for (int q = 0; q < W; ++q) {
        tot += all[q][lane];
        pre += bef[q][lane];
      }
      uint32_t inc = tot;
      for (int o = 1; o < 64; o <<= 1) {
        const uint32_t v = __shfl_up(inc, o);
        if ((int)lane >= o) inc += v;
      }
      const uint32_t start = inc - tot;
      if (t == s.sort_tile0) {
        st.start[(size_t)tl.seg * (kSplitMax + 1) + lane] = start;
        if (lane == 63) st.start[(size_t)tl.seg * (kSplitMax + 1) + 64] = inc;
      }
      dst0[lane] = start + pre;
      uint32_t run = 0;
      for (int q = 0; q < W; ++q) {
        const uint32_t c = wcnt[q][lane];
        wcnt[q][lane] = run;
        run += c;
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kSortItems; ++j) {
      if (dig[j] < 64u) {
        const uint32_t p = dst0[dig[j]] + wcnt[w][dig[j]] + rank[j];
        keys_out[p] = key[j];
        vals_out[p] = val[j];
      }
    }
    __syncthreads();
  }
}

// LDS of the local sort.
template <class K>
struct LocalSort {
  static constexpr int W = kLocalThreads / 64;
  K key[kLocalCap];
  uint32_t val[kLocalCap];
  uint32_t wcnt[W][256];
  uint32_t dstart[256];
  uint32_t shw[W];
  unsigned long long diff;
};

// Rank of this lane's item with digit d (256: none) among the wave's items so far; the
// wave's counters in `cnt` move on.
__device__ __forceinline__ uint32_t wave_rank8(uint32_t d, uint32_t* cnt) {
  unsigned long long peers = ~0ull;
#pragma unroll
  for (int b = 0; b <= 8; ++b) {
    const unsigned long long bal = __ballot((d >> b) & 1u);
    peers &= (d >> b) & 1u ? bal : ~bal;
  }
  const uint32_t below = lanes_below(peers);
  uint32_t r = 0;
  if (d < 256u) {
    const uint32_t before = cnt[d];
    r = before + below;
    if (below == 0u) cnt[d] = before + (uint32_t)__popcll(peers);
  }
  return r;
}

// The waves' counts per digit to their first places within the digit, and in dstart the
// digits' starts within their quarter (64 digits), whose totals go to shw[0..3].
template <class K>
__device__ __forceinline__ void local_starts(LocalSort<K>& L) {
  if (threadIdx.x >= 256u) return;
  const uint32_t d = threadIdx.x, lane = d & 63u;
  uint32_t c[LocalSort<K>::W], tot = 0;
#pragma unroll
  for (int q = 0; q < LocalSort<K>::W; ++q) c[q] = L.wcnt[q][d];
#pragma unroll
  for (int q = 0; q < LocalSort<K>::W; ++q) {
    L.wcnt[q][d] = tot;
    tot += c[q];
  }
  uint32_t inc = tot;
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t v = __shfl_up(inc, o);
    if ((int)lane >= o) inc += v;
  }
  L.dstart[d] = inc - tot;
  if (lane == 63u) L.shw[d >> 6] = inc;
}

// A bucket beyond the LDS: its range of the buffers sorted by digit passes of this block
// alone, chunks of kLocalThreads one after the other. Ends in the buffer it starts in (an
// even number of passes).
template <class K>
__device__ void bucket_through_memory(const SegDesc& s, LocalSort<K>& L, uint32_t lo,
                                      uint32_t hi, int src) {
  const uint32_t w = threadIdx.x >> 6;
  for (uint32_t shift = 0; shift < 8 * sizeof(K); shift += 8, src ^= 1) {
    const auto* keys = gbl(static_cast<const K*>(s.keys[src]));
    const auto* vals = gbl(s.vals[src]);
    auto* keys_out = gblw(static_cast<K*>(s.keys[src ^ 1]));
    auto* vals_out = gblw(s.vals[src ^ 1]);
    for (uint32_t d = threadIdx.x; d < 256u; d += kLocalThreads) L.val[d] = 0u;
    __syncthreads();
    for (uint32_t p = lo + threadIdx.x; p < hi; p += kLocalThreads)
      atomicAdd(&L.val[(uint32_t)(keys[p] >> shift) & 255u], 1u);
    __syncthreads();
    const uint32_t c = threadIdx.x < 256u ? L.val[threadIdx.x] : 0u;
    const uint32_t first = block_exclusive_scan(c, L.shw);
    if (threadIdx.x < 256u) L.val[threadIdx.x] = lo + first;  // next place per digit
    __syncthreads();
    for (uint32_t p0 = lo; p0 < hi; p0 += kLocalThreads) {
      for (uint32_t e = threadIdx.x; e < LocalSort<K>::W * 256u; e += kLocalThreads)
        L.wcnt[e >> 8][e & 255u] = 0u;
      __syncthreads();
      const uint32_t p = p0 + threadIdx.x;
      const bool valid = p < hi;
      const K k = valid ? keys[p] : (K)0;
      const uint32_t v = valid ? vals[p] : 0u;
      const uint32_t d = valid ? (uint32_t)(k >> shift) & 255u : 256u;
      const uint32_t r = wave_rank8(d, L.wcnt[w]);
      __syncthreads();
      uint32_t tot = 0;
      if (threadIdx.x < 256u) {
        tot = L.val[threadIdx.x];
        for (int q = 0; q < LocalSort<K>::W; ++q) {
          const uint32_t x = L.wcnt[q][threadIdx.x];
          L.wcnt[q][threadIdx.x] = tot;
          tot += x;
        }
      }
      __syncthreads();
      if (valid) {
        keys_out[L.wcnt[w][d] + r] = k;
        vals_out[L.wcnt[w][d] + r] = v;
      }
      if (threadIdx.x < 256u) L.val[threadIdx.x] = tot;
      __syncthreads();
    }
    __threadfence_block();  // this block reads the range it has written
    __syncthreads();
  }
}

// One bucket per block into buffer 0: bucket `start` of system `seg` (Tile: pad = 1, split
// into buffer src ^ 1) or a whole system of up to kLocalDirect bodies (pad = 0, in buffer src).
template <class K>
__global__ void __launch_bounds__(kLocalThreads)
k_sort_local(const SegDesc* __restrict__ segs, const Tile* __restrict__ buckets, uint32_t nbuckets,
             int src, SplitTable st) {
  __shared__ LocalSort<K> L;
  const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
  for (uint32_t q = blockIdx.x; q < nbuckets; q += gridDim.x) {
    const Tile bk = buckets[q];
    const SegDesc& s = segs[bk.seg];
    uint32_t lo = 0, hi = s.n;
    int from = src;
    if (bk.pad) {
      lo = st.start[(size_t)bk.seg * (kSplitMax + 1) + bk.start];
      hi = st.start[(size_t)bk.seg * (kSplitMax + 1) + bk.start + 1];
      from = src ^ 1;
    }
    const uint32_t cnt = hi - lo;
    auto* keys_out = gblw(static_cast<K*>(s.keys[0]));
    auto* vals_out = gblw(s.vals[0]);
    if (cnt > kLocalCap) {
      bucket_through_memory<K>(s, L, lo, hi, from);
      if (from != 0)
        for (uint32_t p = lo + threadIdx.x; p < hi; p += kLocalThreads) {
          keys_out[p] = gbl(static_cast<const K*>(s.keys[from]))[p];
          vals_out[p] = gbl(s.vals[from])[p];
        }
      continue;
    }
    const auto* keys_in = gbl(static_cast<const K*>(s.keys[from])) + lo;
    const auto* vals_in = gbl(s.vals[from]) + lo;
    const int items = (int)((cnt + kLocalThreads - 1) / kLocalThreads);
    const uint32_t base = w * 64u * (uint32_t)items + lane;  // striped: order = (wave, item, lane)
    K key[kLocalItems];
    uint32_t val[kLocalItems];
    if (threadIdx.x == 0) L.diff = 0ull;
    __syncthreads();
    unsigned long long diff = 0ull;
    const K k0 = cnt ? keys_in[0] : (K)0;
#pragma unroll
    for (int j = 0; j < kLocalItems; ++j) {
      const uint32_t e = base + 64u * j;
      const bool valid = j < items && e < cnt;
      key[j] = valid ? keys_in[e] : (K)0;
      val[j] = valid ? vals_in[e] : 0u;
      if (valid) diff |= (unsigned long long)(key[j] ^ k0);
    }
    for (int o = 32; o > 0; o >>= 1) diff |= __shfl_xor(diff, o);
    if (lane == 0 && diff) atomicOr(&L.diff, diff);
    __syncthreads();
    diff = L.diff;
    // a wave clears its own counters: by the time it does, every wave is past the scatter
    // that reads them
    auto clear = [&] {
#pragma unroll
      for (int c = 0; c < 4; ++c) L.wcnt[w][64 * c + lane] = 0u;
    };
    clear();
    for (uint32_t shift = 0; shift < 8 * sizeof(K); shift += 8) {
      if (((diff >> shift) & 255ull) == 0ull) continue;  // no two keys differ here
      uint32_t dig[kLocalItems], rank[kLocalItems];
      wave_lds_order();
#pragma unroll
      for (int j = 0; j < kLocalItems; ++j) {
        dig[j] = 256u;
        if (j < items) {
          const bool valid = base + 64u * j < cnt;
          dig[j] = valid ? (uint32_t)(key[j] >> shift) & 255u : 256u;
          rank[j] = wave_rank8(dig[j], L.wcnt[w]);
        }
      }
      __syncthreads();
      local_starts(L);
      __syncthreads();
      const uint32_t q1 = L.shw[0], q2 = q1 + L.shw[1], q3 = q2 + L.shw[2];
#pragma unroll
      for (int j = 0; j < kLocalItems; ++j)
        if (dig[j] < 256u) {
          const uint32_t quarter = dig[j] >> 6;
          const uint32_t p = L.dstart[dig[j]] + L.wcnt[w][dig[j]] + rank[j] +
                             (quarter == 0u ? 0u : (quarter == 1u ? q1 : (quarter == 2u ? q2 : q3)));
          L.key[p] = key[j];
          L.val[p] = val[j];
        }
      __syncthreads();
      clear();
#pragma unroll
      for (int j = 0; j < kLocalItems; ++j) {
        const uint32_t e = base + 64u * j;
        if (j < items && e < cnt) {
          key[j] = L.key[e];
          val[j] = L.val[e];
        }
      }
    }
#pragma unroll
    for (int j = 0; j < kLocalItems; ++j) {
      const uint32_t e = base + 64u * j;
      if (j < items && e < cnt) {
        keys_out[lo + e] = key[j];
        vals_out[lo + e] = val[j];
      }
    }
    __syncthreads();
  }
}

// ----------------------------------------------------------------------------------
// 4. gather sorted leaves: origin-relative f32 position + mass
//    (solvers/src/lbvh.rs:453-456; gpu/src/fused_core.rs:32-45)
// ----------------------------------------------------------------------------------

// Sorted leaves of a fresh build, or the positions of a cached tree refreshed in its
// existing leaf order (the same arithmetic). 1024 threads per 2048-element tile keep more
// of the random reads in flight.
constexpr int kGatherThreads = 1024;

__global__ void __launch_bounds__(kGatherThreads)
k_gather(const SegDesc* __restrict__ segs, const Tile* __restrict__ tiles, uint32_t ntiles) {
  for (uint32_t t = xcd_block<kXcdBuildRun>(); t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const SegDesc& s = segs[tl.seg];
    const double o0 = s.bounds[5], o1 = s.bounds[6], o2 = s.bounds[7];
    for (uint32_t e = threadIdx.x; e < tl.count; e += kGatherThreads) {
      const uint32_t k = tl.start + e;
      const size_t i = min(gbl(s.vals[0])[k], s.n - 1);
      const auto* x = gbl(s.x);
      auto* lp = gblw(reinterpret_cast<float*>(s.leaf)) + 4 * (size_t)k;
      lp[0] = (float)(x[3 * i] - o0);
      lp[1] = (float)(x[3 * i + 1] - o1);
      lp[2] = (float)(x[3 * i + 2] - o2);
      lp[3] = (float)gbl(s.m)[i];
    }
  }
}

// ----------------------------------------------------------------------------------
// 5. Karras radix-tree build (solvers/src/lbvh.rs:153-240,276-306), signed int
//    indices; each internal node also records its leaf range.
// ----------------------------------------------------------------------------------

// The sorted keys of a tile and kKarrasPad on either side, staged in LDS: the searches
// of most nodes stay inside this window and only the long ranges of nodes near the root
// read global memory.
constexpr int kKarrasPad = 512;

template <class K>
struct KeyWindow {
  const K* codes;
  const K* win;
  int w0, wlen;
  // The window as an LDS read (clamped index) and the global key only outside it, so
  // neither becomes a flat load through a selected pointer.
  __device__ __forceinline__ K at(int g) const {
    const int q = g - w0;
    const bool in = q >= 0 && q < wlen;
    K v = win[in ? q : 0];
    if (!in) v = gbl(codes)[g];
    return v;
  }
};

// delta(a, b) of the node's own key ka (position a) and the key at b; -1 outside [0, n)
template <class K>
__device__ __forceinline__ int kdelta(const KeyWindow<K>& kw, int n, int a, K ka, int b) {
  if (b < 0 || b >= n) return -1;
  const K cb = kw.at(b);
  if (ka == cb) return KeyTraits<K>::tie_base + __clz((int)((uint32_t)a ^ (uint32_t)b));
  return KeyTraits<K>::clz(ka ^ cb);
}

// 1024 threads per 2048-key tile: two nodes per thread, so the binary searches of a tile
// are spread over 16 waves that hide each other's LDS and memory latency.
constexpr int kKarrasThreads = 1024;

template <class K>
__global__ void __launch_bounds__(kKarrasThreads)
k_karras(const SegDesc* __restrict__ segs, const Tile* __restrict__ tiles, uint32_t ntiles) {
  __shared__ K win[kSortTile + 2 * kKarrasPad];
  for (uint32_t t = xcd_block<kXcdBuildRun>(); t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const SegDesc& s = segs[tl.seg];
    const int n = (int)s.n;
    const K* codes = static_cast<const K*>(s.keys[0]);
    KeyWindow<K> kw{codes, win, (int)tl.start - kKarrasPad, (int)tl.count + 2 * kKarrasPad};
    for (int q = threadIdx.x; q < kw.wlen; q += kKarrasThreads) {
      const int g = kw.w0 + q;
      if (g >= 0 && g < n) win[q] = codes[g];
    }
    __syncthreads();
    for (uint32_t e = threadIdx.x; e < tl.count; e += kKarrasThreads) {
      const int i = (int)(tl.start + e);
      if (i >= n - 1) continue;
      const K ki = kw.at(i);
      const int dir = kdelta(kw, n, i, ki, i + 1) > kdelta(kw, n, i, ki, i - 1) ? 1 : -1;
      const int dmin = kdelta(kw, n, i, ki, i - dir);
      int lmax = 2;
      while (kdelta(kw, n, i, ki, i + lmax * dir) > dmin) lmax *= 2;
      int l = 0;
      for (int tt = lmax / 2; tt > 0; tt /= 2)
        if (kdelta(kw, n, i, ki, i + (l + tt) * dir) > dmin) l += tt;
      const int j = i + l * dir;
      const int dnode = kdelta(kw, n, i, ki, j);
      int sp = 0, tt = l;
      for (;;) {
        tt = (tt + 1) / 2;
        if (kdelta(kw, n, i, ki, i + (sp + tt) * dir) > dnode) sp += tt;
        if (tt <= 1) break;
      }
      const int gamma = i + sp * dir + (dir < 0 ? dir : 0);
      const int lo = i < j ? i : j, hi = i < j ? j : i;
      const uint32_t lu = (lo == gamma) ? (uint32_t)gamma : (uint32_t)(n + gamma);
      const uint32_t ru = (hi == gamma + 1) ? (uint32_t)(gamma + 1) : (uint32_t)(n + gamma + 1);
      const uint32_t me = (uint32_t)(n + i);
      // node i's own fields; its parent field is written by its parent (the root's here)
      uint32_t* tp = reinterpret_cast<uint32_t*>(s.topo);
      tp[4 * (size_t)i] = (uint32_t)lo;
      tp[4 * (size_t)i + 1] = (uint32_t)hi;
      tp[4 * (size_t)i + 2] = enc_children(lu, ru, (uint32_t)n);
      if (lu < (uint32_t)n) s.parent_leaf[lu] = me; else tp[4 * (size_t)(lu - n) + 3] = me;
      if (ru < (uint32_t)n) s.parent_leaf[ru] = me; else tp[4 * (size_t)(ru - n) + 3] = me;
      if (i == 0) tp[3] = kNoParent;
      // walk groups: the subtrees of at most group_size (<= 64) bodies whose parent holds
      // more; a node above the limit marks those of its two children
      const int gmax = (int)s.group_size;
      if (hi - lo + 1 > gmax) {
        if (gamma - lo + 1 <= gmax) s.gend[lo] = (uint32_t)gamma;
        if (hi - gamma <= gmax) s.gend[gamma + 1] = (uint32_t)hi;
      } else if (i == 0) {
        s.gend[0] = (uint32_t)(n - 1);
      }
    }
    __syncthreads();  // the window is refilled for the next tile
  }
}

// ----------------------------------------------------------------------------------
// 6. bottom-up aggregate (fold order fixed: left, right; solvers/src/lbvh.rs:623-636),
//    in passes that need only workgroup-scope ordering:
//    (a) per tile of kAggTile sorted leaves, one block folds the nodes whose leaf range
//        lies inside the tile, in LDS, and lists the others that are indexed in it (the
//        straddlers: about 12 a tile, an internal node's range has its own index at one
//        end);
//    (b) for systems of more than kMidMin bodies, one block per super-tile of kMidTiles
//        tiles folds the straddlers inside the super-tile and lists the rest, and again per
//        kMidTiles super-tiles above kMid2Min bodies;
//    (c) one block per segment folds what is listed, up to the root.
//    Each completed node is written once as its walk record (and quadrupole). A node's
//    record depends only on its children's, so the records are the same whichever pass
//    completes a node and in whatever order its children arrive.
// ----------------------------------------------------------------------------------

// 16-byte record i of a float4 array as one global load (a flat load would also hold up
// the LDS waits that follow it).
__device__ __forceinline__ float4 gload4(const float4* p, size_t i) {
  const auto* q = gbl(reinterpret_cast<const float*>(p)) + 4 * i;
  return make_float4(q[0], q[1], q[2], q[3]);
}

// ... and as one global store: a flat store is counted with the LDS operations, so an LDS
// fence after it would wait for it to complete.
__device__ __forceinline__ void gstore4(float4* p, size_t i, float4 v) {
  auto* q = gblw(reinterpret_cast<float*>(p)) + 4 * i;
  q[0] = v.x;
  q[1] = v.y;
  q[2] = v.z;
  q[3] = v.w;
}

// 16 B at a 32-bit byte offset from a wave-uniform base: the global load's scalar-base
// form (base in SGPRs, offset in one VGPR), with no 64-bit address arithmetic per lane
__device__ __forceinline__ float4 gload4_at(const char* base, uint32_t off) {
  const auto* q = gbl(reinterpret_cast<const float*>(base + off));
  return make_float4(q[0], q[1], q[2], q[3]);
}

__device__ __forceinline__ uint4 gload_u4(const uint4* p, size_t i) {
  const auto* q = gbl(reinterpret_cast<const uint32_t*>(p)) + 4 * i;
  return make_uint4(q[0], q[1], q[2], q[3]);
}

struct AggV {
  float3 com, mn, mx;
  float mass;
  float q[6];  // traceless quadrupole xx, yy, zz, xy, xz, yz about com
};

__device__ __forceinline__ AggV leaf_agg(float4 p) {
  AggV r;
  r.com = make_float3(p.x, p.y, p.z);
  r.mn = r.com;
  r.mx = r.com;
  r.mass = p.w;
  for (int c = 0; c < 6; ++c) r.q[c] = 0.f;
  return r;
}

// The fold and the record below are written out without floating-point contraction, so
// a node's record is the same bits whichever kernel computes it (the compiler would
// otherwise fuse multiplies and adds differently in each inlining context).
template <bool QUAD>
__device__ __forceinline__ AggV fold_agg(const AggV& l, const AggV& r) {
#pragma clang fp contract(off)
  AggV o;
  o.mass = l.mass + r.mass;
  if (o.mass > 0.0f) {
    o.com.x = (l.com.x * l.mass + r.com.x * r.mass) / o.mass;
    o.com.y = (l.com.y * l.mass + r.com.y * r.mass) / o.mass;
    o.com.z = (l.com.z * l.mass + r.com.z * r.mass) / o.mass;
  } else {
    o.com.x = (l.mn.x + l.mx.x + r.mn.x + r.mx.x) * 0.25f;
    o.com.y = (l.mn.y + l.mx.y + r.mn.y + r.mx.y) * 0.25f;
    o.com.z = (l.mn.z + l.mx.z + r.mn.z + r.mx.z) * 0.25f;
  }
  o.mn = make_float3(fminf(l.mn.x, r.mn.x), fminf(l.mn.y, r.mn.y), fminf(l.mn.z, r.mn.z));
  o.mx = make_float3(fmaxf(l.mx.x, r.mx.x), fmaxf(l.mx.y, r.mx.y), fmaxf(l.mx.z, r.mx.z));
  for (int c = 0; c < 6; ++c) o.q[c] = 0.f;
  if (QUAD && o.mass > 0.0f) {
    // parallel-axis shift of each child's traceless quadrupole to the parent com
    const AggV* ch[2] = {&l, &r};
    for (int k = 0; k < 2; ++k) {
      const AggV& c = *ch[k];
      const float dx = c.com.x - o.com.x, dy = c.com.y - o.com.y, dz = c.com.z - o.com.z;
      const float d2 = dx * dx + dy * dy + dz * dz, m = c.mass;
      o.q[0] += c.q[0] + m * (3.f * dx * dx - d2);
      o.q[1] += c.q[1] + m * (3.f * dy * dy - d2);
      o.q[2] += c.q[2] + m * (3.f * dz * dz - d2);
      o.q[3] += c.q[3] + m * 3.f * dx * dy;
      o.q[4] += c.q[4] + m * 3.f * dx * dz;
      o.q[5] += c.q[5] + m * 3.f * dy * dz;
    }
  }
  return o;
}

// Walk record of internal node j from its aggregate (solvers/src/lbvh.rs:602-611 for
// centre/half/delta; the acceptance radius follows from :511-514:
// theta*(d - delta) >= s  <=>  d >= s/theta + delta).
// The walk record of internal node j (topology fields given: leaf range [lo, hi] and
// children).
template <bool QUAD>
__device__ __forceinline__ void store_node(const SegDesc& s, uint32_t j, const AggV& r,
                                           float inv_theta, uint32_t lo, uint32_t hi,
                                           uint32_t cl, uint32_t cr,
                                           bool write_box = true) {
#pragma clang fp contract(off)
  const float cx = (r.mn.x + r.mx.x) * 0.5f, cy = (r.mn.y + r.mx.y) * 0.5f,
              cz = (r.mn.z + r.mx.z) * 0.5f;
  const float hx = (r.mx.x - r.mn.x) * 0.5f, hy = (r.mx.y - r.mn.y) * 0.5f,
              hz = (r.mx.z - r.mn.z) * 0.5f;
  const float size = 2.0f * fmaxf(hx, fmaxf(hy, hz));
  const float ddx = r.com.x - cx, ddy = r.com.y - cy, ddz = r.com.z - cz;
  const float delta = sqrtf(ddx * ddx + ddy * ddy + ddz * ddz);
  const float rcrit = size * inv_theta + delta;
  Node nd;
  nd.a = make_float4(r.com.x, r.com.y, r.com.z, r.mass);
  const float ch = __uint_as_float(enc_entries(cl, cr, s.n));
  NodeBox bx;
  bx.lo = make_float4(r.mn.x, r.mn.y, r.mn.z, __uint_as_float(lo));
  bx.hi = make_float4(r.mx.x, r.mx.y, r.mx.z, __uint_as_float(hi));
  // the farthest that a point of the box lies from the com, per axis; without quadrupoles the
  // square of that distance, summed as the per-target walk sums a target's
  const float ex = fmaxf(r.com.x - r.mn.x, r.mx.x - r.com.x),
              ey = fmaxf(r.com.y - r.mn.y, r.mx.y - r.com.y),
              ez = fmaxf(r.com.z - r.mn.z, r.mx.z - r.com.z);
  if (QUAD) {
    // the group walk's classifier radii: squared monopole-band radius (s / (theta
    // mono_ratio) + delta; FLT_MAX when the band is off) and the node's radius about its
    // com (far-field test), negative for a node that is a single point
    const float rn = sqrtf(fmaf(ex, ex, fmaf(ey, ey, ez * ez)));
    const float rm = fmaf(size, s.mono_inv, delta);
    nd.h = make_float4(rcrit * rcrit, ch, s.mono_inv > 0.f ? rm * rm : 3.4e38f,
                       size > 0.f ? rn : -rn);
  } else {
    nd.h = make_float4(rcrit * rcrit, ch, ex * ex + ey * ey + ez * ez, size);
  }
  if (!(rcrit >= 0.0f)) nd.h.x = nd.h.w = INFINITY;  // a NaN com: nobody accepts it
  const size_t j2 = 2 * (size_t)j;
  gstore4(reinterpret_cast<float4*>(s.node), j2, nd.a);
  gstore4(reinterpret_cast<float4*>(s.node), j2 + 1, nd.h);
  if (write_box) {
    gstore4(reinterpret_cast<float4*>(s.box), j2, bx.lo);
    gstore4(reinterpret_cast<float4*>(s.box), j2 + 1, bx.hi);
  }
  if (QUAD) {
    gstore4(s.quad, j2, make_float4(r.q[0], r.q[1], r.q[2], r.q[3]));
    gstore4(s.quad, j2 + 1, make_float4(r.q[4], r.q[5], 0.f, 0.f));
  }
}

template <bool QUAD>
__device__ __forceinline__ AggV global_child(const SegDesc& s, uint32_t c) {
  const uint32_t n = s.n;
  if (c < n) return leaf_agg(gload4(s.leaf, c));
  AggV r;
  const size_t c2 = 2 * (size_t)(c - n);
  const float4 a = gload4(reinterpret_cast<const float4*>(s.node), c2),
               b = gload4(reinterpret_cast<const float4*>(s.box), c2),
               cc = gload4(reinterpret_cast<const float4*>(s.box), c2 + 1);
  r.com = make_float3(a.x, a.y, a.z);
  r.mass = a.w;
  r.mn = make_float3(b.x, b.y, b.z);
  r.mx = make_float3(cc.x, cc.y, cc.z);
  if (QUAD) {
    const float4 q0 = gload4(s.quad, c2), q1 = gload4(s.quad, c2 + 1);
    r.q[0] = q0.x; r.q[1] = q0.y; r.q[2] = q0.z; r.q[3] = q0.w; r.q[4] = q1.x; r.q[5] = q1.y;
  } else {
    for (int k = 0; k < 6; ++k) r.q[k] = 0.f;
  }
  return r;
}

// Tile pass, one block of one thread per leaf per tile, in two phases:
//  A. every leaf climbs with arrival words in LDS, as far as the nodes inside the tile
//     go; an arrival only adds its subtree height, and the second arrival at a node
//     learns the node's height (1 + the taller child's) and climbs on.
//  B. the in-tile nodes, bucketed by height in LDS, are folded one height at a time
//     (every child of a height-h node is lower), so the lanes that fold are packed into
//     as few waves as the bucket needs: the fold, most of a climb step's instructions,
//     runs about once per node instead of once per wave per tree level.
// Topology is staged in LDS first by coalesced loads (an in-tile node j has t0 <= j < t1:
// an internal node's leaf range has its own index at one end), packed tile-relative in
// 8 bytes; each leaf is staged into its parent's LDS record, which the parent's fold
// reads before overwriting it with its own aggregate.
constexpr int kAggThreads = kAggTile;
// Heights of in-tile nodes stay below this: the common prefix of a node's range (key bits,
// then index bits for equal keys: at most 64 + 32) grows strictly from parent to child.
constexpr uint32_t kMaxHeight = 128;
// packed in-tile topology (s_info): x = lo | hi << 10 | inside | parent << 21 | parent in
// tile; y = split | root | leaf flags (kLeftLeaf, kRightLeaf), all tile-relative
constexpr uint32_t kInInside = 1u << 20, kInParent = 1u << 31, kInRoot = 1u << 20;

// Block barrier that orders LDS only: the global stores before it (node records, read by
// later kernels only) are not waited for, as __syncthreads' release fence would.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <bool QUAD, int N>
__device__ __forceinline__ AggV lds_child(const float4 (*agg)[N], uint32_t c) {
  AggV r;
  const float4 p0 = agg[0][c], p1 = agg[1][c], p2 = agg[2][c];
  r.com = make_float3(p0.x, p0.y, p0.z);
  r.mass = p0.w;
  r.mn = make_float3(p1.x, p1.y, p1.z);
  r.mx = make_float3(p2.x, p2.y, p2.z);
  if (QUAD) {
    const float4 p3 = agg[QUAD ? 3 : 0][c];
    r.q[0] = p1.w; r.q[1] = p2.w; r.q[2] = p3.x; r.q[3] = p3.y; r.q[4] = p3.z; r.q[5] = p3.w;
  } else {
    for (int k = 0; k < 6; ++k) r.q[k] = 0.f;
  }
  return r;
}

// Two blocks per CU (the LDS below fits twice into 160 KB): 8 waves per SIMD, so at most
// 64 VGPRs.
template <bool QUAD>
__global__ void __launch_bounds__(kAggThreads) __attribute__((amdgpu_waves_per_eu(8, 8)))
k_aggregate_tile(const SegDesc* __restrict__ segs, const Tile* __restrict__ tiles,
                 uint32_t ntiles, int group) {
  constexpr int NP = QUAD ? 4 : 3;  // com+mass, min(+q0), max(+q1), q2..q5
  __shared__ float4 s_agg[NP][kAggTile];
  __shared__ uint2 s_info[kAggTile];
  __shared__ uint32_t s_hw[kAggTile];  // A: arrivals << 16 | height; B: nodes by height
  __shared__ uint32_t s_hoff[kMaxHeight + 1], s_hcur[kMaxHeight];
  __shared__ uint32_t s_maxh;
  __shared__ uint32_t s_out[kAggThreads / 64];  // straddlers per wave
  const uint32_t e = threadIdx.x;  // this thread's leaf (and staged node) in the tile
  for (uint32_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const SegDesc& s = segs[tl.seg];
    const uint32_t n = s.n;
    if (n < 2) continue;
    const uint32_t t0 = tl.start, cnt = tl.count, t1 = t0 + cnt;
    const float inv_theta = 1.0f / s.theta;
    // every node's box record is read by the per-target walk and by the group walk above
    // theta = 1 (compared as bits, as the walk does) or with buckets
    const bool box_all = !group || __float_as_uint(s.theta) > __float_as_uint(1.0f) ||
                         s.leaf_size > 1u;
    if (e < kMaxHeight) s_hcur[e] = 0u;
    float4 lf = make_float4(0.f, 0.f, 0.f, 0.f);
    uint32_t p = kNoParent;
    bool out = false;  // node t0 + e is not inside the tile
    if (e < cnt) {
      lf = gload4(s.leaf, t0 + e);
      p = gbl(s.parent_leaf)[t0 + e];
      uint2 inf = make_uint2(0u, 0u);
      if (t0 + e < n - 1) {
        const uint4 tj = gload_u4(s.topo, t0 + e);
        if (tj.x >= t0 && tj.y < t1) {
          const uint32_t pr = tj.w - n - t0;  // wraps far past cnt for kNoParent
          inf.x = (tj.x - t0) | (tj.y - t0) << 10 | kInInside;
          if (tj.w != kNoParent && pr < cnt) inf.x |= pr << 21 | kInParent;
          inf.y = ((tj.z & kSplitMask) - t0) | (tj.z & (kLeftLeaf | kRightLeaf)) |
                  (tj.w == kNoParent ? kInRoot : 0u);
        } else {
          out = true;
        }
      }
      s_info[e] = inf;
      s_hw[e] = 0u;
    }
    const unsigned long long outs = __ballot(out);
    if ((e & 63u) == 0u) s_out[e >> 6] = (uint32_t)__popcll(outs);
    lds_barrier();
    {  // the tile's straddlers, in index order
      uint32_t at = 0, all = 0;
      for (uint32_t k = 0; k < kAggThreads / 64; ++k) {
        if (k == e >> 6) at = all;
        all += s_out[k];
      }
      if (out) gblw(s.strad)[t0 + at + lanes_below(outs)] = t0 + e;
      if (e == 0) gblw(s.scount)[t0 / kAggTile] = all;
    }
    // A: climbs (each in-tile node is reached twice; the bound only guards corrupted input)
    if (e < cnt) {
      uint32_t hu = 0;
      for (uint32_t guard = 0; guard < cnt; ++guard) {
        const uint32_t q = p - n - t0;
        const uint32_t ix = q < cnt ? s_info[q].x : 0u;
        if (!(ix & kInInside)) break;  // the rest of the path leaves the tile
        if (hu == 0u)  // the leaf itself: stage it for its parent's fold (left child = split)
          s_agg[(s_info[q].y & 1023u) == e ? 0 : 1][q] = lf;
        const uint32_t old = atomicAdd(&s_hw[q], 0x10000u + hu + 1u);
        if (old < 0x10000u) break;  // first arrival
        const uint32_t h = max(old & 0xFFFFu, hu + 1u);
        const uint32_t hb = h < kMaxHeight ? h : kMaxHeight - 1;
        s_hw[q] = hb;
        atomicAdd(&s_hcur[hb], 1u);
        hu = h;
        if (!(ix & kInParent)) break;
        p = n + t0 + ((ix >> 21) & 1023u);
      }
    }
    lds_barrier();
    // the in-tile nodes in buckets by height: offsets, then each node's slot
    const uint32_t hn = (e < cnt && (s_info[e].x & kInInside)) ? s_hw[e] : 0u;
    if (e < 64) {
      const uint32_t c0 = s_hcur[2 * e], c1 = s_hcur[2 * e + 1], v = c0 + c1;
      uint32_t inc = v;
      for (int o = 1; o < 64; o <<= 1) {
        const uint32_t w = __shfl_up(inc, o);
        if ((int)e >= o) inc += w;
      }
      s_hoff[2 * e] = inc - v;
      s_hoff[2 * e + 1] = inc - v + c0;
      s_hcur[2 * e] = inc - v;
      s_hcur[2 * e + 1] = inc - v + c0;
      if (e == 63) s_hoff[kMaxHeight] = inc;
      // the tallest height present: the last non-empty bucket
      const unsigned long long any = __ballot(v != 0u);
      if (e == 0) s_maxh = any ? 2u * (63u - (uint32_t)__clzll(any)) + 1u : 0u;
    }
    lds_barrier();
    if (hn) s_hw[atomicAdd(&s_hcur[hn], 1u)] = e;
    lds_barrier();
    // B: folds, one height at a time
    const uint32_t H = s_maxh;
    for (uint32_t h = 1; h <= H; ++h) {
      const uint32_t idx = s_hoff[h] + e;
      if (idx < s_hoff[h + 1]) {
        const uint32_t q = s_hw[idx];
        const uint2 inf = s_info[q];
        const uint32_t g = inf.y & 1023u;
        const bool ll = inf.y & kLeftLeaf, rl = inf.y & kRightLeaf;
        const AggV a = ll ? leaf_agg(s_agg[0][q]) : lds_child<QUAD>(s_agg, g);
        const AggV b = rl ? leaf_agg(s_agg[1][q]) : lds_child<QUAD>(s_agg, g + 1);
        const AggV r = fold_agg<QUAD>(a, b);
        s_agg[0][q] = make_float4(r.com.x, r.com.y, r.com.z, r.mass);
        s_agg[1][q] = make_float4(r.mn.x, r.mn.y, r.mn.z, r.q[0]);
        s_agg[2][q] = make_float4(r.mx.x, r.mx.y, r.mx.z, r.q[1]);
        if (QUAD) s_agg[QUAD ? 3 : 0][q] = make_float4(r.q[2], r.q[3], r.q[4], r.q[5]);
      }
      lds_barrier();
    }
    // the records, a node per thread: outside the rounds, whose length is one fold's latency
    // (with them inside, and as flat stores that the LDS fences waited for, 423 us on the
    // 512-system ensemble and 26 us on 16,384 bodies; now 349 and 21)
    if (hn) {
      const uint2 inf = s_info[e];
      const uint32_t g = inf.y & 1023u;
      const bool ll = inf.y & kLeftLeaf, rl = inf.y & kRightLeaf;
      const uint32_t lo = t0 + (inf.x & 1023u), hi = t0 + ((inf.x >> 10) & 1023u);
      const uint32_t cl = ll ? t0 + g : n + t0 + g, cr = rl ? t0 + g + 1 : n + t0 + g + 1;
      // box records: every node's for the builds that read them (per-target walk, the
      // group walk above theta = 1 or with buckets); otherwise only those of the roots
      // handed to the later passes (no in-tile parent), which fold their boxes
      const bool in_parent = (inf.x & kInParent) &&
                             (s_info[(inf.x >> 21) & 1023u].x & kInInside);
      store_node<QUAD>(s, t0 + e, lds_child<QUAD>(s_agg, e), inv_theta, lo, hi, cl, cr,
                       box_all || !in_parent);
    }
    lds_barrier();
  }
}

// The climbing passes: one block folds a span's straddlers. `lists` lists hold them in index
// order, list i holding count[i] of them at strad[i * stride ...].
constexpr int kFoldThreads = 832;  // 13 waves; one thread and one LDS slot per straddler
constexpr uint32_t kSpanLists = 512;  // most lists of a span: 2^29 bodies in spans of 2^20
static_assert(kMidTiles <= kSpanLists && kMidMin / kAggTile <= kSpanLists &&
                  kMid2Min / kMidSpan <= kSpanLists && (1u << 29) / kMid2Span <= kSpanLists,
              "every pass's lists fit");
constexpr uint32_t kNoSlot = 0xFFFFu;

// pre (in LDS) = exclusive prefix of the counts; returns their sum.
__device__ uint32_t list_prefix(const uint32_t* __restrict__ count, uint32_t nlists,
                                uint32_t* pre, uint32_t* sh_wave, uint32_t* sh_carry) {
  uint32_t carry = 0;
  for (uint32_t c0 = 0; c0 < nlists; c0 += blockDim.x) {
    const uint32_t i = c0 + threadIdx.x;
    const uint32_t v = i < nlists ? gbl(count)[i] : 0u;
    const uint32_t ex = block_exclusive_scan(v, sh_wave);
    if (i < nlists) pre[i] = carry + ex;
    if (threadIdx.x == blockDim.x - 1) *sh_carry = carry + ex + v;
    __syncthreads();
    carry = *sh_carry;
    __syncthreads();
  }
  return carry;
}

// The list holding entry r of the concatenation: the last i with pre[i] <= r.
__device__ __forceinline__ uint32_t list_of(const uint32_t* pre, uint32_t nlists, uint32_t r) {
  uint32_t lo = 0, hi = nlists - 1;
  while (lo < hi) {
    const uint32_t mid = (lo + hi + 1) >> 1;
    if (pre[mid] <= r) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// Whether child c (unified) of a straddler is complete: a leaf, or a node inside one span
// of the pass before (tiles or super-tiles).
__device__ __forceinline__ bool complete_child(const SegDesc& s, uint32_t c, uint32_t below) {
  if (c < s.n) return true;
  const uint4 t = gload_u4(s.topo, c - s.n);
  return t.x / below == t.y / below;
}

// A span with more straddlers than LDS slots: the same folds through global memory. A
// straddler with two complete children is folded at once and climbs; one with one has an
// arrival to its name already. Arrival counters at workgroup scope: no other block reaches
// the nodes of this span; they are back at 0 when the climbs end.
template <bool QUAD>
__device__ void fold_global(const SegDesc& s, const uint32_t* strad, uint32_t stride,
                            const uint32_t* pre, uint32_t nlists, uint32_t total, uint32_t below,
                            uint32_t S0, uint32_t S1) {
  const uint32_t n = s.n;
  const float inv_theta = 1.0f / s.theta;
  for (int phase = 0; phase < 2; ++phase) {
    for (uint32_t r = threadIdx.x; r < total; r += blockDim.x) {
      const uint32_t i = list_of(pre, nlists, r);
      uint32_t j = gbl(strad)[(size_t)i * stride + (r - pre[i])];
      uint4 tj = gload_u4(s.topo, j);
      if (tj.x < S0 || tj.y >= S1) continue;
      const uint32_t ext = (uint32_t)complete_child(s, left_child(tj.z, n), below) +
                           (uint32_t)complete_child(s, right_child(tj.z, n), below);
      if (phase == 0) {
        if (ext == 1u)
          __hip_atomic_store(&s.flag[j], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        continue;
      }
      if (ext != 2u) continue;
      for (uint32_t guard = 0; guard < n; ++guard) {
        const uint32_t cl = left_child(tj.z, n), cr = right_child(tj.z, n);
        const AggV a = fold_agg<QUAD>(global_child<QUAD>(s, cl), global_child<QUAD>(s, cr));
        store_node<QUAD>(s, j, a, inv_theta, tj.x, tj.y, cl, cr);
        if (tj.w == kNoParent) break;
        j = tj.w - n;
        tj = gload_u4(s.topo, j);
        if (tj.x < S0 || tj.y >= S1) break;
        const uint32_t old = __hip_atomic_fetch_add(&s.flag[j], 1u, __ATOMIC_ACQ_REL,
                                                    __HIP_MEMORY_SCOPE_WORKGROUP);
        if (old == 0u) break;
        __hip_atomic_store(&s.flag[j], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    }
    __syncthreads();
  }
}

// One span: the super-tile [S0, S1) of a system (MID, level 1 or 2: the straddlers that leave
// it are listed for the next pass) or the whole system. A thread per straddler loads its topology,
// finds its children's and parent's slots by bisection of the sorted index list and loads
// its complete children's records, all in parallel; then the climbs run in LDS: a straddler
// with two complete children is folded by its own thread, one with one holds it in its slot
// with an arrival counted, and the second arrival at a node folds its children's slots.
// Bound: the height of the tree above the tiles (18 to 54 levels) times one fold and an LDS
// round trip. Climbing from the subtree roots through global memory took three dependent
// memory round trips a level: 53 us for 16,384 bodies (16 tiles), now 31; 111 + 73 us (top,
// middle) for a 2^20 collision, now 50 + 36; 114 us for the 512-system ensemble, now 73.
template <bool QUAD, bool MID>
__global__ void __launch_bounds__(kFoldThreads)
k_aggregate_span(const SegDesc* __restrict__ segs, const Tile* __restrict__ spans,
                 uint32_t nspans, int level) {
  constexpr int NP = QUAD ? 4 : 3;
  __shared__ float4 s_agg[NP][kFoldThreads];
  __shared__ uint32_t s_j[kFoldThreads], s_cnt[kFoldThreads];
  __shared__ uint16_t s_l[kFoldThreads], s_r[kFoldThreads], s_up[kFoldThreads];
  __shared__ uint32_t sh_wave[kFoldThreads / 64], sh_carry;
  __shared__ uint32_t pre[MID ? kMidTiles : kSpanLists];
  for (uint32_t sp = blockIdx.x; sp < nspans; sp += gridDim.x) {
    const Tile span = MID ? spans[sp] : Tile{sp, 0, 0, 0};
    const SegDesc& s = segs[span.seg];
    const uint32_t n = s.n;
    if (n < 2) continue;
    const uint32_t S0 = MID ? span.start : 0u, S1 = MID ? span.start + span.count : n;
    // the pass before: 0 the tiles, 1 the super-tiles, 2 the super-tiles' super-tiles
    const int from = MID ? level - 1 : (n > kMid2Min ? 2 : (n > kMidMin ? 1 : 0));
    const uint32_t below = from == 0 ? (uint32_t)kAggTile : (from == 1 ? kMidSpan : kMid2Span);
    const uint32_t* count = from == 0 ? s.scount : (from == 1 ? s.scount2 : s.scount3);
    const uint32_t* strad = (from == 1 ? s.strad2 : s.strad) + S0;
    uint32_t* strad_out = (level == 1 ? s.strad2 : s.strad) + S0;
    const uint32_t nl = (S1 - S0 + below - 1) / below;
    const uint32_t total = list_prefix(count + S0 / below, nl, pre, sh_wave, &sh_carry);
    const uint32_t e = threadIdx.x;
    // this thread's straddler: inside the span, or (MID) listed for the top pass
    const bool all = total <= (uint32_t)kFoldThreads;
    uint32_t out_base = 0;
    uint32_t j = 0;
    uint4 tj = make_uint4(0u, 0u, 0u, kNoParent);
    bool in = false;
    for (uint32_t r0 = 0; r0 < (MID ? total : min(total, (uint32_t)kFoldThreads));
         r0 += kFoldThreads) {
      const uint32_t r = r0 + e;
      bool out = false;
      if (r < total) {
        const uint32_t i = list_of(pre, nl, r);
        j = gbl(strad)[(size_t)i * below + (r - pre[i])];
        tj = gload_u4(s.topo, j);
        in = !MID || (tj.x >= S0 && tj.y < S1);
        out = !in;
      }
      if (MID) {
        const uint32_t at = block_exclusive_scan(out ? 1u : 0u, sh_wave);
        if (out) gblw(strad_out)[out_base + at] = j;
        if (e == kFoldThreads - 1) sh_carry = out_base + at + (out ? 1u : 0u);
        __syncthreads();
        out_base = sh_carry;
        __syncthreads();
      }
    }
    if (MID && e == 0) {
      if (level == 1) s.scount2[S0 / kMidSpan] = out_base;
      else s.scount3[S0 / kMid2Span] = out_base;
    }
    if (!all) {
      fold_global<QUAD>(s, strad, below, pre, nl, total, below, S0, S1);
      continue;
    }
    const float inv_theta = 1.0f / s.theta;
    const uint32_t slot = block_exclusive_scan(in ? 1u : 0u, sh_wave);
    if (e == kFoldThreads - 1) sh_carry = slot + (in ? 1u : 0u);
    if (in) s_j[slot] = j;
    __syncthreads();
    const uint32_t m = sh_carry;
    auto find = [&](uint32_t key) -> uint32_t {  // slot of node `key`, or kNoSlot
      uint32_t lo = 0, hi = m;
      while (lo < hi) {
        const uint32_t q = (lo + hi) >> 1;
        if (s_j[q] < key) lo = q + 1; else hi = q;
      }
      return lo < m && s_j[lo] == key ? lo : kNoSlot;
    };
    auto put = [&](uint32_t q, const AggV& r) {
      s_agg[0][q] = make_float4(r.com.x, r.com.y, r.com.z, r.mass);
      s_agg[1][q] = make_float4(r.mn.x, r.mn.y, r.mn.z, r.q[0]);
      s_agg[2][q] = make_float4(r.mx.x, r.mx.y, r.mx.z, r.q[1]);
      if (QUAD) s_agg[QUAD ? 3 : 0][q] = make_float4(r.q[2], r.q[3], r.q[4], r.q[5]);
    };
    bool climbs = false;
    if (in) {
      const uint32_t g = tj.z & kSplitMask;
      const uint32_t cl = left_child(tj.z, n), cr = right_child(tj.z, n);
      const uint32_t l = (tj.z & kLeftLeaf) ? kNoSlot : find(g);
      const uint32_t r = (tj.z & kRightLeaf) ? kNoSlot : find(g + 1u);
      s_l[slot] = (uint16_t)(l == kNoSlot ? slot : l);  // a complete child waits in the slot
      s_r[slot] = (uint16_t)(r == kNoSlot ? slot : r);
      s_up[slot] = (uint16_t)(tj.w == kNoParent ? kNoSlot : find(tj.w - n));
      s_cnt[slot] = (l == kNoSlot || r == kNoSlot) ? 1u : 0u;
      climbs = l == kNoSlot && r == kNoSlot;
      if (climbs) {
        const AggV a =
            fold_agg<QUAD>(global_child<QUAD>(s, cl), global_child<QUAD>(s, cr));
        put(slot, a);
      } else if (l == kNoSlot) {
        put(slot, global_child<QUAD>(s, cl));
      } else if (r == kNoSlot) {
        put(slot, global_child<QUAD>(s, cr));
      }
    }
    lds_barrier();
    if (climbs) {
      uint32_t q = s_up[slot];
      for (uint32_t guard = 0; q != kNoSlot && guard < m; ++guard) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        const uint32_t old = __hip_atomic_fetch_add(&s_cnt[q], 1u, __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_WORKGROUP);
        if (old == 0u) break;  // first arrival
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        const AggV a = lds_child<QUAD>(s_agg, s_l[q]), b = lds_child<QUAD>(s_agg, s_r[q]);
        const AggV r = fold_agg<QUAD>(a, b);
        put(q, r);
        q = s_up[q];
      }
    }
    lds_barrier();
    if (in)  // the records, off the climbs' path
      store_node<QUAD>(s, j, lds_child<QUAD>(s_agg, slot), inv_theta, tj.x, tj.y,
                       left_child(tj.z, n), right_child(tj.z, n));
    lds_barrier();
  }
}

// ----------------------------------------------------------------------------------
// 6b. flatten, exported for parity only (the walks do not need it): the reference's DFS
//     pre-order layout (solvers/src/lbvh.rs:545-614), every node placed in parallel. In
//     pre-order with the left child first, the nodes before u are its ancestors and the
//     subtrees hanging left of its root path; those cover the leaves [0, lo) and hold
//     2 lo minus their count of nodes, one per right edge of the path, so
//     slot(u) = 2 lo + (left edges on the root path of u).
// ----------------------------------------------------------------------------------

__device__ uint32_t flat_slot(const SegDesc& s, uint32_t u) {
  const uint32_t n = s.n;
  if (n == 1) return 0u;
  const uint32_t lo = u < n ? u : s.topo[u - n].x;
  uint32_t left_edges = 0, v = u;
  uint32_t p = u < n ? gbl(s.parent_leaf)[u] : s.topo[u - n].w;
  for (uint32_t guard = 0; p != kNoParent && guard < n; ++guard) {  // depth < n
    const uint32_t j = p - n;
    if (j >= n - 1) break;
    const uint4 tj = s.topo[j];
    if (left_child(tj.z, n) == v) ++left_edges;
    v = p;
    p = tj.w;
  }
  return 2u * lo + left_edges;
}

__device__ __forceinline__ void flat_store3(float* a, uint32_t q, float x, float y, float z) {
  a[3 * (size_t)q] = x;
  a[3 * (size_t)q + 1] = y;
  a[3 * (size_t)q + 2] = z;
}

// One thread per sorted leaf k places leaf k and internal node k (k < n - 1). Geometry is
// the f32 origin-relative aggregate: centre and half extent of the AABB, com, mass and
// delta = |com - centre|; a leaf's centre is its position and its half extent zero.
__global__ void __launch_bounds__(kBlock)
k_flatten(const SegDesc* __restrict__ segs, const Tile* __restrict__ tiles, uint32_t ntiles,
          FlatOut o) {
  for (uint32_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const SegDesc& s = segs[tl.seg];
    const uint32_t n = s.n;
    for (uint32_t e = threadIdx.x; e < tl.count; e += kBlock) {
      const uint32_t k = tl.start + e;
      {
        const uint32_t q = flat_slot(s, k);
        const float4 lf = s.leaf[k];
        o.next[q] = q + 1u;
        o.body_start[q] = k;
        o.body_count[q] = 1u;
        flat_store3(o.center, q, lf.x, lf.y, lf.z);
        flat_store3(o.half, q, 0.f, 0.f, 0.f);
        flat_store3(o.com, q, lf.x, lf.y, lf.z);
        o.mass[q] = lf.w;
        o.delta[q] = 0.f;
      }
      if (k + 1u < n) {
        const uint32_t q = flat_slot(s, n + k);
        const float4 na = s.node[k].a, nb = s.box[k].lo, nc = s.box[k].hi;
        const uint32_t lo = s.topo[k].x, hi = s.topo[k].y;
        const float cx = (nb.x + nc.x) * 0.5f, cy = (nb.y + nc.y) * 0.5f,
                    cz = (nb.z + nc.z) * 0.5f;
        const float dx = na.x - cx, dy = na.y - cy, dz = na.z - cz;
        o.next[q] = q + 2u * (hi - lo + 1u) - 1u;  // 2 leaves - 1 nodes in the subtree
        o.body_start[q] = 0u;
        o.body_count[q] = 0u;
        flat_store3(o.center, q, cx, cy, cz);
        flat_store3(o.half, q, (nc.x - nb.x) * 0.5f, (nc.y - nb.y) * 0.5f,
                    (nc.z - nb.z) * 0.5f);
        flat_store3(o.com, q, na.x, na.y, na.z);
        o.mass[q] = na.w;
        o.delta[q] = sqrtf(dx * dx + dy * dy + dz * dz);
      }
    }
  }
}

// ----------------------------------------------------------------------------------
// 7. walks. Accelerations are accumulated in origin-relative f32 coordinates with
//    optional Kahan compensation; the epilogue scatters a (x G) to the original
//    index and, in resident mode, applies the closing half-kick
//    (core/src/integrator.rs:70-73).
// ----------------------------------------------------------------------------------

struct Acc3 {
  float x, y, z, cx, cy, cz;
};

template <bool KAHAN>
__device__ __forceinline__ void acc_add(Acc3& a, float tx, float ty, float tz) {
  if (KAHAN) {
    float y, t;
    y = tx - a.cx; t = a.x + y; a.cx = (t - a.x) - y; a.x = t;
    y = ty - a.cy; t = a.y + y; a.cy = (t - a.y) - y; a.y = t;
    y = tz - a.cz; t = a.z + y; a.cz = (t - a.z) - y; a.z = t;
  } else {
    a.x += tx;
    a.y += ty;
    a.z += tz;
  }
}

// Two sums as one. Compensated, the rounding of each addition joins the compensations (the
// exact error of a + b, D. Knuth's two-sum), so that nothing of the lanes' is lost.
template <bool KAHAN>
__device__ __forceinline__ void sum_join(float& v, float& c, float w, float d) {
  const float t = v + w;
  if (KAHAN) {
    const float b = t - v;
    c = (c + d) - ((v - (t - b)) + (w - b));
  }
  v = t;
}
template <bool KAHAN>
__device__ __forceinline__ Acc3 acc_join(Acc3 a, const Acc3& b) {
  sum_join<KAHAN>(a.x, a.cx, b.x, b.cx);
  sum_join<KAHAN>(a.y, a.cy, b.y, b.cy);
  sum_join<KAHAN>(a.z, a.cz, b.z, b.cz);
  return a;
}
template <bool KAHAN>
__device__ __forceinline__ Acc3 acc_shfl(const Acc3& a, int src) {
  Acc3 r = {__shfl(a.x, src), __shfl(a.y, src), __shfl(a.z, src), 0.f, 0.f, 0.f};
  if (KAHAN) {
    r.cx = __shfl(a.cx, src);
    r.cy = __shfl(a.cy, src);
    r.cz = __shfl(a.cz, src);
  }
  return r;
}
template <bool KAHAN>
__device__ __forceinline__ Acc3 acc_shfl_xor(const Acc3& a, int o) {
  Acc3 r = {__shfl_xor(a.x, o), __shfl_xor(a.y, o), __shfl_xor(a.z, o), 0.f, 0.f, 0.f};
  if (KAHAN) {
    r.cx = __shfl_xor(a.cx, o);
    r.cy = __shfl_xor(a.cy, o);
    r.cz = __shfl_xor(a.cz, o);
  }
  return r;
}

template <bool KAHAN>
__device__ __forceinline__ void store_acc(const SegDesc& s, uint32_t k, const Acc3& a, int mode) {
  const uint32_t n = s.n;
  const float g = s.g;
  const float ax = (a.x - (KAHAN ? a.cx : 0.f)) * g;
  const float ay = (a.y - (KAHAN ? a.cy : 0.f)) * g;
  const float az = (a.z - (KAHAN ? a.cz : 0.f)) * g;
  const size_t i = min(s.vals[0][k], n - 1);
  if (s.acc_out) {
    s.acc_out[3 * i] = (double)ax;
    s.acc_out[3 * i + 1] = (double)ay;
    s.acc_out[3 * i + 2] = (double)az;
  } else {
    s.acc[3 * i] = ax;
    s.acc[3 * i + 1] = ay;
    s.acc[3 * i + 2] = az;
    if (mode == 1) {
      const float h = s.half_dt;
      s.v[3 * i] += ax * h;
      s.v[3 * i + 1] += ay * h;
      s.v[3 * i + 2] += az * h;
    }
  }
}

// Squared distance from a node's com to its box's farthest corner, from the second part of its
// record; not less than any target's in the box.
template <bool QUAD>
__device__ __forceinline__ float corner_distance2(const float4& H) {
  return QUAD ? H.w * H.w * 1.000002f : H.z;
}

// Per-target walk (the reference's criterion for every target, solvers/src/lbvh.rs:469-524):
// one wave walks for kTargets Morton-consecutive targets, 64 nodes at a time, one per lane.
// A node carries the mask of the targets that opened all its ancestors; a lane tests its
// node against each of them (their positions are wave-uniform), adds the accepted ones'
// monopole terms and the leaves' bodies to its own partial sums, and pushes the node's
// children's word for the targets that open it. The partial sums are added over the wave
// at the end, compensations included. Every target accepts and opens exactly the nodes of the
// reference's pre-order walk (the distance test is written without contraction, and the box
// is read wherever a target inside it could pass it); only the order of the sum differs.
// Bound: one lane per target, each following its own chain of dependent node loads through
// the pre-order, took 605 to 649 us for 1,000 bodies (16 waves on the chip), 1,782 us for a
// 16,384-body Plummer sphere and 177 ms for a 2^18-body collision. With 64 nodes per step
// the chain is the tree's depth and the wave's loads are in flight together: 23, 55 us and
// 9.4 ms (2,621 -> 231 us at 100,003 bodies), now bound by the node gathers and about 140 VALU
// instructions a round. Sharing each node load between 4 targets measured best over that
// range (2 targets: 20, 64 us, 15 ms; 8: 32, 74 us, 10.7 ms). 64 VGPRs are 8 waves per SIMD,
// worth 4% at 100,003 bodies.
constexpr int kTargets = 4;
constexpr int kTargetLanes = 64 / kTargets;  // lanes that end with one target's sum
// Stack entries (children word of an opened node, mask of the targets that opened it).
// 32 are popped per round while that cannot overflow; above kOpenWide one at a time, depth
// first, which adds at most one entry per level (trees are at most 96 levels deep).
constexpr uint32_t kOpenCap = 512, kOpenWide = kOpenCap - 160;

template <bool KAHAN, bool COUNT, bool QUAD>
__device__ __forceinline__ Acc3 target_walk(const SegDesc& s, uint32_t k0, uint32_t cnt,
                                            bool boxes, uint32_t lane, uint32_t* words,
                                            uint8_t* masks, uint32_t counted,
                                            unsigned long long& n_int,
                                            unsigned long long& n_vis) {
  const uint32_t n = s.n;
  const float eps2 = s.eps2;
  const auto* lf = (const __attribute__((address_space(4))) float*)s.leaf + 4 * (size_t)k0;
  float mx[kTargets], my[kTargets], mz[kTargets];
  Acc3 a[kTargets];
#pragma unroll
  for (int t = 0; t < kTargets; ++t) {
    const int q = (uint32_t)t < cnt ? t : 0;
    mx[t] = lf[4 * q];
    my[t] = lf[4 * q + 1];
    mz[t] = lf[4 * q + 2];
    a[t] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  }
  const uint64_t leaf_base = (uint64_t)s.leaf, node_base = (uint64_t)s.node;
  uint32_t sp = 0, u = n == 1 ? 0u : kEntryNode, mk = lane == 0 ? (1u << cnt) - 1u : 0u;
  // every node is pushed at most once; the bound only guards corrupted trees
  for (uint32_t guard = 0; guard <= n; ++guard) {
    const bool node = (int32_t)u < 0;
    const uint32_t ni = node ? u & ~kEntryNode : 0u;
    const float4 A = gload4(reinterpret_cast<const float4*>(node ? node_base : leaf_base),
                            node ? 2u * ni : u);
    const float4 H = gload4(reinterpret_cast<const float4*>(s.node), 2 * (size_t)ni + 1);
    if (COUNT) n_vis += (uint32_t)__popc(mk & counted);
    float d2[kTargets], dx[kTargets], dy[kTargets], dz[kTargets];
    uint32_t acc = 0;  // bit t: target t accepts the node
    bool edge = false;
    // No target within a node's box accepts it. Such a target lies no farther from the com than
    // the box's farthest corner, whose squared distance is in the record: a target's differences
    // are at most the corner's, and rounding keeps that order through the same operations. So
    // the box is read only where an accepted distance is not beyond it: for theta > 1, and for
    // nodes a few ulps wide, whose com and centre are rounded onto the box's own bodies. (The
    // quadrupole builds' records hold other radii; their rare fallback reads every box.) Without
    // boxes, in the group walk's fallback, nothing that near is accepted, a point excepted.
    const float corner2 = corner_distance2<QUAD>(H);
    const float lim = QUAD ? INFINITY : corner2;
    {
#pragma clang fp contract(off)
#pragma unroll
      for (int t = 0; t < kTargets; ++t) {
        dx[t] = A.x - mx[t];
        dy[t] = A.y - my[t];
        dz[t] = A.z - mz[t];
        d2[t] = dx[t] * dx[t] + dy[t] * dy[t] + dz[t] * dz[t];
        const bool ok = d2[t] >= H.x;
        acc |= ok ? 1u << t : 0u;
        edge |= ok & (d2[t] <= lim);
      }
    }
    const bool massive = A.w > 0.0f;
    if (boxes && __ballot(edge & node & massive) != 0ull) {
      const float4* brec = reinterpret_cast<const float4*>(s.box);
      const float4 B = gload4(brec, 2 * (size_t)ni), C = gload4(brec, 2 * (size_t)ni + 1);
#pragma unroll
      for (int t = 0; t < kTargets; ++t)
        if ((B.x <= mx[t]) & (mx[t] <= C.x) & (B.y <= my[t]) & (my[t] <= C.y) &
            (B.z <= mz[t]) & (mz[t] <= C.z))
          acc &= ~(1u << t);
    }
    if (!boxes) {
#pragma unroll
      for (int t = 0; t < kTargets; ++t)
        if (H.w > 0.0f && d2[t] <= corner2) acc &= ~(1u << t);
    }
    const uint32_t live = massive ? mk : 0u;
    const uint32_t self = u - k0 < (uint32_t)kTargets ? 1u << (u - k0) : 0u;
    const uint32_t sum = live & (node ? acc : ~self);
    const uint32_t open = node ? live & ~acc : 0u;
    if (COUNT) n_int += (uint32_t)__popc(sum & counted);
    // Branches, not a weight of 0: a node or leaf that a target does not take may lie at a NaN
    // or infinity (a massless body there, and every com above it). They cost nothing: a set
    // whose lanes all pass skips the term (16,384 bodies 57.4 us with zero weights, 56.6 so,
    // 61.2 with the differences zeroed too; 2^18-body collision 10.2, 9.7, 10.7 ms).
#pragma unroll
    for (int t = 0; t < kTargets; ++t) {
      if ((sum >> t) & 1u) {
        const float r2 = d2[t] + eps2;
        const float ir = rsqrtf(r2);
        const float w = A.w * ir * ir * ir;
        if (KAHAN) {
          acc_add<true>(a[t], dx[t] * w, dy[t] * w, dz[t] * w);
        } else {
          a[t].x = fmaf(dx[t], w, a[t].x);
          a[t].y = fmaf(dy[t], w, a[t].y);
          a[t].z = fmaf(dz[t], w, a[t].z);
        }
      }
    }
    const unsigned long long mo = __ballot(open != 0u);
    if (open != 0u) {
      const uint32_t q = sp + lanes_below(mo);
      words[q] = __float_as_uint(H.y);
      masks[q] = (uint8_t)open;
    }
    sp += (uint32_t)__popcll(mo);
    wave_lds_order();
    if (sp == 0u) break;
    const uint32_t m = sp <= kOpenWide ? min(sp, 32u) : 1u;
    sp -= m;
    const uint32_t e = lane >> 1;  // two lanes per popped word: left and right child
    u = 0u;
    mk = 0u;
    if (e < m) {
      const uint32_t w = words[sp + e];
      mk = masks[sp + e];
      u = (lane & 1u) ? right_entry(w) : left_entry(w);
    }
    wave_lds_order();
  }
  // Sum over the wave, halving the targets a lane holds with each of the first steps, so
  // that lanes [t kTargetLanes, (t + 1) kTargetLanes) end with target t's sum.
  int o = 32;
#pragma unroll
  for (int h = kTargets / 2; h > 0; h >>= 1, o >>= 1) {
    const bool up = (lane & (uint32_t)o) != 0u;
#pragma unroll
    for (int t = 0; t < h; ++t) {
      const Acc3 give = up ? a[t] : a[t + h];
      a[t] = acc_join<KAHAN>(up ? a[t + h] : a[t], acc_shfl_xor<KAHAN>(give, o));
    }
  }
#pragma unroll
  for (int w = kTargetLanes / 2; w > 0; w >>= 1)
    a[0] = acc_join<KAHAN>(a[0], acc_shfl_xor<KAHAN>(a[0], w));
  return a[0];
}

// One wave per block and kTargets targets per wave; the tiles hold kBlock targets.
constexpr uint32_t kTileQuads = kBlock / kTargets;

template <bool KAHAN, bool COUNT>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(KAHAN || COUNT ? 1 : 8)))
k_walk_target(const SegDesc* __restrict__ segs, const Tile* __restrict__ tiles, uint32_t ntiles,
              int mode) {
  __shared__ uint32_t words[kOpenCap];
  __shared__ uint8_t masks[kOpenCap];
  const uint32_t lane = threadIdx.x;
  for (uint32_t b = xcd_block<kXcdTargetRun>(); b < ntiles * kTileQuads; b += gridDim.x) {
    const Tile tl = tiles[b / kTileQuads];
    const SegDesc& s = segs[tl.seg];
    const uint32_t q = (b % kTileQuads) * kTargets;
    if (tl.start == 0 && q == 0 && lane < 6) bbox_neutral(s.bbox, lane);
    if (q >= tl.count) continue;
    const uint32_t k0 = __builtin_amdgcn_readfirstlane(tl.start + q);
    const uint32_t cnt = min(tl.count - q, (uint32_t)kTargets);
    // lanes t kTargetLanes store target t
    const uint32_t t = lane / kTargetLanes, k = k0 + min(t, cnt - 1u);
    bool on = t < cnt && lane % kTargetLanes == 0u;
    if (s.active) {
      on = on && s.active[min(s.vals[0][k], s.n - 1)];
      if (__ballot(on) == 0ull) continue;
    }
    unsigned long long n_int = 0, n_vis = 0;
    const Acc3 a = target_walk<KAHAN, COUNT, false>(s, k0, cnt, true, lane, words, masks, ~0u,
                                                    n_int, n_vis);
    if (on) store_acc<KAHAN>(s, k, a, mode);
    if (COUNT) {
      n_int = wave_sum_u64(n_int);
      n_vis = wave_sum_u64(n_vis);
      if (lane == 0) {
        atomicAdd(&s.counters[kCntInteractions], n_int);
        atomicAdd(&s.counters[kCntVisits], n_vis);
      }
    }
    __syncthreads();
  }
}

// Group walk: one wave walks the tree for 64 Morton-consecutive targets. Nodes to
// test are popped 64 at a time from an LDS stack (one node per lane); a node is
// accepted for the whole group when its centre of mass is at least the reference
// acceptance radius (s/theta + delta) from every point of the group's bounding box
// and the group box does not overlap the node box — so each target's own reference
// test (solvers/src/lbvh.rs:506-514) holds for every accepted node. Accepted nodes
// and reached leaves are appended to LDS interaction lists which the 64 lanes then
// evaluate against their own targets (LDS broadcast reads, no divergence). Opened
// nodes push both children. If the stack would overflow, the group falls back to
// the per-target walk.
constexpr int kStackCap = 896;  // the deepest stack measured is 520 entries
static_assert(kStackCap * 4 >= kOpenCap * 5, "the per-target fallback's stack fits");
constexpr int kListCap = 64;   // lists are drained every round, which adds at most 64
constexpr int kRangeCap = 64;
constexpr int kFarCap = 128;  // far nodes are drained 64 at a time, one per lane

// Floor on the softened r^2 of a point term: a source at the target's position (dx = 0
// exactly, the target itself included) then adds 0 * finite rather than 0 * inf when the
// softening is 0. It is far below any separation f32 positions resolve at unit scale.
constexpr float kR2Floor = 1e-20f;

// Point-mass term of one source on the lane's target: a += m d / (|d|^2 + eps^2)^1.5.
// The raw v_rsq (1 ulp) serves as rsqrt: r^2 is never denormal here. FLOOR applies the
// r^2 floor; with eps^2 >= the floor, r^2 >= eps^2 already and the floor is left out.
template <bool KAHAN, bool FLOOR = true>
__device__ __forceinline__ void point_term(Acc3& a, const float4& me, const float4& p, float eps2) {
  const float dx = p.x - me.x, dy = p.y - me.y, dz = p.z - me.z;
  const float r2s = fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, eps2)));
  const float r2 = FLOOR ? fmaxf(r2s, kR2Floor) : r2s;
  const float ir = __builtin_amdgcn_rsqf(r2);
  const float w = p.w * (ir * ir) * ir;
  if (KAHAN) {
    acc_add<true>(a, dx * w, dy * w, dz * w);
  } else {
    a.x = fmaf(dx, w, a.x);
    a.y = fmaf(dy, w, a.y);
    a.z = fmaf(dz, w, a.z);
  }
}

// Monopole + quadrupole term of one node (com/mass P, traceless Q = {xx,yy,zz,xy}, {xz,yz})
// with the softened radius r^2 = |d|^2 + eps^2, d = com - x:
//   a = m d / r^3 - Q d / r^5 + 2.5 (d.Q.d) d / r^7
//     = r^-5 [(m r^2 + 2.5 (d.Q.d) / r^2) d - Q d]
// An accepted node is never at the target (its box is disjoint from the group's), so
// r^2 > 0.
template <bool KAHAN>
__device__ __forceinline__ void quad_term(Acc3& a, const float4& me, const float4& P,
                                          const float4& B, const float2& Cq, float eps2) {
  const float dx = P.x - me.x, dy = P.y - me.y, dz = P.z - me.z;
  const float r2 = fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, eps2)));
  const float ir = __builtin_amdgcn_rsqf(r2), ir2 = ir * ir, ir5 = (ir2 * ir2) * ir;
  const float qx = fmaf(B.x, dx, fmaf(B.w, dy, Cq.x * dz));
  const float qy = fmaf(B.w, dx, fmaf(B.y, dy, Cq.y * dz));
  const float qz = fmaf(Cq.x, dx, fmaf(Cq.y, dy, B.z * dz));
  const float dqd = fmaf(dx, qx, fmaf(dy, qy, dz * qz));
  const float c = fmaf(P.w, r2, 2.5f * dqd * ir2);
  const float tx = fmaf(c, dx, -qx), ty = fmaf(c, dy, -qy), tz = fmaf(c, dz, -qz);
  if (KAHAN) {
    acc_add<true>(a, ir5 * tx, ir5 * ty, ir5 * tz);
  } else {
    a.x = fmaf(ir5, tx, a.x);
    a.y = fmaf(ir5, ty, a.y);
    a.z = fmaf(ir5, tz, a.z);
  }
}

// Far field of a group: a node (com at d from the group centre, mass m, traceless Q) is
// folded into a local expansion of the softened acceleration about the centre,
// a(c + y) = A0 + A1 y + A2 y y / 2 + A3 y y y / 6 (R^2 = |d|^2 + eps^2):
//   monopole   A0 = m d / R^3,  A1_ij = m (3 d_i d_j / R^5 - delta_ij / R^3),
//              A2_ijk = m (15 d_i d_j d_k / R^7
//                          - 3 (delta_ij d_k + delta_ik d_j + delta_jk d_i) / R^5),
//              A3_ijkl = m (105 d_i d_j d_k d_l / R^9 - 15 (delta_ij d_k d_l + 5 more
//                           pairings) / R^7 + 3 (delta_ij delta_kl + 2 more) / R^5)
//   quadrupole A0 = -q / R^5 + 2.5 s d / R^7 (q = Q d, s = d.q),
//              A1_ij = Q_ij / R^5 - 5 (q_i d_j + q_j d_i) / R^7 - 2.5 s delta_ij / R^7
//                      + 17.5 s d_i d_j / R^9
// (the successive derivatives of the field in y: each order adds one factor |y| / R to
// the truncation error; the quadrupole's second-order term is dropped: it is smaller than
// the neglected fourth-order monopole term for well-separated nodes). Coefficients:
// L[0..2] = A0, L[3..8] = A1 {xx,yy,zz,xy,xz,yz},
// L[9..18] = A2 {xxx,xxy,xxz,xyy,xyz,xzz,yyy,yyz,yzz,zzz},
// L[19..33] = A3 {xxxx,xxxy,xxxz,xxyy,xxyz,xxzz,xyyy,xyyz,xyzz,xzzz,yyyy,yyyz,yyzz,yzzz,zzzz}.
constexpr int kLocal = 34;

__device__ __forceinline__ void far_m2l(float* L, float x, float y, float z, float m,
                                        const float4& Q0, const float4& Q1, float eps2) {
  const float R2 = fmaf(x, x, fmaf(y, y, fmaf(z, z, eps2)));
  const float ir = __builtin_amdgcn_rsqf(R2), ir2 = ir * ir;
  const float mr3 = m * ir * ir2, ir5 = ir * ir2 * ir2, ir7 = ir5 * ir2;
  const float xx = x * x, yy = y * y, zz = z * z, xy = x * y, xz = x * z, yz = y * z;
  // monopole
  L[0] = fmaf(mr3, x, L[0]);
  L[1] = fmaf(mr3, y, L[1]);
  L[2] = fmaf(mr3, z, L[2]);
  const float t = 3.0f * m * ir5;
  L[3] += fmaf(t, xx, -mr3);
  L[4] += fmaf(t, yy, -mr3);
  L[5] += fmaf(t, zz, -mr3);
  L[6] = fmaf(t, xy, L[6]);
  L[7] = fmaf(t, xz, L[7]);
  L[8] = fmaf(t, yz, L[8]);
  const float w = 15.0f * m * ir7;
  L[9] += x * fmaf(w, xx, -3.0f * t);
  L[10] += y * fmaf(w, xx, -t);
  L[11] += z * fmaf(w, xx, -t);
  L[12] += x * fmaf(w, yy, -t);
  L[13] = fmaf(w * xy, z, L[13]);
  L[14] += x * fmaf(w, zz, -t);
  L[15] += y * fmaf(w, yy, -3.0f * t);
  L[16] += z * fmaf(w, yy, -t);
  L[17] += y * fmaf(w, zz, -t);
  L[18] += z * fmaf(w, zz, -3.0f * t);
  // third order: 105 m X / R^9 - w (sum over equal-index pairs of the other two d's)
  // + t (number of pairings into equal pairs), X the component's product of four d's
  const float a9 = 7.0f * w * ir2;  // 105 m / R^9
  L[19] += fmaf(a9 * xx, xx, fmaf(-6.0f * w, xx, 3.0f * t));
  L[20] += xy * fmaf(a9, xx, -3.0f * w);
  L[21] += xz * fmaf(a9, xx, -3.0f * w);
  L[22] += fmaf(a9 * xx, yy, fmaf(-w, xx + yy, t));
  L[23] += yz * fmaf(a9, xx, -w);
  L[24] += fmaf(a9 * xx, zz, fmaf(-w, xx + zz, t));
  L[25] += xy * fmaf(a9, yy, -3.0f * w);
  L[26] += xz * fmaf(a9, yy, -w);
  L[27] += xy * fmaf(a9, zz, -w);
  L[28] += xz * fmaf(a9, zz, -3.0f * w);
  L[29] += fmaf(a9 * yy, yy, fmaf(-6.0f * w, yy, 3.0f * t));
  L[30] += yz * fmaf(a9, yy, -3.0f * w);
  L[31] += fmaf(a9 * yy, zz, fmaf(-w, yy + zz, t));
  L[32] += yz * fmaf(a9, zz, -3.0f * w);
  L[33] += fmaf(a9 * zz, zz, fmaf(-6.0f * w, zz, 3.0f * t));
  // quadrupole {xx,yy,zz,xy} = Q0, {xz,yz} = Q1.xy
  const float qx = fmaf(Q0.x, x, fmaf(Q0.w, y, Q1.x * z));
  const float qy = fmaf(Q0.w, x, fmaf(Q0.y, y, Q1.y * z));
  const float qz = fmaf(Q1.x, x, fmaf(Q1.y, y, Q0.z * z));
  const float s = fmaf(x, qx, fmaf(y, qy, z * qz));
  const float f = 2.5f * s * ir7, e = 7.0f * f * ir2, g5 = 5.0f * ir7;
  L[0] += fmaf(f, x, -qx * ir5);
  L[1] += fmaf(f, y, -qy * ir5);
  L[2] += fmaf(f, z, -qz * ir5);
  L[3] += fmaf(Q0.x, ir5, fmaf(e, xx, -f)) - 2.0f * g5 * qx * x;
  L[4] += fmaf(Q0.y, ir5, fmaf(e, yy, -f)) - 2.0f * g5 * qy * y;
  L[5] += fmaf(Q0.z, ir5, fmaf(e, zz, -f)) - 2.0f * g5 * qz * z;
  L[6] += fmaf(Q0.w, ir5, e * xy) - g5 * fmaf(qx, y, qy * x);
  L[7] += fmaf(Q1.x, ir5, e * xz) - g5 * fmaf(qx, z, qz * x);
  L[8] += fmaf(Q1.y, ir5, e * yz) - g5 * fmaf(qy, z, qz * y);
}

// a(c + y) from the local coefficients: a_i = A0_i + A1_ij y_j + A2_ijk y_j y_k / 2
// + A3_ijkl y_j y_k y_l / 6, the symmetric sums written over distinct monomials.
__device__ __forceinline__ void far_l2p(const float* L, float x, float y, float z, float& ax,
                                        float& ay, float& az) {
  const float xx = x * x, yy = y * y, zz = z * z, xy = x * y, xz = x * z, yz = y * z;
  ax = L[0] + fmaf(L[3], x, fmaf(L[6], y, L[7] * z)) +
       0.5f * fmaf(L[9], xx, fmaf(L[12], yy, fmaf(L[14], zz,
              2.0f * fmaf(L[10], xy, fmaf(L[11], xz, L[13] * yz)))));
  ay = L[1] + fmaf(L[6], x, fmaf(L[4], y, L[8] * z)) +
       0.5f * fmaf(L[10], xx, fmaf(L[15], yy, fmaf(L[17], zz,
              2.0f * fmaf(L[12], xy, fmaf(L[13], xz, L[16] * yz)))));
  az = L[2] + fmaf(L[7], x, fmaf(L[8], y, L[5] * z)) +
       0.5f * fmaf(L[11], xx, fmaf(L[16], yy, fmaf(L[18], zz,
              2.0f * fmaf(L[13], xy, fmaf(L[14], xz, L[17] * yz)))));
  // third order over the cubic monomials scaled by 1 / (p! q! r!)
  const float c0 = xx * x * (1.0f / 6.0f), c1 = 0.5f * xx * y, c2 = 0.5f * xx * z,
              c3 = 0.5f * x * yy, c4 = xy * z, c5 = 0.5f * x * zz, c6 = yy * y * (1.0f / 6.0f),
              c7 = 0.5f * yy * z, c8 = 0.5f * y * zz, c9 = zz * z * (1.0f / 6.0f);
  ax += fmaf(L[19], c0, fmaf(L[20], c1, fmaf(L[21], c2, fmaf(L[22], c3, fmaf(L[23], c4,
        fmaf(L[24], c5, fmaf(L[25], c6, fmaf(L[26], c7, fmaf(L[27], c8, L[28] * c9)))))))));
  ay += fmaf(L[20], c0, fmaf(L[22], c1, fmaf(L[23], c2, fmaf(L[25], c3, fmaf(L[26], c4,
        fmaf(L[27], c5, fmaf(L[29], c6, fmaf(L[30], c7, fmaf(L[31], c8, L[32] * c9)))))))));
  az += fmaf(L[21], c0, fmaf(L[23], c1, fmaf(L[24], c2, fmaf(L[26], c3, fmaf(L[27], c4,
        fmaf(L[28], c5, fmaf(L[30], c6, fmaf(L[31], c7, fmaf(L[32], c8, L[33] * c9)))))))));
}

// The queued far nodes (node indices) into this lane's share of the local expansion:
// lane e takes entries e, e + 64, ...
__device__ __forceinline__ void far_drain(float* L, const SegDesc& s, const uint32_t* fl,
                                          uint32_t nf, uint32_t lane, float cx, float cy,
                                          float cz, float eps2) {
  for (uint32_t e = lane; e < nf; e += kGroup) {
    const uint32_t j = fl[e];
    const float4 A = gload4(reinterpret_cast<const float4*>(s.node), 2 * (size_t)j);
    far_m2l(L, A.x - cx, A.y - cy, A.z - cz, A.w, gload4(s.quad, 2 * (size_t)j),
            gload4(s.quad, 2 * (size_t)j + 1), eps2);
  }
}

// Bodies of the buckets in `rl[0, nr)` (first leaf, count) on the lane's target. The
// range is wave-uniform, so the body records come through scalar loads (the leaf array
// is read-only during the walk: a constant-address-space pointer gives s_load).
template <bool KAHAN>
__device__ __forceinline__ uint32_t bucket_terms(Acc3& a, const float4& me, const SegDesc& s,
                                                 const uint2* rl, uint32_t nr, float eps2) {
  const auto* leaf = (const __attribute__((address_space(4))) float*)s.leaf;
  uint32_t total = 0;
  for (uint32_t r = 0; r < nr; ++r) {
    const uint2 rg = rl[r];
    const uint32_t lo = __builtin_amdgcn_readfirstlane(rg.x);
    const uint32_t c = __builtin_amdgcn_readfirstlane(rg.y);
    for (uint32_t e = 0; e < c; ++e) {
      const auto* q = leaf + 4 * (size_t)(lo + e);
      point_term<KAHAN>(a, me, make_float4(q[0], q[1], q[2], q[3]), eps2);
    }
    total += c;
  }
  return total;
}

// Per-segment constants of the group walk (wave-uniform).
struct WalkSeg {
  uint32_t n, bucket, scap;
  bool loose_theta;      // theta > 1: the disjoint-box test is needed
  bool fits;             // the record offsets below fit (always in the wide form)
  const char* lbase;     // leaf array
  uint32_t dn32, dq32;   // classifier records and quadrupoles from it
};

template <bool WIDE>
__device__ __forceinline__ WalkSeg walk_seg(const SegDesc& s) {
  WalkSeg w;
  w.n = s.n;
  w.bucket = s.leaf_size;
  // the disjoint-box test is needed only above theta = 1 (theta >= 0: compared as bits, a
  // scalar test)
  w.loose_theta = __float_as_uint(s.theta) > __float_as_uint(1.0f);
  // The compact form addresses leaves, classifier records and quadrupoles by 32-bit byte
  // offsets from the leaf array (the launch takes the wide form when a segment's arrays do
  // not fit; a segment that does not fit here is walked per target)
  const uint64_t leaf_base = (uint64_t)s.leaf, node_base = (uint64_t)s.node;
  w.fits = WIDE || walk_off32(leaf_base, node_base, (uint64_t)s.quad, w.n);
  w.lbase = reinterpret_cast<const char*>(s.leaf);
  w.dn32 = (uint32_t)(node_base - leaf_base);
  w.dq32 = (uint32_t)((uint64_t)s.quad - leaf_base);
  // stack entries before a group falls back to the per-target walk
  w.scap = s.stack_cap && s.stack_cap < (uint32_t)kStackCap ? s.stack_cap : (uint32_t)kStackCap;
  return w;
}

// One walk group: its bodies' lanes, its box (centre c, half extent h) and radius.
struct WalkGroup {
  uint32_t g0, gcount, rep, sub, k, e0;
  bool owner, valid;
  float4 me;
  float gx0, gy0, gz0, gx1, gy1, gz1, cx, cy, cz, hx, hy, hz, rg;
  float near2;  // squared distance within which no node is accepted (theta <= 1), points excepted
};

template <bool FAR>
__device__ __forceinline__ WalkGroup walk_group(const SegDesc& s, uint32_t n, uint32_t g0,
                                                uint32_t gl, uint32_t lane) {
  WalkGroup g;
  g.g0 = g0;
  g.gcount = min(min(gl - g0 + 1u, (uint32_t)kGroup), n - g0);
  // A group of at most 32 bodies gives each body rep lanes (2, 3 or 4): the lists are
  // drained with stride rep, and the partial sums are folded into the body's first lane
  // (its owner) before the store.
  // (at most group_lanes; rep >= 1 also lets the compiler count the drains' trips)
  g.rep = max(min(g.gcount > 32u ? 1u : (g.gcount > 21u ? 2u : (g.gcount > 16u ? 3u : 4u)),
                  s.group_lanes), 1u);
  g.sub = (uint32_t)(lane >= g.gcount) + (uint32_t)(lane >= 2u * g.gcount) +
          (uint32_t)(lane >= 3u * g.gcount);
  g.owner = lane < g.gcount;
  g.valid = lane < g.rep * g.gcount;
  g.k = g0 + (g.valid ? lane - g.sub * g.gcount : 0u);
  g.e0 = g.valid ? g.sub : 0xFFFFu;  // this lane's first list entry
  return g;
}

template <bool FAR>
__device__ __forceinline__ void walk_group_box(const SegDesc& s, WalkGroup& g) {
  const float4 me = gload4(s.leaf, g.k);
  g.me = me;
  g.gx0 = wave_minf(me.x);
  g.gy0 = wave_minf(me.y);
  g.gz0 = wave_minf(me.z);
  g.gx1 = wave_maxf(me.x);
  g.gy1 = wave_maxf(me.y);
  g.gz1 = wave_maxf(me.z);
  g.cx = 0.5f * (g.gx0 + g.gx1);
  g.cy = 0.5f * (g.gy0 + g.gy1);
  g.cz = 0.5f * (g.gz0 + g.gz1);
  g.hx = 0.5f * (g.gx1 - g.gx0);
  g.hy = 0.5f * (g.gy1 - g.gy0);
  g.hz = 0.5f * (g.gz1 - g.gz0);
  // Distances from the box come from its centre and half extent, each rounded to 2^-24 of its
  // coordinates, so they may be 7 of these too large: a node much smaller than that at the box's
  // edge would be accepted by the group that holds its bodies. Nothing within near_coord of the
  // coordinates is accepted, which is farther than any such node (near_share).
  const float most = fmaxf(fmaxf(fmaxf(-g.gx0, g.gx1), fmaxf(-g.gy0, g.gy1)),
                           fmaxf(-g.gz0, g.gz1));
  const float t = most * s.near_coord;
  g.near2 = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(fmaxf(t * t, 1.2e-38f))));
  g.rg = FAR ? sqrtf(fmaf(g.hx, g.hx, fmaf(g.hy, g.hy, g.hz * g.hz))) : 0.0f;
}

// The interaction lists of one round (at most 64 entries each; far nodes queue up). The
// quadrupole list holds com and mass with the moments, or (SPLIT) with the node's index, the
// moments then being fetched by the wave that uses them. (LDS comes in granules of 1,280 B:
// one word more than the 7,680 B of the build without far field costs a wave per SIMD, 3%.)
template <bool QUAD, bool SPLIT>
struct WalkLists {
  float4 pl[kListCap];
  float4 qa[QUAD ? kListCap : 1], qb[QUAD && !SPLIT ? kListCap : 1];
  float2 qc[QUAD && !SPLIT ? kListCap : 1];
  uint32_t qi[QUAD && SPLIT ? kListCap : 0];
  uint2 rl[kRangeCap];
};
struct ListCounts {
  uint32_t np, nq, nr;
};

// Traceless quadrupole {xx,yy,zz,xy}, {xz,yz} of node ni.
template <bool WIDE>
__device__ __forceinline__ void node_moments(const SegDesc& s, const WalkSeg& w, uint32_t ni,
                                             float4& q0, float2& q1) {
  float4 hi;
  if (!WIDE) {
    const uint32_t qoff = w.dq32 + (ni << 5);
    q0 = gload4_at(w.lbase, qoff);
    hi = gload4_at(w.lbase + 16, qoff);
  } else {
    q0 = gload4(s.quad, 2 * (size_t)ni);
    hi = gload4(s.quad, 2 * (size_t)ni + 1);
  }
  q1 = make_float2(hi.x, hi.y);
}

// One round: tests the wave's stack entries u (live: lanes below the round's count), fills
// the lists, queues far nodes and pushes the children of opened nodes. False: the stack
// would overflow.
template <bool QUAD, bool FAR, bool WIDE, bool BOX, bool SPLIT>
__device__ __forceinline__ bool walk_round(const SegDesc& s, const WalkSeg& w, const WalkGroup& g,
                                           bool live, uint32_t u, uint32_t* stk, uint32_t& sp,
                                           WalkLists<QUAD, SPLIT>& L, ListCounts& c,
                                           uint32_t* fl,
                                           uint32_t& nf) {
  // Classify without divergent branches: every lane loads one record and the node
  // fields, and the predicates below are balloted, so the ballots that build the
  // lists always see the full wave.
  // Lists: point/monopole, quadrupole node, open (children pushed), bucket (a node of
  // at most leaf_size bodies that is not accepted: its bodies are summed directly),
  // far (local expansion).
  const bool is_node = live & ((int32_t)u < 0);
  const bool is_leaf = live & ((int32_t)u >= 0);
  // node index (0 on a leaf lane, which reads node 0's record, a line every such
  // lane shares, and ignores it) and leaf index
  const uint32_t ni = is_node ? u & ~kEntryNode : 0u, li = u;
  const size_t nr2 = 2 * (size_t)ni;  // record as two float4
  const char* const lbase16 = w.lbase + 16;  // second float4 of a record
  // a leaf's record (position, mass) has the layout of a node's first float4 (com,
  // mass), so one load serves both kinds
  float4 A, H;
  if (!WIDE) {
    const uint32_t noff = w.dn32 + (ni << 5);
    A = gload4_at(w.lbase, is_leaf ? li << 4 : noff);
    H = gload4_at(lbase16, noff);
  } else {
    const uint64_t abase = is_leaf ? (uint64_t)s.leaf : (uint64_t)s.node;
    A = gload4(reinterpret_cast<const float4*>(abase), is_leaf ? li : 2u * ni);
    H = gload4(reinterpret_cast<const float4*>(s.node), nr2 + 1);
  }
  // The box record only where it is needed (wave-uniform): the disjoint-box test
  // (apart) and the bucket test's leaf range
  bool apart = true;
  uint32_t nlo = 0u, ncount = 2u;  // an internal node holds at least two bodies
  if (BOX) {
    const float4* brec = reinterpret_cast<const float4*>(s.box);
    const float4 B = gload4(brec, nr2), Cc = gload4(brec, nr2 + 1);
    // Every point of the node's box lies within sqrt(3) s / 2 + delta of its com
    // (half its diagonal from the box centre, delta from there to the com), and an
    // accepted com is at least s / theta + delta from the group box, so for theta <= 1
    // (1 / theta > sqrt(3) / 2 with a margin) acceptance implies disjoint boxes, beyond
    // near2. (A node of size 0 is one point, whose monopole is exact for every body.)
    if (w.loose_theta)
      apart = (Cc.x < g.gx0) | (B.x > g.gx1) | (Cc.y < g.gy0) | (B.y > g.gy1) |
              (Cc.z < g.gz0) | (B.z > g.gz1);
    nlo = __float_as_uint(B.w);
    ncount = __float_as_uint(Cc.w) - nlo + 1u;
  }
  // com relative to the group centre; distance from the group box to the com
  const float dx = A.x - g.cx, dy = A.y - g.cy, dz = A.z - g.cz;
  const float ex = fmaxf(fabsf(dx) - g.hx, 0.f);
  const float ey = fmaxf(fabsf(dy) - g.hy, 0.f);
  const float ez = fmaxf(fabsf(dz) - g.hz, 0.f);
  const float dmin2 = ex * ex + ey * ey + ez * ez;
  const bool massive = A.w > 0.0f;
  const bool node_live = is_node & massive;
  // the acceptance radius, at least near2 for a node that is not a single point (one
  // instruction more: H.w > 0 there); above theta = 1 the boxes have been compared
  const float lim = BOX && w.loose_theta ? H.x : __builtin_amdgcn_fmed3f(H.x, g.near2, H.w * 1e30f);
  const bool accept = node_live & apart & (dmin2 >= lim);  // boxes disjoint too
  const bool near = node_live & !accept;
  const bool bkt = BOX & near & (ncount <= w.bucket);  // (leaf_size > 1 needs boxes)
  const bool open = near & !bkt;
  // accepted and well separated from the whole group -> local expansion (node radius
  // about its com from the record)
  bool far = false;
  if (FAR) {
    const float rn = fabsf(H.w) + g.rg;
    far = accept & (rn * rn <= s.far2 * fmaf(dx, dx, fmaf(dy, dy, dz * dz)));
  }
  // an accepted node that also passes the opening test at theta * mono_ratio is a
  // monopole: the squared band radius is in the record
  const bool mono = QUAD && accept && dmin2 >= H.z;
  const bool point = (is_leaf & massive) | (!QUAD & accept) | (mono & !far);
  const bool quadn = QUAD & accept & !point & !far;
  const uint32_t cl = left_entry(__float_as_uint(H.y)), cr = right_entry(__float_as_uint(H.y));
  const unsigned long long m1 = __ballot(point), m2 = __ballot(quadn), m3 = __ballot(open);
  unsigned long long m4 = 0ull;
  if (BOX) m4 = __ballot(bkt);
  const uint32_t c3 = (uint32_t)__popcll(m3);
  if (sp + 2u * c3 > w.scap) return false;
  if (point) L.pl[lanes_below(m1)] = A;
  if (QUAD && quadn) {  // only accepted nodes fetch their moments
    const uint32_t q = lanes_below(m2);
    L.qa[q] = A;
    if (SPLIT) {
      L.qi[q] = ni;
    } else {
      float4 q0;
      float2 q1;
      node_moments<WIDE>(s, w, ni, q0, q1);
      L.qb[q] = q0;
      L.qc[q] = q1;
    }
  }
  if (open) {
    const uint32_t q = sp + 2u * lanes_below(m3);
    stk[q] = cr;
    stk[q + 1] = cl;  // left child popped first
  }
  if (bkt) L.rl[lanes_below(m4)] = make_uint2(nlo, ncount);
  if (FAR) {
    const unsigned long long m5 = __ballot(far);
    if (far) fl[nf + lanes_below(m5)] = ni;
    nf += (uint32_t)__popcll(m5);
  }
  c.np = (uint32_t)__popcll(m1);
  c.nq = (uint32_t)__popcll(m2);
  c.nr = (uint32_t)__popcll(m4);
  sp += 2u * c3;
  return true;
}

// The point list of one round: entries of stride rep from the lane's first. With one lane
// per body (groups of more than 32 bodies) every lane takes every entry, so the loop runs
// on a wave-uniform index (scalar loop control, LDS reads at immediate offsets); the lanes
// beyond the group are masked off (their terms would never be stored; masked, the walk
// measured 1.4% faster at the same instruction count).
template <bool KAHAN, int U, class Lists>
__device__ __forceinline__ uint32_t drain_points(Acc3& a, const SegDesc& s, const WalkGroup& g,
                                                 const Lists& L, const ListCounts& c,
                                                 float eps2, bool soft) {
  const uint32_t np = c.np;
  if (np != 0u) {
    if (g.rep == 1u && soft) {
      if (g.valid)
#pragma unroll U
        for (uint32_t e = 0; e < np; ++e) point_term<KAHAN, false>(a, g.me, L.pl[e], eps2);
    } else if (g.rep == 1u) {
      if (g.valid)
#pragma unroll U
        for (uint32_t e = 0; e < np; ++e) point_term<KAHAN>(a, g.me, L.pl[e], eps2);
    } else {
#pragma unroll U
      for (uint32_t e = g.e0; e < np; e += g.rep) point_term<KAHAN>(a, g.me, L.pl[e], eps2);
    }
  }
  uint32_t terms = 0;
  if (c.nr != 0u) {  // bucket bodies come through scalar loads: owners only
    if (g.owner) terms = bucket_terms<KAHAN>(a, g.me, s, L.rl, c.nr, eps2);
  }
  return terms;
}

// The quadrupole list of one round (its moments in qb, qc), as the points.
template <bool KAHAN, int U>
__device__ __forceinline__ void drain_quads(Acc3& a, const WalkGroup& g, const float4* qa,
                                            const float4* qb, const float2* qc, uint32_t nq,
                                            float eps2) {
  if (nq == 0u) return;
  if (g.rep == 1u) {
    if (g.valid)
#pragma unroll U
      for (uint32_t e = 0; e < nq; ++e) quad_term<KAHAN>(a, g.me, qa[e], qb[e], qc[e], eps2);
  } else {
#pragma unroll U
    for (uint32_t e = g.e0; e < nq; e += g.rep)
      quad_term<KAHAN>(a, g.me, qa[e], qb[e], qc[e], eps2);
  }
}

// Per-target fallback of a group whose stack would overflow: the aligned target sets of the
// per-target walk that hold the group's bodies, so that a body's sum is the reference
// build's bit for bit (but for nodes a few ulps wide, opened there without their boxes). The
// stack array serves as that walk's stack.
template <bool KAHAN, bool COUNT, bool QUAD>
__device__ __forceinline__ Acc3 group_fallback(const SegDesc& s, const WalkGroup& g, uint32_t n,
                                               bool boxes, uint32_t lane, uint32_t* stk,
                                               unsigned long long& f_int,
                                               unsigned long long& n_vis) {
  // what depends on the lane is computed here, not kept in registers through every walk
  if (!QUAD) asm volatile("" : "+v"(lane));
  Acc3 a = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (uint32_t q = g.g0 / kTargets * kTargets; q < g.g0 + g.gcount; q += kTargets) {
    uint32_t mine = 0;  // the set's targets in this group (counted once)
    for (uint32_t i = 0; i < (uint32_t)kTargets; ++i) mine |= q + i - g.g0 < g.gcount ? 1u << i : 0u;
    const Acc3 r = target_walk<KAHAN, COUNT, QUAD>(
        s, __builtin_amdgcn_readfirstlane(q), min(n - q, (uint32_t)kTargets), boxes, lane, stk,
        reinterpret_cast<uint8_t*>(stk + kOpenCap), mine, f_int, n_vis);
    const int src = (int)((g.k - q) & (kTargets - 1)) * kTargetLanes;
    const Acc3 mine_sum = acc_shfl<KAHAN>(r, src);
    if (g.owner && g.k - q < (uint32_t)kTargets) a = mine_sum;
    wave_lds_order();
  }
  return a;
}

// Folds each body's lanes into its owner (lanes lane + j gcount < 64).
template <bool KAHAN>
__device__ __forceinline__ void fold_lanes(Acc3& a, const WalkGroup& g, uint32_t lane) {
  if (g.rep <= 1u) return;
  const float px = a.x - (KAHAN ? a.cx : 0.f), py = a.y - (KAHAN ? a.cy : 0.f),
              pz = a.z - (KAHAN ? a.cz : 0.f);
  for (uint32_t j = 1; j < g.rep; ++j) {
    const int src = (int)((lane + j * g.gcount) & 63u);
    const float qx = __shfl(px, src), qy = __shfl(py, src), qz = __shfl(pz, src);
    if (g.owner) acc_add<KAHAN>(a, qx, qy, qz);
  }
}

template <bool B>
struct BoolTag {
  static constexpr bool value = B;
};

// The far-field build holds a 34-coefficient local expansion per lane: without a bound
// the compiler takes about 147 VGPRs (3 waves per SIMD: walk +21%); at 4 waves per SIMD it
// fits 128 VGPRs without spilling. The builds without quadrupoles are held to 80 VGPRs (6
// waves per SIMD): the inlined per-target fallback took 84 (5 waves), 96 compensated. 2^22
// bodies, theta = 0.5 / 1 / 1.3: 5,345 / 1,591 / 1,401 us at 5 waves, 5,289 / 1,514 / 1,315 at 6;
// compensated 7,394 / 2,167 / 1,741 and 7,406 / 2,143 / 1,670. Those with quadrupoles and no
// far field fit 96 VGPRs (5 waves). The counting build is left unbounded (it only counts).
template <bool KAHAN, bool COUNT, bool QUAD, bool FAR, bool WIDE>
__global__ void __launch_bounds__(kGroup)
__attribute__((amdgpu_waves_per_eu(COUNT ? 1 : (QUAD ? (FAR ? 4 : 5) : 6))))
k_walk_group(const SegDesc* __restrict__ segs, const Tile* __restrict__ tiles, uint32_t ntiles,
             int mode) {
  __shared__ uint32_t stk[kStackCap];
  __shared__ WalkLists<QUAD, false> lists;
  __shared__ uint32_t fl[FAR ? kFarCap : 1];
  const uint32_t lane = threadIdx.x;
  for (uint32_t t = xcd_block(); t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const SegDesc& s = segs[tl.seg];
    if (tl.start == 0 && lane < 6) bbox_neutral(s.bbox, lane);
    const WalkSeg w = walk_seg<WIDE>(s);
    const uint32_t n = w.n;
    const float eps2 = s.eps2;
    const bool soft = eps2 >= kR2Floor;  // r^2 >= eps^2 needs no floor
    const bool need_box = w.loose_theta || w.bucket > 1u;  // box records (bounds, leaf range)
    // the walk groups (subtrees of at most kGroup bodies, marked by the tree build)
    // that start in this chunk of sorted leaves, one after the other
    const uint32_t ge = lane < tl.count ? gbl(s.gend)[tl.start + lane] : kEnd;
    unsigned long long starts = __ballot(ge != kEnd);
    unsigned long long t_int = 0, t_vis = 0, t_quad = 0, t_far = 0, t_rounds = 0;
    uint32_t t_peak = 0;
    while (starts != 0ull) {
      const uint32_t l0 = (uint32_t)__builtin_ctzll(starts);
      starts &= starts - 1ull;
      WalkGroup g = walk_group<FAR>(s, n, tl.start + l0, (uint32_t)__shfl((int)ge, (int)l0), lane);
      if (s.active) {  // masked walk: a group without an active body is skipped
        const bool on = g.owner && s.active[min(s.vals[0][g.k], n - 1)] != 0;
        if (__ballot(on) == 0ull) continue;
      }
      walk_group_box<FAR>(s, g);
      float loc[FAR ? kLocal : 1];  // this lane's share of the local expansion
#pragma unroll
      for (int c = 0; c < (FAR ? kLocal : 1); ++c) loc[c] = 0.0f;
      Acc3 a = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      unsigned long long n_int = 0, n_vis = 0, n_quad = 0, n_far = 0, n_rounds = 0, f_int = 0;
      uint32_t sp = w.fits ? 1u : 0u, nf = 0, peak = 1;
      bool overflow = !w.fits;
      // stack entries: leaf g -> g, internal node g -> g | 2^31 (the root is node 0)
      if (lane == 0) stk[0] = (n == 1) ? 0u : kEntryNode;
      __syncthreads();
      // The rounds, specialised on whether the node tests need the box record (wave-
      // uniform per segment), so that the common case carries none of its instructions
      auto rounds = [&](auto box_tag) {
        constexpr bool BOX = decltype(box_tag)::value;
        // every node is pushed at most once, so a round count above 2n only happens on a
        // corrupted tree; the bound keeps such input from spinning forever
        for (uint32_t round = 0; sp > 0; ++round) {
          if (round > 2 * n + 2) {
            overflow = true;
            break;
          }
          const uint32_t m = sp < 64u ? sp : 64u;
          const bool live = lane < m;
          sp -= m;
          const uint32_t u = live ? stk[sp + lane] : 0u;  // beyond the round: leaf 0, not live
          if (COUNT && lane == 0) {
            n_vis += m;
            ++n_rounds;
          }
          ListCounts c;
          if (!walk_round<QUAD, FAR, WIDE, BOX, false>(s, w, g, live, u, stk, sp, lists, c, fl,
                                                       nf)) {
            overflow = true;
            break;
          }
          peak = sp > peak ? sp : peak;
          __syncthreads();
          const uint32_t bt = drain_points<KAHAN, 2>(a, s, g, lists, c, eps2, soft);
          if (QUAD) drain_quads<KAHAN, 2>(a, g, lists.qa, lists.qb, lists.qc, c.nq, eps2);
          if (COUNT) {
            n_int += bt;
            if (g.e0 < c.np) n_int += (c.np - g.e0 + g.rep - 1u) / g.rep;
            if (g.e0 < c.nq) n_quad += (c.nq - g.e0 + g.rep - 1u) / g.rep;
          }
          if (FAR && nf >= 64u) {  // one far node per lane
            far_drain(loc, s, fl, nf, lane, g.cx, g.cy, g.cz, eps2);
            if (COUNT && lane == 0) n_far += nf;
            nf = 0;
          }
          __syncthreads();
        }
      };
      if (need_box) rounds(BoolTag<true>{});
      else rounds(BoolTag<false>{});
      if (overflow) {
        n_int = 0;
        n_quad = 0;
        a = group_fallback<KAHAN, COUNT, QUAD>(s, g, n, need_box, lane, stk, f_int, n_vis);
        if (lane == 0) atomicAdd(&s.counters[kCntOverflow], 1ull);
      } else {  // the lists were drained in the last round
        fold_lanes<KAHAN>(a, g, lane);
      }
      if (FAR && !overflow) {
        far_drain(loc, s, fl, nf, lane, g.cx, g.cy, g.cz, eps2);
        if (COUNT && lane == 0) n_far += nf;
#pragma unroll
        for (int c = 0; c < (FAR ? kLocal : 1); ++c) loc[c] = wave_sumf(loc[c]);
        if (g.owner) {  // the other lanes' partial sums are folded already
          float fx, fy, fz;
          far_l2p(loc, g.me.x - g.cx, g.me.y - g.cy, g.me.z - g.cz, fx, fy, fz);
          acc_add<KAHAN>(a, fx, fy, fz);
        }
      }
      if (g.owner) store_acc<KAHAN>(s, g.k, a, mode);
      if (COUNT) {
        // n_int is per target (uniform over valid lanes unless the group fell back)
        t_int += wave_sum_u64((g.valid ? n_int : 0ull) + f_int);
        t_quad += wave_sum_u64(g.valid ? n_quad : 0ull);
        t_vis += wave_sum_u64(n_vis);
        t_far += wave_sum_u64(n_far);
        t_rounds += wave_sum_u64(n_rounds);
        t_peak = peak > t_peak ? peak : t_peak;
      }
      __syncthreads();
    }
    if (COUNT && lane == 0 && (t_int | t_quad | t_vis)) {
      atomicAdd(&s.counters[kCntInteractions], t_int);
      atomicAdd(&s.counters[kCntQuad], t_quad);
      atomicAdd(&s.counters[kCntVisits], t_vis);
      atomicMax(&s.counters[kCntMaxStack], (unsigned long long)t_peak);
      atomicAdd(&s.counters[kCntFar], t_far);
      atomicAdd(&s.counters[kCntRounds], t_rounds);
    }
  }
}

// The same walk with its work on two waves of a block (three with the far field), for
// launches that would leave the chip idle: wave 0 pops, classifies and fills the lists of a
// round, wave 1 drains them in order, fetching a round's quadrupole moments while it drains
// its points, and wave 2 folds the queued far nodes. A ring of rounds in LDS lets the
// producer run ahead, so that neither waits for the other's long rounds. Lists, queue order
// and every sum are those of k_walk_group: the results are the same bits and the launch may
// choose by size. One wave alone spends a group's time in turn on the rounds' dependent
// loads, the terms' chains and the far nodes' fetches; here they overlap. Plummer spheres at
// theta = 0.5, one wave / split: with far field 155 / 54 us at 2,000 bodies, 194 / 88 at
// 16,384 (61 of it the producer's chain of loads), 282 / 208 at 100,003; quadrupoles only
// 193 / 81, 367 / 179 (now the slowest group's terms, 58 without them) and 566 / 484 us.
// With a barrier per round instead of the ring: 58, 96 and 234 us with far field.
constexpr uint32_t kSplitSlots = 4;  // blocks per walk tile: the tile's groups go to them in turn
// Rounds in flight: 8 with the far field (4: +5% at 40,000 and 100,003 bodies); the longer
// lists without it fill the LDS at 8 (100,003 bodies: 552 us against 484 at 4).
constexpr uint32_t split_ring(bool far) { return far ? 8u : 4u; }

template <bool QUAD>
struct SplitRound {
  WalkLists<QUAD, true> lists;
  ListCounts c;
  uint32_t last;  // 1: the walk's last round, 2: the stack overflowed
};

// A value that is the same in every lane, as a scalar.
__device__ __forceinline__ uint32_t uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// Progress counters in LDS between the waves of a block: a wave publishes after its LDS
// writes (release) and reads after it has seen the count (acquire). All waves of a block
// are resident and every wait ends: the producer's rounds are bounded, and what it waits
// for is drained by waves that wait only for it.
__device__ __forceinline__ void publish(uint32_t* count, uint32_t v, uint32_t lane) {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  if (lane == 0) __hip_atomic_store(count, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// Until *count >= v (counts only grow); returns the count seen.
__device__ __forceinline__ uint32_t await_count(const uint32_t* count, uint32_t v) {
  uint32_t c;
  while ((c = uniform(__hip_atomic_load(count, __ATOMIC_RELAXED,
                                        __HIP_MEMORY_SCOPE_WORKGROUP))) < v)
    __builtin_amdgcn_s_sleep(1);
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  return c;
}

template <bool KAHAN, bool QUAD, bool FAR, bool WIDE>
__global__ void __launch_bounds__(64 * (2 + FAR))
k_walk_split(const SegDesc* __restrict__ segs, const Tile* __restrict__ tiles, uint32_t ntiles,
             int mode) {
  __shared__ uint32_t stk[kStackCap];
  constexpr uint32_t kRing = split_ring(FAR);
  __shared__ SplitRound<QUAD> ring[kRing];
  __shared__ float4 qb[QUAD ? kListCap : 1];  // moments of the round being drained
  __shared__ float2 qc[QUAD ? kListCap : 1];
  __shared__ uint32_t fl[2][FAR ? kFarCap : 1];  // far nodes: one queue fills, one is folded
  __shared__ uint32_t fn[2], flast[2];
  __shared__ float expansion[FAR ? kLocal : 1];
  __shared__ uint32_t made, drained, far_made, far_done;
  const uint32_t lane = threadIdx.x & 63u, role = threadIdx.x >> 6;
  // blocks [slot * ntiles, (slot + 1) * ntiles) take the tiles' groups slot, slot +
  // kSplitSlots, ...: most tiles hold one or two groups, so the blocks with work come first
  // and lie on every XCD
  const uint32_t slot = blockIdx.x / ntiles;
  const Tile tl = tiles[blockIdx.x % ntiles];
  const SegDesc& s = segs[tl.seg];
  if (tl.start == 0 && slot == 0 && threadIdx.x < 6) bbox_neutral(s.bbox, threadIdx.x);
  const WalkSeg w = walk_seg<WIDE>(s);
  const uint32_t n = w.n;
  const float eps2 = s.eps2;
  const bool soft = eps2 >= kR2Floor;
  const bool need_box = w.loose_theta || w.bucket > 1u;
  const uint32_t ge = lane < tl.count ? gbl(s.gend)[tl.start + lane] : kEnd;
  unsigned long long starts = __ballot(ge != kEnd);
  for (uint32_t i = 0; starts != 0ull; ++i, starts &= starts - 1ull) {
    if (i % kSplitSlots != slot) continue;
    const uint32_t l0 = (uint32_t)__builtin_ctzll(starts);
    WalkGroup g = walk_group<FAR>(s, n, tl.start + l0, (uint32_t)__shfl((int)ge, (int)l0), lane);
    if (s.active) {
      const bool on = g.owner && s.active[min(s.vals[0][g.k], n - 1)] != 0;
      if (__ballot(on) == 0ull) continue;
    }
    if (threadIdx.x == 0) made = drained = far_made = far_done = 0u;
    walk_group_box<FAR>(s, g);
    __syncthreads();
    if (role == 0) {
      uint32_t sp = w.fits ? 1u : 0u, nf = 0, hand = 0, seen = 0;
      if (lane == 0) stk[0] = (n == 1) ? 0u : kEntryNode;
      auto rounds = [&](auto box_tag) {
        constexpr bool BOX = decltype(box_tag)::value;
        for (uint32_t round = 0;; ++round) {
          if (round >= seen + kRing) seen = await_count(&drained, round + 1u - kRing);
          SplitRound<QUAD>& r = ring[round % kRing];
          const uint32_t m = sp < 64u ? sp : 64u;
          const bool live = lane < m;
          sp -= m;
          wave_lds_order();  // this wave's own stack
          const uint32_t u = live ? stk[sp + lane] : 0u;
          ListCounts c = {0u, 0u, 0u};
          const bool ok = w.fits && round <= 2 * n + 2 &&
                          walk_round<QUAD, FAR, WIDE, BOX, true>(
                              s, w, g, live, u, stk, sp, r.lists, c, fl[FAR ? hand & 1u : 0u], nf);
          const uint32_t last = !ok ? 2u : (sp == 0u ? 1u : 0u);
          if (lane == 0) {
            r.c = c;
            r.last = last;
          }
          publish(&made, round + 1u, lane);
          // far nodes go over 64 or more at a time, as one wave would drain them, and the
          // rest after the last round; the queue filled next was handed over before this one
          if (FAR && (nf >= 64u || last != 0u)) {
            if (lane == 0) {
              fn[hand & 1u] = last == 2u ? 0u : nf;
              flast[hand & 1u] = last;
            }
            publish(&far_made, ++hand, lane);
            nf = 0;
            if (last == 0u && hand >= 2u) await_count(&far_done, hand - 1u);
          }
          if (last != 0u) break;
        }
      };
      if (need_box) rounds(BoolTag<true>{});
      else rounds(BoolTag<false>{});
      __syncthreads();
    } else if (role == 1) {
      Acc3 a = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      uint32_t last = 0, seen = 0;
      for (uint32_t round = 0; last == 0u; ++round) {
        if (round >= seen) seen = await_count(&made, round + 1u);
        const SplitRound<QUAD>& r = ring[round % kRing];
        last = uniform(r.last);
        if (last != 2u) {
          const ListCounts c = {uniform(r.c.np), uniform(r.c.nq), uniform(r.c.nr)};
          const uint32_t nq = c.nq;
          float4 m0 = make_float4(0.f, 0.f, 0.f, 0.f);
          float2 m1 = make_float2(0.f, 0.f);
          if (QUAD && lane < nq) node_moments<WIDE>(s, w, r.lists.qi[QUAD ? lane : 0], m0, m1);
          drain_points<KAHAN, 4>(a, s, g, r.lists, c, eps2, soft);
          if (QUAD && nq != 0u) {
            wave_lds_order();  // this wave's own moments
            if (lane < nq) {
              qb[QUAD ? lane : 0] = m0;
              qc[QUAD ? lane : 0] = m1;
            }
            wave_lds_order();
            drain_quads<KAHAN, 4>(a, g, r.lists.qa, qb, qc, nq, eps2);
          }
        }
        publish(&drained, round + 1u, lane);
      }
      __syncthreads();
      if (last == 2u) {
        unsigned long long unused = 0;
        a = group_fallback<KAHAN, false, QUAD>(s, g, n, need_box, lane, stk, unused, unused);
        if (lane == 0) atomicAdd(&s.counters[kCntOverflow], 1ull);
      } else {
        fold_lanes<KAHAN>(a, g, lane);
        if (FAR && g.owner) {
          float fx, fy, fz;
          far_l2p(expansion, g.me.x - g.cx, g.me.y - g.cy, g.me.z - g.cz, fx, fy, fz);
          acc_add<KAHAN>(a, fx, fy, fz);
        }
      }
      if (g.owner) store_acc<KAHAN>(s, g.k, a, mode);
    } else if constexpr (FAR) {
      float loc[kLocal];
#pragma unroll
      for (int c = 0; c < kLocal; ++c) loc[c] = 0.0f;
      uint32_t last = 0;
      for (uint32_t hand = 0; last == 0u; ++hand) {
        await_count(&far_made, hand + 1u);
        last = uniform(flast[hand & 1u]);
        far_drain(loc, s, fl[hand & 1u], uniform(fn[hand & 1u]), lane, g.cx, g.cy, g.cz, eps2);
        publish(&far_done, hand + 1u, lane);
      }
#pragma unroll
      for (int c = 0; c < kLocal; ++c) {
        loc[c] = wave_sumf(loc[c]);
        if (lane == 0) expansion[c] = loc[c];
      }
      __syncthreads();
    }
    __syncthreads();  // the lists, expansion and stack are free for the next group
  }
}

// ----------------------------------------------------------------------------------
// 8. FP64 diagnostics (core/src/diagnostics.rs:8-68): per-tile partial sums in a
//    fixed reduction order, then a fixed-order sum over each segment's tiles.
//    Partial record: KE, P xyz, L xyz, sum m*x xyz, sum m  (11 doubles).
// ----------------------------------------------------------------------------------

__global__ void __launch_bounds__(kBlock)
k_diag_partial(const SegDesc* __restrict__ segs, const Tile* __restrict__ tiles, uint32_t ntiles,
               double* __restrict__ partial) {
  __shared__ double sh[kDiagRecord][kBlock / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (uint32_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const SegDesc& s = segs[tl.seg];
    double acc[kDiagRecord];
    for (int q = 0; q < kDiagRecord; ++q) acc[q] = 0.0;
    for (uint32_t e = threadIdx.x; e < tl.count; e += kBlock) {
      const size_t i = tl.start + e;
      const double m = s.m[i];
      const double x = s.x[3 * i], y = s.x[3 * i + 1], z = s.x[3 * i + 2];
      const double vx = s.v[3 * i], vy = s.v[3 * i + 1], vz = s.v[3 * i + 2];
      acc[0] += 0.5 * m * (vx * vx + vy * vy + vz * vz);
      acc[1] += vx * m;
      acc[2] += vy * m;
      acc[3] += vz * m;
      acc[4] += (y * vz - z * vy) * m;
      acc[5] += (z * vx - x * vz) * m;
      acc[6] += (x * vy - y * vx) * m;
      acc[7] += x * m;
      acc[8] += y * m;
      acc[9] += z * m;
      acc[10] += m;
    }
    for (int q = 0; q < kDiagRecord; ++q) {
      const double r = wave_sum(acc[q]);
      if (lane == 0) sh[q][w] = r;
    }
    __syncthreads();
    if (threadIdx.x < kDiagRecord) {
      double r = 0.0;
      for (int k = 0; k < kBlock / 64; ++k) r += sh[threadIdx.x][k];
      partial[(size_t)t * kDiagRecord + threadIdx.x] = r;
    }
    __syncthreads();
  }
}

__global__ void k_diag_final(const SegDesc* __restrict__ segs, uint32_t nseg,
                             const double* __restrict__ partial, double* __restrict__ out) {
  const uint32_t sidx = blockIdx.x;
  if (sidx >= nseg || threadIdx.x >= kDiagRecord) return;
  const SegDesc& s = segs[sidx];
  double r = 0.0;
  for (uint32_t t = s.sort_tile0; t < s.sort_tile0 + s.sort_tiles; ++t)
    r += partial[(size_t)t * kDiagRecord + threadIdx.x];
  out[(size_t)sidx * kDiagRecord + threadIdx.x] = r;
}

// ----------------------------------------------------------------------------------
// 9. FP64 direct summation (solvers/src/direct_sum.rs:25-45 pair kernel) onto a
//    target subset, and the FP64 softened potential (solvers/src/potential.rs:17-27)
//    as per-wave partials.
// ----------------------------------------------------------------------------------

// A wave takes 64 bodies, one per lane, against a range of sources. The source index is
// wave-uniform, so positions and masses come through scalar loads and reach the arithmetic
// as SGPR operands: no LDS, no barriers, any number of independent waves.
// Bound: FP64 issue. Per pair about 21 instructions for the force and 18 for the potential
// (3 differences, 3 FMAs for r^2, the f32 estimate and its two conversions, the refinement,
// the sums). Before, 27 and 25 with two Newton steps, LDS reads of every source by every
// wave, and, for the potential, one block per 256 rows of which the first met all n sources
// and the last 256. 4,096 targets x 2^20 sources: 4.65 -> 3.24 ms; potential of 131,072
// bodies: 21.1 -> 5.4 ms (1.6e12 pairs/s), of 1,000: 0.19 -> 0.03 ms. Two bodies per lane
// measured slower for the force (3.56 ms, twice the registers) and 2% faster for the
// potential; batches of 3 or 6 sources 4% and 7% slower than 4.
constexpr int kUnroll = 4;  // sources per batch: their estimates are checked together

template <class T>
__device__ __forceinline__ const __attribute__((address_space(4))) T* cst(const T* p) {
  return (const __attribute__((address_space(4))) T*)p;
}

// y ~ x^-1/2 from the f32 hardware estimate (relative error below 2^-22 with the conversion
// of x) and e = 1 - x y^2, |e| < 1e-6: x^-1/2 = y (1 - e)^-1/2. Where x is not a normal f32
// (or is 0, infinite or NaN) e is not small and the caller takes the IEEE square root and
// division instead.
__device__ __forceinline__ bool small_e(double e) { return fabs(e) < 1e-3; }

// m x^-3/2 = m y^3 (1 - e)^-3/2, the series to e^2 (the next term is below 3e-18)
__device__ __forceinline__ double inv_cube(double m, double x, bool& bad) {
  const double y = (double)__builtin_amdgcn_rsqf((float)x), y2 = y * y;
  const double e = fma(-x, y2, 1.0);
  bad |= !small_e(e);
  return (m * y) * (y2 * fma(fma(1.875, e, 1.5), e, 1.0));
}
__device__ __forceinline__ double inv_cube_ieee(double m, double x) {
  const double y = 1.0 / sqrt(x);
  return m * (y * y * y);
}
// x^-1/2, the series to e^2 (the next term is below 4e-19)
__device__ __forceinline__ double inv_root(double x, bool& bad) {
  const double y = (double)__builtin_amdgcn_rsqf((float)x);
  const double e = fma(-x * y, y, 1.0);
  bad |= !small_e(e);
  return fma(fma(0.375, e, 0.5), y * e, y);
}

// The sources [j0, j1) in batches of kUnroll, the next batch's scalar loads issued before
// this one's arithmetic (they return out of order, so a batch waits for all of its own).
template <class PX, class PM, class F>
__device__ __forceinline__ void sweep(PX sx, PM sm, uint32_t j0, uint32_t j1, F&& batch) {
  uint32_t j = j0;
  if (j + kUnroll <= j1) {
    double bx[3 * kUnroll], bm[kUnroll];
#pragma unroll
    for (int q = 0; q < 3 * kUnroll; ++q) bx[q] = (sx + 3 * (size_t)j)[q];
#pragma unroll
    for (int q = 0; q < kUnroll; ++q) bm[q] = (sm + j)[q];
    for (;;) {
      const uint32_t jn = j + kUnroll;
      const bool more = jn + kUnroll <= j1;
      const uint32_t jl = more ? jn : j;  // (the last batch loads itself again)
      double nx[3 * kUnroll], nm[kUnroll];
#pragma unroll
      for (int q = 0; q < 3 * kUnroll; ++q) nx[q] = (sx + 3 * (size_t)jl)[q];
#pragma unroll
      for (int q = 0; q < kUnroll; ++q) nm[q] = (sm + jl)[q];
      batch(j, bx, bm, std::integral_constant<int, kUnroll>{});
      j = jn;
      if (!more) break;
#pragma unroll
      for (int q = 0; q < 3 * kUnroll; ++q) bx[q] = nx[q];
#pragma unroll
      for (int q = 0; q < kUnroll; ++q) bm[q] = nm[q];
    }
  }
  for (; j < j1; ++j) {
    const double bx[3] = {sx[3 * (size_t)j], sx[3 * (size_t)j + 1], sx[3 * (size_t)j + 2]};
    const double bm[1] = {sm[j]};
    batch(j, bx, bm, std::integral_constant<int, 1>{});
  }
}

// Targets [64 blockIdx.x, +64) against the sources of chunk blockIdx.y, [c * len, min(n,
// (c + 1) * len)), self excluded: by its zero distance where that gives a zero term (each of
// the wave's own weights is finite: neither the mass nor the softening's inverse cube is
// extreme), else by index, a compare and two selects a pair. With one chunk the sums go
// straight to out (3 per target); with several, chunk c writes partial[(c * nt + t) * 3 +
// axis] and k_direct_reduce adds the chunks in a fixed order, so results do not depend on
// timing. (64 VGPRs, 8 waves per SIMD: at the 66 the compiler takes unasked, 2^20 sources and
// 4,096 targets take 1.5% longer.)
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(8)))
k_direct_f64(const double* __restrict__ x, const double* __restrict__ m, uint32_t n,
             const uint32_t* __restrict__ targets, uint32_t nt, double g, double eps2,
             uint32_t chunk_len, double* __restrict__ out) {
  const uint32_t t = blockIdx.x * 64u + threadIdx.x;
  const uint32_t id = targets[min(t, nt - 1u)];
  const double xi = x[3 * (size_t)id], yi = x[3 * (size_t)id + 1], zi = x[3 * (size_t)id + 2];
  double ax = 0.0, ay = 0.0, az = 0.0;
  const uint32_t j0 = blockIdx.y * chunk_len;
  const uint32_t j1 = (n - j0 < chunk_len) ? n : j0 + chunk_len;
  auto sum = [&](auto by_index) {
    sweep(cst(x), cst(m), j0, j1, [&](uint32_t j, const double* bx, const double* bm, auto count) {
      constexpr int U = decltype(count)::value;
      double dx[U], dy[U], dz[U], r2[U], w[U];
      bool bad = false;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        dx[u] = bx[3 * u] - xi;
        dy[u] = bx[3 * u + 1] - yi;
        dz[u] = bx[3 * u + 2] - zi;
        r2[u] = fma(dx[u], dx[u], fma(dy[u], dy[u], fma(dz[u], dz[u], eps2)));
        w[u] = inv_cube(bm[u], r2[u], bad);
      }
      if (__builtin_expect(bad, 0)) {
#pragma unroll
        for (int u = 0; u < U; ++u) w[u] = inv_cube_ieee(bm[u], r2[u]);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const double q = (decltype(by_index)::value && j + u == id) ? 0.0 : w[u];
        ax = fma(dx[u], q, ax);
        ay = fma(dy[u], q, ay);
        az = fma(dz[u], q, az);
      }
    });
  };
  if (__ballot(!(fabs(inv_cube_ieee(m[id], eps2)) < 1e300)) == 0ull) sum(std::false_type{});
  else sum(std::true_type{});
  if (t < nt) {
    double* o = out + ((size_t)blockIdx.y * nt + t) * 3;
    o[0] = g * ax;
    o[1] = g * ay;
    o[2] = g * az;
  }
}

// out[3 t + axis] = sum over chunks c of partial[(c * nt + t) * 3 + axis]: a block takes 64
// outputs, each of its 16 waves one sixteenth of the chunks in index order, and the first
// wave adds the sixteenths in order.
constexpr int kReduceWaves = 16;

__global__ void __launch_bounds__(64 * kReduceWaves)
k_direct_reduce(const double* __restrict__ partial, uint32_t nt, uint32_t chunks,
                double* __restrict__ out) {
  __shared__ double part[kReduceWaves][64];
  const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const size_t e = (size_t)blockIdx.x * 64 + lane, rows = 3 * (size_t)nt;
  const uint32_t per = (chunks + kReduceWaves - 1) / kReduceWaves;
  const uint32_t c0 = min(chunks, w * per), c1 = min(chunks, c0 + per);
  double r = 0.0;
  if (e < rows) {
#pragma unroll 4
    for (uint32_t c = c0; c < c1; ++c) r += partial[(size_t)c * rows + e];
  }
  part[w][lane] = r;
  __syncthreads();
  if (w == 0 && e < rows) {
    for (int k = 1; k < kReduceWaves; ++k) r += part[k][lane];
    out[e] = r;
  }
}

// Softened potential of the pairs i < j: rows [64 blockIdx.x, +64) against the sources of
// chunk blockIdx.y, counted from the block's first row (a chunk past the end adds nothing);
// one partial per wave. Only the sources among the rows need the j > i test.
__global__ void __launch_bounds__(64)
k_potential_f64(const double* __restrict__ x, const double* __restrict__ m, uint32_t n, double g,
                double eps2, uint32_t chunk_len, double* __restrict__ partial) {
  const uint32_t base = blockIdx.x * 64u;
  const uint64_t first = (uint64_t)base + (uint64_t)blockIdx.y * chunk_len;
  double* o = partial + (size_t)blockIdx.y * gridDim.x + blockIdx.x;
  if (first >= n) {
    if (threadIdx.x == 0) *o = 0.0;
    return;
  }
  const uint32_t j0 = (uint32_t)first, j1 = (uint32_t)min((uint64_t)n, first + chunk_len);
  const uint32_t diag_end = min(j1, base + 64u);
  const uint32_t row = base + threadIdx.x;
  const size_t i = min(row, n - 1u);
  const double xi = x[3 * i], yi = x[3 * i + 1], zi = x[3 * i + 2];
  double pot = 0.0;
  auto batch = [&](uint32_t j, const double* bx, const double* bm, auto count, auto masked) {
    constexpr int U = decltype(count)::value;
    double r2[U], y[U];
    bool bad = false;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const double dx = bx[3 * u] - xi, dy = bx[3 * u + 1] - yi, dz = bx[3 * u + 2] - zi;
      r2[u] = fma(dx, dx, fma(dy, dy, fma(dz, dz, eps2)));
      y[u] = inv_root(r2[u], bad);
    }
    if (__builtin_expect(bad, 0)) {
#pragma unroll
      for (int u = 0; u < U; ++u) y[u] = 1.0 / sqrt(r2[u]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // pairs j > i only (selected, not multiplied: the self pair and the mass may be infinite)
      const double t = fma(bm[u], y[u], pot);
      pot = decltype(masked)::value && j + u <= row ? pot : t;
    }
  };
  sweep(cst(x), cst(m), j0, max(j0, diag_end),
        [&](uint32_t j, const double* bx, const double* bm, auto count) {
          batch(j, bx, bm, count, std::true_type{});
        });
  sweep(cst(x), cst(m), max(j0, diag_end), j1,
        [&](uint32_t j, const double* bx, const double* bm, auto count) {
          batch(j, bx, bm, count, std::false_type{});
        });
  pot = row < n && pot != 0.0 ? -g * m[row] * pot : 0.0;  // (0: no source of this chunk counts)
  pot = wave_sum(pot);
  if (threadIdx.x == 0) *o = pot;
}

// Sum of n doubles in a fixed order: thread t adds in[t], in[t + 1024], ..., then a tree.
__global__ void __launch_bounds__(1024)
k_sum_f64(const double* __restrict__ in, uint32_t n, double* __restrict__ out) {
  __shared__ double part[16];
  double r = 0.0;
#pragma unroll 4
  for (uint32_t i = threadIdx.x; i < n; i += 1024) r += in[i];
  r = wave_sum(r);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = r;
  __syncthreads();
  if (threadIdx.x == 0) {
    r = 0.0;
    for (int k = 0; k < 16; ++k) r += part[k];
    *out = r;
  }
}

__global__ void k_seg_reset(const SegDesc* __restrict__ segs, uint32_t nseg) {
  const uint32_t q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nseg * 6u) return;
  bbox_neutral(segs[q / 6u].bbox, (int)(q % 6u));
}

// ----------------------------------------------------------------------------------
// host-side launch wrappers
// ----------------------------------------------------------------------------------

static inline uint32_t grid_for(uint32_t ntiles, uint32_t cap = 65535u) {
  return ntiles == 0 ? 1u : (ntiles < cap ? ntiles : cap);
}

// Grid for the XCD-ordered kernels: a multiple of the span (idle blocks skip the tile loop).
template <uint32_t RUN = kXcdRun>
static inline uint32_t xcd_grid(uint32_t ntiles, uint32_t max_blocks = 65535u) {
  const uint32_t span = kXcds * RUN, cap = max_blocks / span * span;
  if (ntiles < span) return ntiles == 0 ? 1u : ntiles;
  const uint32_t g = (ntiles + span - 1) / span * span;
  return g < cap ? g : cap;
}

hipError_t launch_seg_reset(hipStream_t st, const SegDesc* segs, uint32_t nseg) {
  if (nseg == 0) return hipSuccess;
  hipLaunchKernelGGL(k_seg_reset, dim3((nseg * 6 + 255) / 256), dim3(256), 0, st, segs, nseg);
  return hipGetLastError();
}

hipError_t launch_bbox(hipStream_t st, const SegDesc* segs, const Tile* et, uint32_t net) {
  hipLaunchKernelGGL(k_bbox, dim3(grid_for(net)), dim3(kBlock), 0, st, segs, et, net);
  return hipGetLastError();
}

hipError_t launch_kick_drift_bbox(hipStream_t st, const SegDesc* segs, const Tile* et,
                                  uint32_t net) {
  hipLaunchKernelGGL(k_kick_drift_bbox, dim3(grid_for(net)), dim3(kBlock), 0, st, segs, et, net);
  return hipGetLastError();
}

hipError_t launch_encode(hipStream_t st, const Mode& md, const SegDesc* segs, const Tile* et,
                         uint32_t net, uint32_t* lanes_out) {
  const int dst = sort_start(md.key63, md.radix_bits);
  if (md.key63)
    hipLaunchKernelGGL(k_encode<uint64_t>, dim3(grid_for(net)), dim3(kBlock), 0, st, segs, et, net,
                       lanes_out, dst);
  else
    hipLaunchKernelGGL(k_encode<uint32_t>, dim3(grid_for(net)), dim3(kBlock), 0, st, segs, et, net,
                       lanes_out, dst);
  return hipGetLastError();
}

hipError_t launch_bounds_only(hipStream_t st, const Mode& md, const SegDesc* segs, uint32_t nseg) {
  hipLaunchKernelGGL(k_bounds, dim3((nseg + 63) / 64), dim3(64), 0, st, segs, nseg,
                     md.key63 ? 21 : 10);
  return hipGetLastError();
}

hipError_t launch_iota(hipStream_t st, const Mode& md, const SegDesc* segs, const Tile* et,
                       uint32_t net) {
  hipLaunchKernelGGL(k_iota, dim3(grid_for(net)), dim3(kBlock), 0, st, segs, et, net,
                     sort_start(md.key63, md.radix_bits));
  return hipGetLastError();
}

// The keys start in buffer sort_start() and end in buffer 0.
template <class K, int B>
static void sort_passes(hipStream_t st, const SegDesc* segs, uint32_t nseg, const Tile* et,
                        uint32_t net, const SortScratch& sc) {
  constexpr bool key63 = sizeof(K) == 8;
  int src = sort_start(key63, B);
  for (int pass = 0; pass < sort_passes_for(key63, B); ++pass) {
    const int shift = pass * B;
    hipLaunchKernelGGL((k_radix_upsweep<K, B>), dim3(xcd_grid<kXcdBuildRun>(net)),
                       dim3(kSortThreads), 0, st, segs, et, net, sc.tile_hist, shift, src);
    hipLaunchKernelGGL(k_radix_scan<B>, dim3(grid_for(sc.nchunks * ((1 << B) / kScanDigits))),
                       dim3(kScanThreads), 0, st, sc.chunks, sc.nchunks, sc.tile_hist, sc.chunk_rows);
    hipLaunchKernelGGL((sc.chunked ? k_radix_downsweep<K, B, true> : k_radix_downsweep<K, B, false>),
                       dim3(xcd_grid<kXcdBuildRun>(net)), dim3(kSortThreads), 0, st, segs, et, net,
                       sc.tile_hist, sc.chunk_rows, shift, src);
    src ^= 1;
  }
}

template <class K>
static void sort_local(hipStream_t st, int radix_bits, const SegDesc* segs, uint32_t nseg,
                       const Tile* et, uint32_t net, const SortScratch& sc) {
  const int src = sort_start(sizeof(K) == 8, radix_bits);
  if (sc.split) {
    hipLaunchKernelGGL(k_split<K>, dim3(grid_for(nseg)), dim3(1024), 0, st, segs, nseg, src,
                       sc.table);
    hipLaunchKernelGGL(k_bucket_count<K>, dim3(grid_for(net)), dim3(kSortThreads), 0, st, segs, et,
                       net, sc.tile_hist, src, sc.table);
    hipLaunchKernelGGL(k_bucket_scatter<K>, dim3(grid_for(net)), dim3(kSortThreads), 0, st, segs,
                       et, net, sc.tile_hist, src, sc.table);
  }
  hipLaunchKernelGGL(k_sort_local<K>, dim3(grid_for(sc.nbuckets)), dim3(kLocalThreads), 0, st,
                     segs, sc.buckets, sc.nbuckets, src, sc.table);
}

template <class K>
static void sort_width(hipStream_t st, int bits, const SegDesc* segs, uint32_t nseg,
                       const Tile* et, uint32_t net, const SortScratch& sc) {
  if (bits == 10)
    sort_passes<K, 10>(st, segs, nseg, et, net, sc);
  else if (bits == 9)
    sort_passes<K, 9>(st, segs, nseg, et, net, sc);
  else
    sort_passes<K, 8>(st, segs, nseg, et, net, sc);
}

hipError_t launch_sort(hipStream_t st, const Mode& md, const SegDesc* segs, uint32_t nseg,
                       const Tile* et, uint32_t net, const SortScratch& sc) {
  if (md.radix_bits < 8 || md.radix_bits > kRadixBitsMax) return hipErrorInvalidValue;
  if (sc.nbuckets && md.key63)
    sort_local<uint64_t>(st, md.radix_bits, segs, nseg, et, net, sc);
  else if (sc.nbuckets)
    sort_local<uint32_t>(st, md.radix_bits, segs, nseg, et, net, sc);
  else if (md.key63)
    sort_width<uint64_t>(st, md.radix_bits, segs, nseg, et, net, sc);
  else
    sort_width<uint32_t>(st, md.radix_bits, segs, nseg, et, net, sc);
  return hipGetLastError();
}

hipError_t launch_gather(hipStream_t st, const SegDesc* segs, const Tile* et, uint32_t net) {
  hipLaunchKernelGGL(k_gather, dim3(xcd_grid<kXcdBuildRun>(net)), dim3(kGatherThreads), 0, st,
                     segs, et, net);
  return hipGetLastError();
}

hipError_t launch_refresh_leaves(hipStream_t st, const SegDesc* segs, const Tile* et,
                                 uint32_t net) {
  hipLaunchKernelGGL(k_gather, dim3(xcd_grid<kXcdBuildRun>(net)), dim3(kGatherThreads), 0, st,
                     segs, et, net);
  return hipGetLastError();
}

hipError_t launch_flatten(hipStream_t st, const SegDesc* segs, const Tile* et, uint32_t net,
                          const FlatOut& out) {
  hipLaunchKernelGGL(k_flatten, dim3(grid_for(net)), dim3(kBlock), 0, st, segs, et, net, out);
  return hipGetLastError();
}

hipError_t launch_karras(hipStream_t st, const Mode& md, const SegDesc* segs, const Tile* et,
                         uint32_t net) {
  if (md.key63)
    hipLaunchKernelGGL(k_karras<uint64_t>, dim3(xcd_grid<kXcdBuildRun>(net)), dim3(kKarrasThreads),
                       0, st, segs, et, net);
  else
    hipLaunchKernelGGL(k_karras<uint32_t>, dim3(xcd_grid<kXcdBuildRun>(net)), dim3(kKarrasThreads),
                       0, st, segs, et, net);
  return hipGetLastError();
}

template <bool QUAD>
static void aggregate_q(hipStream_t st, bool group, const SegDesc* segs, uint32_t nseg,
                        const AggTiles& t) {
  const dim3 fb(kFoldThreads);
  hipLaunchKernelGGL(k_aggregate_tile<QUAD>, dim3(grid_for(t.nat)), dim3(kAggThreads), 0, st, segs,
                     t.at, t.nat, (int)group);
  if (t.nmt)
    hipLaunchKernelGGL((k_aggregate_span<QUAD, true>), dim3(grid_for(t.nmt)), fb, 0, st, segs, t.mt,
                       t.nmt, 1);
  if (t.nm2)
    hipLaunchKernelGGL((k_aggregate_span<QUAD, true>), dim3(grid_for(t.nm2)), fb, 0, st, segs, t.m2,
                       t.nm2, 2);
  if (t.top)
    hipLaunchKernelGGL((k_aggregate_span<QUAD, false>), dim3(grid_for(nseg)), fb, 0, st, segs,
                       nullptr, nseg, 0);
}

hipError_t launch_aggregate(hipStream_t st, const Mode& md, const SegDesc* segs, uint32_t nseg,
                            const AggTiles& t) {
  if (md.quad) aggregate_q<true>(st, md.group, segs, nseg, t);
  else aggregate_q<false>(st, md.group, segs, nseg, t);
  return hipGetLastError();
}

// Launches of at most this many walk tiles (64 bodies each) take the split form: up to here
// a group's latency counts, above it the waves that one group occupies. Plummer spheres at
// theta = 0.5, one wave / split: far field 282 / 208 us at 100,003 bodies, 351 / 386 at
// 200,000; quadrupoles only 898 / 820 at 200,000, 1,164 / 1,134 at 300,000 (compensated 1,406
// / 1,419); monopoles 498 / 389 and 644 / 531.
constexpr uint32_t split_tiles(bool quad, bool far) {
  return far ? 2304u : (quad ? 4096u : 8192u);
}

template <bool KAHAN, bool COUNT, bool WIDE>
static void walk_group_q(hipStream_t st, bool quad, bool far, const SegDesc* segs, const Tile* gt,
                         uint32_t ngt, int mode) {
  if (!COUNT && ngt <= split_tiles(quad, far)) {
    const dim3 sg(ngt * kSplitSlots);
    if (quad && far)
      hipLaunchKernelGGL((k_walk_split<KAHAN, true, true, WIDE>), sg, dim3(192), 0, st, segs,
                         gt, ngt, mode);
    else if (quad)
      hipLaunchKernelGGL((k_walk_split<KAHAN, true, false, WIDE>), sg, dim3(128), 0, st, segs,
                         gt, ngt, mode);
    else
      hipLaunchKernelGGL((k_walk_split<KAHAN, false, false, WIDE>), sg, dim3(128), 0, st,
                         segs, gt, ngt, mode);
    return;
  }
  // one block per walk tile (up to 2^25 blocks of one wave): a block that took a second
  // tile a grid's length later would mix two distant regions in its XCD's L2
  const dim3 g(xcd_grid(ngt, 1u << 25)), b(kGroup);
  if (quad && far)
    hipLaunchKernelGGL((k_walk_group<KAHAN, COUNT, true, true, WIDE>), g, b, 0, st, segs, gt, ngt,
                       mode);
  else if (quad)
    hipLaunchKernelGGL((k_walk_group<KAHAN, COUNT, true, false, WIDE>), g, b, 0, st, segs, gt,
                       ngt, mode);
  else
    hipLaunchKernelGGL((k_walk_group<KAHAN, COUNT, false, false, WIDE>), g, b, 0, st, segs, gt,
                       ngt, mode);
}

template <bool KAHAN, bool COUNT>
static void walk_group_w(hipStream_t st, bool wide, bool quad, bool far, const SegDesc* segs,
                         const Tile* gt, uint32_t ngt, int mode) {
  if (wide) walk_group_q<KAHAN, COUNT, true>(st, quad, far, segs, gt, ngt, mode);
  else walk_group_q<KAHAN, COUNT, false>(st, quad, far, segs, gt, ngt, mode);
}

hipError_t launch_walk(hipStream_t st, const Mode& md, const SegDesc* segs, const Tile* wt,
                       uint32_t nwt, const Tile* gt, uint32_t ngt, int mode, bool count,
                       bool wide) {
  if (md.group) {
    if (md.kahan) {
      if (count) walk_group_w<true, true>(st, wide, md.quad, md.far, segs, gt, ngt, mode);
      else walk_group_w<true, false>(st, wide, md.quad, md.far, segs, gt, ngt, mode);
    } else {
      if (count) walk_group_w<false, true>(st, wide, md.quad, md.far, segs, gt, ngt, mode);
      else walk_group_w<false, false>(st, wide, md.quad, md.far, segs, gt, ngt, mode);
    }
    return hipGetLastError();
  }
  const dim3 g(xcd_grid<kXcdTargetRun>(nwt * kTileQuads, 1u << 25)), b(64);
  if (md.kahan) {
    if (count)
      hipLaunchKernelGGL((k_walk_target<true, true>), g, b, 0, st, segs, wt, nwt, mode);
    else
      hipLaunchKernelGGL((k_walk_target<true, false>), g, b, 0, st, segs, wt, nwt, mode);
  } else {
    if (count)
      hipLaunchKernelGGL((k_walk_target<false, true>), g, b, 0, st, segs, wt, nwt, mode);
    else
      hipLaunchKernelGGL((k_walk_target<false, false>), g, b, 0, st, segs, wt, nwt, mode);
  }
  return hipGetLastError();
}

hipError_t launch_diag(hipStream_t st, const SegDesc* segs, uint32_t nseg, const Tile* et,
                       uint32_t net, double* partial, double* out) {
  hipLaunchKernelGGL(k_diag_partial, dim3(grid_for(net)), dim3(kBlock), 0, st, segs, et, net,
                     partial);
  hipLaunchKernelGGL(k_diag_final, dim3(nseg), dim3(64), 0, st, segs, nseg, partial, out);
  return hipGetLastError();
}

DirectPlan direct_plan(uint32_t n, uint32_t nt, size_t partial_bytes) {
  DirectPlan p{1u, n ? n : 1u};
  if (nt == 0 || n == 0) return p;
  // about 8192 waves (8 per SIMD) of one target block x one source chunk
  const uint32_t tblocks = (nt + 63u) / 64u;
  uint32_t c = (8192u + tblocks - 1) / tblocks;
  const uint32_t by_src = (n + 127u) / 128u;  // at least 128 sources per chunk
  if (c > by_src) c = by_src;
  const size_t fit = partial_bytes / (3 * sizeof(double) * (size_t)nt);
  if ((size_t)c > fit) c = (uint32_t)fit;
  if (c < 2u) return p;
  uint32_t len = (n + c - 1) / c;
  len = (len + kUnroll - 1) / kUnroll * kUnroll;
  p.chunks = (n + len - 1) / len;
  p.chunk_len = len;
  if (p.chunks < 2u) p = DirectPlan{1u, n};
  return p;
}

hipError_t launch_direct_f64(hipStream_t st, const double* x, const double* m, uint32_t n,
                             const uint32_t* targets, uint32_t nt, double g, double eps2,
                             const DirectPlan& plan, double* partial, double* out) {
  if (nt == 0) return hipSuccess;
  const bool whole = plan.chunks < 2u;
  const dim3 grid((nt + 63u) / 64u, whole ? 1u : plan.chunks), b(64);
  double* to = whole ? out : partial;
  hipLaunchKernelGGL(k_direct_f64, grid, b, 0, st, x, m, n, targets, nt, g, eps2, plan.chunk_len,
                     to);
  if (whole) return hipGetLastError();
  const uint32_t rblocks = (uint32_t)((3 * (size_t)nt + 63) / 64);
  hipLaunchKernelGGL(k_direct_reduce, dim3(rblocks), dim3(64 * kReduceWaves), 0, st, partial, nt,
                     plan.chunks, out);
  return hipGetLastError();
}

// Row blocks x source chunks of the potential: about 16,384 waves, of which half lie in the
// triangle j > i, with chunks of at least 64 sources.
struct PotentialPlan {
  uint32_t blocks, chunks, chunk_len;
};
static PotentialPlan potential_plan(uint32_t n) {
  PotentialPlan p;
  p.blocks = (n + 63u) / 64u;
  const uint32_t c = (16384u + p.blocks - 1) / p.blocks, most = (n + 63u) / 64u;
  const uint32_t chunks = c < most ? c : most;
  p.chunk_len = (n + chunks - 1) / chunks;
  p.chunks = (n + p.chunk_len - 1) / p.chunk_len;
  return p;
}

size_t potential_doubles(uint32_t n) {
  if (n == 0) return 1;
  const PotentialPlan p = potential_plan(n);
  return (size_t)p.blocks * p.chunks + 1;
}

hipError_t launch_potential_f64(hipStream_t st, const double* x, const double* m, uint32_t n,
                                double g, double eps2, double* work) {
  if (n == 0) return hipSuccess;
  const PotentialPlan p = potential_plan(n);
  double* partial = work + 1;
  const dim3 grid(p.blocks, p.chunks), b(64);
  hipLaunchKernelGGL(k_potential_f64, grid, b, 0, st, x, m, n, g, eps2, p.chunk_len, partial);
  hipLaunchKernelGGL(k_sum_f64, dim3(1), dim3(1024), 0, st, partial, p.blocks * p.chunks, work);
  return hipGetLastError();
}

}  // namespace glx
