// Scatter of VM factor gradients with far fewer memory-side atomics: the
// transpose of TensorVM.interpolate (tensor_vm.py:42-89, 226-250) for a
// batch of rows, split into
//   * planes: the (row, mode) pairs are counting-sorted by plane cell (the 2x2
//     texel block a row's bilinear taps read); a group of lanes walks a run of
//     pairs and sums the texels of the current cell in registers, so a texel
//     costs one add per stretch of cells that share it instead of one per pair;
//   * lines: the same walk in ray order, or over the pairs sorted by line cell.
// Fields that the walks do not take add the lines in ray order, one 16-lane
// group per row, equal texels among the four rows of a wave merged.
// Float atomics to device memory are performed at the memory side on this
// part and adds to one address serialise there; the transaction count is
// what bounds a scatter.
#pragma once

#include "tfh_vm_kernels.h"

namespace tfh {

// Grids up to this size use the sorted plane scatter.
constexpr int kSortMaxGrid = 512;
// Rows up to this many can be sorted: their pairs, three a row, are counted and
// placed with 32-bit signed integers.
constexpr int64_t kSortMaxRows = INT32_MAX / 3;

// Code of one axis' tap pair: the lower texel when the pair is (i, i+1),
// G-1 for the pair clamped at the low edge (0, 0), G for the high edge
// (G-1, G-1) -- lin_tap never yields other equal pairs.
__device__ __forceinline__ int tap_code(const Tap& t, int g) {
  if (t.i1 == t.i0 + 1) return t.i0;
  return t.i0 == 0 ? g - 1 : g;
}

// Taps of mode m only: (v, a, b) = (x, y, z), (z, x, y), (y, z, x)
// (tensor_vm.py:50-52).
__device__ __forceinline__ void one_mode_taps(float x, float y, float z, int g, int m, Tap& v,
                                              Tap& a, Tap& b) {
  const float pv = m == 0 ? x : (m == 1 ? z : y);
  const float pa = m == 0 ? y : (m == 1 ? x : z);
  const float pb = m == 0 ? z : (m == 1 ? y : x);
  v = lin_tap(pv, g);
  a = lin_tap(pa, g);
  b = lin_tap(pb, g);
}

__device__ __forceinline__ int plane_bin(int m, const Tap& a, const Tap& b, int g) {
  return (m * (g + 1) + tap_code(a, g)) * (g + 1) + tap_code(b, g);
}

// Upstream gradient of a row's feature (mode m, channel c): a row-major
// (M, 3C) array (appearance features), or one scalar per row that every
// channel of every mode receives (the density head: sigma = softplus(sum of
// the 3C features + shift), so dL/dfeature = dL/ds for all of them).
struct RowGrad {
  const float* g;
  int C;
  __device__ __forceinline__ float at(int64_t row, int m, int c) const {
    return g[row * 3 * C + m * C + c];
  }
  // channels c4 .. c4+3 (16-byte aligned rows: C % 4 == 0)
  __device__ __forceinline__ float4 at4(int64_t row, int m, int c4) const {
    return *reinterpret_cast<const float4*>(g + row * 3 * C + m * C + c4);
  }
  bool aligned16() const { return (reinterpret_cast<uintptr_t>(g) & 15) == 0 && C % 4 == 0; }
};

struct ScalarGrad {
  const float* g;
  __device__ __forceinline__ float at(int64_t row, int, int) const { return g[row]; }
  __device__ __forceinline__ float4 at4(int64_t row, int, int) const {
    const float v = g[row];
    return make_float4(v, v, v, v);
  }
  bool aligned16() const { return true; }
};

// Two-level sort of the (row, mode) pairs by plane cell. Cells are grouped
// into tiles of kTile x kTile cells per mode. (A) every workgroup ranks its
// pairs within their tiles in LDS and reserves each tile's share with one
// global atomic; (B) one workgroup scans the tile counts; (C) every pair
// moves to its tile's segment; (D) every chunk of up to kSortChunk pairs of
// one tile is counting-sorted by cell in LDS in place. Equal cells are then
// adjacent within a chunk (a tile larger than a chunk repeats a cell in each
// of its chunks). Global atomics: one per (workgroup, tile) instead of two
// per pair.
constexpr int kTile = 16;
constexpr int kSortMaxTiles = 3 * ((kSortMaxGrid + 1 + kTile - 1) / kTile) *
                              ((kSortMaxGrid + 1 + kTile - 1) / kTile);
constexpr int kRowsPerRankGroup = 1024;  // rows of one workgroup of pass A
constexpr int kSortChunk = 4096;         // pairs sorted by cell in one workgroup

struct SortWs {
  uint32_t* order = nullptr;    // (3 M) pairs row*4 + mode, sorted by cell
  uint16_t* tile_of = nullptr;  // (3 M) tile of pair row*3 + mode
  uint32_t* rank_of = nullptr;  // (3 M) position of the pair within its tile
  int32_t* tile_count = nullptr;  // (tiles) pairs per tile
  int32_t* tile_start = nullptr;  // (tiles + 1) first pair of each tile
  int32_t* chunk_start = nullptr; // (tiles + 1) first chunk of each tile
};

__device__ __forceinline__ int tiles_per_axis(int g) { return (g + 1 + kTile - 1) / kTile; }

// Tile and cell (0..kTile^2-1) of mode m's plane taps.
__device__ __forceinline__ void pair_tile(int m, const Tap& a, const Tap& b, int g, int& tile,
                                          int& cell) {
  const int ca = tap_code(a, g), cb = tap_code(b, g), nt = tiles_per_axis(g);
  tile = (m * nt + ca / kTile) * nt + cb / kTile;
  cell = (ca % kTile) * kTile + cb % kTile;
}

// (A) Per workgroup of kRowsPerRankGroup rows: LDS ranks within tiles, one
// global reservation per tile present. LINE: the bins are instead the line
// cells of each mode (m (g+1) + the line tap code, 3 (g+1) bins), with no
// cell pass after.
template <class Src, bool LINE = false>
__global__ void __launch_bounds__(256) k_tile_rank(Src src, int64_t M, int g,
                                                   int32_t* __restrict__ tile_count,
                                                   uint16_t* __restrict__ tile_of,
                                                   uint32_t* __restrict__ rank_of) {
  constexpr int RPT = kRowsPerRankGroup / 256;
  __shared__ int32_t cnt[kSortMaxTiles];
  const int nt = tiles_per_axis(g), tiles = LINE ? 3 * (g + 1) : 3 * nt * nt;
  for (int t = threadIdx.x; t < tiles; t += 256) cnt[t] = 0;
  __syncthreads();
  const int64_t r0 = (int64_t)blockIdx.x * kRowsPerRankGroup;
  int tl[RPT][3], rk[RPT][3];
#pragma unroll
  for (int j = 0; j < RPT; ++j) {
    const int64_t s = r0 + j * 256 + threadIdx.x;
#pragma unroll
    for (int m = 0; m < 3; ++m) tl[j][m] = -1;
    if (s < M) {
      float x, y, z;
      src.get(s, x, y, z);
      ModeTaps mt[3];
      mode_taps(x, y, z, g, mt);
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        if constexpr (LINE) {
          tl[j][m] = m * (g + 1) + tap_code(mt[m].v, g);
        } else {
          int cell;
          pair_tile(m, mt[m].a, mt[m].b, g, tl[j][m], cell);
        }
        rk[j][m] = atomicAdd(&cnt[tl[j][m]], 1);
      }
    }
  }
  __syncthreads();
  for (int t = threadIdx.x; t < tiles; t += 256) {
    const int c = cnt[t];
    if (c > 0) cnt[t] = atomicAdd(tile_count + t, c);  // this workgroup's base in the tile
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < RPT; ++j) {
    const int64_t s = r0 + j * 256 + threadIdx.x;
    if (s < M) {
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        tile_of[3 * s + m] = (uint16_t)tl[j][m];
        rank_of[3 * s + m] = (uint32_t)(cnt[tl[j][m]] + rk[j][m]);
      }
    }
  }
}

// (B) Exclusive scans of the tile counts and of the chunks per tile (one
// workgroup; tiles <= kSortMaxTiles).
static __global__ void __launch_bounds__(1024) k_tile_scan(
    const int32_t* __restrict__ tile_count, int tiles, int32_t* __restrict__ tile_start,
    int32_t* __restrict__ chunk_start) {
  __shared__ int32_t wsum[2][16];
  __shared__ int32_t carry[2];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (threadIdx.x == 0) carry[0] = carry[1] = 0;
  __syncthreads();
  for (int t0 = 0; t0 < tiles; t0 += 1024) {
    const int t = t0 + threadIdx.x;
    const int32_t c = t < tiles ? tile_count[t] : 0;
    const int32_t ch = (c + kSortChunk - 1) / kSortChunk;
    int32_t ic = c, ih = ch;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int32_t a = __shfl_up(ic, o, 64), b = __shfl_up(ih, o, 64);
      if (lane >= o) {
        ic += a;
        ih += b;
      }
    }
    if (lane == 63) {
      wsum[0][w] = ic;
      wsum[1][w] = ih;
    }
    __syncthreads();
    int32_t bc = carry[0], bh = carry[1];
    for (int j = 0; j < w; ++j) {
      bc += wsum[0][j];
      bh += wsum[1][j];
    }
    if (t < tiles) {
      tile_start[t] = bc + ic - c;
      chunk_start[t] = bh + ih - ch;
    }
    __syncthreads();
    if (threadIdx.x == 1023) {
      carry[0] = bc + ic;
      carry[1] = bh + ih;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    tile_start[tiles] = carry[0];
    chunk_start[tiles] = carry[1];
  }
}

// (C) Every pair to its tile's segment.
static __global__ void __launch_bounds__(256) k_tile_place(int64_t pairs,
                                                    const uint16_t* __restrict__ tile_of,
                                                    const uint32_t* __restrict__ rank_of,
                                                    const int32_t* __restrict__ tile_start,
                                                    uint32_t* __restrict__ order) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p >= pairs) return;
  const int64_t row = p / 3;
  const int m = (int)(p - 3 * row);
  order[tile_start[tile_of[p]] + rank_of[p]] = (uint32_t)row * 4u + (uint32_t)m;
}

// (D) One chunk of a tile: counting sort by cell in LDS, written back in
// place. Workgroup w finds its tile by binary search of chunk_start;
// workgroups past the last chunk return.
template <class Src>
__global__ void __launch_bounds__(256) k_chunk_sort(Src src, int g, int tiles,
                                                    const int32_t* __restrict__ tile_start,
                                                    const int32_t* __restrict__ chunk_start,
                                                    uint32_t* __restrict__ order) {
  constexpr int PT = kSortChunk / 256, NC = kTile * kTile;
  __shared__ int32_t hist[NC];
  __shared__ int32_t wsum[4];
  const int w = blockIdx.x;
  if (w >= chunk_start[tiles]) return;
  int lo = 0, hi = tiles - 1;  // last tile with chunk_start <= w
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (chunk_start[mid] <= w) lo = mid; else hi = mid - 1;
  }
  const int t = lo;
  const int64_t base = (int64_t)tile_start[t] + (int64_t)(w - chunk_start[t]) * kSortChunk;
  const int len = (int)min((int64_t)kSortChunk, (int64_t)tile_start[t + 1] - base);
  for (int c = threadIdx.x; c < NC; c += 256) hist[c] = 0;
  __syncthreads();
  uint32_t pk[PT];
  int cl[PT], rk[PT];
#pragma unroll
  for (int j = 0; j < PT; ++j) {
    const int i = j * 256 + threadIdx.x;
    cl[j] = -1;
    if (i < len) {
      pk[j] = order[base + i];
      float x, y, z;
      src.get((int64_t)(pk[j] >> 2), x, y, z);
      Tap tv, ta, tb;
      one_mode_taps(x, y, z, g, (int)(pk[j] & 3u), tv, ta, tb);
      int tile;
      pair_tile((int)(pk[j] & 3u), ta, tb, g, tile, cl[j]);
      rk[j] = atomicAdd(&hist[cl[j]], 1);
    }
  }
  __syncthreads();
  // exclusive scan of the 256 cell counts (one per thread)
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int32_t c0 = hist[threadIdx.x];
  int32_t inc = c0;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int32_t a = __shfl_up(inc, o, 64);
    if (lane >= o) inc += a;
  }
  if (lane == 63) wsum[wv] = inc;
  __syncthreads();
  int32_t before = 0;
  for (int j = 0; j < wv; ++j) before += wsum[j];
  __syncthreads();
  hist[threadIdx.x] = before + inc - c0;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < PT; ++j)
    if (cl[j] >= 0) order[base + hist[cl[j]] + rk[j]] = pk[j];
}

// ---- walks over pairs -----------------------------------------------------------
// A group of LPS lanes walks `per` consecutive pairs and sums the gradients of
// the texels of the current cell in registers; a texel is added to memory
// when the walk leaves it. A walk that steps to a neighbouring cell keeps the
// texels the two share. Long walks save adds, short ones fill the chip: 64
// pairs where that leaves kWalkGroups groups, fewer (a power of two, at
// least 8) where it does not. A training step of 256 rays with 24 of 160
// samples shaded (16 + 48 channels, G = 128) takes 513 us with 64 pairs
// everywhere and 264 us with this rule; one of 1024 rays with all shaded 572
// and 505. With twice as many groups asked for, the latter takes 555 us
// (more adds), with half as many 509.
constexpr int kPairsPerGroup = 64;
constexpr int64_t kWalkGroups = 32768;
inline int walk_pairs(int64_t pairs) {
  int per = 8;
  while (per < kPairsPerGroup && pairs > per * kWalkGroups) per *= 2;
  return per;
}

// The taps of one pair, computed once by the lane that loads it and handed to
// its group lane by lane (every lane computing them for every pair is what
// bounded these passes: 40 of 60 vector instructions a pair).
struct PairTaps {
  uint32_t pk;      // row * 4 + mode
  int kl, kp;       // line0 * 2 + (line1 - line0); p00 * 4 + (row step) * 2 + (column step)
  float wv, wa, wb; // upper weights (the lower one is 1 - w)
};

__device__ __forceinline__ PairTaps make_pair_taps(uint32_t pk, float x, float y, float z, int g) {
  const int m = (int)(pk & 3u);
  Tap tv, ta, tb;
  one_mode_taps(x, y, z, g, m, tv, ta, tb);
  PairTaps t;
  t.pk = pk;
  t.kl = (m * g + tv.i0) * 2 + (tv.i1 - tv.i0);
  t.kp = ((m * g + ta.i0) * g + tb.i0) * 4 + (ta.i1 - ta.i0) * 2 + (tb.i1 - tb.i0);
  t.wv = tv.w1;
  t.wa = ta.w1;
  t.wb = tb.w1;
  return t;
}

__device__ __forceinline__ PairTaps shfl_pair(const PairTaps& t, int from) {
  PairTaps r;
  r.pk = __shfl(t.pk, from, 64);
  r.kl = __shfl(t.kl, from, 64);
  r.kp = __shfl(t.kp, from, 64);
  r.wv = __shfl(t.wv, from, 64);
  r.wa = __shfl(t.wa, from, 64);
  r.wb = __shfl(t.wb, from, 64);
  return r;
}

// Channel 16q + l of a 16-lane group whose lane j holds channels
// 4j .. 4j+3 (v): the sums go back to one channel per lane before they are
// added, so that each atomic instruction of a group covers 64 contiguous
// bytes (one memory-side transaction); with the quads the lanes' adds were
// 16 bytes apart, three transactions per instruction (the plane pass took
// 1.54 ms instead of 0.69). All 16 lanes of the group must call it (gl0: the
// group's first lane in the wave).
__device__ __forceinline__ float quad_to_lane(const float (&v)[4], int q, int l, int gl0) {
  const int from = gl0 + 4 * q + (l >> 2);
  const float t0 = __shfl(v[0], from, 64), t1 = __shfl(v[1], from, 64);
  const float t2 = __shfl(v[2], from, 64), t3 = __shfl(v[3], from, 64);
  const int u = l & 3;
  return u == 0 ? t0 : (u == 1 ? t1 : (u == 2 ? t2 : t3));
}

// One field of a walk: its factors, the upstream gradients (RowGrad or
// ScalarGrad) and where its sums go.
template <class GS>
struct WalkField {
  tfh_vm vm;
  GS g;
  float* out;  // the plane gradient, or nlc copies of the line gradient
  int nlc;
};
struct NoField {};

// A field of 16 < C <= 64 channels, C % 4 == 0, 16-byte aligned: lane l of 16
// owns channels 4l .. 4l+3.
template <class GS, int NT>
struct QuadLanes {
  const WalkField<GS>& f;
  float* out;
  int C, l, gl0;
  bool on;
  float4 acc[NT];
  __device__ __forceinline__ QuadLanes(const WalkField<GS>& f_, float* out_, int l_, int gl0_)
      : f(f_), out(out_), C((int)f_.vm.channels), l(l_), gl0(gl0_), on(4 * l_ < C) {
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  __device__ __forceinline__ float4 load(const float* base, int texel) const {
    return on ? *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(base) +
                                                 (uint32_t)((texel * C + 4 * l) * 4))
              : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  __device__ __forceinline__ float4 grad(uint32_t pk) const {
    return on ? f.g.at4((int64_t)(pk >> 2), (int)(pk & 3u), 4 * l)
              : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  __device__ __forceinline__ void add(int t, float w, const float4& v) {
    acc[t].x += w * v.x;
    acc[t].y += w * v.y;
    acc[t].z += w * v.z;
    acc[t].w += w * v.w;
  }
  __device__ __forceinline__ void flush(int t, int texel) {
    const float v[4] = {acc[t].x, acc[t].y, acc[t].z, acc[t].w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (16 * q < C) {  // group-uniform
        const float val = quad_to_lane(v, q, l, gl0);
        const int c = 16 * q + l;
        if (c < C && val != 0.0f) unsafeAtomicAdd(out + (size_t)texel * C + c, val);
      }
    }
    acc[t] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  __device__ __forceinline__ void move(int to, int from) {
    acc[to] = acc[from];
    acc[from] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
};

// A field of at most LPS channels: lane l owns channel l.
template <class GS, int NT>
struct LaneLanes {
  const WalkField<GS>& f;
  float* out;
  int C, l;
  bool on;
  float acc[NT];
  __device__ __forceinline__ LaneLanes(const WalkField<GS>& f_, float* out_, int l_, int)
      : f(f_), out(out_), C((int)f_.vm.channels), l(l_), on(l_ < C) {
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = 0.0f;
  }
  __device__ __forceinline__ float load(const float* base, int texel) const {
    return on ? *reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) +
                                                (uint32_t)((texel * C + l) * 4))
              : 0.0f;
  }
  __device__ __forceinline__ float grad(uint32_t pk) const {
    return on ? f.g.at((int64_t)(pk >> 2), (int)(pk & 3u), l) : 0.0f;
  }
  __device__ __forceinline__ void add(int t, float w, float v) { acc[t] += w * v; }
  __device__ __forceinline__ void flush(int t, int texel) {
    if (on && acc[t] != 0.0f) unsafeAtomicAdd(out + (size_t)texel * C + l, acc[t]);
    acc[t] = 0.0f;
  }
  __device__ __forceinline__ void move(int to, int from) {
    acc[to] = acc[from];
    acc[from] = 0.0f;
  }
};

struct NoLanes {
  template <class... T>
  __device__ __forceinline__ explicit NoLanes(T&&...) {}
  __device__ __forceinline__ void flush(int, int) {}
  __device__ __forceinline__ void move(int, int) {}
};

__device__ __forceinline__ float4 mul4(const float4& a, const float4& b) {
  return make_float4(a.x * b.x, a.y * b.y, a.z * b.z, a.w * b.w);
}
__device__ __forceinline__ float mul4(float a, float b) { return a * b; }
__device__ __forceinline__ float4 mix2(float w0, const float4& a, float w1, const float4& b) {
  return make_float4(w0 * a.x + w1 * b.x, w0 * a.y + w1 * b.y, w0 * a.z + w1 * b.z,
                     w0 * a.w + w1 * b.w);
}
__device__ __forceinline__ float mix2(float w0, float a, float w1, float b) {
  return w0 * a + w1 * b;
}
__device__ __forceinline__ float4 mix4(const float (&w)[4], const float4& a, const float4& b,
                                       const float4& c, const float4& d) {
  return make_float4(((w[0] * a.x + w[1] * b.x) + w[2] * c.x) + w[3] * d.x,
                     ((w[0] * a.y + w[1] * b.y) + w[2] * c.y) + w[3] * d.y,
                     ((w[0] * a.z + w[1] * b.z) + w[2] * c.z) + w[3] * d.z,
                     ((w[0] * a.w + w[1] * b.w) + w[2] * c.w) + w[3] * d.w);
}
__device__ __forceinline__ float mix4(const float (&w)[4], float a, float b, float c, float d) {
  return ((w[0] * a + w[1] * b) + w[2] * c) + w[3] * d;
}

template <class F>
struct IsNone {
  static constexpr bool v = false;
};
template <>
struct IsNone<NoField> {
  static constexpr bool v = true;
};
// The lane view of a field: quads for FA, one channel per lane for FD.
template <class F, int NT>
struct QuadOf;
template <class GS, int NT>
struct QuadOf<WalkField<GS>, NT> {
  using T = QuadLanes<GS, NT>;
};
template <int NT>
struct QuadOf<NoField, NT> {
  using T = NoLanes;
};
template <class F, int NT>
struct LaneOf;
template <class GS, int NT>
struct LaneOf<WalkField<GS>, NT> {
  using T = LaneLanes<GS, NT>;
};
template <int NT>
struct LaneOf<NoField, NT> {
  using T = NoLanes;
};
template <class GS>
__device__ __forceinline__ float* copy_of(const WalkField<GS>& f, int g) {
  return f.out + (int64_t)(blockIdx.x % f.nlc) * 3 * g * f.vm.channels;
}
__device__ __forceinline__ float* copy_of(const NoField&, int) { return nullptr; }
template <class GS>
__device__ __forceinline__ float* whole_of(const WalkField<GS>& f) { return f.out; }
__device__ __forceinline__ float* whole_of(const NoField&) { return nullptr; }

// Plane gradients from pairs sorted by plane cell: dL/dplane[m][texel][c] +=
// w_texel * line_m(c) * gout[row][m*C + c], of field FA (quad lanes, LPS = 16)
// and field FD (a channel per lane); either may be NoField. Both fields' line
// taps and upstream gradients are requested before the flush: one memory round
// trip per pair.
template <class Src, class FA, class FD, int LPS>
__global__ void __launch_bounds__(256) k_plane_walk(Src src, int g, int64_t pairs, int per,
                                                    const uint32_t* __restrict__ order, FA fa,
                                                    FD fd) {
  constexpr bool A = !IsNone<FA>::v, D = !IsNone<FD>::v;
  static_assert(!A || LPS == 16, "quad lanes are 16 to a pair");
  const int l = threadIdx.x % LPS;
  const int gl0 = (threadIdx.x - l) & 63;
  const int64_t first = ((int64_t)blockIdx.x * (256 / LPS) + threadIdx.x / LPS) * per;
  if (first >= pairs) return;  // whole group: no cross-group exchange below
  const int64_t last = min(first + per, pairs);
  typename QuadOf<FA, 4>::T la(fa, whole_of(fa), l, gl0);
  typename LaneOf<FD, 4>::T ld(fd, whole_of(fd), l, gl0);
  int cur = -1;
  int tex[4] = {0, 0, 0, 0};
  auto flush = [&](int t) __attribute__((always_inline)) {
    la.flush(t, tex[t]);
    ld.flush(t, tex[t]);
  };
  for (int64_t b0 = first; b0 < last; b0 += LPS) {
    const int64_t e = b0 + l;
    PairTaps mine{};
    if (e < last) {
      const uint32_t pk = order[e];
      float x, y, z;
      src.get((int64_t)(pk >> 2), x, y, z);
      mine = make_pair_taps(pk, x, y, z, g);
    }
    const int nb = (int)min((int64_t)LPS, last - b0);
    for (int j = 0; j < nb; ++j) {
      const PairTaps p = shfl_pair(mine, gl0 + j);
      const int i0 = p.kl >> 1, i1 = i0 + (p.kl & 1);
      const float w0 = 1.0f - p.wv;
      float4 a0, a1, ag;
      float d0, d1, dg;
      if constexpr (A) {
        a0 = la.load(fa.vm.line, i0);
        a1 = la.load(fa.vm.line, i1);
        ag = la.grad(p.pk);
      }
      if constexpr (D) {
        d0 = ld.load(fd.vm.line, i0);
        d1 = ld.load(fd.vm.line, i1);
        dg = ld.grad(p.pk);
      }
      if (p.kp != cur) {
        int nt[4];
        nt[0] = p.kp >> 2;
        nt[1] = nt[0] + (p.kp & 1);
        nt[2] = nt[0] + ((p.kp >> 1) & 1) * g;
        nt[3] = nt[2] + (p.kp & 1);
        if (cur >= 0) {
          flush(0);
          flush(2);
          if (nt[0] == tex[1] && nt[2] == tex[3]) {  // the next cell of the row
            la.move(0, 1);
            la.move(2, 3);
            ld.move(0, 1);
            ld.move(2, 3);
          } else {
            flush(1);
            flush(3);
          }
        }
        cur = p.kp;
#pragma unroll
        for (int t = 0; t < 4; ++t) tex[t] = nt[t];
      }
      const float wa0 = 1.0f - p.wa, wb0 = 1.0f - p.wb;
      const float w[4] = {wa0 * wb0, wa0 * p.wb, p.wa * wb0, p.wa * p.wb};
      if constexpr (A) {
        const float4 v = mul4(ag, mix2(w0, a0, p.wv, a1));
#pragma unroll
        for (int t = 0; t < 4; ++t) la.add(t, w[t], v);
      }
      if constexpr (D) {
        const float v = dg * mix2(w0, d0, p.wv, d1);
#pragma unroll
        for (int t = 0; t < 4; ++t) ld.add(t, w[t], v);
      }
    }
  }
  if (cur >= 0) {
#pragma unroll
    for (int t = 0; t < 4; ++t) flush(t);
  }
}

// Line gradients: dL/dline[m][v][c] += w_v * plane_m(c) * gout[row][m*C + c],
// over pairs sorted by line cell (order), or with RAY in ray order, mode by
// mode (pair e = (row e % M, mode e / M)): a run is then a stretch of a ray
// inside one line cell, and the adds go to copies of the line gradient (block
// b into copy b % nlc), since every ray crosses the same few line texels.
template <class Src, class FA, class FD, int LPS, bool RAY>
__global__ void __launch_bounds__(256) k_line_walk(Src src, int g, int64_t pairs, int per, int64_t M,
                                                   const uint32_t* __restrict__ order, FA fa,
                                                   FD fd) {
  constexpr bool A = !IsNone<FA>::v, D = !IsNone<FD>::v;
  static_assert(!A || LPS == 16, "quad lanes are 16 to a pair");
  const int l = threadIdx.x % LPS;
  const int gl0 = (threadIdx.x - l) & 63;
  const int64_t first = ((int64_t)blockIdx.x * (256 / LPS) + threadIdx.x / LPS) * per;
  if (first >= pairs) return;  // whole group: no cross-group exchange below
  const int64_t last = min(first + per, pairs);
  typename QuadOf<FA, 2>::T la(fa, copy_of(fa, g), l, gl0);
  typename LaneOf<FD, 2>::T ld(fd, copy_of(fd, g), l, gl0);
  int cur = -1, t0 = 0, t1 = 0;
  int cell = -1;  // the plane cell whose values are in a and d
  float4 a[4];
  float d[4];
  for (int64_t b0 = first; b0 < last; b0 += LPS) {
    const int64_t e = b0 + l;
    PairTaps mine{};
    if (e < last) {
      uint32_t pk;
      if constexpr (RAY) {
        const int m = e >= 2 * M ? 2 : (e >= M ? 1 : 0);
        pk = (uint32_t)(e - m * M) << 2 | (uint32_t)m;
      } else {
        pk = order[e];
      }
      float x, y, z;
      src.get((int64_t)(pk >> 2), x, y, z);
      mine = make_pair_taps(pk, x, y, z, g);
    }
    const int nb = (int)min((int64_t)LPS, last - b0);
    for (int j = 0; j < nb; ++j) {
      const PairTaps p = shfl_pair(mine, gl0 + j);
      float4 ag;
      float dg;
      if constexpr (A) ag = la.grad(p.pk);
      if constexpr (D) dg = ld.grad(p.pk);
      if (p.kp != cell) {
        const int p00 = p.kp >> 2, p01 = p00 + (p.kp & 1);
        const int p10 = p00 + ((p.kp >> 1) & 1) * g, p11 = p10 + (p.kp & 1);
        if constexpr (A) {
          a[0] = la.load(fa.vm.plane, p00);
          a[1] = la.load(fa.vm.plane, p01);
          a[2] = la.load(fa.vm.plane, p10);
          a[3] = la.load(fa.vm.plane, p11);
        }
        if constexpr (D) {
          d[0] = ld.load(fd.vm.plane, p00);
          d[1] = ld.load(fd.vm.plane, p01);
          d[2] = ld.load(fd.vm.plane, p10);
          d[3] = ld.load(fd.vm.plane, p11);
        }
        cell = p.kp;
      }
      if (p.kl != cur) {
        const int n0 = p.kl >> 1, n1 = n0 + (p.kl & 1);
        if (cur >= 0) {
          if (n1 == t0 && n0 != t1) {  // one texel down
            la.flush(1, t1);
            ld.flush(1, t1);
            la.move(1, 0);
            ld.move(1, 0);
          } else {
            la.flush(0, t0);
            ld.flush(0, t0);
            if (n0 == t1) {  // one texel up
              la.move(0, 1);
              ld.move(0, 1);
            } else {
              la.flush(1, t1);
              ld.flush(1, t1);
            }
          }
        }
        cur = p.kl;
        t0 = n0;
        t1 = n1;
      }
      const float wa0 = 1.0f - p.wa, wb0 = 1.0f - p.wb, w0 = 1.0f - p.wv;
      const float w[4] = {wa0 * wb0, wa0 * p.wb, p.wa * wb0, p.wa * p.wb};
      if constexpr (A) {
        const float4 v = mul4(ag, mix4(w, a[0], a[1], a[2], a[3]));
        la.add(0, w0, v);
        la.add(1, p.wv, v);
      }
      if constexpr (D) {
        const float v = dg * mix4(w, d[0], d[1], d[2], d[3]);
        ld.add(0, w0, v);
        ld.add(1, p.wv, v);
      }
    }
  }
  if (cur >= 0) {
    la.flush(0, t0);
    la.flush(1, t1);
    ld.flush(0, t0);
    ld.flush(1, t1);
  }
}

// Plane gradients from the sorted pairs: dL/dplane[m][texel][c] +=
// w_texel * line_m(c) * gout[row][m*C + c]. Each 16-lane group owns kPairsPerGroup
// consecutive sorted pairs; lane l owns channels l, l+16, ... . The group
// walks its pairs in batches of 16 (one pair's index and point loaded per
// lane, then broadcast), sums the four taps' gradients of the current bin in
// registers and adds them when the bin changes and at the end.
template <class Src, class GS>
__global__ void __launch_bounds__(256) k_plane_scatter_sorted(tfh_vm vm, Src src, int64_t pairs,
                                                              const uint32_t* __restrict__ order,
                                                              GS gsrc,
                                                              float* __restrict__ gplane) {
  constexpr int LPS = 16, NQ = 64 / LPS;
  const int G = (int)vm.grid_dim, C = (int)vm.channels;
  const int l = threadIdx.x & 15;
  const int gbase = threadIdx.x & ~15;  // first lane of the group in the block
  const int64_t first = ((int64_t)blockIdx.x * (256 / LPS) + threadIdx.x / LPS) * kPairsPerGroup;
  if (first >= pairs) return;  // whole group: no cross-group exchange below
  const int64_t last = min(first + (int64_t)kPairsPerGroup, pairs);
  float acc[4][NQ];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int q = 0; q < NQ; ++q) acc[t][q] = 0.0f;
  int cur = -1;  // bin being summed
  int tex[4] = {0, 0, 0, 0};
  auto flush = [&]() {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const int c = l + LPS * q;
        if (c < C && acc[t][q] != 0.0f) unsafeAtomicAdd(gplane + (size_t)tex[t] * C + c, acc[t][q]);
        acc[t][q] = 0.0f;
      }
  };
  for (int64_t b0 = first; b0 < last; b0 += LPS) {
    // lane l fetches pair b0 + l: its packed index and the row's point
    const int64_t e = b0 + l;
    uint32_t pk = 0xffffffffu;
    float px = 0.f, py = 0.f, pz = 0.f;
    if (e < last) {
      pk = order[e];
      src.get((int64_t)(pk >> 2), px, py, pz);
    }
    const int nb = (int)min((int64_t)LPS, last - b0);
    for (int j = 0; j < nb; ++j) {
      const uint32_t p = __shfl(pk, gbase + j, 64);
      const float x = __shfl(px, gbase + j, 64), y = __shfl(py, gbase + j, 64),
                  z = __shfl(pz, gbase + j, 64);
      const int64_t row = (int64_t)(p >> 2);
      const int m = (int)(p & 3u);
      Tap tv, ta, tb;
      one_mode_taps(x, y, z, G, m, tv, ta, tb);
      const int bin = plane_bin(m, ta, tb, G);
      if (bin != cur) {
        if (cur >= 0) flush();
        cur = bin;
        const int base = m * G;
        tex[0] = (base + ta.i0) * G + tb.i0;
        tex[1] = (base + ta.i0) * G + tb.i1;
        tex[2] = (base + ta.i1) * G + tb.i0;
        tex[3] = (base + ta.i1) * G + tb.i1;
      }
      const float w[4] = {ta.w0 * tb.w0, ta.w0 * tb.w1, ta.w1 * tb.w0, ta.w1 * tb.w1};
      const float* lrow0 = vm.line + (size_t)(m * G + tv.i0) * C;
      const float* lrow1 = vm.line + (size_t)(m * G + tv.i1) * C;
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const int c = l + LPS * q;
        if (LPS * q < C && c < C) {
          const float lv = tv.w0 * lrow0[c] + tv.w1 * lrow1[c];
          const float gl = gsrc.at(row, m, c) * lv;
#pragma unroll
          for (int t = 0; t < 4; ++t) acc[t][q] += w[t] * gl;
        }
      }
    }
  }
  if (cur >= 0) flush();
}

// Line gradients in row order: dL/dline[m][v][c] += w_v * plane_m(c) *
// gout[row][m*C + c]; 16-lane groups, equal line texels of the wave's four
// rows (in either tap slot) added once. grad_line holds nlc copies; block b
// adds into copy b % nlc.
template <class Src, class GS>
__global__ void __launch_bounds__(kGatherThreads) k_line_scatter(tfh_vm vm, Src src, int64_t M,
                                                                 GS gsrc,
                                                                 float* __restrict__ gline,
                                                                 int nlc) {
  constexpr int LPS = 16, SPB = kGatherThreads / LPS, NQ = 64 / LPS;
  const int grp = threadIdx.x / LPS, l = threadIdx.x % LPS;
  const int64_t s0 = (int64_t)blockIdx.x * SPB;
  if (s0 >= M) return;
  const int64_t s = s0 + grp;
  const bool active = s < M;
  const int G = (int)vm.grid_dim, C = (int)vm.channels;
  gline += (int64_t)(blockIdx.x % nlc) * 3 * G * C;
  float x = 0.f, y = 0.f, z = 0.f;
  if (active) src.get(s, x, y, z);
  ModeTaps mt[3];
  mode_taps(x, y, z, G, mt);
  const int wg = grp & 3;  // group within the wave
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    TapAddr a;
    tap_addrs(mt[m], m, G, a);
    // merge plan of the two line slots over the wave's four groups
    int k0 = active ? a.line0 : -1 - 2 * wg, k1 = active ? a.line1 : -2 - 2 * wg;
    const bool fold = active && k1 == k0;  // clamped at the grid edge
    if (fold) k1 = INT_MIN + wg;
    int src0[3], src1[3];
    bool lead0 = active, lead1 = active && !fold;
#pragma unroll
    for (int oi = 0; oi < 3; ++oi) {
      const int o = LPS * (oi + 1);
      const bool lower = (wg ^ (oi + 1)) < wg;
      const int p0 = __shfl_xor(k0, o, 64), p1 = __shfl_xor(k1, o, 64);
      src0[oi] = p0 == k0 ? 0 : (p1 == k0 ? 1 : -1);
      src1[oi] = p0 == k1 ? 0 : (p1 == k1 ? 1 : -1);
      if (src0[oi] >= 0 && lower) lead0 = false;
      if (src1[oi] >= 0 && lower) lead1 = false;
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int c = l + LPS * q;
      if (LPS * q < C) {  // wave-uniform: every lane joins the exchange
        const bool on = active && c < C;
        float v0 = 0.f, v1 = 0.f;
        if (on) {
          float lv, pv;
          tap_values(vm.plane, vm.line, C, c, a, lv, pv);
          const float gp = gsrc.at(s, m, c) * pv;
          v0 = a.wl0 * gp;
          v1 = a.wl1 * gp;
          if (fold) {
            v0 += v1;
            v1 = 0.f;
          }
        }
        float acc0 = v0, acc1 = v1;
#pragma unroll
        for (int oi = 0; oi < 3; ++oi) {
          const int o = LPS * (oi + 1);
          const float q0 = __shfl_xor(v0, o, 64), q1 = __shfl_xor(v1, o, 64);
          acc0 += src0[oi] == 0 ? q0 : (src0[oi] == 1 ? q1 : 0.0f);
          acc1 += src1[oi] == 0 ? q0 : (src1[oi] == 1 ? q1 : 0.0f);
        }
        if (lead0 && acc0 != 0.0f) unsafeAtomicAdd(gline + (size_t)k0 * C + c, acc0);
        if (lead1 && acc1 != 0.0f) unsafeAtomicAdd(gline + (size_t)k1 * C + c, acc1);
      }
    }
  }
}

// Orders the (row, mode) pairs by line cell (3 (g+1) bins: rank, scan,
// place; the bin is the whole key).
template <class Src>
inline int32_t sort_lines(int g, const Src& src, int64_t M, const SortWs& s, hipStream_t st) {
  const int bins = 3 * (g + 1);
  const int64_t pairs = 3 * M;
  ProfScope ps("line_sort", st);
  TFH_TRY(zero_copies(reinterpret_cast<float*>(s.tile_count), bins, st));  // all-zero bits
  hipLaunchKernelGGL((k_tile_rank<Src, true>), dim3((unsigned)ceil_div(M, kRowsPerRankGroup)),
                     dim3(256), 0, st, src, M, g, s.tile_count, s.tile_of, s.rank_of);
  hipLaunchKernelGGL(k_tile_scan, dim3(1), dim3(1024), 0, st, s.tile_count, bins, s.tile_start,
                     s.chunk_start);
  hipLaunchKernelGGL(k_tile_place, dim3((unsigned)ceil_div(pairs, 256)), dim3(256), 0, st, pairs,
                     s.tile_of, s.rank_of, s.tile_start, s.order);
  return check_launch("vm scatter: line sort");
}

// The plane pass of field(s) fa (quad lanes) and fd (a channel per lane) over
// the pairs sort_pairs ordered.
template <int LPS, class Src, class FA, class FD>
inline int32_t launch_plane_walk(const Src& src, int g, int64_t M, const SortWs& s, const FA& fa,
                                 const FD& fd, const char* stage, hipStream_t st) {
  ProfScope ps(stage, st);
  const int per = walk_pairs(3 * M);
  const int64_t blocks = ceil_div(ceil_div(3 * M, per), 256 / LPS);
  hipLaunchKernelGGL((k_plane_walk<Src, FA, FD, LPS>), dim3((unsigned)blocks), dim3(256), 0, st,
                     src, g, 3 * M, per, s.order, fa, fd);
  return check_launch("vm scatter: planes");
}

// The line pass; sorted: over the pairs sort_lines ordered, else in ray order.
template <int LPS, class Src, class FA, class FD>
inline int32_t launch_line_walk(bool sorted, const Src& src, int g, int64_t M, const SortWs& s,
                                const FA& fa, const FD& fd, const char* stage, hipStream_t st) {
  ProfScope ps(stage, st);
  const int per = walk_pairs(3 * M);
  const int64_t blocks = ceil_div(ceil_div(3 * M, per), 256 / LPS);
  if (sorted)
    hipLaunchKernelGGL((k_line_walk<Src, FA, FD, LPS, false>), dim3((unsigned)blocks), dim3(256),
                       0, st, src, g, 3 * M, per, M, s.order, fa, fd);
  else
    hipLaunchKernelGGL((k_line_walk<Src, FA, FD, LPS, true>), dim3((unsigned)blocks), dim3(256), 0,
                       st, src, g, 3 * M, per, M, nullptr, fa, fd);
  return check_launch("vm scatter: lines");
}

// Bytes of the sort's workspace for up to M rows.
inline size_t sort_ws_bytes(int64_t M) {
  return align_up((size_t)(3 * M) * 4, 256) * 2 + align_up((size_t)(3 * M) * 2, 256) +
         3 * align_up((size_t)(kSortMaxTiles + 1) * 4, 256);
}

inline void take_sort_ws(Carve& cv, int64_t M, SortWs& s) {
  s.order = cv.take<uint32_t>(3 * M);
  s.rank_of = cv.take<uint32_t>(3 * M);
  s.tile_of = cv.take<uint16_t>(3 * M);
  s.tile_count = cv.take<int32_t>(kSortMaxTiles + 1);
  s.tile_start = cv.take<int32_t>(kSortMaxTiles + 1);
  s.chunk_start = cv.take<int32_t>(kSortMaxTiles + 1);
}

// Whether a field takes the sorted scatter: at most 64 channels, a grid
// within the bin budget, and a row count whose pairs fit the sort's counters
// (packed (row, mode) indices fit 32 bits then, too).
inline bool sorted_scatter_ok(const tfh_vm& vm, int64_t M, const SortWs& s) {
  return s.order && vm.channels <= 64 && vm.grid_dim <= kSortMaxGrid && M <= kSortMaxRows;
}

// Whether the sort pays for a field by itself. Up to 8 channels the direct scatter
// adds 32 bytes a tap from 8 lanes a row, and for few rows it is done before the
// sort's four launches are: 8 channels, compositing backward and scatter, direct and
// sorted, us: 2 thousand rows 24 and 73, 33 thousand 54 and 79, 102 thousand 95 and
// 102 (G = 128; 127 and 105 at G = 24), 226 thousand 167 and 131; the appearance
// scatter of 34 thousand 36 and 77. Wider fields take the sort from the first row
// (16 and 48 channels, 256 rows: 334 and 115).
constexpr int64_t kSortNarrowRows = 3 << 15;
inline bool sorted_scatter_pays(const tfh_vm& vm, int64_t M) {
  return vm.channels > 8 || M >= kSortNarrowRows;
}

// Whether a field can take the walks' quad lanes.
template <class GS>
inline bool quad_lanes_ok(const tfh_vm& vm, const GS& g) {
  return vm.channels > 16 && vm.channels <= 64 && vm.channels % 4 == 0 &&
         (reinterpret_cast<uintptr_t>(vm.plane) & 15) == 0 &&
         (reinterpret_cast<uintptr_t>(vm.line) & 15) == 0 && g.aligned16();
}

// Whether both fields can go in one walk (every sample shaded, one grid).
inline bool two_field_scatter_ok(const tfh_vm& den, const tfh_vm& app, const RowGrad& ga) {
  return den.grid_dim == app.grid_dim && den.channels >= 1 && den.channels <= 16 &&
         quad_lanes_ok(app, ga);
}

// Sorts the (row, mode) pairs of M rows by plane cell of a grid of size g.
template <class Src>
inline int32_t sort_pairs(int g, const Src& src, int64_t M, const SortWs& s, const char* stage,
                          hipStream_t st) {
  const int nt = (g + 1 + kTile - 1) / kTile, tiles = 3 * nt * nt;
  const int64_t pairs = 3 * M;
  ProfScope ps(stage, st);
  TFH_TRY(zero_copies(reinterpret_cast<float*>(s.tile_count), tiles, st));  // all-zero bits
  hipLaunchKernelGGL(k_tile_rank<Src>, dim3((unsigned)ceil_div(M, kRowsPerRankGroup)), dim3(256),
                     0, st, src, M, g, s.tile_count, s.tile_of, s.rank_of);
  hipLaunchKernelGGL(k_tile_scan, dim3(1), dim3(1024), 0, st, s.tile_count, tiles, s.tile_start,
                     s.chunk_start);
  hipLaunchKernelGGL(k_tile_place, dim3((unsigned)ceil_div(pairs, 256)), dim3(256), 0, st, pairs,
                     s.tile_of, s.rank_of, s.tile_start, s.order);
  // at most one partial chunk per tile beyond pairs / kSortChunk full ones
  const int64_t chunk_bound = pairs / kSortChunk + tiles;
  hipLaunchKernelGGL(k_chunk_sort<Src>, dim3((unsigned)chunk_bound), dim3(256), 0, st, src, g,
                     tiles, s.tile_start, s.chunk_start, s.order);
  return check_launch("vm scatter: pair sort");
}

// The scatter of a field's feature gradients (gsrc) for M rows whose pairs
// sort_pairs has ordered: planes into grad.plane, lines in ray order into
// grad.line (nlc copies). Fields of more than 16 channels that quad lanes
// cannot take keep the general passes (four channel slots per lane). stages:
// profile names of the plane and line passes.
template <class Src, class GS>
inline int32_t scatter_sorted_pairs(const tfh_vm& vm, const Src& src, int64_t M, const GS& gsrc,
                                    const tfh_vm_grad& grad, int nlc, const SortWs& s,
                                    const char* plane_stage, const char* line_stage,
                                    hipStream_t st) {
  if (M <= 0) return TFH_OK;
  const int g = (int)vm.grid_dim;
  const WalkField<GS> fp{vm, gsrc, grad.plane, 1}, fl{vm, gsrc, grad.line, nlc};
  const NoField none;
  if (quad_lanes_ok(vm, gsrc)) {
    TFH_TRY(launch_plane_walk<16>(src, g, M, s, fp, none, plane_stage, st));
    return launch_line_walk<16>(false, src, g, M, s, fl, none, line_stage, st);
  }
  if (vm.channels <= 8) {
    TFH_TRY(launch_plane_walk<8>(src, g, M, s, none, fp, plane_stage, st));
    return launch_line_walk<8>(false, src, g, M, s, none, fl, line_stage, st);
  }
  if (vm.channels <= 16) {
    TFH_TRY(launch_plane_walk<16>(src, g, M, s, none, fp, plane_stage, st));
    return launch_line_walk<16>(false, src, g, M, s, none, fl, line_stage, st);
  }
  {
    ProfScope ps(plane_stage, st);
    const int64_t pairs = 3 * M;
    const int64_t groups = ceil_div(pairs, kPairsPerGroup);
    hipLaunchKernelGGL((k_plane_scatter_sorted<Src, GS>), dim3((unsigned)ceil_div(groups, 16)),
                       dim3(256), 0, st, vm, src, pairs, s.order, gsrc, grad.plane);
    TFH_TRY(check_launch("vm scatter: planes"));
  }
  ProfScope ps(line_stage, st);
  hipLaunchKernelGGL((k_line_scatter<Src, GS>), dim3((unsigned)ceil_div(M, kGatherThreads / 16)),
                     dim3(kGatherThreads), 0, st, vm, src, M, gsrc, grad.line, nlc);
  return check_launch("vm scatter: lines");
}

// Whether a field takes the walks by itself.
template <class GS>
inline bool walk_ok(const tfh_vm& vm, const GS& g) {
  return vm.channels <= 16 || quad_lanes_ok(vm, g);
}

// The scatter of M rows in no particular order (walk_ok, sorted_scatter_ok): both
// passes over sorted pairs.
template <class Src, class GS>
inline int32_t scatter_scattered_rows(const tfh_vm& vm, const Src& src, int64_t M, const GS& gsrc,
                                      const tfh_vm_grad& grad, const SortWs& s, hipStream_t st) {
  const int g = (int)vm.grid_dim;
  const WalkField<GS> fp{vm, gsrc, grad.plane, 1}, fl{vm, gsrc, grad.line, 1};
  const NoField none;
  TFH_TRY(sort_pairs(g, src, M, s, "scatter_sort", st));
  if (vm.channels > 16)
    TFH_TRY(launch_plane_walk<16>(src, g, M, s, fp, none, "scatter_planes", st));
  else if (vm.channels > 8)
    TFH_TRY(launch_plane_walk<16>(src, g, M, s, none, fp, "scatter_planes", st));
  else
    TFH_TRY(launch_plane_walk<8>(src, g, M, s, none, fp, "scatter_planes", st));
  TFH_TRY(sort_lines(g, src, M, s, st));
  if (vm.channels > 16)
    return launch_line_walk<16>(true, src, g, M, s, fl, none, "scatter_lines", st);
  if (vm.channels > 8)
    return launch_line_walk<16>(true, src, g, M, s, none, fl, "scatter_lines", st);
  return launch_line_walk<8>(true, src, g, M, s, none, fl, "scatter_lines", st);
}

}  // namespace tfh
