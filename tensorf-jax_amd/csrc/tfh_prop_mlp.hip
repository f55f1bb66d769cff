// MLP of the proposal density field (no counterpart in the reference):
// z = W3 relu(W2 relu(W1 f + b1) + b2) + b3, sigma = softplus(z), with
// f the 3C <= 32 VM features of a sample, 64 hidden units, FP32 MFMA.
// Forward: 32 rows per wave, in registers. Backward (input dL/dz): persistent
// teams of four waves recompute the forward of 64 rows at a time, keep the weight
// gradients in registers and store them once per team; k_prop_reduce sums the
// teams.
#include <algorithm>

#include "tfh_mfma.h"
#include "tfh_vm_kernels.h"

namespace tfh {

constexpr int kPH = 64;       // hidden width
constexpr int kPF = 32;       // padded feature width
constexpr int kPNW = 8;       // waves per workgroup

struct PropW {
  const float *w1, *b1, *w2, *b2, *w3, *b3;
  int F;
};

// packed gradient partial: w1 (F x 64) | b1 | w2 (64 x 64) | b2 | w3 (64) | b3
struct PropPack {
  int w1, b1, w2, b2, w3, b3, total;
};

__host__ __device__ inline PropPack prop_pack(int F) {
  PropPack p;
  int o = 0;
  p.w1 = o; o += F * kPH;
  p.b1 = o; o += kPH;
  p.w2 = o; o += kPH * kPH;
  p.b2 = o; o += kPH;
  p.w3 = o; o += kPH;
  p.b3 = o; o += 1;
  p.total = (o + 63) / 64 * 64;
  return p;
}

// ---- forward --------------------------------------------------------------------
// A wave computes 32 rows in registers, the products transposed: the operand
// with 16 rows of the result is a table of the weights, the one with 16
// columns the wave's rows. A result tile holds, in lane (r, kq) = r + 16 kq,
// entries 4 kq .. 4 kq + 3 of row r; with unit 16 c + 4 e + kq of tile c at
// entry 4 kq + e (kUnit), register e of tile c is the operand that product
// 4 c + e of the next layer (inputs 16 c + 4 e + kq) reads, and no activation
// passes through LDS. Every FP32 sum runs over the inputs in ascending order,
// four to a product.
//
// Bound by the FP32 matrix rate: 24 + 64 + 16 products of 16x16x4 per 16 rows
// (the last 16 for one output), 1.35 ms for 12.6 M rows. With activations of a
// 64-row tile in LDS, read by single values, and the weights loaded per tile it
// took 2885 us there after a gather of 517, 607 after 116 for the 3.1 M rows of
// a training step; with the gather in this kernel 1770 and 414. Ten or twelve
// waves per workgroup (5 or 6 per SIMD) took 2167 and 1812.
constexpr int kPRows = 32;            // rows per wave
constexpr int kPLdT = 28;             // row stride of a wave's features: 16 rows x 4 inputs of a
                                      // product are 64 different banks

struct PropTables {
  float4 a1[4][2][64];  // [unit tile][four products][lane]
  float4 a2[4][4][64];
  float4 b1[4][4], b2[4][4];  // [unit tile][kq]
};

struct PropFwdLds {
  PropTables t;
  float4 a3[4][64];  // the output's weights in rows 0 and 4, zero elsewhere
};

__device__ __forceinline__ int prop_unit(int tile, int entry) {
  return 16 * tile + 4 * (entry & 3) + (entry >> 2);
}

__device__ __forceinline__ void prop_tables(const PropW& w, PropTables& t) {
  float* a1 = &t.a1[0][0][0].x;
  for (int e = threadIdx.x; e < 4 * 2 * 256; e += blockDim.x) {
    const int lane = (e >> 2) & 63, k = 4 * (4 * ((e >> 8) & 1) + (e & 3)) + (lane >> 4);
    a1[e] = k < w.F ? w.w1[k * kPH + prop_unit(e >> 9, lane & 15)] : 0.0f;
  }
  float* a2 = &t.a2[0][0][0].x;
  for (int e = threadIdx.x; e < 4 * 4 * 256; e += blockDim.x) {
    const int lane = (e >> 2) & 63, k = 4 * (4 * ((e >> 8) & 3) + (e & 3)) + (lane >> 4);
    a2[e] = w.w2[k * kPH + prop_unit(e >> 10, lane & 15)];
  }
  if (threadIdx.x < 64) {
    const int u = prop_unit(threadIdx.x >> 4, threadIdx.x & 15);
    (&t.b1[0][0].x)[threadIdx.x] = w.b1[u];
    (&t.b2[0][0].x)[threadIdx.x] = w.b2[u];
  }
}

__device__ __forceinline__ void prop_fwd_tables(const PropW& w, PropFwdLds& t) {
  prop_tables(w, t.t);
  float* a3 = &t.a3[0][0].x;
  for (int e = threadIdx.x; e < 4 * 256; e += blockDim.x) {
    const int lane = (e >> 2) & 63, k = 4 * (4 * (e >> 8) + (e & 3)) + (lane >> 4);
    a3[e] = (lane & 11) == 0 ? w.w3[k] : 0.0f;
  }
}

// One layer's products i < N for S sets of 16 rows and C tiles of its outputs;
// in(s, i) is the operand of set s.
template <int N, int S, int C, int G, class In>
__device__ __forceinline__ void prop_layer(const float4 (&a)[C][G][64], int lane, In in,
                                           f32x4 (&acc)[S][C]) {
#pragma unroll
  for (int s = 0; s < S; ++s) zero_acc(acc[s]);
#pragma unroll
  for (int g = 0; 4 * g < N; ++g) {
    float4 av[C];
#pragma unroll
    for (int c = 0; c < C; ++c) av[c] = a[c][g][lane];
#pragma unroll
    for (int e = 0; e < 4 && 4 * g + e < N; ++e)
#pragma unroll
      for (int c = 0; c < C; ++c)
#pragma unroll
        for (int s = 0; s < S; ++s)
          acc[s][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(
              e == 0 ? av[c].x : (e == 1 ? av[c].y : (e == 2 ? av[c].z : av[c].w)), in(s, 4 * g + e),
              acc[s][c], 0, 0, 0);
  }
}

template <int S>
__device__ __forceinline__ void prop_relu(const float4 (&b)[4][4], int kq, f32x4 (&acc)[S][4]) {
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const float4 bias = b[c][kq];
#pragma unroll
    for (int s = 0; s < S; ++s) {
      acc[s][c][0] = fmaxf(acc[s][c][0] + bias.x, 0.0f);
      acc[s][c][1] = fmaxf(acc[s][c][1] + bias.y, 0.0f);
      acc[s][c][2] = fmaxf(acc[s][c][2] + bias.z, 0.0f);
      acc[s][c][3] = fmaxf(acc[s][c][3] + bias.w, 0.0f);
    }
  }
}

// The features come from feats, or (GATHER: 8 channels, F = 24) from the
// field at pts, two lanes per sample with four channels each (the arithmetic
// of k_vm_gather4), and go to feats too. N1: first-layer products, 4 N1 >= F.
template <int N1, bool GATHER>
__global__ void __launch_bounds__(kPNW * 64, 4)
    k_prop_mlp_fwd(PropW w, float* __restrict__ feats, tfh_vm vm, const float* __restrict__ pts,
                   int64_t M, float* __restrict__ z, float* __restrict__ sigma) {
  static_assert(!GATHER || N1 == 6, "8 channels");
  __shared__ PropFwdLds t;
  __shared__ float4 rows[GATHER ? kPNW : 1][GATHER ? kPRows * kPLdT / 4 : 1];
  prop_fwd_tables(w, t);
  __syncthreads();
  const int wave = threadIdx.x >> 6;
  const int64_t tiles = (M + kPRows - 1) / kPRows;
  for (int64_t tile = (int64_t)blockIdx.x * kPNW + wave; tile < tiles;
       tile += (int64_t)gridDim.x * kPNW) {
    // (computed per tile: the tables' 128 registers would be kept otherwise)
    const int lane = lane_here(), n = lane & 15, kq = lane >> 4;
    const int64_t row0 = tile * kPRows;
    float f[2][N1];
    if constexpr (GATHER) {
      const int i = lane >> 1, c4 = 4 * (lane & 1);
      const int64_t row = row0 + i;
      const bool valid = row < M;
      const int G = (int)vm.grid_dim;
      float x = 0.f, y = 0.f, zc = 0.f;
      if (valid) {
        x = pts[row * 3];
        y = pts[row * 3 + 1];
        zc = pts[row * 3 + 2];
      }
      ModeTaps mt[3];
      mode_taps(x, y, zc, G, mt);
      float4* to = &rows[wave][i * (kPLdT / 4)];
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        TapAddr a;
        tap_addrs(mt[m], m, G, a);
        float4 lv, pv;
        tap_values4(vm.plane, vm.line, 8, c4, a, lv, pv);
        const float4 v = make_float4(lv.x * pv.x, lv.y * pv.y, lv.z * pv.z, lv.w * pv.w);
        to[2 * m + (lane & 1)] = v;
        if (valid) *reinterpret_cast<float4*>(feats + row * 24 + 8 * m + c4) = v;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      const float* from = &rows[wave][0].x;
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int j = 0; j < N1; ++j) f[s][j] = from[(16 * s + n) * kPLdT + 4 * j + kq];
      // (the next tile's writes follow these reads in the wave's LDS order)
      __builtin_amdgcn_wave_barrier();
    } else {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int64_t row = row0 + 16 * s + n;
#pragma unroll
        for (int j = 0; j < N1; ++j)
          f[s][j] = row < M && 4 * j + kq < w.F ? feats[row * w.F + 4 * j + kq] : 0.0f;
      }
    }
    f32x4 h1[2][4], h2[2][4];
    prop_layer<N1>(t.t.a1, lane, [&](int s, int j) TFH_INLINE { return f[s][j]; }, h1);
    prop_relu(t.t.b1, kq, h1);
    prop_layer<16>(t.t.a2, lane, [&](int s, int j) TFH_INLINE { return h1[s][j >> 2][j & 3]; }, h2);
    prop_relu(t.t.b2, kq, h2);
    f32x4 o[2];
    zero_acc(o);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const float4 av = t.a3[g][lane];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        o[s] = __builtin_amdgcn_mfma_f32_16x16x4f32(av.x, h2[s][g][0], o[s], 0, 0, 0);
        o[s] = __builtin_amdgcn_mfma_f32_16x16x4f32(av.y, h2[s][g][1], o[s], 0, 0, 0);
        o[s] = __builtin_amdgcn_mfma_f32_16x16x4f32(av.z, h2[s][g][2], o[s], 0, 0, 0);
        o[s] = __builtin_amdgcn_mfma_f32_16x16x4f32(av.w, h2[s][g][3], o[s], 0, 0, 0);
      }
    }
    // rows 0 and 4 of the output tile are the output: lanes 0 .. 15 take the
    // first set's, lanes 16 .. 31 the second's
    const float zv = (lane < 16 ? o[0][0] : o[1][0]) + w.b3[0];
    const int64_t row = row0 + lane;
    if (lane < kPRows && row < M) {
      if (z) z[row] = zv;
      sigma[row] = softplus(zv);
    }
  }
}

// ---- backward -------------------------------------------------------------------
// Four waves share a tile of 64 rows, 16 each through the forward and back,
// transposed as in the forward: a lane's activations and their gradients (units
// 16 c + 4 e + kq of row r) stay in registers. The products of the weight
// gradients run over the rows, so their operands cross lanes through LDS, and
// each wave sums a quarter of the 28 tiles (dW3 64 x 1, dW2 64 x 64, dW1 32 x 64) in
// registers for all its tiles. A workgroup holds two such teams, which share
// the weights' LDS. A team's tiles and the order of every sum are those that
// its number (of two per CU) and the row order give: the gradients of a batch
// do not change from run to run.
//
// Bound by the FP32 matrix rate: 296 products of 16x16x4 per 16 rows, 510 us
// for the 1.72 M rows with a gradient of a step with 16384 rays x (128 + 64)
// samples. With the activations in LDS only, read by single values, the weights
// from memory per tile and seven barriers it took 1240 us; this one takes 714.
constexpr int kPTM = 64;   // rows per tile
constexpr int kPLdH = 68;  // rows of 64 values: rows 0, 4, 8, 12 x 16 values are 64 banks

// A team's LDS: activations and gradients of the tile's rows, value 16 c +
// 4 kq + e of a row for unit 16 c + 4 e + kq.
struct PropTeam {
  float h1[kPTM * kPLdH];  // h1, then dZ1
  float d2[kPTM * kPLdH];  // dZ2, then the features
  float h2[kPTM * kPLdH];
  float g[kPTM];           // dL/dz
};

struct PropBwdLds {
  PropTables t;
  float4 a2t[4][4][64];  // W2 and W1 as operands of the input gradients
  float4 a1t[2][4][64];
  float4 w3[4][4];       // [unit tile][kq]
  PropTeam team[2];
};
static_assert(kPNW == 8 && sizeof(PropBwdLds) <= 160 * 1024, "two teams of four, one workgroup per CU");

// A workgroup barrier that orders LDS only: loads from memory stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// 16 rows x 64 values (value 16 c + 4 kq + e of row r in register e of tile c)
// to LDS.
__device__ __forceinline__ void prop_put(float* to, int n, int kq, const f32x4 (&v)[4]) {
#pragma unroll
  for (int c = 0; c < 4; ++c)
    *reinterpret_cast<f32x4*>(to + n * kPLdH + 16 * c + 4 * kq) = v[c];
}

// acc[c] += X[:, 16 c ..]^T Y[:, col ..] over a tile's rows, 4 kq + i of each 16
// in product i.
template <int C>
__device__ __forceinline__ void prop_wgrad(const float* X, const float* Y, int col, int n, int kq,
                                           f32x4 (&acc)[C]) {
#pragma unroll
  for (int k0 = 0; k0 < kPTM; k0 += 16) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = (k0 + 4 * kq + i) * kPLdH;
      const float b = Y[row + col + n];
#pragma unroll
      for (int c = 0; c < C; ++c)
        acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(X[row + 16 * c + n], b, acc[c], 0, 0, 0);
    }
  }
}

// Rows: all M, or the first min(M, *count) entries of idx (feature and dz row
// of each); dfeat is written per processed row. teams: the partials; workgroup
// b's teams are 2b and 2b + 1. N1: as in the forward.
template <int N1>
__global__ void __launch_bounds__(kPNW * 64, 2)
    k_prop_mlp_bwd(PropW w, const float* __restrict__ feats, const float* __restrict__ dz,
                   int64_t M_max, const int32_t* __restrict__ idx,
                   const int32_t* __restrict__ count, float* __restrict__ dfeat,
                   float* __restrict__ partials, int teams) {
  extern __shared__ float4 prop_lds[];
  PropBwdLds& s = *reinterpret_cast<PropBwdLds*>(prop_lds);
  const int64_t M = count ? min(M_max, (int64_t)*count) : M_max;
  prop_tables(w, s.t);
  float* a2t = &s.a2t[0][0][0].x;
  for (int e = threadIdx.x; e < 4 * 4 * 256; e += blockDim.x) {
    const int lane = (e >> 2) & 63, u = 4 * (4 * ((e >> 8) & 3) + (e & 3)) + (lane >> 4);
    a2t[e] = w.w2[prop_unit(e >> 10, lane & 15) * kPH + u];
  }
  float* a1t = &s.a1t[0][0][0].x;
  for (int e = threadIdx.x; e < 2 * 4 * 256; e += blockDim.x) {
    const int lane = (e >> 2) & 63, u = 4 * (4 * ((e >> 8) & 3) + (e & 3)) + (lane >> 4);
    const int k = 16 * (e >> 10) + (lane & 15);
    a1t[e] = k < w.F ? w.w1[k * kPH + u] : 0.0f;
  }
  if (threadIdx.x < 64)
    (&s.w3[0][0].x)[threadIdx.x] = w.w3[prop_unit(threadIdx.x >> 4, threadIdx.x & 15)];
  const int wave = (threadIdx.x >> 6) & 3;  // of the team
  PropTeam& tm = s.team[threadIdx.x >> 8];
  const int team = 2 * blockIdx.x + (threadIdx.x >> 8);
  __syncthreads();
  f32x4 dw3[1], dw2[4], dw1[2];
  zero_acc(dw3);
  zero_acc(dw2);
  zero_acc(dw1);
  float db = 0.0f;   // lane u of wave 0: db2, of wave 1: db1 of value u
  float db3 = 0.0f;  // wave 2
  // the same number of rounds for both teams; a team past the end has no rows
  const int64_t tiles = (M + kPTM - 1) / kPTM;
  int64_t tile = team < teams ? team : tiles;
  // the features and dL/dz of a tile's rows are requested one tile ahead
  float f[1][N1], g;
  auto request = [&](int64_t at, int n, int kq) TFH_INLINE {
    const int64_t i = at * kPTM + 16 * wave + n;
    const bool valid = i < M;
    const int64_t row = valid ? (idx ? (int64_t)idx[i] : i) : 0;
#pragma unroll
    for (int j = 0; j < N1; ++j)
      f[0][j] = valid && 4 * j + kq < w.F ? feats[row * w.F + 4 * j + kq] : 0.0f;
    g = valid ? dz[row] : 0.0f;
  };
  request(tile, lane_id() & 15, lane_id() >> 4);
  for (int64_t first = 2 * blockIdx.x; first < tiles; first += teams, tile += teams) {
    const int lane = lane_here(), n = lane & 15, kq = lane >> 4;
    const int row0 = 16 * wave * kPLdH;  // the wave's rows
    float f0[1][N1];
    const float gz = g;
    f32x4 h1[1][4], h2[1][4], d1[1][4];
#pragma unroll
    for (int j = 0; j < N1; ++j) f0[0][j] = f[0][j];
    prop_layer<N1>(s.t.a1, lane, [&](int, int j) TFH_INLINE { return f0[0][j]; }, h1);
    request(tile + teams, n, kq);
    prop_relu(s.t.b1, kq, h1);
    prop_put(tm.h1 + row0, n, kq, h1[0]);
    prop_layer<16>(s.t.a2, lane, [&](int, int j) TFH_INLINE { return h1[0][j >> 2][j & 3]; }, h2);
    prop_relu(s.t.b2, kq, h2);
    prop_put(tm.h2 + row0, n, kq, h2[0]);
    if (kq == 0) tm.g[16 * wave + n] = gz;
    // dZ2 = dz W3^T where h2 > 0
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float4 w3 = s.w3[c][kq];
      const float wv[4] = {w3.x, w3.y, w3.z, w3.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) h2[0][c][e] = h2[0][c][e] > 0.0f ? gz * wv[e] : 0.0f;
    }
    prop_put(tm.d2 + row0, n, kq, h2[0]);
    lds_barrier();
    // dW3 += h2^T dz, dW2 += h1^T dZ2
#pragma unroll
    for (int k0 = 0; k0 < kPTM; k0 += 16)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = k0 + 4 * kq + i;
        dw3[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(tm.h2[row * kPLdH + 16 * wave + n],
                                                      n == 0 ? tm.g[row] : 0.0f, dw3[0], 0, 0, 0);
      }
    prop_wgrad(tm.h1, tm.d2, 16 * wave, n, kq, dw2);
    if (wave == 0) {
#pragma unroll 16
      for (int i = 0; i < kPTM; ++i) db += tm.d2[i * kPLdH + lane];
    } else if (wave == 2) {
#pragma unroll 16
      for (int i = 0; i < kPTM; ++i) db3 += tm.g[i];
    }
    // dZ1 = dZ2 W2^T where h1 > 0
    prop_layer<16>(s.a2t, lane, [&](int, int j) TFH_INLINE { return h2[0][j >> 2][j & 3]; }, d1);
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) d1[0][c][e] = h1[0][c][e] > 0.0f ? d1[0][c][e] : 0.0f;
    lds_barrier();
    prop_put(tm.h1 + row0, n, kq, d1[0]);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      tm.d2[row0 + n * kPLdH + 4 * j + kq] = j < N1 ? f0[0][j < N1 ? j : 0] : 0.0f;
    lds_barrier();
    // dW1 += F^T dZ1, dF = dZ1 W1^T
    prop_wgrad(tm.d2, tm.h1, 16 * wave, n, kq, dw1);
    if (wave == 1) {
#pragma unroll 16
      for (int i = 0; i < kPTM; ++i) db += tm.h1[i * kPLdH + lane];
    }
    if (dfeat) {
      f32x4 df[1][2];
      prop_layer<16>(s.a1t, lane, [&](int, int j) TFH_INLINE { return d1[0][j >> 2][j & 3]; }, df);
      const int64_t row = tile * kPTM + 16 * wave + n;
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int k = 16 * c + 4 * kq + e;
          if (row < M && k < w.F) dfeat[row * w.F + k] = df[0][c][e];
        }
    }
    lds_barrier();
  }
  if (team >= teams) return;
  const int lane = lane_id(), n = lane & 15, kq = lane >> 4;
  const PropPack pp = prop_pack(w.F);
  float* part = partials + (int64_t)team * pp.total;
  const int u = prop_unit(wave, n);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
#pragma unroll
    for (int c = 0; c < 4; ++c) part[pp.w2 + prop_unit(c, 4 * kq + e) * kPH + u] = dw2[c][e];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int k = 16 * c + 4 * kq + e;
      if (k < w.F) part[pp.w1 + k * kPH + u] = dw1[c][e];
    }
    if (n == 0) part[pp.w3 + prop_unit(wave, 4 * kq + e)] = dw3[0][e];
  }
  if (wave == 0) part[pp.b2 + prop_unit(lane >> 4, lane & 15)] = db;
  if (wave == 1) part[pp.b1 + prop_unit(lane >> 4, lane & 15)] = db;
  if (wave == 2 && lane == 0) part[pp.b3] = db3;
}

// Sum of the workgroup partials: a workgroup owns 64 consecutive entries and
// its kPRedWaves waves split the partials (wave w adds rows w, w + kPRedWaves,
// ...), so every load is one coalesced 256-byte row segment; the waves' sums
// meet in LDS and are added in a fixed order.
constexpr int kPRedWaves = 16;

__global__ void __launch_bounds__(64 * kPRedWaves) k_prop_reduce(const float* __restrict__ partials,
                                                                int64_t nblk, PropPack pp,
                                                                tfh_prop_mlp_grad g) {
  __shared__ float red[kPRedWaves][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int n = pp.b3 + 1;
  const int e = blockIdx.x * 64 + lane;
  float part = 0.0f;
  if (e < n) {
#pragma unroll 8
    for (int64_t b = w; b < nblk; b += kPRedWaves) part += partials[b * pp.total + e];
  }
  red[w][lane] = part;
  __syncthreads();
  if (w == 0 && e < n) {
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < kPRedWaves; ++i) s += red[i][lane];
    float* dst;
    int o;
    if (e >= pp.b3) { dst = g.b3; o = e - pp.b3; }
    else if (e >= pp.w3) { dst = g.w3; o = e - pp.w3; }
    else if (e >= pp.b2) { dst = g.b2; o = e - pp.b2; }
    else if (e >= pp.w2) { dst = g.w2; o = e - pp.w2; }
    else if (e >= pp.b1) { dst = g.b1; o = e - pp.b1; }
    else { dst = g.w1; o = e - pp.w1; }
    dst[o] += s;
  }
}

// Persistent backward: two teams per CU.
static int64_t prop_bwd_teams(int64_t M) {
  return std::max<int64_t>(1, std::min<int64_t>(ceil_div(M, kPTM), 2 * (int64_t)num_cus()));
}

int32_t check_prop_mlp(const tfh_prop_mlp* p, const char* who) {
  TFH_REQUIRE(p != nullptr, "%s: null tfh_prop_mlp", who);
  TFH_REQUIRE(p->w1 && p->b1 && p->w2 && p->b2 && p->w3 && p->b3, "%s: null proposal weight", who);
  TFH_REQUIRE(p->feat_dim >= 1 && p->feat_dim <= kPF, "%s: proposal feat_dim %lld outside [1, %d]",
              who, (long long)p->feat_dim, kPF);
  return TFH_OK;
}

static PropW to_pw(const tfh_prop_mlp* p) {
  return PropW{p->w1, p->b1, p->w2, p->b2, p->w3, p->b3, (int)p->feat_dim};
}

static unsigned prop_fwd_blocks(int64_t M) {
  return (unsigned)std::min<int64_t>(ceil_div(M, kPNW * kPRows), 2 * (int64_t)num_cus());
}

int32_t prop_mlp_fwd(const tfh_prop_mlp* p, const float* feats, int64_t M, float* z, float* sigma,
                     hipStream_t st) {
  if (M == 0) return TFH_OK;
  ProfScope ps("prop_mlp_fwd", st);
  auto kernel = p->feat_dim <= 24 ? k_prop_mlp_fwd<6, false> : k_prop_mlp_fwd<8, false>;
  hipLaunchKernelGGL(kernel, dim3(prop_fwd_blocks(M)), dim3(kPNW * 64), 0, st, to_pw(p),
                     const_cast<float*>(feats), tfh_vm{}, nullptr, M, z, sigma);
  return check_launch("proposal mlp fwd");
}

// The features of the field at pts (M, 3) to feats and the MLP on them: one
// kernel for 8 channels behind 16-byte aligned pointers, the gather and the
// MLP by themselves otherwise.
int32_t prop_mlp_fwd_gather(const tfh_prop_mlp* p, const tfh_vm& field, const float* pts,
                            int64_t M, float* feats, float* sigma, hipStream_t st) {
  if (M == 0) return TFH_OK;
  const uintptr_t any = reinterpret_cast<uintptr_t>(field.plane) |
                        reinterpret_cast<uintptr_t>(field.line) |
                        reinterpret_cast<uintptr_t>(feats);
  if (field.channels == 8 && p->feat_dim == 24 && (any & 15) == 0) {
    ProfScope ps("prop_mlp_fwd", st);
    hipLaunchKernelGGL((k_prop_mlp_fwd<6, true>), dim3(prop_fwd_blocks(M)), dim3(kPNW * 64), 0,
                       st, to_pw(p), feats, field, pts, M, nullptr, sigma);
    return check_launch("proposal mlp fwd with the gather");
  }
  {
    ProfScope ps("prop_gather", st);
    const RaySamples src{pts, nullptr, 1, 1};
    TFH_TRY((launch_vm_gather<RaySamples, true>(field, src, M, feats, st)));
  }
  return prop_mlp_fwd(p, feats, M, nullptr, sigma, st);
}

size_t prop_mlp_bwd_workspace(const tfh_prop_mlp* p, int64_t M) {
  return align_up((size_t)prop_bwd_teams(M) * prop_pack((int)p->feat_dim).total * sizeof(float),
                  256);
}

int32_t prop_mlp_bwd(const tfh_prop_mlp* p, const float* feats, const float* dz, int64_t M,
                     float* dfeat, const tfh_prop_mlp_grad* g, void* ws, size_t ws_bytes,
                     hipStream_t st, const int32_t* idx = nullptr,
                     const int32_t* count = nullptr) {
  if (M == 0) return TFH_OK;
  const int64_t teams = prop_bwd_teams(M);
  const PropPack pp = prop_pack((int)p->feat_dim);
  TFH_REQUIRE(ws_bytes >= prop_mlp_bwd_workspace(p, M), "proposal mlp bwd: workspace too small");
  float* partials = static_cast<float*>(ws);
  {
    ProfScope ps("prop_mlp_bwd", st);
    auto kernel = p->feat_dim <= 24 ? k_prop_mlp_bwd<6> : k_prop_mlp_bwd<8>;
    allow_lds(kernel, sizeof(PropBwdLds));
    hipLaunchKernelGGL(kernel, dim3((unsigned)ceil_div(teams, 2)), dim3(kPNW * 64),
                       sizeof(PropBwdLds), st, to_pw(p), feats, dz, M, idx, count, dfeat,
                       partials, (int)teams);
  }
  TFH_TRY(check_launch("proposal mlp bwd"));
  hipLaunchKernelGGL(k_prop_reduce, dim3((unsigned)ceil_div(pp.b3 + 1, 64)),
                     dim3(64 * kPRedWaves), 0, st, partials, teams, pp, *g);
  return check_launch("proposal mlp reduce");
}

}  // namespace tfh

using namespace tfh;

extern "C" {

int32_t tfh_prop_mlp_fwd(const tfh_prop_mlp* mlp, const float* features, int64_t num_rows,
                         float* z, float* sigma, tfh_stream_t stream) {
  TFH_TRY(check_prop_mlp(mlp, "tfh_prop_mlp_fwd"));
  TFH_REQUIRE(num_rows >= 0, "tfh_prop_mlp_fwd: negative num_rows");
  if (num_rows == 0) return TFH_OK;
  TFH_REQUIRE(features && sigma, "tfh_prop_mlp_fwd: null pointer");
  TFH_TRY(require_device());
  return prop_mlp_fwd(mlp, features, num_rows, z, sigma, as_stream(stream));
}

size_t tfh_prop_mlp_bwd_workspace_size(const tfh_prop_mlp* mlp, int64_t num_rows) {
  if (check_prop_mlp(mlp, "tfh_prop_mlp_bwd_workspace_size") != TFH_OK || num_rows < 0) return 0;
  return prop_mlp_bwd_workspace(mlp, num_rows);
}

int32_t tfh_prop_mlp_bwd(const tfh_prop_mlp* mlp, const float* features, int64_t num_rows,
                         const float* grad_z, float* grad_features,
                         const tfh_prop_mlp_grad* grad, void* workspace, size_t workspace_bytes,
                         tfh_stream_t stream) {
  TFH_TRY(check_prop_mlp(mlp, "tfh_prop_mlp_bwd"));
  TFH_REQUIRE(num_rows >= 0, "tfh_prop_mlp_bwd: negative num_rows");
  if (num_rows == 0) return TFH_OK;
  TFH_REQUIRE(features && grad_z && grad && grad->w1 && grad->b1 && grad->w2 && grad->b2 &&
                  grad->w3 && grad->b3 && workspace,
              "tfh_prop_mlp_bwd: null pointer");
  TFH_TRY(require_device());
  return prop_mlp_bwd(mlp, features, grad_z, num_rows, grad_features, grad, workspace,
                      workspace_bytes, as_stream(stream));
}

}  // extern "C"
