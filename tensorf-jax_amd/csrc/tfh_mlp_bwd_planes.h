// Backward of the FeatureMlp shapes with compile-time dims (networks.py:38-121)
// that reads the activations the forward kernel kept: relu(z1), relu(z2)
// (before any FiLM camera embedding) and the output.
//
// Every product runs on v_mfma_f32_16x16x32_bf16. NP is the number of BF16
// planes an operand is held in:
//   NP = 1  the BF16 MLP: operands rounded to BF16, as everywhere in that mode.
//   NP = 3  the FP32 MLP: v = hi + mid + lo, three BF16 values (round to nearest
//           each; 24 significant bits, so the sum is v exactly, but for values
//           below 2^-110, whose lo falls under BF16's range: their error is at
//           most 2^-126), and a product is six MFMAs (hi hi, hi mid, mid hi,
//           mid mid, hi lo, lo hi) with FP32 accumulation. The dropped terms are below 2^-25 of a
//           product, under the rounding of an FP32 multiply-add. Six BF16
//           products of K = 32 take 96 SIMD cycles where the eight
//           v_mfma_f32_16x16x4_f32 they replace take 256. An operand that is
//           infinite (or above BF16's largest finite value) makes NaN of every
//           sum it enters: a workgroup that finds NaN in its sums says so in
//           its flag, and k_mlp_bwd, launched behind this kernel, then does the
//           batch again with FP32 products.
//
// One workgroup of 8 waves per CU walks tiles of TM rows; every weight-gradient
// tile stays in registers of its owning wave for the whole kernel: wave w owns
// column tile w of dW2 and dW1, whose Y operand (dZ2, dZ1) it has just
// computed: a lane's results of two row tiles are its operand of a K = 32
// product over the rows in the order 16 (e / 4) + 4 (lane / 16) + e % 4, which
// the X operands follow. Per tile, with one barrier after each step:
//   commit  the tile's inputs, loaded during the previous tile, go to LDS
//   B       layer 0 (h0, in K parts) ; dZ2 = (dZ3 W3^T) [z2 > 0], db2, dW3 ;
//           dW2 += H1^T dZ2
//   C       the encoding -> X ; dZ1 = (dZ2 W2^T) [z1 > 0], db1
//   D       dW1 += X^T dZ1 ; dX = dZ1 W1^T for the columns that feed h0
//   E       the next tile's loads are issued ; dH0 from dX and the encoding's
//           sines and cosines
//   F       dW0 += F^T dH0 ; dF = dH0 W0^T
//
// Measured against the FP32-MFMA / FP32-rows-in-LDS kernel this replaces
// (32-row tiles, weight-gradient operands read a float at a time): 2.1 M rows
// FP32 4.22 -> 2.71 ms; BF16 1.05 M rows 1.29 -> 0.63 ms; with the embedding,
// BF16, 4.2 M rows 5.85 -> 2.77 ms. What bounds it (counters, FP32): LDS busy
// 52% of the cycles, MFMA 37%, vector ALU 35%, one workgroup per CU (its
// 140-160 KB of LDS and 250 registers), so the steps' latencies show.
// 64-row tiles in BF16 halve the weight-table reads and barriers per row
// (0.73 -> 0.64 ms per 1 M rows with them against 32); three planes of 64 rows
// do not fit the LDS.
#pragma once

#include "tfh_mlp_kernels.h"

namespace tfh {

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

// The encoded input X in this kernel: its columns in NH groups (one after the
// other in the same LDS when a shape's X does not fit whole), each the Fourier
// features (nf sines, nf cosines per value) of some of the values of h0, then
// those values; the last group also those of the direction, then the
// direction. x_orig maps a column of a group to its row of W1.
template <int F_, int NF_, int NH_>
struct BwdShape {
  static constexpr int F = F_, S = 27, NF = NF_, FEW = 2 * NF_, NH = NH_;
  static constexpr int E = S + 3 + FEW * (S + 3);
  static constexpr int FK = (F + 31) / 32 * 32;        // K of layer 0
  static constexpr int FT = (F + 15) / 16;             // feature column tiles
  static constexpr int HF = (S + NH - 1) / NH;
  static constexpr int first(int h) { return h * HF; }               // first value of group h
  static constexpr int count(int h) { return h < NH - 1 ? HF : S - (NH - 1) * HF; }
  static constexpr int values(int h) { return count(h) + (h == NH - 1 ? 3 : 0); }
  static constexpr int XT(int h) { return (values(h) * (FEW + 1) + 15) / 16; }  // column tiles
  static constexpr int DXT(int h) { return (count(h) * (FEW + 1) + 15) / 16; }  // that feed h0
  static constexpr int xt0(int h) { return h == 0 ? 0 : xt0(h - 1) + XT(h - 1); }
  static constexpr int dxt0(int h) { return h == 0 ? 0 : dxt0(h - 1) + DXT(h - 1); }
  static constexpr int maxXT() { return NH == 1 || XT(0) > XT(NH - 1) ? XT(0) : XT(NH - 1); }
  static constexpr int maxDXT() { return NH == 1 || DXT(0) > DXT(NH - 1) ? DXT(0) : DXT(NH - 1); }
  __host__ __device__ static constexpr int x_orig(int h, int c) {
    const int n = count(h), d = c - n * (FEW + 1);
    return c < n * FEW ? S + 3 + FEW * first(h) + c
                       : (d < 0 ? first(h) + c - n * FEW
                                : (h < NH - 1 ? -1
                                              : (d < 3 * FEW ? S + 3 + FEW * S + d
                                                             : (d < 3 * FEW + 3 ? S + d - 3 * FEW
                                                                                : -1))));
  }
};
using BwdStd = BwdShape<144, 2, 1>;  // 48 channels, 2 frequencies
using BwdDef = BwdShape<72, 6, 2>;   // 24 channels, 6 frequencies: the reference's defaults

// Operand tables of the backward (B operands; B(k, j) below), zero padded:
//   f0: W0[k][j], FK x 32    g0: W0[j][k], 32 x 16 FT    g2: W2[j][k], U x U
//   g1: W1[j][k], U x 16 per dX tile (j in X's column order)     g3: W3[j][k], 32 x U
// in the order the lanes read them: for each column tile and chunk of 32 k,
// NP planes of 64 lanes x 8 values, so a lane's load is 16 bytes of a
// contiguous kilobyte.
template <class SH>
struct BwdTables {
  static constexpr int f0 = 32 * SH::FK, g0 = 16 * SH::FT * 32, g1 = 16 * SH::dxt0(SH::NH) * kU,
                       g2 = kU * kU, g3 = kU * 32;
  static constexpr int o_g0 = f0, o_g1 = o_g0 + g0, o_g2 = o_g1 + g1, o_g3 = o_g2 + g2,
                       total = o_g3 + g3;  // values; a table of NP planes starts at NP * o
};

constexpr int kPackThreads = 256;
constexpr float kBf16Max = 3.38953139e38f;  // BF16's largest finite value

__device__ __forceinline__ void split3(float v, __bf16& h, __bf16& m, __bf16& l) {
  h = (__bf16)v;
  const float r = v - (float)h;
  m = (__bf16)r;
  l = (__bf16)(r - (float)m);
}

// flags (three planes): one per workgroup, whether it met a weight that the planes
// cannot hold.
template <class SH, int NP>
__global__ void __launch_bounds__(kPackThreads) k_pack_bwd(MlpW w, __bf16* __restrict__ t,
                                                          int32_t* __restrict__ flags) {
  using T = BwdTables<SH>;
  static_assert(T::total % kPackThreads == 0, "every thread has an entry");
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  const int base = e < T::o_g0 ? 0 : (e < T::o_g1 ? T::o_g0 : (e < T::o_g2 ? T::o_g1
                 : (e < T::o_g3 ? T::o_g2 : T::o_g3)));
  const int kc = base == 0 ? SH::FK / 32 : (base == T::o_g1 || base == T::o_g2 ? kU / 32 : 1);
  const int f = e - base, blk = f >> 9, lane = (f >> 3) & 63;
  const int j = 16 * (blk / kc) + (lane & 15), k = 32 * (blk % kc) + 8 * (lane >> 4) + (f & 7);
  float v = 0.0f;
  if (base == 0) {
    if (j < SH::S && k < SH::F) v = w.w0[k * SH::S + j];
  } else if (base == T::o_g0) {
    if (j < SH::F && k < SH::S) v = w.w0[j * SH::S + k];
  } else if (base == T::o_g1) {
    const bool tail = SH::NH > 1 && j >= 16 * SH::dxt0(SH::NH - 1);
    const int o = tail ? SH::x_orig(SH::NH - 1, j - 16 * SH::dxt0(SH::NH - 1)) : SH::x_orig(0, j);
    if (o >= 0) v = w.w1[o * kU + k];
  } else if (base == T::o_g2) {
    v = w.w2[j * kU + k];
  } else if (k < 3) {
    v = w.w3[j * 3 + k];
  }
  __bf16* o = t + NP * base + blk * NP * 512 + (f & 511);
  if constexpr (NP == 1) {
    o[0] = (__bf16)v;
  } else {
    split3(v, o[0], o[512], o[1024]);
    __shared__ int bad;
    if (threadIdx.x == 0) bad = 0;
    __syncthreads();
    if (!(fabsf(v) <= kBf16Max)) bad = 1;
    __syncthreads();
    if (threadIdx.x == 0) flags[blockIdx.x] = bad;
  }
}

// One lane's operand of a K = 32 product: 8 values in each plane.
template <int NP>
struct Frag {
  bf16x8 p[NP];
};

// acc + low += A B. With three planes the five small products go to `low`,
// whose values stay small: the unit aligns an MFMA's products to the largest of
// them and C and cuts off what falls below, so small products added to a large
// C would leave a bias towards minus infinity (-7e-9 of the result's rms at
// K = 128, 50 times that of the separate sum, and 1e-6 in a bias gradient's
// sum over 20,000 rows). The error of a K = 128 product against float64 is
// 0.65e-7 of the rms, of the FP32 unit's 2.0e-7. Weight gradients summed over
// 2.1 M rows (256 tiles a workgroup, gradients of one sign) against float64, rms
// error over rms: W1 4.8e-7, W2 2.7e-7, b1 3.8e-7, b2 2.5e-7, W0 7.5e-6 (ReLU edges,
// in FP32 products too); with FP32 products 4.9e-7, 2.9e-7, 4.0e-7, 2.4e-7, 7.5e-6.
template <int NP>
__device__ __forceinline__ void mma(f32x4& acc, f32x4& low, const Frag<NP>& a, const Frag<NP>& b) {
  if constexpr (NP == 3) {
    low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.p[0], b.p[2], low, 0, 0, 0);
    low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.p[2], b.p[0], low, 0, 0, 0);
    low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.p[1], b.p[1], low, 0, 0, 0);
    low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.p[0], b.p[1], low, 0, 0, 0);
    low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.p[1], b.p[0], low, 0, 0, 0);
  }
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.p[0], b.p[0], acc, 0, 0, 0);
}
// acc += low, here: left alone, the adds of a whole step move to its end and
// hold its registers.
template <int NP>
__device__ __forceinline__ void fold(f32x4& acc, const f32x4& low) {
  if constexpr (NP == 3) {
    acc += low;
    asm volatile("" : "+v"(acc));
  }
}
// The same for one product onto a running sum.
template <int NP>
__device__ __forceinline__ void mma_add(f32x4& acc, const Frag<NP>& a, const Frag<NP>& b) {
  f32x4 low{0.f, 0.f, 0.f, 0.f};
  mma<NP>(acc, low, a, b);
  fold<NP>(acc, low);
}

// A matrix of BF16 planes in LDS: TM rows of LD values per plane.
template <int NP, int TM, int LD>
struct Planes {
  static constexpr int ps = TM * LD;     // one plane
  static constexpr int bytes = NP * ps * 2;
  __bf16* m;
  // Operand over columns: row `row`, values k .. k + 7.
  __device__ __forceinline__ Frag<NP> row8(int row, int k) const {
    Frag<NP> f;
#pragma unroll
    for (int p = 0; p < NP; ++p)
      f.p[p] = *reinterpret_cast<const bf16x8*>(m + p * ps + row * LD + k);
    return f;
  }
  // Operand over rows (transposed read): column col0 + lane % 16, rows
  // 32 k + 16 (e / 4) + 4 (lane / 16) + e % 4 for e < 8. The 16 lanes of a group
  // point at a block of 4 rows by 16 columns (lane i at row i / 4, columns
  // 4 (i % 4) ..) and each receives one column of it. 64 bytes a clock for any
  // row stride that is not a multiple of 64 dwords.
  __device__ __forceinline__ Frag<NP> over_rows(int col0, int k, int lane) const {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s16x4* lds_ptr;
    const int i = lane & 15, kq = lane >> 4;
    Frag<NP> f;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const __bf16* at = m + p * ps + (32 * k + 4 * kq + (i >> 2)) * LD + col0 + 4 * (i & 3);
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(at));
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(at + 16 * LD));
      typedef short s16x8 __attribute__((ext_vector_type(8)));
      f.p[p] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
    return f;
  }
  __device__ __forceinline__ void put(int row, int col, float v) const {
    if constexpr (NP == 1) {
      m[row * LD + col] = (__bf16)v;
    } else {
      split3(v, m[row * LD + col], m[ps + row * LD + col], m[2 * ps + row * LD + col]);
    }
  }
  __device__ __forceinline__ void put4(int row, int col, const float (&v)[4]) const {
    bf16x4 h, md, l;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if constexpr (NP == 1) {
        h[q] = (__bf16)v[q];
      } else {
        __bf16 a, b, c;
        split3(v[q], a, b, c);
        h[q] = a; md[q] = b; l[q] = c;
      }
    }
    *reinterpret_cast<bf16x4*>(m + row * LD + col) = h;
    if constexpr (NP == 3) {
      *reinterpret_cast<bf16x4*>(m + ps + row * LD + col) = md;
      *reinterpret_cast<bf16x4*>(m + 2 * ps + row * LD + col) = l;
    }
  }
};

// The transpose in LDS: per column TM rows, in groups of 32 ordered so that a
// lane's operand over the rows is one 16-byte read (row_pos).
__device__ __forceinline__ int row_pos(int row) {
  return (row & ~31) + 8 * ((row & 15) >> 2) + 4 * ((row >> 4) & 1) + (row & 3);
}
template <int NP, int TM, int COLS>
struct PlanesT {
  static constexpr int LD = TM + 8;
  static constexpr int ps = COLS * LD;
  static constexpr int bytes = NP * ps * 2;
  __bf16* m;
  __device__ __forceinline__ Frag<NP> over_rows(int col0, int k, int lane) const {
    Frag<NP> f;
#pragma unroll
    for (int p = 0; p < NP; ++p)
      f.p[p] = *reinterpret_cast<const bf16x8*>(m + p * ps + (col0 + (lane & 15)) * LD + 32 * k +
                                                8 * (lane >> 4));
    return f;
  }
  __device__ __forceinline__ void put_frag(int col, int k, int kq, const Frag<NP>& f) const {
#pragma unroll
    for (int p = 0; p < NP; ++p)
      *reinterpret_cast<bf16x8*>(m + p * ps + col * LD + 32 * k + 8 * kq) = f.p[p];
  }
  __device__ __forceinline__ void put(int pos, int col, float v) const {
    __bf16* at = m + col * LD + pos;
    if constexpr (NP == 1)
      at[0] = (__bf16)v;
    else
      split3(v, at[0], at[ps], at[2 * ps]);
  }
};

template <int NP>
__device__ __forceinline__ void set_frag(Frag<NP>& f, int e, float v) {
  if constexpr (NP == 1) {
    f.p[0][e] = (__bf16)v;
  } else {
    __bf16 a, b, c;
    split3(v, a, b, c);
    f.p[0][e] = a; f.p[1][e] = b; f.p[2][e] = c;
  }
}

// A table of KC chunks of 32 k per column tile as the B operand.
template <int NP, int KC>
struct TableB {
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ TableB(const __bf16* t, int values)
      : r(buffer_rsrc(t, NP * values * 2)) {}
  __device__ __forceinline__ Frag<NP> load(int ct, int c) const {
    typedef int i32x4 __attribute__((ext_vector_type(4)));
    const int lane = lane_here();
    Frag<NP> f;
#pragma unroll
    for (int p = 0; p < NP; ++p)
      f.p[p] = __builtin_bit_cast(
          bf16x8, (i32x4)__builtin_amdgcn_raw_buffer_load_b128(
                      r, lane * 16 + p * 1024, (ct * KC + c) * NP * 1024, 0));
    return f;
  }
};

// acc[rt] += A(rows row0 + 16 rt .., values 32 c0 ..) B(., column tile ct) over
// the chunks [c0, c0 + KC) of 32; the first PD chunks of B are in ring, the
// rest are requested PD chunks ahead of their use.
template <int NP, bool AHEAD, int RT, int KC, int PD, class AP, class BT>
__device__ __forceinline__ void strip(const AP& A, int row0, int c0, const BT& b, int ct,
                                      f32x4 (&acc)[RT], Frag<NP> (&ring)[PD]) {
  const int lane = lane_here();
  const int r = lane & 15, kq = lane >> 4;
  f32x4 low[RT];
  zero_acc(low);
  // AHEAD: the next chunk's A is read ahead of this chunk's products
  Frag<NP> a[AHEAD ? 2 : 1][RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) a[0][rt] = A.row8(row0 + 16 * rt + r, 32 * c0 + 8 * kq);
#pragma unroll
  for (int c = 0; c < KC; ++c) {
    const int n = AHEAD ? c + 1 : c;
    if (n > 0 && n < KC) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
        a[AHEAD ? n & 1 : 0][rt] = A.row8(row0 + 16 * rt + r, 32 * (c0 + n) + 8 * kq);
    }
    if (AHEAD) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) mma<NP>(acc[rt], low[rt], a[AHEAD ? c & 1 : 0][rt], ring[c % PD]);
    if (c + PD < KC) ring[c % PD] = b.load(ct, c0 + c + PD);
    __builtin_amdgcn_sched_barrier(0);
  }
  if constexpr (NP == 3) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) acc[rt] += low[rt];
  }
}

// Weight-gradient tiles: acc[AT + i] += X[:, tile i]^T y over the 32 rows of
// group k, i < NX. AHEAD: the next X operand is read ahead.
template <int NP, bool AHEAD, int NX, int AT, int NA, class XP>
__device__ __forceinline__ void wgrad(const XP& X, int k, const Frag<NP>& y, f32x4 (&acc)[NA]) {
  const int lane = lane_here();
  Frag<NP> x[AHEAD ? 2 : 1];
  f32x4 low[2];  // folded a tile later: the sum waits for no product
  x[0] = X.over_rows(0, k, lane);
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    const int n = AHEAD ? i + 1 : i;
    if (n > 0 && n < NX) x[AHEAD ? n & 1 : 0] = X.over_rows(16 * n, k, lane);
    if (AHEAD) __builtin_amdgcn_sched_barrier(0);
    low[i & 1] = f32x4{0.f, 0.f, 0.f, 0.f};
    mma<NP>(acc[AT + i], low[i & 1], x[AHEAD ? i & 1 : 0], y);
    if (i > 0) fold<NP>(acc[AT + i - 1], low[(i - 1) & 1]);
    __builtin_amdgcn_sched_barrier(0);
  }
  fold<NP>(acc[AT + NX - 1], low[(NX - 1) & 1]);
}

template <int NP, int PD, class BT>
__device__ __forceinline__ void strip_pre(const BT& b, int ct, int c0, Frag<NP> (&ring)[PD]) {
#pragma unroll
  for (int c = 0; c < PD; ++c) ring[c] = b.load(ct, c0 + c);
}

// The thread index like lane_here: offsets derived from it are computed where
// they are used instead of being hoisted out of the tile loop and spilled.
__device__ __forceinline__ int thread_here() {
  int t = (int)threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

// Runs two independent parts of a step. With SWAP half of the waves (`late`,
// one per SIMD) take them in the other order, so that one part's vector-ALU
// work runs beside the other's LDS reads and MFMAs. It pays with one plane
// (0.73 -> 0.64 ms per 1 M rows); with three, whose LDS traffic is three times
// that, it does not (1.44 against 1.51 ms, both before the separate low sums).
template <bool SWAP, class A, class B>
__device__ __forceinline__ void either_order(bool late, A&& a, B&& b) {
  if (SWAP && late) {
    b();
    a();
  } else {
    a();
    b();
  }
}

template <class SH, int NP, bool SPLIT0>
struct BwdLds {
  static constexpr int TM = NP == 1 ? 64 : 32;
  static constexpr int ldF = SH::FK + 8, ldH = kU + 8, ldD = 40;
  using PF = Planes<NP, TM, ldF>;
  using PX = PlanesT<NP, TM, 16 * SH::maxXT()>;
  using PH = Planes<NP, TM, ldH>;
  using PHT = PlanesT<NP, TM, kU>;
  using PD = Planes<NP, TM, ldD>;
  static constexpr int ldDX = 16 * SH::maxDXT() + 4;   // dX rows (FP32)
  static constexpr int ldP = 33;                  // h0 parts (FP32)
  static constexpr int max2(int a, int b) { return a > b ? a : b; }
  static constexpr int oF = 0;
  static constexpr int oX = oF + PF::bytes;
  static constexpr int oH1 = oX + PX::bytes;      // relu(z1), then dZ1
  static constexpr int oZ2 = oH1 + max2(PH::bytes, PHT::bytes);
  // dX lies over dZ2 (dead after step C)
  static constexpr int oZ3p = oZ2 + max2(TM * ldDX * 4, PH::bytes);  // BF16: dZ3's operand
  static constexpr int oP = oZ3p + (NP == 1 ? PD::bytes : 0);
  static constexpr int p_bytes = ((SPLIT0 ? 2 : 1) * TM * ldP * 4 + 15) / 16 * 16;
  // dH0 over the h0 parts, which a second group's encoding still reads
  static constexpr int oD = oP + (SH::NH == 1 ? 0 : p_bytes);
  static constexpr int oZ3 = max2(oP + p_bytes, oD + PD::bytes);
  static constexpr int oDs = oZ3 + TM * 12;       // dZ3 (FP32, 3 x TM), then the directions
  static constexpr int oCs = oDs + TM * 12;       // cameras
  static constexpr int oE = oCs + TM * 4;         // FiLM: running embedding gradient, 2 ids
  static constexpr int oA0 = oE + kU * 4 + 16;    // dW0's sums
  static constexpr int bytes = oA0 + SH::FT * 2 * 64 * 16;
};

// FILM: cams (per ray; null: camera 0), gembed (ncam x U, added to) and ncam >= 1.
// SPLIT0: layer 0 in two K parts and the doubled frequency from the first by
// the double-angle identities (the training steps); else one K chain and a
// sincosf per frequency.
// KB: the kept activations are BF16 (else FP32).
// flags (three planes): one per workgroup, whether its sums hold NaN.
template <class SH, int NP, bool FILM, bool SPLIT0, bool KB>
__global__ void __launch_bounds__(512) k_mlp_bwd_planes(
    MlpW w, const __bf16* __restrict__ tables, const float* __restrict__ feats,
    const float* __restrict__ dirs, const float* __restrict__ grgb, int64_t M, int64_t rpr,
    float* __restrict__ gfeat, float* __restrict__ partials, GradPack gp,
    const float* __restrict__ act, const float* __restrict__ rgb_in,
    const uint32_t* __restrict__ cams, float* __restrict__ gembed, int ncam,
    int32_t* __restrict__ flags) {
  using L = BwdLds<SH, NP, SPLIT0>;
  using T = BwdTables<SH>;
  static_assert(!KB || NP == 1, "BF16 activations are the BF16 MLP's");
  static_assert(!SPLIT0 || SH::NF == 2, "the double-angle identities reach two frequencies");
  constexpr int TM = L::TM, RT = TM / 16, NT = 512, NW = 8, KR = TM / 32;
  constexpr bool BF = NP == 1;
  // reading operands a step ahead takes registers that three planes lack and
  // brings them nothing: the LDS is their bound (1.59 ms per 1 M rows either
  // way, the wide shape 2.55 without and 2.78 with)
  constexpr bool AHEAD = NP == 1;
  extern __shared__ __attribute__((aligned(16))) char smem_b[];
  const typename L::PF Fp{reinterpret_cast<__bf16*>(smem_b + L::oF)};
  const typename L::PX Xp{reinterpret_cast<__bf16*>(smem_b + L::oX)};
  const typename L::PHT H1t{reinterpret_cast<__bf16*>(smem_b + L::oH1)};  // relu(z1)
  const typename L::PH Z1{reinterpret_cast<__bf16*>(smem_b + L::oH1)};    // dZ1 over it
  const typename L::PH Z2{reinterpret_cast<__bf16*>(smem_b + L::oZ2)};  // dZ2
  const typename L::PD Z3p{reinterpret_cast<__bf16*>(smem_b + L::oZ3p)};  // BF16: dZ3
  const typename L::PD Dp{reinterpret_cast<__bf16*>(smem_b + L::oD)};   // dH0
  float* DX = reinterpret_cast<float*>(smem_b + L::oZ2);
  float* P0 = reinterpret_cast<float*>(smem_b + L::oP);                 // h0 parts
  float* Z3 = reinterpret_cast<float*>(smem_b + L::oZ3);                // [3][TM]
  float* Ds = reinterpret_cast<float*>(smem_b + L::oDs);                // [3][TM]
  int* Cs = reinterpret_cast<int*>(smem_b + L::oCs);
  float* Eacc = reinterpret_cast<float*>(smem_b + L::oE);
  int* Run = reinterpret_cast<int*>(Eacc + kU);
  const TableB<NP, SH::FK / 32> t_f0(tables, T::f0);
  const TableB<NP, 1> t_g0(tables + NP * T::o_g0, T::g0);
  const TableB<NP, kU / 32> t_g1(tables + NP * T::o_g1, T::g1);
  const TableB<NP, kU / 32> t_g2(tables + NP * T::o_g2, T::g2);
  const TableB<NP, 1> t_g3(tables + NP * T::o_g3, T::g3);

  const int wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & (NW - 1));
  const bool late = wave >= NW / 2;
  float* part = partials + (int64_t)blockIdx.x * gp.total;

  // weight-gradient tiles in registers: column tile `wave` of dW2 and dW1, every
  // row tile. Those of dW0 (feature tile ft, wave ft % 8) lie in LDS, a lane's
  // four values in 16 bytes: in registers they were the ones the compiler
  // spilled, and their reload in step F waited for the next tile's loads.
  constexpr int XTN = SH::xt0(SH::NH);
  f32x4 a2[kU / 16], a1[XTN];
  f32x4* A0 = reinterpret_cast<f32x4*>(smem_b + L::oA0);
#pragma unroll
  for (int i = 0; i < kU / 16; ++i) a2[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < XTN; ++i) a1[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float db1 = 0.f, db2 = 0.f, db3 = 0.f, dw3[3] = {0.f, 0.f, 0.f};
  float w3r[3] = {0.f, 0.f, 0.f};
  if constexpr (!BF) {
#pragma unroll
    for (int c = 0; c < 3; ++c) w3r[c] = w.w3[(16 * wave + (lane_id() & 15)) * 3 + c];
  }

  // zero padding that no tile overwrites: everything once
  const int tid = threadIdx.x;
  for (int e = tid; e < L::oP / 16; e += NT)
    *reinterpret_cast<uint4*>(smem_b + 16 * e) = make_uint4(0, 0, 0, 0);
  for (int e = tid; e < SH::FT * 2 * 64; e += NT) A0[e] = f32x4{0.f, 0.f, 0.f, 0.f};
  if constexpr (FILM) {
    for (int c = tid; c < kU; c += NT) Eacc[c] = 0.0f;
    if (tid == 0) Run[1] = -1;
  }

  // ---- the next tile's inputs in registers -------------------------------------
  typedef int i32x4 __attribute__((ext_vector_type(4)));
  constexpr int F4 = SH::F / 4, nF = (TM * F4 + NT - 1) / NT;
  static_assert(SH::F % 4 == 0 && kKeptGroup == 32, "whole loads");
  constexpr int nA = KB ? 1 : 2;  // 16-byte loads of the lane's 8 values of a group
  i32x4 vf[nF], va[KR][nA], vb[KR][nA];
  float vs = 0.f, vg = 0.f, vd = 0.f;
  int vcam = 0;
  // ray of the next tile to issue, advanced by a grid of tiles at a time
  const unsigned rp = (unsigned)rpr;
  const int64_t step_rows = (int64_t)gridDim.x * TM, first = (int64_t)blockIdx.x * TM;
  const int64_t step_rays = step_rows / rpr;
  const unsigned step_rem = (unsigned)(step_rows - step_rays * rpr);
  int64_t ray0 = first / rpr;
  unsigned rem0 = (unsigned)(first - ray0 * rpr);
  auto issue = [&](int64_t row0) TFH_INLINE {
    const int t = thread_here();
    const int nv = (int)max((int64_t)0, min((int64_t)TM, M - row0));
    // rays of the tile: rows [row0, row0 + nv) start rem0 rows into ray0
    const bool one = rp >= (unsigned)TM;  // at most two rays: no division
    const unsigned last = rem0 + (unsigned)(nv > 0 ? nv - 1 : 0);
    const int nray = nv > 0 ? (int)(one ? (last >= rp ? 1u : 0u) : last / rp) + 1 : 0;
    const float* fbase = feats + row0 * SH::F;
    asm volatile("" : "+s"(fbase));
    const auto rf = buffer_rsrc(fbase, nv * SH::F * 4);
    const auto ra = buffer_rsrc(
        reinterpret_cast<const char*>(act) + row0 / kKeptGroup * kKeptGroupBytes<KB>,
        (nv + kKeptGroup - 1) / kKeptGroup * kKeptGroupBytes<KB>);
    const auto rs = buffer_rsrc(rgb_in + row0 * 3, nv * 12);
    const auto rg = buffer_rsrc(grgb + row0 * 3, nv * 12);
    const auto rd = buffer_rsrc(dirs + ray0 * 3, nray * 12);
#pragma unroll
    for (int k = 0; k < nF; ++k) {
      const int e = t + k * NT;
      vf[k] = __builtin_amdgcn_raw_buffer_load_b128(rf, e < TM * F4 ? e * 16 : kOOB, 0, 0);
    }
#pragma unroll
    for (int k = 0; k < KR; ++k)
#pragma unroll
      for (int h = 0; h < nA; ++h) {
        const int off = t * 16 * nA + h * 16;  // (wave, lane) in order
        va[k][h] = __builtin_amdgcn_raw_buffer_load_b128(ra, off, k * kKeptGroupBytes<KB>, 0);
        vb[k][h] = __builtin_amdgcn_raw_buffer_load_b128(
            ra, off, k * kKeptGroupBytes<KB> + kKeptGroupBytes<KB> / 2, 0);
      }
    const int i3 = t / 3, c3 = t - 3 * i3;
    const bool own3 = t < TM * 3;
    vs = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, own3 ? t * 4 : kOOB, 0, 0));
    vg = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rg, own3 ? t * 4 : kOOB, 0, 0));
    const unsigned at3 = rem0 + (unsigned)i3;
    const unsigned rel = one ? (at3 >= rp ? 1u : 0u) : at3 / rp;
    vd = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
        rd, (own3 && i3 < nv) ? (int)(rel * 3 + c3) * 4 : kOOB, 0, 0));
    if constexpr (FILM) {
      const auto rc = buffer_rsrc(cams ? static_cast<const void*>(cams + ray0) : dirs,
                                  cams ? nray * 4 : 0);
      const unsigned atc = rem0 + (unsigned)t;
      const unsigned relc = one ? (atc >= rp ? 1u : 0u) : atc / rp;
      vcam = (int)__builtin_amdgcn_raw_buffer_load_b32(rc, t < nv ? (int)relc * 4 : kOOB, 0, 0);
    }
    // the loads stay here, ahead of their use
    asm volatile("" ::: "memory");
    // to the next tile of this workgroup
    ray0 += step_rays;
    rem0 += step_rem;
    if (rem0 >= rp) {
      rem0 -= rp;
      ++ray0;
    }
  };

  // layer 0's items: (K part, column tile, row tile), the first one's B chunks
  // (ringf) requested behind the tile's own loads
  constexpr int KC0 = SH::FK / 32, KA = SPLIT0 ? (KC0 + 1) / 2 : KC0, KR0 = KC0 - KA;
  constexpr int PARTS = SPLIT0 ? 2 : 1, NI0 = 2 * RT * PARTS;
  constexpr int PD0 = NP == 3 || KR0 == 1 ? 1 : 2;
  Frag<NP> ringf[PD0];
  auto issue_f0 = [&]() TFH_INLINE {
    strip_pre<NP>(t_f0, (wave / PARTS) & 1, (SPLIT0 && (wave & 1)) ? KA : 0, ringf);
  };

  const int64_t ntiles = (M + TM - 1) / TM;
  issue((int64_t)blockIdx.x * TM);
  issue_f0();
  for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int64_t row0 = tile * TM;
    __syncthreads();
    // ---- commit ----
    unsigned pos1 = 0;  // bit q: the lane's relu(z1) value q is positive
    {
      const int t = thread_here();
#pragma unroll
      for (int k = 0; k < nF; ++k) {
        const int e = t + k * NT, i = e / F4, c4 = e - i * F4;
        if (e < TM * F4) {
          const float4 v = __builtin_bit_cast(float4, vf[k]);
          const float f[4] = {v.x, v.y, v.z, v.w};
          Fp.put4(i, 4 * c4, f);
        }
      }
      const int kq4 = (t >> 4) & 3, ucol = 16 * wave + (t & 15);
#pragma unroll
      for (int k = 0; k < KR; ++k) {
        Frag<NP> f;
        if constexpr (KB) {
          f.p[0] = __builtin_bit_cast(bf16x8, va[k][0]);
#pragma unroll
          for (int e = 0; e < 8; ++e)
            pos1 |= (float)f.p[0][e] > 0.0f ? 1u << (8 * k + e) : 0u;
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float h = __uint_as_float((unsigned)va[k][KB ? 0 : e / 4][e % 4]);
            set_frag<NP>(f, e, h);
            pos1 |= h > 0.0f ? 1u << (8 * k + e) : 0u;
          }
        }
        H1t.put_frag(ucol, k, kq4, f);
      }
      if (t < TM * 3) {
        const int i3 = t / 3, c3 = t - 3 * i3;
        Ds[c3 * TM + i3] = vd;
        const float z = vg * vs * (1.0f - vs);
        Z3[c3 * TM + i3] = z;
        db3 += z;
        if constexpr (BF) Z3p.m[i3 * L::ldD + c3] = (__bf16)z;
      }
      if constexpr (FILM) {
        if (t < TM) Cs[t] = (vcam < 0 || vcam >= ncam) ? 0 : vcam;
      }
    }
    // dZ2's B chunk
    Frag<NP> ring3[1];
    if constexpr (BF) strip_pre<NP>(t_g3, wave, 0, ring3);
    __syncthreads();
    if constexpr (FILM) {
      // wave 0 hands the running embedding gradient over when the camera changes
      const int lane = lane_here();
      const int nvalid = (int)min((int64_t)TM, M - row0);
      const int c0 = Cs[0];
      const int tc = __all(lane >= nvalid || Cs[lane < TM ? lane : 0] == c0) ? c0 : -1;
      if (wave == 0) {
        const int rc = Run[1];
        if (tc >= 0 && rc >= 0 && rc != tc) {
          for (int c = lane; c < kU; c += 64) {
            unsafeAtomicAdd(gembed + (size_t)rc * kU + c, Eacc[c]);
            Eacc[c] = 0.0f;
          }
        }
        if (lane == 0) {
          Run[0] = tc;
          if (tc >= 0) Run[1] = tc;
        }
      }
      __syncthreads();
    }
    // dZ1's first B chunks
    constexpr int PD2 = NP == 1 ? 4 : (SH::NH == 1 ? 2 : 1);
    Frag<NP> ring2[PD2];
    strip_pre<NP>(t_g2, wave, 0, ring2);
    // ---- B: layer 0 -> P0 ----
    auto layer0 = [&]() TFH_INLINE {
      for (int it = wave; it < NI0; it += NW) {
        const int kp = SPLIT0 ? it & 1 : 0, ct = (it / PARTS) & 1, rt = it / (2 * PARTS);
        f32x4 acc[1];
        zero_acc(acc);
        if (it != wave) strip_pre<NP>(t_f0, ct, kp ? KA : 0, ringf);
        if (kp == 0)
          strip<NP, AHEAD, 1, KA, PD0>(Fp, 16 * rt, 0, t_f0, ct, acc, ringf);
        else
          strip<NP, AHEAD, 1, (KR0 > 0 ? KR0 : 1), PD0>(Fp, 16 * rt, KA, t_f0, ct, acc, ringf);
        const int ln = lane_here(), r16 = ln & 15, kq4 = ln >> 4;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          P0[(kp * TM + 16 * rt + 4 * kq4 + e) * L::ldP + 16 * ct + r16] = acc[0][e];
      }
    };
    // ---- B: dZ2 = (dZ3 W3^T) [z2 > 0] -> Z2 ; db2 ; dW3 ; dW2 += H1^T dZ2 ----
    auto layer3 = [&]() TFH_INLINE {
      Frag<NP> y[KR];
      f32x4 acc[RT];
      zero_acc(acc);
      if constexpr (BF) strip<NP, AHEAD, RT, 1, 1>(Z3p, 0, 0, t_g3, wave, acc, ring3);
      const int lane = lane_here(), r16 = lane & 15, kq4 = lane >> 4, ucol = 16 * wave + r16;
      const bool film = FILM && 16 * wave >= kU / 2;  // wave-uniform
      int tcam = -1;
      float esc = 1.0f, esh = 0.0f, sh = 0.0f, sg = 0.0f;
      if constexpr (FILM) {
        tcam = Run[0];
        if (film && tcam >= 0) {
          esc = w.embed[(size_t)tcam * kU + ucol - kU / 2];
          esh = w.embed[(size_t)tcam * kU + ucol];
        }
      }
      // dL/dh2 (rt, e) and relu(z2) of the lane
      const auto grad_of = [&](int rt, int e, const float (&z)[3][4]) TFH_INLINE {
        if constexpr (BF)
          return acc[rt][e];
        else
          return z[0][e] * w3r[0] + z[1][e] * w3r[1] + z[2][e] * w3r[2];
      };
      const auto kept_of = [&](int rt, int e) TFH_INLINE {
        if constexpr (KB)
          return (float)__builtin_bit_cast(bf16x8, vb[rt / 2][0])[4 * (rt & 1) + e];
        else
          return __uint_as_float((unsigned)vb[rt / 2][KB ? 0 : rt & 1][e]);
      };
      const auto load_z = [&](int rt, float (&z)[3][4]) TFH_INLINE {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const float4 v = *reinterpret_cast<const float4*>(Z3 + c * TM + 16 * rt + 4 * kq4);
          z[c][0] = v.x; z[c][1] = v.y; z[c][2] = v.z; z[c][3] = v.w;
        }
      };
      if constexpr (FILM) {
        if (film && tcam < 0) {
          // A tile of several cameras: a lane sums its runs of rows of one camera,
          // and lanes whose last runs are of one camera add once. With an add per
          // row, 64-row tiles of 96 samples a ray took 4.8 ns a row (BF16, 5 cameras;
          // now 0.87).
#pragma unroll
          for (int rt = 0; rt < RT; ++rt) {
            int rcam = -1;
            float rsh = 0.0f, rsg = 0.0f;
            const auto end_run = [&]() TFH_INLINE {
              if (rcam >= 0) {
                float* gemb = gembed + (size_t)rcam * kU;
                unsafeAtomicAdd(gemb + ucol - kU / 2, rsh);
                unsafeAtomicAdd(gemb + ucol, rsg);
              }
              rsh = rsg = 0.0f;
            };
            float z[3][4];
            if constexpr (!BF) load_z(rt, z);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int row = 16 * rt + 4 * kq4 + e;
              if (row0 + row < M) {
                const int cam = Cs[row];
                if (cam != rcam) end_run();
                rcam = cam;
                const float g = grad_of(rt, e, z);
                rsh += g * kept_of(rt, e);
                rsg += g;
              }
            }
#pragma unroll
            for (int o = 16; o <= 32; o <<= 1) {
              const int pc = __shfl_xor(rcam, o, 64);
              const float ph = __shfl_xor(rsh, o, 64), pg = __shfl_xor(rsg, o, 64);
              if (pc == rcam) {
                rsh = lane & o ? 0.0f : rsh + ph;
                rsg = lane & o ? 0.0f : rsg + pg;
                if (lane & o) rcam = -1;
              }
            }
            end_run();
          }
        }
      }
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        float z[3][4];
        load_z(rt, z);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int row = 16 * rt + 4 * kq4 + e;
          float g = grad_of(rt, e, z);
          const float hp = kept_of(rt, e);
          float hf = hp;  // the layer-3 input
          if constexpr (FILM) {
            if (film) {
              if (tcam >= 0) {
                if (row0 + row < M) {
                  sh += g * hp;
                  sg += g;
                }
                hf = esc * hp + esh;
                g = g * esc;
              } else {
                const float* emb = w.embed + (size_t)Cs[row] * kU;
                hf = emb[ucol - kU / 2] * hp + emb[ucol];
                g = g * emb[ucol - kU / 2];
              }
            }
          }
          if constexpr (BF) hf = (float)(__bf16)hf;  // the operands' BF16 rounding
#pragma unroll
          for (int c = 0; c < 3; ++c)
            dw3[c] += hf * (BF ? (float)(__bf16)z[c][e] : z[c][e]);
          const float dz = hp > 0.0f ? g : 0.0f;
          db2 += dz;
          Frag<NP>& f = y[rt / 2];
          const int at = 4 * (rt & 1) + e;
          set_frag<NP>(f, at, dz);
#pragma unroll
          for (int p = 0; p < NP; ++p) Z2.m[p * L::PH::ps + row * L::ldH + ucol] = f.p[p][at];
        }
      }
      if constexpr (FILM) {
        if (film && tcam >= 0) {
          sh += __shfl_xor(sh, 16, 64);
          sh += __shfl_xor(sh, 32, 64);
          sg += __shfl_xor(sg, 16, 64);
          sg += __shfl_xor(sg, 32, 64);
          if (lane < 16) {  // the wave covers every row of the column: plain adds
            Eacc[ucol - kU / 2] += sh;
            Eacc[ucol] += sg;
          }
        }
      }
#pragma unroll
      for (int k = 0; k < KR; ++k)
        wgrad<NP, AHEAD, kU / 16, 0>(H1t, k, y[k], a2);
    };
    either_order<BF>(late, layer0, layer3);
    __syncthreads();
    // ---- C: encoding of a group -> X ----
    // slots (value u, row i) of 512 threads, the same in the encoding and in
    // step E, which finds the sines and cosines in registers (of the first
    // frequency alone where the second is derived)
    constexpr int nI = TM * ((SH::HF + (SH::NH == 1 ? 3 : 2) + 7) / 8 * 8) / NT;
    constexpr int JN = nI * NT / TM, NK = SPLIT0 ? 2 : SH::FEW;
    static_assert(JN >= SH::values(0) && JN >= SH::values(SH::NH - 1), "a slot per value");
    float sc[nI][NK];
    auto encode = [&](auto hc) TFH_INLINE {
      constexpr int h = decltype(hc)::value, n = SH::count(h);
#pragma unroll
      for (int m = 0; m < nI; ++m) {
        const int e = thread_here() + m * NT, i = e % TM, u = e / TM, pos = row_pos(i);
        float v = 0.f;
        if (u < n) {
          v = P0[i * L::ldP + SH::first(h) + u];
          if constexpr (SPLIT0) v += P0[(TM + i) * L::ldP + SH::first(h) + u];
        } else if (u < SH::values(h)) {
          v = Ds[(u - n) * TM + i];
        }
        float fe[SH::FEW];
        sincosf(v, &fe[0], &fe[SH::NF]);
        sc[m][0] = fe[0];
        sc[m][NK / 2] = fe[SH::NF];
#pragma unroll
        for (int q = 1; q < SH::NF; ++q) {
          if constexpr (SPLIT0) {
            fe[1] = 2.0f * fe[0] * fe[2];
            fe[3] = (fe[2] - fe[0]) * (fe[2] + fe[0]);
          } else {
            sincosf(v * (float)(1 << q), &fe[q], &fe[SH::NF + q]);
            sc[m][q] = fe[q];
            sc[m][SH::NF + q] = fe[SH::NF + q];
          }
        }
        if (u < SH::values(h)) {
          const int fc = u < n ? SH::FEW * u : n * (SH::FEW + 1) + SH::FEW * (u - n);
#pragma unroll
          for (int q = 0; q < SH::FEW; ++q) Xp.put(pos, fc + q, fe[q]);
          Xp.put(pos, u < n ? n * SH::FEW + u : n * (SH::FEW + 1) + 3 * SH::FEW + (u - n), v);
        }
      }
    };
    // ---- C: dZ1 = (dZ2 W2^T) [z1 > 0] over relu(z1) ; db1 ----
    Frag<NP> y1[KR];
    auto layer2 = [&]() TFH_INLINE {
      f32x4 acc[RT];
      zero_acc(acc);
      strip<NP, AHEAD, RT, 4, PD2>(Z2, 0, 0, t_g2, wave, acc, ring2);
      const int lane = lane_here(), kq4 = lane >> 4, ucol = 16 * wave + (lane & 15);
#pragma unroll
      for (int q = 0; q < 4 * RT; ++q) {
        const int rt = q / 4, e = q % 4;
        const int row = 16 * rt + 4 * kq4 + e;
        const float dz = (pos1 >> q) & 1 ? acc[rt][e] : 0.0f;
        db1 += dz;
        Frag<NP>& f = y1[rt / 2];
        const int at = 4 * (rt & 1) + e;
        set_frag<NP>(f, at, dz);
#pragma unroll
        for (int p = 0; p < NP; ++p) Z1.m[p * L::PH::ps + row * L::ldH + ucol] = f.p[p][at];
      }
    };
    either_order<BF>(late, [&]() TFH_INLINE { encode(std::integral_constant<int, 0>{}); }, layer2);
    // ---- D: dW1 += X^T dZ1 ; dX = dZ1 W1^T (group h; its first B chunks in ring2) ----
    auto layer1 = [&](auto hc) TFH_INLINE {
      constexpr int h = decltype(hc)::value, ct0 = SH::dxt0(h);
#pragma unroll
      for (int k = 0; k < KR; ++k) wgrad<NP, AHEAD, SH::XT(h), SH::xt0(h)>(Xp, k, y1[k], a1);
      // the column tiles past the last whole round go one row tile to a wave
      constexpr int DXF = SH::DXT(h) / NW, DXR = SH::DXT(h) % NW;
#pragma unroll 1
      for (int i = 0; i < DXF; ++i) {
        const int ct = wave + NW * i;
        if (i > 0) strip_pre<NP>(t_g1, ct0 + ct, 0, ring2);
        f32x4 acc[RT];
        zero_acc(acc);
        strip<NP, AHEAD, RT, 4, PD2>(Z1, 0, 0, t_g1, ct0 + ct, acc, ring2);
        const int lane = lane_here(), r16 = lane & 15, kq4 = lane >> 4;
#pragma unroll
        for (int q = 0; q < 4 * RT; ++q)
          DX[(16 * (q / 4) + 4 * kq4 + q % 4) * L::ldDX + 16 * ct + r16] = acc[q / 4][q % 4];
      }
#pragma unroll 1
      for (int it = wave; it < DXR * RT; it += NW) {
        const int ct = NW * DXF + it / RT, rt = it % RT;
        strip_pre<NP>(t_g1, ct0 + ct, 0, ring2);
        f32x4 acc[1];
        zero_acc(acc);
        strip<NP, AHEAD, 1, 4, PD2>(Z1, 16 * rt, 0, t_g1, ct0 + ct, acc, ring2);
        const int lane = lane_here(), r16 = lane & 15, kq4 = lane >> 4;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          DX[(16 * rt + 4 * kq4 + e) * L::ldDX + 16 * ct + r16] = acc[0][e];
      }
    };
    // ---- E: dH0[j] = dX[h_j] + sum_q 2^q (dX[sin_q] cos(2^q h) - dX[cos_q] sin(2^q h)) ----
    auto squash = [&](auto hc) TFH_INLINE {
      constexpr int h = decltype(hc)::value, n = SH::count(h);
#pragma unroll
      for (int m = 0; m < nI; ++m) {
        const int e = thread_here() + m * NT, i = e % TM, j = e / TM;
        if (j < n) {
          const float* dx = DX + i * L::ldDX;
          float d[SH::FEW];
#pragma unroll
          for (int q = 0; q < SH::FEW; q += 4) {
            const float4 v = *reinterpret_cast<const float4*>(dx + SH::FEW * j + q);
            d[q] = v.x; d[q + 1] = v.y; d[q + 2] = v.z; d[q + 3] = v.w;
          }
          float g = dx[n * SH::FEW + j];
#pragma unroll
          for (int q = 0; q < SH::NF; ++q) {
            float sq, cq;
            if constexpr (SPLIT0) {
              const float s0 = sc[m][0], c0 = sc[m][1];
              sq = q == 0 ? s0 : 2.0f * s0 * c0;
              cq = q == 0 ? c0 : (c0 - s0) * (c0 + s0);
            } else {
              sq = sc[m][q];
              cq = sc[m][SH::NF + q];
            }
            const float s = (float)(1 << q);
            g += d[q] * s * cq;
            g -= d[SH::NF + q] * s * sq;
          }
          Dp.put(i, SH::first(h) + j, g);
        } else if (h == SH::NH - 1) {  // the zero padding to 32 columns
          for (int c = SH::S + (j - n); c < 32; c += JN - n) Dp.put(i, c, 0.0f);
        }
      }
    };
    strip_pre<NP>(t_g1, wave, 0, ring2);
    __syncthreads();
    layer1(std::integral_constant<int, 0>{});
    if constexpr (SH::NH == 2) {
      strip_pre<NP>(t_g1, SH::dxt0(1) + wave, 0, ring2);
      __syncthreads();
      squash(std::integral_constant<int, 0>{});
      encode(std::integral_constant<int, 1>{});
      __syncthreads();
      layer1(std::integral_constant<int, 1>{});
    }
    // dF's B chunks: column tile wave for every row tile, then one (column
    // tile, row tile) of those past the first 8, counted down from the last
    // wave (the first waves hold the extra dW0 tiles)
    constexpr int DFX = SH::FT > NW ? (SH::FT - NW) * RT : 0;
    static_assert(DFX <= NW, "one extra dF item per wave");
    const int xdf = NW - 1 - wave;
    Frag<NP> ringg[2];
    if (wave < SH::FT) ringg[0] = t_g0.load(wave, 0);
    if (xdf < DFX) ringg[1] = t_g0.load(NW + xdf / RT, 0);
    __syncthreads();
    // the next tile's loads: steps E and F wait for nothing behind them
    either_order<BF>(late, [&]() TFH_INLINE { issue(row0 + (int64_t)gridDim.x * TM); },
                     [&]() TFH_INLINE { squash(std::integral_constant<int, SH::NH - 1>{}); });
    __syncthreads();
    // ---- F: dF = dH0 W0^T ; dW0 += F^T dH0 ----
    if (gfeat) {
      // a buffer over the tile's valid rows drops the others
      const auto rgf = buffer_rsrc(gfeat + row0 * SH::F,
                                   (int)min((int64_t)TM, M - row0) * SH::F * 4);
      auto store = [&](const f32x4& v, int ct, int rt) TFH_INLINE {
        const int ln = lane_here(), kq4 = ln >> 4, col = 16 * ct + (ln & 15);
        const int off = ((16 * rt + 4 * kq4) * SH::F + col) * 4;
        if (SH::F % 16 == 0 || col < SH::F) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v[e]), rgf,
                                                  off + e * SH::F * 4, 0, 0);
        }
      };
      if (wave < SH::FT) {
        const int ln = lane_here();
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          f32x4 acc{0.f, 0.f, 0.f, 0.f};
          mma_add<NP>(acc, Dp.row8(16 * rt + (ln & 15), 8 * (ln >> 4)), ringg[0]);
          store(acc, wave, rt);
        }
      }
      if (xdf < DFX) {
        const int ln = lane_here(), rt = xdf % RT;
        f32x4 acc{0.f, 0.f, 0.f, 0.f};
        mma_add<NP>(acc, Dp.row8(16 * rt + (ln & 15), 8 * (ln >> 4)), ringg[1]);
        store(acc, NW + xdf / RT, rt);
      }
    }
    for (int ft = wave; ft < SH::FT; ft += NW) {
      const int ln = lane_here();
      f32x4* slot = A0 + ft * 2 * 64 + ln;
      f32x4 acc[2] = {slot[0], slot[64]};
#pragma unroll
      for (int k = 0; k < KR; ++k) {
        const Frag<NP> x = Fp.over_rows(16 * ft, k, ln);
#pragma unroll
        for (int j = 0; j < 2; ++j) mma_add<NP>(acc[j], x, Dp.over_rows(16 * j, k, ln));
      }
      slot[0] = acc[0];
      slot[64] = acc[1];
    }
    issue_f0();
  }

  // ---- the workgroup's sums -> its partial ----
  const int t = threadIdx.x, lane = lane_id(), r16 = lane & 15, kq4 = lane >> 4;
  const int ucol = 16 * wave + r16;
  __syncthreads();
  if constexpr (FILM) {
    const int rc = Run[1];
    if (rc >= 0)
      for (int c = t; c < kU; c += NT) unsafeAtomicAdd(gembed + (size_t)rc * kU + c, Eacc[c]);
  }
#pragma unroll
  for (int o = 16; o <= 32; o <<= 1) {
    db1 += __shfl_xor(db1, o, 64);
    db2 += __shfl_xor(db2, o, 64);
#pragma unroll
    for (int c = 0; c < 3; ++c) dw3[c] += __shfl_xor(dw3[c], o, 64);
  }
  if (lane < 16) {
    part[gp.b1 + ucol] = db1;
    part[gp.b2 + ucol] = db2;
#pragma unroll
    for (int c = 0; c < 3; ++c) part[gp.w3 + ucol * 3 + c] = dw3[c];
  }
  if (t < 3 * TM) Z3[t] = db3;  // thread t: colour t % 3
  int* Bad = Cs;
  if (t == 0) Bad[0] = 0;
  __syncthreads();
  bool nan = false;
  const auto put = [&](int64_t at, float v) TFH_INLINE {
    part[at] = v;
    nan |= v != v;
  };
  if (t < 3) {
    float s = 0.0f;
    for (int i = 0; i < TM; ++i) s += Z3[3 * i + t];
    part[gp.b3 + t] = s;
  }
#pragma unroll
  for (int i = 0; i < kU / 16; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      put(gp.w2 + (16 * i + 4 * kq4 + e) * kU + ucol, a2[i][e]);
#pragma unroll
  for (int i = 0; i < XTN; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int h = SH::NH > 1 && i >= SH::xt0(SH::NH - 1) ? SH::NH - 1 : 0;
      const int o = SH::x_orig(h, 16 * (i - SH::xt0(h)) + 4 * kq4 + e);
      if (o >= 0) put(gp.w1 + o * kU + ucol, a1[i][e]);
    }
  for (int ft = wave; ft < SH::FT; ft += NW)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const f32x4 v = A0[(ft * 2 + j) * 64 + lane];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int f = 16 * ft + 4 * kq4 + e, scol = 16 * j + r16;
        if (f < SH::F && scol < SH::S) put(gp.w0 + f * SH::S + scol, v[e]);
      }
    }
  if constexpr (NP == 3) {
    if (nan) Bad[0] = 1;
    __syncthreads();
    if (t == 0) flags[blockIdx.x] = Bad[0];
  }
}

template <class SH, int NP, bool FILM, bool SPLIT0, bool KB>
int32_t run_planes(const MlpW& w, const BwdPlanesArgs& a, hipStream_t st) {
  using L = BwdLds<SH, NP, SPLIT0>;
  static_assert(L::bytes <= 160 * 1024, "the tile fits the LDS of a CU");
  auto kernel = k_mlp_bwd_planes<SH, NP, FILM, SPLIT0, KB>;
  allow_lds(kernel, L::bytes);
  static_assert(L::TM == (NP == 1 ? kBwdRowsBf16 : kBwdRowsFp32), "bwd_planes_blocks");
  hipLaunchKernelGGL(kernel, dim3((unsigned)bwd_planes_blocks(NP == 1, a.M, a.max_blocks)), dim3(512), L::bytes, st, w,
                     static_cast<const __bf16*>(a.tables), a.feats, a.dirs, a.grgb, a.M, a.rpr,
                     a.gfeat, a.partials, a.gp, a.act, a.rgb, a.cams, a.gembed, a.ncam, a.flags);
  return check_launch("mlp bwd");
}

template <class SH>
int32_t pack_planes(bool bf, const MlpW& w, void* tables, int32_t* flags, hipStream_t st) {
  const dim3 grid(BwdTables<SH>::total / kPackThreads);
  if (bf)
    hipLaunchKernelGGL((k_pack_bwd<SH, 1>), grid, dim3(kPackThreads), 0, st, w,
                       static_cast<__bf16*>(tables), flags);
  else
    hipLaunchKernelGGL((k_pack_bwd<SH, 3>), grid, dim3(kPackThreads), 0, st, w,
                       static_cast<__bf16*>(tables), flags);
  return check_launch("mlp bwd: operand tables");
}

}  // namespace tfh
