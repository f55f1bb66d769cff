// MFMA tile helpers shared by the MLP kernels (gfx950, wave64).
//
// D layout of a 16x16 tile: lane l, element r -> row 4*(l/16)+r, col l%16.
// FP32 (K=4):  A[l%16][k0 + l/16],        B[k0 + l/16][l%16]
// BF16 (K=32): A[l%16][k0 + 8(l/16) + e], B[k0 + 8(l/16) + e][l%16], e < 8
#pragma once

#include <type_traits>

#include "tfh_common.h"

// for lambdas: one that is not inlined passes its captured arrays through scratch
#define TFH_INLINE __attribute__((always_inline))

namespace tfh {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));


// The lane index behind an empty volatile asm: each call computes it afresh,
// so operand addresses derived from it are computed where a tile product
// runs. With the plain index, loop-invariant code motion hoists every
// product's addresses out of a persistent kernel's tile loop, where a kernel
// at its register limit spills them and reloads each one (a scratch round
// trip) in front of its MFMA.
__device__ __forceinline__ int lane_here() {
  int l = (int)(threadIdx.x & 63);
  asm volatile("" : "+v"(l));
  return l;
}

template <int NR>
__device__ __forceinline__ void zero_acc(f32x4 (&acc)[NR]) {
#pragma unroll
  for (int i = 0; i < NR; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
}

__device__ __forceinline__ bf16x8 to_bf16x8(const float4& lo, const float4& hi) {
  bf16x8 v;
  v[0] = (__bf16)lo.x; v[1] = (__bf16)lo.y; v[2] = (__bf16)lo.z; v[3] = (__bf16)lo.w;
  v[4] = (__bf16)hi.x; v[5] = (__bf16)hi.y; v[6] = (__bf16)hi.z; v[7] = (__bf16)hi.w;
  return v;
}

// Raw buffer resource over `bytes` bytes at `base`: loads take a 32-bit VGPR
// byte offset (no per-load 64-bit scalar address) and read 0 past the end.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_rsrc(const void* base, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, bytes, 0x00020000);
}
constexpr int kOOB = 0x7ffffff0;  // a byte offset past every buffer: loads return 0

// A table of B operands in the order the strips read it: one block of 1 KB per
// column tile of 16 and chunk of KC = 16 (FP32) or 32 (BF16) inputs, in it a
// lane's 16 bytes at 16 * lane: lane (r, kq) = r + 16 kq holds column r's
// inputs kq * KC / 4 .. + KC / 4 - 1 of the chunk. A load of a wave is one
// contiguous KB; from a row-major table it was 16 rows' 64-byte pieces, and the
// forward (which reads its 80 or 160 KB of tables once per 32 rows) took 2218
// us instead of 2055 for 2.1 M rows in FP32, 2329 instead of 2040 for 4.2 M in
// BF16, 2205 instead of 1740 for 4.1 M rendered ones.
template <typename T>
struct Table {
  static constexpr int kChunk = sizeof(T) == 2 ? 32 : 16;
  __amdgpu_buffer_rsrc_t r;
  int chunks;  // per column tile
  __device__ __forceinline__ Table(const T* t, int K, int cols)
      : r(buffer_rsrc(t, K * cols * (int)sizeof(T))), chunks(K / kChunk) {}
  // lane16: 16 * lane; the block's offset is the same in every lane
  __device__ __forceinline__ auto load(int chunk, int tile, int lane16) const {
    using V = typename std::conditional<sizeof(T) == 2, bf16x8, float4>::type;
    typedef int i32x4 __attribute__((ext_vector_type(4)));
    const i32x4 v =
        __builtin_amdgcn_raw_buffer_load_b128(r, lane16, (tile * chunks + chunk) * 1024, 0);
    return __builtin_bit_cast(V, v);
  }
};
// The (input, column) of entry e of such a table.
template <typename T>
__device__ __forceinline__ void table_entry(int64_t e, int K, int& k, int& col) {
  constexpr int KC = Table<T>::kChunk, n = KC / 4;
  const int block = (int)(e / (16 * KC)), lane = (int)(e % (16 * KC)) / n, chunks = K / KC;
  col = block / chunks * 16 + (lane & 15);
  k = block % chunks * KC + (lane >> 4) * n + (int)(e % n);
}
using PackedB = Table<__bf16>;
using PackedB32 = Table<float>;

// FP32 strip with a permuted K order: within each chunk of 16, MFMA c (c < 4)
// sums k = 16i + 4*kq + c over the four lane groups kq, so that a lane's four
// A operands (row r, k = 16i + 4kq .. +3) are one 16-byte LDS read and its
// four B operands one 16-byte buffer load. The sum over k is unchanged; only
// the order of the FP32 accumulation differs from a k-ascending chain.
// Requires K % 16 == 0, lda % 4 == 0 and a 16-byte aligned A.
template <int NR, int KMAX>
__device__ __forceinline__ void mma_strip(const float* __restrict__ A, int lda, int K,
                                          PackedB32 b, int col0, f32x4 (&acc)[NR]) {
  const int lane = lane_here();
  const int r = lane & 15, kq = lane >> 4;
  const int ct = __builtin_amdgcn_readfirstlane(col0) >> 4;
  constexpr int NS = KMAX / 16;
  for (int kc = 0; kc < K; kc += KMAX) {  // one pass for K <= KMAX
    // B chunks stream through a ring PD deep: chunk i + PD is requested
    // before chunk i is multiplied, so PD L2 round trips overlap the products.
    // The scheduling barriers pin that order; left to itself the scheduler
    // sinks each load next to its use under register pressure (one round trip
    // per chunk), and hoisting all NS loads costs NS * 4 registers.
    constexpr int PD = NS < 4 ? NS : 4;
    float4 bb[NS];
#pragma unroll
    for (int i = 0; i < PD; ++i)
      if (kc + 16 * i < K) bb[i] = b.load(kc / 16 + i, ct, 16 * lane);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      if (i + PD < NS && kc + 16 * (i + PD) < K) bb[i + PD] = b.load(kc / 16 + i + PD, ct, 16 * lane);
      if (kc + 16 * i < K) {
#pragma unroll
        for (int rt = 0; rt < NR; ++rt) {
          const float4 a = *reinterpret_cast<const float4*>(A + (16 * rt + r) * lda + kc +
                                                            16 * i + 4 * kq);
          acc[rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, bb[i].x, acc[rt], 0, 0, 0);
          acc[rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, bb[i].y, acc[rt], 0, 0, 0);
          acc[rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, bb[i].z, acc[rt], 0, 0, 0);
          acc[rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, bb[i].w, acc[rt], 0, 0, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// A lane's 8 A operands of a BF16 strip: FP32 rows rounded per use, or rows
// kept in BF16 (one 16-byte read).
__device__ __forceinline__ bf16x8 strip_a8(const float* ap) {
  return to_bf16x8(*reinterpret_cast<const float4*>(ap), *reinterpret_cast<const float4*>(ap + 4));
}
__device__ __forceinline__ bf16x8 strip_a8(const __bf16* ap) {
  return *reinterpret_cast<const bf16x8*>(ap);
}

// BF16 strip (AT: float, or __bf16 with lda in BF16 values and 16-byte aligned
// rows). Its whole column of B is loaded before the first product.
template <int NR, int KMAX, class AT>
__device__ __forceinline__ void mma_strip_b16(const AT* __restrict__ A, int lda, int K, PackedB b,
                                              int col0, f32x4 (&acc)[NR]) {
  const int lane = lane_here();
  const int r = lane & 15, kq = lane >> 4;
  const int ct = __builtin_amdgcn_readfirstlane(col0) >> 4;
  constexpr int NS = (KMAX + 31) / 32;
  for (int kc = 0; kc < K; kc += 32 * NS) {  // one pass for K <= KMAX
    bf16x8 bb[NS];
#pragma unroll
    for (int i = 0; i < NS; ++i)
      if (kc + 32 * i < K) bb[i] = b.load(kc / 32 + i, ct, 16 * lane);
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      if (kc + 32 * i < K) {
#pragma unroll
        for (int rt = 0; rt < NR; ++rt) {
          const bf16x8 av = strip_a8(A + (16 * rt + r) * lda + kc + 32 * i + 8 * kq);
          acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bb[i], acc[rt], 0, 0, 0);
        }
      }
    }
  }
}

template <int NR, int KMAX>
__device__ __forceinline__ void mma_strip(const float* __restrict__ A, int lda, int K, PackedB b,
                                          int col0, f32x4 (&acc)[NR]) {
  mma_strip_b16<NR, KMAX>(A, lda, K, b, col0, acc);
}
template <int NR, int KMAX>
__device__ __forceinline__ void mma_strip(const __bf16* __restrict__ A, int lda, int K, PackedB b,
                                          int col0, f32x4 (&acc)[NR]) {
  mma_strip_b16<NR, KMAX>(A, lda, K, b, col0, acc);
}

// Weight-gradient tile: acc(i, j) = sum_k X[k][row0 + i] * Y[k][col0 + j],
// k < K (the rows of the tile). Each lane reads single floats down a column,
// so the four lane groups of one read instruction hit the rows of four
// different k; the k order is permuted so that those rows are 4 apart
// (FP32: k = 16m + 4kq + c for MFMA c of chunk m; BF16: element e of lane
// group kq is k = 32m + 16(e/4) + 4kq + e%4). With row strides of 4 mod 8
// floats, 4 rows are 16 mod 32 floats apart: the four groups' 16-float
// segments fall in disjoint banks. The sum over k is unchanged; only the
// order of the FP32 accumulation differs. Requires K % 16 == 0 (32 for BF16).
template <bool BF, int K>
__device__ __forceinline__ f32x4 mma_wgrad(const float* __restrict__ X, int ldx, int row0,
                                           const float* __restrict__ Y, int ldy, int col0) {
  f32x4 acc{0.f, 0.f, 0.f, 0.f};
  const int lane = lane_here();
  const int r = lane & 15, kq = lane >> 4;
  if constexpr (BF) {
    static_assert(K % 32 == 0, "BF16 weight-gradient tiles take K in steps of 32");
#pragma unroll
    for (int k0 = 0; k0 < K; k0 += 32) {
      bf16x8 av, bv;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int k = k0 + 16 * (e >> 2) + 4 * kq + (e & 3);
        av[e] = (__bf16)X[k * ldx + row0 + r];
        bv[e] = (__bf16)Y[k * ldy + col0 + r];
      }
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, acc, 0, 0, 0);
    }
  } else {
    static_assert(K % 16 == 0, "FP32 weight-gradient tiles take K in steps of 16");
#pragma unroll
    for (int k0 = 0; k0 < K; k0 += 16) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int k = k0 + 4 * kq + c;
        const float a = X[k * ldx + row0 + r];
        const float b = Y[k * ldy + col0 + r];
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0);
      }
    }
  }
  return acc;
}

}  // namespace tfh
