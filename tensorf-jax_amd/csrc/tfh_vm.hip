// TensorVM.interpolate (tensor_vm.py:42-89, 140-167, 226-250), its VJP and
// TensorVM.resize (tensor_vm.py:91-100, 183-223) as gfx950 kernels.
#include <algorithm>

#include "tfh_vm.h"
#include "tfh_scatter_sorted.h"

namespace tfh {

// Align-corners linear resampling of the channel-last factors; one thread per
// output float, channel fastest (coalesced). Output texel o samples input
// position o*(G-1)/(G'-1) (jax.image.scale_and_translate with
// scale=(G'-1)/(G-1), translation=0.5-scale/2, tensor_vm.py:210-223).
__device__ __forceinline__ void resample_pos(int64_t o, int64_t gin, int64_t gout, int& i0,
                                             int& i1, float& f) {
  double x = gout > 1 ? (double)o * (double)(gin - 1) / (double)(gout - 1) : 0.0;
  int i = (int)floor(x);
  if (i > gin - 1) i = (int)gin - 1;
  if (i < 0) i = 0;
  f = (float)(x - (double)i);
  i0 = i;
  i1 = i + 1 < gin ? i + 1 : (int)gin - 1;
}

__global__ void __launch_bounds__(256) k_resize_plane(const float* __restrict__ src,
                                                      float* __restrict__ dst, int64_t C,
                                                      int64_t gin, int64_t gout) {
  const int64_t total = 3 * gout * gout * C;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t c = e % C;
    int64_t t = e / C;
    const int64_t col = t % gout;
    t /= gout;
    const int64_t row = t % gout;
    const int64_t m = t / gout;
    int r0, r1, c0, c1;
    float fr, fc;
    resample_pos(row, gin, gout, r0, r1, fr);
    resample_pos(col, gin, gout, c0, c1, fc);
    const float* s = src + (size_t)m * gin * gin * C;
    const float v00 = s[((size_t)r0 * gin + c0) * C + c];
    const float v01 = s[((size_t)r0 * gin + c1) * C + c];
    const float v10 = s[((size_t)r1 * gin + c0) * C + c];
    const float v11 = s[((size_t)r1 * gin + c1) * C + c];
    // separable: along columns first, then rows
    const float top = (1.0f - fc) * v00 + fc * v01;
    const float bot = (1.0f - fc) * v10 + fc * v11;
    dst[e] = (1.0f - fr) * top + fr * bot;
  }
}

__global__ void __launch_bounds__(256) k_resize_line(const float* __restrict__ src,
                                                     float* __restrict__ dst, int64_t C,
                                                     int64_t gin, int64_t gout) {
  const int64_t total = 3 * gout * C;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t c = e % C;
    int64_t t = e / C;
    const int64_t o = t % gout;
    const int64_t m = t / gout;
    int i0, i1;
    float f;
    resample_pos(o, gin, gout, i0, i1, f);
    const float* s = src + (size_t)m * gin * C;
    dst[e] = (1.0f - f) * s[(size_t)i0 * C + c] + f * s[(size_t)i1 * C + c];
  }
}

__global__ void __launch_bounds__(256) k_zero_copies(float* __restrict__ p, int64_t n) {
  for (int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4; e < n;
       e += (int64_t)gridDim.x * 256 * 4) {
    if (e + 4 <= n)
      *reinterpret_cast<float4*>(p + e) = make_float4(0.f, 0.f, 0.f, 0.f);
    else
      for (int64_t j = e; j < n; ++j) p[j] = 0.0f;
  }
}

// Several arrays in one launch: workgroup b clears kZeroChunk floats of the
// array whose chunks it falls in (each a launch of its own took 4 us of host time
// per array, 12 arrays for a render's gradients).
constexpr int kZeroArrays = 16;
constexpr int64_t kZeroChunk = 16384;
struct ZeroList {
  float* p[kZeroArrays];
  int64_t n[kZeroArrays];
};

__global__ void __launch_bounds__(256) k_zero_arrays(ZeroList z) {
  int64_t b = blockIdx.x;
  int i = 0;
  for (; i < kZeroArrays - 1; ++i) {
    const int64_t chunks = (z.n[i] + kZeroChunk - 1) / kZeroChunk;
    if (b < chunks) break;
    b -= chunks;
  }
  const int64_t e0 = b * kZeroChunk, e1 = min(e0 + kZeroChunk, z.n[i]);
  float* p = z.p[i];
  if ((reinterpret_cast<uintptr_t>(p) & 15) == 0) {
    for (int64_t e = e0 + threadIdx.x * 4; e < e1; e += 1024) {
      if (e + 4 <= e1)
        *reinterpret_cast<float4*>(p + e) = make_float4(0.f, 0.f, 0.f, 0.f);
      else
        for (int64_t j = e; j < e1; ++j) p[j] = 0.0f;
    }
  } else {
    for (int64_t e = e0 + threadIdx.x; e < e1; e += 256) p[e] = 0.0f;
  }
}

// A workgroup adds up 64 consecutive entries at a time; its kSumWaves waves
// split the copies (wave w adds copies w, w + kSumWaves, ...), so every load
// is one coalesced 256-byte segment, and the waves' sums meet in LDS in a
// fixed order. The chunk loop's trip count is the same for every thread.
constexpr int kSumWaves = 16;

__global__ void __launch_bounds__(64 * kSumWaves) k_sum_copies(const float* __restrict__ copies,
                                                              int ncopy, int64_t len,
                                                              float* __restrict__ dst) {
  __shared__ float red[kSumWaves][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int64_t e0 = (int64_t)blockIdx.x * 64; e0 < len; e0 += (int64_t)gridDim.x * 64) {
    const int64_t e = e0 + lane;
    float part = 0.0f;
    if (e < len) {
#pragma unroll 4
      for (int k = w; k < ncopy; k += kSumWaves) part += copies[(int64_t)k * len + e];
    }
    red[w][lane] = part;
    __syncthreads();
    if (w == 0 && e < len) {
      float sum = 0.0f;
#pragma unroll
      for (int i = 0; i < kSumWaves; ++i) sum += red[i][lane];
      dst[e] += sum;
    }
    __syncthreads();
  }
}

// p must be 16-byte aligned (a workspace region).
int32_t zero_copies(float* p, int64_t n, hipStream_t st) {
  if (n <= 0) return TFH_OK;
  const int64_t blocks = std::min<int64_t>(ceil_div(n, 1024), 4096);
  hipLaunchKernelGGL(k_zero_copies, dim3((unsigned)blocks), dim3(256), 0, st, p, n);
  return check_launch("clear gradient copies");
}

int32_t sum_copies(const float* copies, int ncopy, int64_t len, float* dst, hipStream_t st) {
  if (len <= 0) return TFH_OK;
  const int64_t blocks = std::min<int64_t>(ceil_div(len, 64), 8192);
  hipLaunchKernelGGL(k_sum_copies, dim3((unsigned)blocks), dim3(64 * kSumWaves), 0, st, copies,
                     ncopy, len, dst);
  return check_launch("sum gradient copies");
}

// (rows, m), rows `ld` apart, -> (m, rows): 64 x 64 tiles through LDS, 256
// contiguous bytes each way.
__global__ void __launch_bounds__(256) k_transpose(const float* __restrict__ in, int rows,
                                                   int64_t m, int64_t ld,
                                                   float* __restrict__ out) {
  __shared__ float tile[64][65];
  const int x = threadIdx.x & 63, y = threadIdx.x >> 6;
  const int64_t s0 = (int64_t)blockIdx.x * 64;
  const int c0 = blockIdx.y * 64;
  for (int c = y; c < 64 && c0 + c < rows; c += 4)
    if (s0 + x < m) tile[c][x] = in[(int64_t)(c0 + c) * ld + s0 + x];
  __syncthreads();
  for (int i = y; i < 64 && s0 + i < m; i += 4)
    if (c0 + x < rows) out[(s0 + i) * rows + c0 + x] = tile[x][i];
}

// The walks over scattered points read a point's channels together: row-major
// gradients, and room for the sort. bytes 0: the direct scatter is the better one
// or the only one. The direct scatter is bound by its adds (54 transactions of 64
// bytes a point at 48 channels), the walks by the reads of the rows and of
// the other factor. Forward and backward at G = 300, 48 channels, direct and sorted:
// 66 thousand points 246 and 258 us, 130 thousand 450 and 358, 250 thousand 849
// and 571; at G = 128 a million 3224 and 1648. A point takes 12C + 30 bytes, so
// larger batches go in equal parts of at most kInterpPart points (2.5 GB at 48
// channels).
struct InterpWs {
  int64_t part;  // points at a time
  float* rows;   // (part, 3C)
  SortWs sort;
};
constexpr int64_t kInterpSortPoints = 5 << 14, kInterpPart = 1 << 22;
static_assert(kInterpPart <= kSortMaxRows, "a part can be sorted");

static size_t carve_interp(Carve& cv, const tfh_vm* vm, int64_t M, InterpWs& ws) {
  if (M < kInterpSortPoints || vm->grid_dim > kSortMaxGrid ||
      !walk_ok(*vm, RowGrad{nullptr, (int)vm->channels}))
    return 0;
  ws.part = ceil_div(M, ceil_div(M, kInterpPart));
  ws.rows = cv.take<float>(ws.part * 3 * vm->channels);
  take_sort_ws(cv, ws.part, ws.sort);
  return cv.off;
}

}  // namespace tfh

using namespace tfh;

extern "C" {

int32_t tfh_vm_interpolate(const tfh_vm* vm, const float* ijk, int64_t num_points, float* out,
                           tfh_stream_t stream) {
  TFH_TRY(check_vm(vm, "tfh_vm_interpolate"));
  TFH_REQUIRE(num_points >= 0, "tfh_vm_interpolate: negative num_points");
  if (num_points == 0) return TFH_OK;
  TFH_REQUIRE(ijk && out, "tfh_vm_interpolate: null pointer");
  TFH_TRY(require_device());
  PlanarPoints src{ijk, num_points};
  return launch_vm_gather<PlanarPoints, false>(*vm, src, num_points, out, as_stream(stream));
}

int32_t tfh_vm_interpolate_bwd(const tfh_vm* vm, const float* ijk, int64_t num_points,
                               const float* grad_out, const tfh_vm_grad* grad,
                               tfh_stream_t stream) {
  TFH_TRY(check_vm(vm, "tfh_vm_interpolate_bwd"));
  TFH_REQUIRE(num_points >= 0, "tfh_vm_interpolate_bwd: negative num_points");
  if (num_points == 0) return TFH_OK;
  TFH_REQUIRE(ijk && grad_out && grad && grad->plane && grad->line,
              "tfh_vm_interpolate_bwd: null pointer");
  TFH_TRY(require_device());
  PlanarPoints src{ijk, num_points};
  return launch_vm_scatter<PlanarPoints, false>(*vm, src, num_points, grad_out, *grad,
                                                as_stream(stream));
}

size_t tfh_vm_interpolate_bwd_workspace_size(const tfh_vm* vm, int64_t num_points) {
  if (check_vm(vm, "tfh_vm_interpolate_bwd_workspace_size") != TFH_OK || num_points < 0) return 0;
  Carve cv(nullptr, 0);
  InterpWs ws;
  return carve_interp(cv, vm, num_points, ws);
}

int32_t tfh_vm_interpolate_bwd_sorted(const tfh_vm* vm, const float* ijk, int64_t num_points,
                                      const float* grad_out, const tfh_vm_grad* grad,
                                      void* workspace, size_t workspace_bytes,
                                      tfh_stream_t stream) {
  TFH_TRY(check_vm(vm, "tfh_vm_interpolate_bwd_sorted"));
  TFH_REQUIRE(num_points >= 0, "tfh_vm_interpolate_bwd_sorted: negative num_points");
  Carve cv(workspace, workspace_bytes);
  InterpWs ws;
  if (carve_interp(cv, vm, num_points, ws) == 0)
    return tfh_vm_interpolate_bwd(vm, ijk, num_points, grad_out, grad, stream);
  TFH_REQUIRE(ijk && grad_out && grad && grad->plane && grad->line,
              "tfh_vm_interpolate_bwd_sorted: null pointer");
  if (!cv.ok)
    return fail(TFH_ERR_WORKSPACE, "tfh_vm_interpolate_bwd_sorted: workspace of %zu bytes, need %zu",
                workspace_bytes, cv.off);
  TFH_TRY(require_device());
  const hipStream_t st = as_stream(stream);
  const int rows = 3 * (int)vm->channels;
  for (int64_t at = 0; at < num_points; at += ws.part) {
    const int64_t n = std::min<int64_t>(ws.part, num_points - at);
    {
      ProfScope ps("scatter_transpose", st);
      hipLaunchKernelGGL(k_transpose,
                         dim3((unsigned)ceil_div(n, 64), (unsigned)ceil_div(rows, 64)), dim3(256),
                         0, st, grad_out + at, rows, n, num_points, ws.rows);
      TFH_TRY(check_launch("tfh_vm_interpolate_bwd_sorted: transpose"));
    }
    const PlanarPoints src{ijk + at, num_points};
    TFH_TRY(scatter_scattered_rows(*vm, src, n, RowGrad{ws.rows, (int)vm->channels}, *grad,
                                   ws.sort, st));
  }
  return TFH_OK;
}

int32_t tfh_zero_arrays(float* const* arrays, const int64_t* counts, int32_t num,
                        tfh_stream_t stream) {
  TFH_REQUIRE(num >= 0 && num <= kZeroArrays, "tfh_zero_arrays: %d arrays", num);
  TFH_REQUIRE(num == 0 || (arrays && counts), "tfh_zero_arrays: null pointer");
  ZeroList z{};
  int64_t blocks = 0;
  for (int i = 0; i < num; ++i) {
    TFH_REQUIRE(counts[i] >= 0 && (arrays[i] || counts[i] == 0), "tfh_zero_arrays: array %d", i);
    z.p[i] = arrays[i];
    z.n[i] = counts[i];
    blocks += ceil_div(counts[i], kZeroChunk);
  }
  if (blocks == 0) return TFH_OK;
  TFH_REQUIRE(blocks < (1ll << 31), "tfh_zero_arrays: too many values");
  TFH_TRY(require_device());
  hipLaunchKernelGGL(k_zero_arrays, dim3((unsigned)blocks), dim3(256), 0, as_stream(stream), z);
  return check_launch("tfh_zero_arrays");
}

int32_t tfh_vm_resize(const tfh_vm* vm, int64_t grid_dim_out, float* out_plane, float* out_line,
                      tfh_stream_t stream) {
  TFH_TRY(check_vm(vm, "tfh_vm_resize"));
  TFH_REQUIRE(out_plane && out_line, "tfh_vm_resize: null output");
  TFH_REQUIRE(grid_dim_out >= vm->grid_dim && grid_dim_out <= 4096,
              "tfh_vm_resize: grid_dim_out %lld must be in [G=%lld, 4096] (upsampling only)",
              (long long)grid_dim_out, (long long)vm->grid_dim);
  TFH_TRY(require_device());
  const int64_t C = vm->channels, gin = vm->grid_dim, gout = grid_dim_out;
  int64_t blocks = ceil_div(3 * gout * gout * C, 256);
  if (blocks > 65535) blocks = 65535;
  hipLaunchKernelGGL(k_resize_plane, dim3((unsigned)blocks), dim3(256), 0, as_stream(stream),
                     vm->plane, out_plane, C, gin, gout);
  TFH_TRY(check_launch("tfh_vm_resize(plane)"));
  blocks = ceil_div(3 * gout * C, 256);
  if (blocks > 65535) blocks = 65535;
  hipLaunchKernelGGL(k_resize_line, dim3((unsigned)blocks), dim3(256), 0, as_stream(stream),
                     vm->line, out_line, C, gin, gout);
  return check_launch("tfh_vm_resize(line)");
}

}  // extern "C"
