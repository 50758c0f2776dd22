// fp32 Linear y = x W^T + b for few rows, on the fp32 matrix cores (gfx950).
//
// For the projections of small fp32 models (a few hundred rows, K and N of a
// few hundred), where a library GEMM of large tiles leaves most CUs idle
// (256 x 256 -> 1024 ran as one workgroup, 63 us).  What bounds it is the
// latency of one tile, so tiles are small and the K of a tile is split:
//  * One workgroup per 32 x 32 output tile; its four waves take a quarter of
//    K each and merge through LDS, so a wave issues K / 8 MFMAs
//    (v_mfma_f32_32x32x2, full-precision fp32) of 64 cycles.  (Eight waves
//    were slower: 5.7 against 4.8 us at 256 x 256 -> 256.)
//  * Operands go straight to registers, 16 bytes a lane (lane half h of slice
//    u holds K 8 u + 4 h .. + 3 of its row on both sides), 32 of K ahead of
//    their use.  Neighbouring tiles share x and W through L2.
// The sums of the quarters are added in ascending order, then the bias.
// Measured (us, GPU time, library -> this): 256 x 256 -> 256 63 -> 4.8, 256 x
// 256 -> 1024 5.7 -> 5.1, 100 x 128 -> 128 11.4 -> 3.9; with more tiles than
// CUs or a longer K the library is faster (512 x 256 -> 768 5.8 against 7.8,
// 256 x 1024 -> 256 5.8 against 10.0: the 32-byte row segments of the loads).
#include "sah_common.hpp"

namespace sah {
namespace {

constexpr int kTile = 32;
constexpr int kSplit = 4;    // waves sharing a tile's K
constexpr int kAhead = 4;    // slices of 8 loaded ahead (32 of K)

__device__ __forceinline__ f32x16 mfma32x2(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

struct LinearF32Params {
  const float* x;
  const float* w;
  const float* bias;  // or null
  float* y;
  int64_t rows, x_ld, y_ld;
  int n, k;
};

__global__ __launch_bounds__(kSplit * 64) void linear_f32_kernel(LinearF32Params p) {
  __shared__ __attribute__((aligned(16))) float part[kSplit][kTile][kTile + 4];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l32 = lane & 31;
  const int half = lane >> 5;
  const int tiles_n = p.n / kTile;
  const int64_t tile_m = blockIdx.x / (unsigned)tiles_n;
  const int n0 = (int)(blockIdx.x - (unsigned)tile_m * (unsigned)tiles_n) * kTile;
  const int64_t m0 = tile_m * kTile;
  const int range = p.k / kSplit;  // a multiple of 8 kAhead
  // rows past the end read the last row; they are not stored
  const int64_t row = m0 + l32 < p.rows ? m0 + l32 : p.rows - 1;
  const float* x = p.x + row * p.x_ld + wave * range + 4 * half;
  const float* w = p.w + (int64_t)(n0 + l32) * p.k + wave * range + 4 * half;

  f32x4 xa[kAhead], wa[kAhead];
#pragma unroll
  for (int u = 0; u < kAhead; ++u) {
    xa[u] = *reinterpret_cast<const f32x4*>(x + 8 * u);
    wa[u] = *reinterpret_cast<const f32x4*>(w + 8 * u);
  }
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
  for (int k0 = 0; k0 < range; k0 += 8 * kAhead) {
    // the next slices (the last ones again at the end: in bounds, not used)
    const int next = k0 + 8 * kAhead < range ? k0 + 8 * kAhead : k0;
    f32x4 xb[kAhead], wb[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      xb[u] = *reinterpret_cast<const f32x4*>(x + next + 8 * u);
      wb[u] = *reinterpret_cast<const f32x4*>(w + next + 8 * u);
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc = mfma32x2(wa[u][i], xa[u][i], acc);
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      xa[u] = xb[u];
      wa[u] = wb[u];
    }
  }
  // acc[r]: column 8 (r / 4) + 4 half + r % 4 of row l32
#pragma unroll
  for (int g = 0; g < 4; ++g)
    *reinterpret_cast<f32x4*>(&part[wave][l32][8 * g + 4 * half]) =
        f32x4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
  __syncthreads();
  const int out_row = threadIdx.x >> 3;
  const int col = (threadIdx.x & 7) * 4;
  if (m0 + out_row >= p.rows) return;
  f32x4 sum = *reinterpret_cast<const f32x4*>(&part[0][out_row][col]);
#pragma unroll
  for (int s = 1; s < kSplit; ++s) sum += *reinterpret_cast<const f32x4*>(&part[s][out_row][col]);
  if (p.bias != nullptr) sum += *reinterpret_cast<const f32x4*>(p.bias + n0 + col);
  *reinterpret_cast<f32x4*>(p.y + (m0 + out_row) * p.y_ld + n0 + col) = sum;
}

}  // namespace
}  // namespace sah

using namespace sah;

extern "C" int sah_linear_f32(const float* x, const float* weight, const float* bias, float* y, int64_t rows,
                              int64_t in_features, int64_t out_features, int64_t x_row_stride,
                              int64_t y_row_stride, sah_stream_t stream) {
  if (rows < 0 || in_features <= 0 || out_features <= 0)
    return fail(SAH_ERR_INVALID_ARGUMENT, "sah_linear_f32: bad sizes rows=%lld in=%lld out=%lld", (long long)rows,
                (long long)in_features, (long long)out_features);
  if (in_features % (8 * kAhead * kSplit) != 0 || out_features % kTile != 0 || in_features > (1 << 20) ||
      out_features > (1 << 20))
    return fail(SAH_ERR_UNSUPPORTED,
                "sah_linear_f32: in_features must be a multiple of %d and out_features of %d (got %lld, %lld)",
                8 * kAhead * kSplit, kTile, (long long)in_features, (long long)out_features);
  if (x_row_stride < in_features || y_row_stride < out_features || x_row_stride % 4 != 0 || y_row_stride % 4 != 0)
    return fail(SAH_ERR_INVALID_ARGUMENT,
                "sah_linear_f32: row strides must cover the row and be multiples of 4 (x %lld, y %lld)",
                (long long)x_row_stride, (long long)y_row_stride);
  if (rows == 0) return SAH_OK;
  if (x == nullptr || weight == nullptr || y == nullptr)
    return fail(SAH_ERR_INVALID_ARGUMENT, "sah_linear_f32: null tensor pointer");
  if (!aligned16(x) || !aligned16(weight) || !aligned16(y) || (bias != nullptr && !aligned16(bias)))
    return fail(SAH_ERR_INVALID_ARGUMENT, "sah_linear_f32: tensors must be 16-byte aligned");
  const int64_t tiles = ceil_div(rows, kTile) * (out_features / kTile);
  if (tiles > (1 << 23))
    return fail(SAH_ERR_UNSUPPORTED, "sah_linear_f32: %lld rows is too many", (long long)rows);
  LinearF32Params p = {};
  p.x = x;
  p.w = weight;
  p.bias = bias;
  p.y = y;
  p.rows = rows;
  p.x_ld = x_row_stride;
  p.y_ld = y_row_stride;
  p.n = (int)out_features;
  p.k = (int)in_features;
  hipLaunchKernelGGL(linear_f32_kernel, dim3((unsigned)tiles), dim3(kSplit * 64), 0,
                     reinterpret_cast<hipStream_t>(stream), p);
  return check_hip(hipGetLastError(), "fp32 linear kernel launch");
}
