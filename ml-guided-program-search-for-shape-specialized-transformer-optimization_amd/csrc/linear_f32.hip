// fp32 Linear y = act(x W^T + b) for few rows, on the fp32 matrix cores (gfx950).
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
//  * A longer K takes 16 x 16 tiles and eight waves (v_mfma_f32_16x16x4):
//    four times the workgroups, and up to K 1024 a wave's loads are one batch.
// The sums of the ranges are added in ascending order, then the bias, then
// GELU (its pass over memory and its launch go: 256 x 256 -> 1024 with it 8.2
// us by library and elementwise kernel, 5.3 here).
// Measured (us, GPU time, library -> this): 256 x 256 -> 256 63 -> 4.7, 256 x
// 256 -> 1024 5.6 -> 4.9, 100 x 128 -> 128 11.4 -> 3.8, 256 x 512 -> 256 117
// -> 5.9, 256 x 1024 -> 256 5.8 -> 6.0, 100 x 640 -> 512 4.9 -> 6.0, 16 x 512 ->
// 512 4.5 -> 5.8; with more tiles than CUs or a longer K
// the library is faster (512 x 256 -> 768 5.8 against 7.8, 256 x 2048 -> 256
// 7.1 against 10.4: the short row segments of the loads).
#include "sah_common.hpp"

namespace sah {
namespace {

constexpr int kTile = 32;
constexpr int kSmallTile = 16;
constexpr int kSmallSplit = 8;
constexpr int kSmallAhead = 8;  // slices of 16 loaded ahead (128 of K: all of a wave's up to K 1024)
// The small tiles serve a longer K, while they fit one round of the CUs (us,
// 32 x 32 / 16 x 16): 256 x 256 -> 256 4.7 / 5.7, 100 x 384 -> 384 5.5 / 5.7,
// 256 x 512 -> 256 6.4 / 5.9, 256 x 1024 -> 256 9.8 / 6.0.
constexpr int kMaxWide = 384;
constexpr int kMaxTiles = 256;
constexpr int kSplit = 4;    // waves sharing a tile's K
constexpr int kAhead = 4;    // slices of 8 loaded ahead (32 of K)

__device__ __forceinline__ f32x16 mfma32x2(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f32x4 mfma16x4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// v Phi(v) by the device library's erff, as the framework's own fp32 GELU has
// it (16-bit outputs take the cheaper gelu_exact).
__device__ __forceinline__ float gelu_f32(float v) { return 0.5f * v * (1.0f + erff(v * 7.071067812e-01f)); }

struct LinearF32Params {
  const float* x;
  const float* w;
  const float* bias;  // or null
  float* y;
  int64_t rows, x_ld, y_ld;
  int n, k;
};

template <bool GELU>
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
  if (GELU)
#pragma unroll
    for (int i = 0; i < 4; ++i) sum[i] = gelu_f32(sum[i]);
  *reinterpret_cast<f32x4*>(p.y + (m0 + out_row) * p.y_ld + n0 + col) = sum;
}

// The same on 16 x 16 tiles, eight waves an eighth of K each: for so few
// outputs that these tiles still fit one round of the CUs.
template <bool GELU>
__global__ __launch_bounds__(kSmallSplit * 64) void linear_f32_small_kernel(LinearF32Params p) {
  __shared__ __attribute__((aligned(16))) float part[kSmallSplit][kSmallTile][kSmallTile + 4];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15;
  const int quarter = lane >> 4;
  const unsigned tiles_n = (unsigned)(p.n / kSmallTile);
  const unsigned tile_m = blockIdx.x / tiles_n;
  const int n0 = (int)(blockIdx.x - tile_m * tiles_n) * kSmallTile;
  const int64_t m0 = (int64_t)tile_m * kSmallTile;
  const int range = p.k / kSmallSplit;  // a multiple of 16
  const int slices = range / 16;
  // rows past the end read the last row; they are not stored
  const int64_t row = m0 + l16 < p.rows ? m0 + l16 : p.rows - 1;
  // slice u: lane quarter q holds K 16 u + 4 q .. + 3 of its row on both sides
  const float* x = p.x + row * p.x_ld + wave * range + 4 * quarter;
  const float* w = p.w + (int64_t)(n0 + l16) * p.k + wave * range + 4 * quarter;

  f32x4 xa[kSmallAhead], wa[kSmallAhead];
#pragma unroll
  for (int u = 0; u < kSmallAhead; ++u) {
    const int at = 16 * (u < slices ? u : slices - 1);
    xa[u] = *reinterpret_cast<const f32x4*>(x + at);
    wa[u] = *reinterpret_cast<const f32x4*>(w + at);
  }
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int s = 0; s < slices; s += kSmallAhead) {
    // the next slices (past the end the last one again: in bounds, not used)
    f32x4 xb[kSmallAhead] = {}, wb[kSmallAhead] = {};
    if (s + kSmallAhead < slices)
#pragma unroll
      for (int u = 0; u < kSmallAhead; ++u) {
        const int next = s + kSmallAhead + u;
        const int at = 16 * (next < slices ? next : slices - 1);
        xb[u] = *reinterpret_cast<const f32x4*>(x + at);
        wb[u] = *reinterpret_cast<const f32x4*>(w + at);
      }
#pragma unroll
    for (int u = 0; u < kSmallAhead; ++u)
      if (s + u < slices)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc = mfma16x4(wa[u][i], xa[u][i], acc);
#pragma unroll
    for (int u = 0; u < kSmallAhead; ++u) {
      xa[u] = xb[u];
      wa[u] = wb[u];
    }
  }
  // acc[r]: column 4 quarter + r of row l16
  *reinterpret_cast<f32x4*>(&part[wave][l16][4 * quarter]) = acc;
  __syncthreads();
  if (wave != 0) return;
  const int out_row = lane >> 2;
  const int col = (lane & 3) * 4;
  if (m0 + out_row >= p.rows) return;
  f32x4 sum = *reinterpret_cast<const f32x4*>(&part[0][out_row][col]);
#pragma unroll
  for (int s = 1; s < kSmallSplit; ++s) sum += *reinterpret_cast<const f32x4*>(&part[s][out_row][col]);
  if (p.bias != nullptr) sum += *reinterpret_cast<const f32x4*>(p.bias + n0 + col);
  if (GELU)
#pragma unroll
    for (int i = 0; i < 4; ++i) sum[i] = gelu_f32(sum[i]);
  *reinterpret_cast<f32x4*>(p.y + (m0 + out_row) * p.y_ld + n0 + col) = sum;
}

}  // namespace
}  // namespace sah

using namespace sah;

extern "C" int sah_linear_f32(const float* x, const float* weight, const float* bias, float* y, int64_t rows,
                              int64_t in_features, int64_t out_features, int64_t x_row_stride,
                              int64_t y_row_stride, int activation, sah_stream_t stream) {
  if (activation != SAH_ACTIVATION_NONE && activation != SAH_ACTIVATION_GELU_EXACT)
    return fail(SAH_ERR_INVALID_ARGUMENT, "sah_linear_f32: unknown activation %d", activation);
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
  const bool gelu = activation == SAH_ACTIVATION_GELU_EXACT;
  const int64_t small_tiles = ceil_div(rows, kSmallTile) * (out_features / kSmallTile);
  const bool small = in_features > kMaxWide && small_tiles <= kMaxTiles;
  auto* kernel = small ? (gelu ? linear_f32_small_kernel<true> : linear_f32_small_kernel<false>)
                       : (gelu ? linear_f32_kernel<true> : linear_f32_kernel<false>);
  hipLaunchKernelGGL(kernel, dim3((unsigned)(small ? small_tiles : tiles)),
                     dim3(64 * (small ? kSmallSplit : kSplit)), 0, reinterpret_cast<hipStream_t>(stream), p);
  return check_hip(hipGetLastError(), "fp32 linear kernel launch");
}
