// The output tile of the projection kernels: parameters, epilogues and the
// launch of the direct-to-LDS tile kernels (linear_tiles.hip).
#pragma once

#include "gemm_mainloop.hpp"

namespace sah {

// Epilogues: row-major y (optionally through exact GELU), or the head-major
// Q / K / V scatter.
constexpr int kEpiRows = 0;
constexpr int kEpiRowsGelu = 1;
constexpr int kEpiHeads = 2;
constexpr int kEpiHeadsSeqValue = 3;  // tile kernels: the value seq-contiguous

struct LinearParams {
  const void* x;     // [rows][K], row stride x_ld
  const void* w;     // [N][K], contiguous
  const void* bias;  // [N] or null, same dtype as x
  void* y;           // [rows][N], row stride y_ld (row-major epilogues)
  int64_t rows, x_ld, y_ld;
  int n, k;
  int tiles_n, num_tiles;
  int tiles_m, group_m;
  uint32_t seq_magic, seq_shift;  // row / seq_len as a multiplication (seq_div)
  // Head-major epilogue: output columns [0, D) -> q, [D, 2D) -> k,
  // [2D, 3D) -> v, column c of a block -> head c / head_dim, element
  // c % head_dim; row r -> token (r / seq_len, r % seq_len).
  void* q;
  void* kk;
  void* v;
  int64_t v_ld;      // seq stride of a seq-contiguous value
  int seq_len, heads, head_dim, d_model;
  int v_seq_major;   // value as [B][H][head_dim][v_ld] instead of [B][H][S][head_dim]
  int seq_aligned;   // seq_len % 8 == 0: 8-token runs never cross a sequence
  // LayerNorm on the x rows: weight / bias [K] in the x dtype and each
  // row's (mean, 1/std).
  const void* ln_w;
  const void* ln_b;
  const float2* ln_stats;
};

// Row strides (elements) whose 256 rows the 32-bit offsets of the direct-to-LDS
// loads reach.
constexpr int64_t kMaxTileStride = 1 << 22;

// The kernel that suits the size (rows, n, k) and epilogue: a tile kernel, or
// linear_gelu.hip's.
enum LinearKernel { kRing64, kRing128, kDeep128, kDeep256, kRegisterStaged };
LinearKernel linear_kernel_for(const LinearParams& prm, int epilogue);

// Launch a tile kernel on the stream (prm.x_ld <= kMaxTileStride; tiles and
// grid are set here).
template <typename T, int EPI>
int launch_linear_tiles(LinearParams prm, LinearKernel kernel, hipStream_t stream);

// The epilogue of the register-staged kernel's TM x TN tile at (m0, n0): bias,
// activation, one rounding; the tile is staged in smem (TM rows of TN + 8 elements; every wave is past
// its last operand read) and leaves as 16-byte stores.
template <typename T, int EPI, int TM, int TN, int WM, int WN>
__device__ __forceinline__ void store_tile(const LinearParams& p, unsigned char* smem, int64_t m0, int n0,
                                           const f32x16 (&acc)[TN / WN / 32][TM / WM / 32]) {
  typedef typename Vec8<T>::type V8;
  typedef typename Vec8<T>::half_type V4;
  constexpr bool GELU = EPI == kEpiRowsGelu;
  constexpr int NI = TN / WN / 32, NJ = TM / WM / 32, ROWS = TM / WM, COLS = TN / WN;
  constexpr int THREADS = WM * WN * 64;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int l32 = lane & 31;
  const int half = lane >> 5;
  const int wave_m = wave / WN;
  const int wave_n = wave % WN;
  T(*y_lds)[TN + 8] = reinterpret_cast<T(*)[TN + 8]>(smem);

  // Accumulator register r of acc[i][j] holds output column
  // 32 i + 8 (r / 4) + 4 half + r % 4 (within the wave's slab) of row 32 j + l32.
  const T* bg = static_cast<const T*>(p.bias);
#pragma unroll
  for (int i = 0; i < NI; ++i) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int n_l = wave_n * COLS + 32 * i + 8 * g + 4 * half;
      float bv[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      if (bg != nullptr) {
        const V4 raw = *reinterpret_cast<const V4*>(bg + n0 + n_l);
#pragma unroll
        for (int q = 0; q < 4; ++q) bv[q] = to_f32(raw[q]);
      }
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        V4 out;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float v = acc[i][j][4 * g + q] + bv[q];
          if (GELU) v = fp32_result<T>(gelu_exact(v));
          out[q] = from_f32<T>(v);
        }
        *reinterpret_cast<V4*>(&y_lds[wave_m * ROWS + 32 * j + l32][n_l]) = out;
      }
    }
  }
  __syncthreads();

  constexpr int kChunks = (TM * TN / 8) / THREADS;  // 16-byte chunks per thread
  if constexpr (EPI != kEpiHeads) {
    // ---- coalesced 16-byte stores of the valid rows.
    T* yg = static_cast<T*>(p.y);
#pragma unroll
    for (int s2 = 0; s2 < kChunks; ++s2) {
      const int c = tid + THREADS * s2;
      const int row = c / (TN / 8);
      const int col = (c % (TN / 8)) * 8;
      const int64_t m = m0 + row;
      if (m < p.rows) store16(yg + m * p.y_ld + n0 + col, *reinterpret_cast<const u32x4*>(&y_lds[row][col]));
    }
  } else {
    // ---- head-major scatter.  d_model is a multiple of kBN, so the whole
    // tile belongs to one of q / k / v.  Token indices fit in 32 bits (the
    // host checks rows < 2^31).
    const int which = n0 / p.d_model;
    const int c0 = n0 - which * p.d_model;
    T* dst = static_cast<T*>(which == 0 ? p.q : which == 1 ? p.kk : p.v);
    const unsigned seq = (unsigned)p.seq_len;
    const int hd = p.head_dim;
    if (which != 2 || !p.v_seq_major) {
      // [B][H][S][hd]: a 16-byte chunk is 8 consecutive elements of one head
      // (head_dim is a multiple of 8).
#pragma unroll 4
      for (int s2 = 0; s2 < kChunks; ++s2) {
        const int c = tid + THREADS * s2;
        const int row = c / (TN / 8);
        const int col = (c % (TN / 8)) * 8;
        const int64_t m = m0 + row;
        if (m >= p.rows) continue;
        const unsigned b = (unsigned)m / seq;
        const unsigned s = (unsigned)m - b * seq;
        const int within = c0 + col;
        const int head = within / hd;
        const int e = within - head * hd;
        T* out = dst + (((int64_t)b * p.heads + head) * (int64_t)seq + s) * hd + e;
        store16(out, *reinterpret_cast<const u32x4*>(&y_lds[row][col]));
      }
    } else {
      // [B][H][hd][v_ld]: a 16-byte chunk is 8 consecutive tokens of one
      // column, read down an LDS column (consecutive lanes take consecutive
      // columns: conflict-free).
#pragma unroll 4
      for (int s2 = 0; s2 < kChunks; ++s2) {
        const int c = tid + THREADS * s2;
        const int col = c % TN;
        const int row0 = (c / TN) * 8;
        const int64_t m = m0 + row0;
        if (m >= p.rows) continue;
        const int within = c0 + col;
        const int head = within / hd;
        const int e = within - head * hd;
        if (p.seq_aligned && m + 8 <= p.rows) {
          const unsigned b = (unsigned)m / seq;
          const unsigned s = (unsigned)m - b * seq;
          V8 run;
#pragma unroll
          for (int t = 0; t < 8; ++t) run[t] = y_lds[row0 + t][col];
          T* out = dst + (((int64_t)b * p.heads + head) * hd + e) * p.v_ld + s;
          store16(out, __builtin_bit_cast(u32x4, run));
        } else {
          for (int t = 0; t < 8 && m + t < p.rows; ++t) {
            const unsigned b = (unsigned)(m + t) / seq;
            const unsigned s = (unsigned)(m + t) - b * seq;
            dst[(((int64_t)b * p.heads + head) * hd + e) * p.v_ld + s] = y_lds[row0 + t][col];
          }
        }
      }
    }
  }
}

}  // namespace sah
