// Matrix-product main loops of the projection kernels (gfx950).
//
// acc = W X^T over K for one output tile of a row-major x [rows][K] and
// w [N][K], on v_mfma_f32_32x32x16 with the K order ascending in slices of
// 16, so every tile shape and schedule sums in the same order and gives the
// same bits.
//
// Staging.  Both operands go from global memory straight into LDS
// (global_load_lds_dwordx4: 1 KB per wave instruction, no staging registers
// and no LDS stores) as rows of 128 bytes, 64 elements of K.  A direct-to-LDS
// write is contiguous, so the rows cannot be padded; instead 16-byte chunk c
// of row r sits in slot c ^ swizzle(r), and the lane that fills a slot reads
// the matching chunk of its row from global memory.  swizzle() is the linear
// map that makes the slots of any 8 and of any 16 consecutive rows distinct
// where they meet in the banks, so the 16-byte operand reads (32 rows, one
// chunk column) are conflict-free.  A row past the end of x is read as the
// last row (in bounds); its results are not stored.
#pragma once

#include "sah_common.hpp"

namespace sah {

__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mfma32(f16x8 a, f16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

constexpr int kTileK = 64;                 // K per stage: 128-byte rows
constexpr int kTileRowBytes = kTileK * 2;

__device__ __forceinline__ int tile_swizzle(int row) { return (row & 7) ^ ((row >> 3) & 1); }

// One 16-byte direct-to-LDS load per lane: lane i's bytes from base + offset
// land at LDS byte lds + 16 i (base and lds wave-uniform).  Assembly, so that
// the compiler does not wait for it before unrelated LDS reads; the loops
// below wait explicitly.
__device__ __forceinline__ void tile_dma16(const void* base, uint32_t offset, uint32_t lds) {
  const uint64_t b = (uint64_t)(uintptr_t)base;
  const uint64_t sbase = ((uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(b >> 32)) << 32) |
                         (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)b);
  asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1"
               :
               : "v"(offset), "s"(sbase), "s"(__builtin_amdgcn_readfirstlane(lds))
               : "memory", "m0");
}

// Workgroup barrier that waits for nothing but the waves (__syncthreads would
// also wait for every load in flight), pinned in the instruction order.
__device__ __forceinline__ void tile_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}

// One output tile of TM x rows by TN w rows for WM x WN wavefronts, wave
// (wm, wn) holding TM/WM x rows by TN/WN w rows as NI x NJ accumulator
// blocks of 32 x 32: acc[i][j] is Y^T of w rows 32 i.. and x rows 32 j.. of
// the wave.
template <typename T, int TM, int TN, int WM, int WN>
struct GemmTile {
  typedef typename Vec8<T>::type V8;
  static constexpr int WAVES = WM * WN;
  static constexpr int THREADS = WAVES * 64;
  static constexpr int ROWS = TM / WM;        // x rows per wave
  static constexpr int COLS = TN / WN;        // w rows (output columns) per wave
  static constexpr int NI = COLS / 32;        // w blocks per wave
  static constexpr int NJ = ROWS / 32;        // x blocks per wave
  static constexpr int XL = TM / 8 / WAVES;   // x loads per wave and stage (8 rows each)
  static constexpr int WL = TN / 8 / WAVES;   // w loads per wave and stage
  static constexpr uint32_t XSTAGE = TM * kTileRowBytes;
  static constexpr uint32_t WSTAGE = TN * kTileRowBytes;
  static_assert(NI >= 1 && NJ >= 1, "a wave holds at least one block");

  // A load covers 8 rows, and neighbouring loads of a wave swizzle their
  // chunks by one bit, so two lane offsets serve all loads of an operand.
  uint32_t x_row;                   // lane's row of this wave's first x load
  uint32_t x_chunk[2], w_off[2];    // lane's chunk byte (x) and row + chunk bytes (w) of even and odd loads
  uint32_t x_last, x_stride;        // last valid x row; bytes from x row to x row
  uint32_t w_step;                  // bytes from w load to w load
  uint32_t x_lds, w_lds;            // this wave's first load's LDS byte in stage 0
  uint32_t x_read, w_read;          // lane's LDS byte of the first operand read, K slice 0
  const char* xb;                   // first x row of the tile
  const char* wb;                   // first w row of the tile

  // LDS addresses: smem holds the x stages, then the w stages at w_offset.
  __device__ __forceinline__ void init(unsigned char* smem, uint32_t w_offset) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
    x_lds = lds0 + wave * XL * 1024;
    w_lds = lds0 + w_offset + wave * WL * 1024;
    const int wm = wave / WN, wn = wave % WN;
    const uint32_t slot = (uint32_t)(half ^ tile_swizzle(l32)) * 16;  // K slice kk: slot ^ 32 kk
    x_read = (wm * ROWS + l32) * kTileRowBytes + slot;
    w_read = w_offset + (wn * COLS + l32) * kTileRowBytes + slot;
  }
  // The tile's operands.  x: first row, x_ld elements apart (at most 2^22),
  // valid_rows of the TM rows valid; w: first row, k elements apart.
  __device__ __forceinline__ void operands(const T* x, int64_t x_ld, int valid_rows, const T* w, int k) {
    static_assert(XL % 2 == 0 && WL % 2 == 0, "loads alternate between the two lane offsets");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    xb = reinterpret_cast<const char*>(x);
    x_last = (uint32_t)(valid_rows - 1);
    x_stride = (uint32_t)x_ld * 2;
    x_row = wave * XL * 8 + (lane >> 3);
    w_step = (uint32_t)k * 16;
    wb = reinterpret_cast<const char*>(w) + (int64_t)wave * WL * w_step;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t chunk = (uint32_t)((lane & 7) ^ tile_swizzle(i * 8 + (lane >> 3))) * 16;
      x_chunk[i] = chunk;
      w_off[i] = (uint32_t)(lane >> 3) * (uint32_t)(k * 2) + chunk;
    }
  }

  // Load l of this wave's XL + WL loads of a K step (x, w: the step's operand
  // bases) into stage s.
  __device__ __forceinline__ void load_one(int l, const char* x, const char* w, uint32_t s) const {
    if (l < XL) {
      const uint32_t row = min(x_row + 8 * l, x_last);
      tile_dma16(x, __umul24(row, x_stride) + x_chunk[l & 1], x_lds + s * XSTAGE + l * 1024);
    } else {
      tile_dma16(w + (uint64_t)w_step * (l - XL), w_off[l & 1], w_lds + s * WSTAGE + (l - XL) * 1024);
    }
  }
  // Loads FIRST .. LAST - 1 of K step t into stage s.
  template <int FIRST, int LAST>
  __device__ __forceinline__ void load_range(int t, uint32_t s) const {
    const char* x = xb + (int64_t)t * kTileRowBytes;
    const char* w = wb + (int64_t)t * kTileRowBytes;
#pragma unroll
    for (int l = FIRST; l < LAST; ++l) load_one(l, x, w, s);
  }
  __device__ __forceinline__ void load(int t, uint32_t s) const { load_range<0, XL + WL>(t, s); }

  // Operands of K slices kk0 .. kk0 + N - 1 of stage s.
  template <int N>
  struct Operands {
    V8 w[N][NI], x[N][NJ];
  };
  template <int N>
  __device__ __forceinline__ void read(Operands<N>& o, const unsigned char* smem, int kk0,
                                       uint32_t s) const {
#pragma unroll
    for (int n = 0; n < N; ++n) {
#pragma unroll
      for (int i = 0; i < NI; ++i)
        o.w[n][i] = *reinterpret_cast<const V8*>(smem + (w_read ^ (32 * (kk0 + n))) + s * WSTAGE + i * 32 * kTileRowBytes);
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        o.x[n][j] = *reinterpret_cast<const V8*>(smem + (x_read ^ (32 * (kk0 + n))) + s * XSTAGE + j * 32 * kTileRowBytes);
    }
  }
  template <int N>
  __device__ __forceinline__ static void multiply(const Operands<N>& o, f32x16 (&acc)[NI][NJ]) {
#pragma unroll
    for (int n = 0; n < N; ++n)
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = mfma32(o.w[n][i], o.x[n][j], acc[i][j]);
  }

  // A ring of R stages, one barrier per step: the loads of step t + R - 1 are
  // issued right after the barrier of step t, so R - 1 steps are in flight
  // while one is read and multiplied.  For tiles whose loads bound them (few
  // rows): reading the operands a step ahead of the products, from a second
  // register set, made every product wait for one more step's loads (777 x
  // 1024 -> 4096 with GELU 15.1 -> 15.7 us).
  template <int R>
  __device__ __forceinline__ void ring(const unsigned char* smem, int steps, f32x16 (&acc)[NI][NJ]) const {
    constexpr int L = XL + WL;
    static_assert((R - 2) * L < 64, "the wait counts loads in six bits");
#pragma unroll
    for (int t = 0; t < R - 1; ++t)
      if (t < steps) load(t, t);
    uint32_t s = 0, s_load = R - 1;
    for (int t = 0; t < steps; ++t) {
      if (t + R - 1 <= steps)  // steps t + 1 .. t + R - 2 may still be under way
        wait_loads<(R - 2) * L>();
      else
        wait_loads<0>();
      tile_barrier();  // step t is in LDS; every wave has read step t - 1
      if (t + R - 1 < steps) load(t + R - 1, s_load);
      Operands<4> o;
      read(o, smem, 0, s);
      multiply(o, acc);
      __builtin_amdgcn_sched_barrier(0);
      s = s + 1 == R ? 0 : s + 1;
      s_load = s_load + 1 == R ? 0 : s_load + 1;
    }
  }

  // Two stages, one wave per SIMD: every operand read and every load is
  // placed between two MFMAs, one K slice of 16 ahead of its use, so the
  // matrix cores wait only at the one barrier per step.  Slices 0-2 of step t
  // read the operands of the next slice; after slice 2 the step's stage has
  // been read and the other stage (step t + 1) has landed (wait, barrier), so
  // slice 3 reads the first slice of step t + 1, and the loads of step t + 2
  // follow in slice 3 (first half) and in slice 0 of step t + 1 (second
  // half), at least two slices ahead of their wait.
  static constexpr int HALF = (XL + WL) / 2;
  template <bool READ, bool LOAD, int FIRST>
  __device__ __forceinline__ void deep_slice(const Operands<1>& now, Operands<1>& next,
                                             const unsigned char* smem, int kk, uint32_t s,
                                             const char* x, const char* w, uint32_t load_s,
                                             f32x16 (&acc)[NI][NJ]) const {
    constexpr int MF = NI * NJ, RD = NI + NJ;
    const uint32_t xr = (x_read ^ (32 * kk)) + s * XSTAGE, wr = (w_read ^ (32 * kk)) + s * WSTAGE;
#pragma unroll
    for (int m = 0; m < MF; ++m) {
      const int i = m / NJ, j = m % NJ;
      if (READ && m * RD % MF < RD) {
        // in the order of their use: w 0, every x, the other w
        const int r = m * RD / MF;
        if (r == 0 || r > NJ)
          next.w[0][r == 0 ? 0 : r - NJ] = *reinterpret_cast<const V8*>(smem + wr + (r == 0 ? 0 : r - NJ) * 32 * kTileRowBytes);
        else
          next.x[0][r - 1] = *reinterpret_cast<const V8*>(smem + xr + (r - 1) * 32 * kTileRowBytes);
      }
      if (LOAD && (m + MF - 1) * HALF % MF < HALF) load_one(FIRST + (m + MF - 1) % MF * HALF / MF, x, w, load_s);
      acc[i][j] = mfma32(now.w[0][i], now.x[0][j], acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // Step t in stage s.  LOAD1: step t + 1 exists (its second half is loaded
  // here); LOAD2: step t + 2 exists (its first half is).
  template <bool LOAD1, bool LOAD2>
  __device__ __forceinline__ void deep_step(const unsigned char* smem, int t, uint32_t s,
                                            Operands<1>& p0, Operands<1>& p1, f32x16 (&acc)[NI][NJ]) const {
    const char* x1 = xb + (int64_t)(t + 1) * kTileRowBytes;
    const char* w1 = wb + (int64_t)(t + 1) * kTileRowBytes;
    deep_slice<true, LOAD1, HALF>(p0, p1, smem, 1, s, x1, w1, s ^ 1, acc);
    deep_slice<true, false, 0>(p1, p0, smem, 2, s, x1, w1, s, acc);
    deep_slice<true, false, 0>(p0, p1, smem, 3, s, x1, w1, s, acc);
    if (LOAD1) {
      wait_lds();
      wait_loads<0>();
      tile_barrier();
    }
    deep_slice<LOAD1, LOAD2, 0>(p1, p0, smem, 0, s ^ 1, x1 + kTileRowBytes, w1 + kTileRowBytes, s, acc);
  }
  // The loads that deep() expects to be under way: step 0 into stage 0 and
  // the first half of step 1 into stage 1; part PART of PARTS.
  static constexpr int PREFETCH = XL + WL + HALF;
  template <int PART, int PARTS>
  __device__ __forceinline__ void deep_prefetch(int steps) const {
#pragma unroll
    for (int l = PART * PREFETCH / PARTS; l < (PART + 1) * PREFETCH / PARTS; ++l) {
      if (l < XL + WL)
        load_one(l, xb, wb, 0);
      else if (steps > 1)
        load_one(l - (XL + WL), xb + kTileRowBytes, wb + kTileRowBytes, 1);
    }
  }
  // The product over all steps, once step 0 has landed (waited for by every
  // wave, then a barrier).  Returns with a barrier: the stages are free.
  __device__ __forceinline__ void deep(const unsigned char* smem, int steps, f32x16 (&acc)[NI][NJ]) const {
    static_assert((XL + WL) % 2 == 0, "two halves");
    Operands<1> p0, p1;
    read(p0, smem, 0, 0);
    uint32_t s = 0;
    int t = 0;
    if (steps > 1) {
      for (; t + 2 < steps; ++t) {
        deep_step<true, true>(smem, t, s, p0, p1, acc);
        s ^= 1;
      }
      deep_step<true, false>(smem, t, s, p0, p1, acc);
      s ^= 1;
      ++t;
    }
    deep_step<false, false>(smem, t, s, p0, p1, acc);
    tile_barrier();
  }
};

}  // namespace sah
