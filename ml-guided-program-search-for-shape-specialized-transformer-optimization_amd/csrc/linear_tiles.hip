// Direct-to-LDS tile kernels of the projections (gfx950): Linear, Linear +
// exact GELU, and the packed QKV projection with its head-major stores.
//
// What bounds them: the matrix cores, under the power limit, and the epilogue
// that nothing covers.  The register-staged 8-wave kernel of linear_gelu.hip
// waits at one __syncthreads per K step with every load behind it, reads
// 192 KB of operands per step and CU, loads its bias in scalars in the epilogue,
// and leaves most CUs idle for few rows.  Here a 256 x 256 tile is held by four
// waves, one per SIMD, 128 x 128 each: a third fewer LDS reads per MFMA, and
// one wave's instruction stream keeps its matrix core busy: 70% of all cycles
// at 65536 x 2048 -> 8192, where the chip holds 1.4-1.6 GHz; a tile takes 93 K
// cycles, 65.5 K of them MFMAs, and 116 K with GELU (counters:
// profiles/linear_tiles_sq_counters.md).  Measured with the same inputs on one
// box, before -> after:
//   65536 x 2048 -> 8192    2567 -> 1710 us (1286 TFLOP/s), GELU 2786 -> 1960 us
//   20002 x 1024 -> 3072     154 ->  118 us, GELU 179 -> 157 us
//   777 x 1024 -> 4096        36 ->   13 us, GELU  44 ->  15 us
//   64 x 4096 -> 1024        102 ->   20 us
// Few rows take smaller tiles on more CUs: one CU loads 50-70 GB/s whatever its
// tile (first row of the table at linear_kernel_for: (TM + TN) rows of 8 KB each
// in that time), and a tile's K steps wait for that.
// Tried and slower at 65536 x 2048 -> 8192: two groups of four waves half a
// step apart on 128 x 64 wave tiles (1983 us); stores of a tile spread over
// the next tile's main loop from registers (1790 us: 32-byte segments and
// spills); loads of the next tile between the epilogue's blocks (1830 us,
// spills; kept for the 128 x 256 tile, which has the registers).

#include <atomic>

#include "linear_tiles.hpp"

namespace sah {
namespace {

// The bias of a wave's NI * 32 columns, two per lane (one register): dword d
// is columns 2 d and 2 d + 1.
template <typename T, int NI>
struct WaveBias {
  uint32_t pair;
  __device__ __forceinline__ void load(const T* bias, int n_wave) {
    const int lane = threadIdx.x & 63;
    pair = 0;
    if (bias != nullptr && lane < NI * 16) pair = *reinterpret_cast<const uint32_t*>(bias + n_wave + 2 * lane);
  }
  // Columns 32 i + 8 g + 4 half .. + 3, as accumulator registers 4 g .. 4 g + 3
  // of acc[i][j] hold them.
  __device__ __forceinline__ void get(int i, int g, float (&out)[4]) const {
    typedef typename Vec8<T>::half_type V4;
    const int half = (threadIdx.x & 63) >> 5;
    const int source = (16 * i + 4 * g + 2 * half) * 4;
    u32x2 raw;
    raw[0] = (uint32_t)__builtin_amdgcn_ds_bpermute(source, (int)pair);
    raw[1] = (uint32_t)__builtin_amdgcn_ds_bpermute(source + 4, (int)pair);
    const V4 v = __builtin_bit_cast(V4, raw);
#pragma unroll
    for (int q = 0; q < 4; ++q) out[q] = to_f32(v[q]);
  }
};

// row / seq_len and its remainder, exact for rows below 2^31
// (LinearParams::seq_magic; seq_len 1 has magic 0).
__device__ __forceinline__ void seq_div(const LinearParams& p, uint32_t row, uint32_t& b, uint32_t& s) {
  b = p.seq_magic == 0 ? row : __umulhi(row, p.seq_magic) >> p.seq_shift;
  s = row - b * (uint32_t)p.seq_len;
}

// The epilogue of one wave's NJ x NI blocks: bias, activation, one rounding.
// 32 rows at a time pass through the wave's own LDS area (32 rows of NI * 64
// bytes, 16-byte chunk c of row r in slot c ^ f(r): conflict-free both ways)
// and leave as 16-byte stores of whole NI * 64 byte row segments, so the waves
// need no barrier and the stages stay free for the next tile's loads.
// (Stored straight from the accumulator layout, 32-byte segments, the 65536 x
// 2048 -> 8192 Linear ran 5% slower.)  m_wave, n_wave: the wave's first row
// and column.  With every row valid the wave issues exactly NJ * NI * 2
// stores (seq-contiguous values apart), the last two blocks' after
// prefetch(NJ - 1).  prefetch(j) runs before the arithmetic of block j.
template <typename T, int EPI, int NI, int NJ, typename F>
__device__ __forceinline__ void store_wave(const LinearParams& p, unsigned char* area, int64_t m_wave,
                                           int n_wave, const WaveBias<T, NI>& bias,
                                           const f32x16 (&acc)[NI][NJ], const F& prefetch) {
  typedef typename Vec8<T>::type V8;
  typedef typename Vec8<T>::half_type V4;
  constexpr bool kHeads = EPI == kEpiHeads || EPI == kEpiHeadsSeqValue;
  constexpr int CPR = NI * 4;         // 16-byte chunks per row
  constexpr int ROWS_PER = 64 / CPR;  // rows per store instruction
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));  // addresses formed here, not kept over the main loop
  const int l32 = lane & 31;
  const int half = lane >> 5;
  auto slot = [](int row, int chunk) { return chunk ^ ((row >> (CPR == 16 ? 0 : CPR == 8 ? 1 : 2)) & (CPR - 1)); };

  const int chunk = lane % CPR;
  const int col = n_wave + chunk * 8;
  // head-major: the wave's columns lie in one of q / k / v (d_model is a
  // multiple of the tile width), a chunk in one head
  T* dst = nullptr;
  int head = 0, e = 0;
  const bool v_seq = EPI == kEpiHeadsSeqValue && n_wave >= 2 * p.d_model;
  if constexpr (kHeads) {
    const int which = n_wave / p.d_model;
    dst = static_cast<T*>(which == 0 ? p.q : which == 1 ? p.kk : p.v);
    const int within = col - which * p.d_model;
    head = within / p.head_dim;
    e = within - head * p.head_dim;
  }

  float bv[NI][4][4];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int g = 0; g < 4; ++g) bias.get(i, g, bv[i][g]);

  // Block j: compute, write to the area, read back row segments; the reads'
  // latency passes under the next block's first arithmetic, then they are
  // stored (LDS keeps a wave's reads before its later writes).
  constexpr int NS = 32 / ROWS_PER;  // stores per block
  u32x4 segment[NS];
  auto store_segments = [&](int j) {
#pragma unroll
    for (int r = 0; r < NS; ++r) {
      const int64_t m = m_wave + 32 * j + r * ROWS_PER + lane / CPR;
      if (kHeads) __builtin_amdgcn_sched_barrier(0);
      if (m >= p.rows) continue;
      if constexpr (kHeads) {
        uint32_t b, s;
        seq_div(p, (uint32_t)m, b, s);
        store16(dst + (((int64_t)b * p.heads + head) * (int64_t)p.seq_len + s) * p.head_dim + e, segment[r]);
      } else {
        store16(static_cast<T*>(p.y) + m * p.y_ld + col, segment[r]);
      }
    }
  };
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    prefetch(j);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        V4 out;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float v = acc[i][j][4 * g + q] + bv[i][g][q];
          if (EPI == kEpiRowsGelu) v = fp32_result<T>(gelu_exact(v));
          out[q] = from_f32<T>(v);
        }
        *reinterpret_cast<V4*>(area + l32 * (CPR * 16) + slot(l32, 4 * i + g) * 16 + half * 8) = out;
      }
      __builtin_amdgcn_sched_barrier(0);
      if (i == 0 && j > 0 && !v_seq) store_segments(j - 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
    if (EPI == kEpiHeadsSeqValue && v_seq) {
      // [B][H][hd][v_ld]: 8 consecutive tokens of one column per 16 bytes
#pragma unroll 1
      for (int c = lane; c < 4 * CPR * 8; c += 64) {
        const int vcol = c % (CPR * 8);
        const int row0 = c / (CPR * 8) * 8;
        const int64_t m = m_wave + 32 * j + row0;
        if (m >= p.rows) continue;
        const int within = n_wave + vcol - 2 * p.d_model;
        const int vh = within / p.head_dim;
        const int ve = within - vh * p.head_dim;
        V8 run;
#pragma unroll
        for (int t = 0; t < 8; ++t)
          run[t] = *reinterpret_cast<const T*>(area + (row0 + t) * (CPR * 16) + slot(row0 + t, vcol >> 3) * 16 + (vcol & 7) * 2);
        uint32_t b, s;
        seq_div(p, (uint32_t)m, b, s);
        if (m + 8 <= p.rows && s + 8 <= (uint32_t)p.seq_len) {
          // 16-byte aligned only where seq_len % 8 == 0; the copy is one 16-byte store all the
          // same, which takes any element's address (B3 S5001 D768 167 -> 92 us against
          // element stores, register-staged 134; D1024 167 -> 103)
          __builtin_memcpy(dst + (((int64_t)b * p.heads + vh) * p.head_dim + ve) * p.v_ld + s, &run, 16);
        } else {
#pragma unroll
          for (int t = 0; t < 8; ++t) {
            if (m + t >= p.rows) break;
            seq_div(p, (uint32_t)(m + t), b, s);
            dst[(((int64_t)b * p.heads + vh) * p.head_dim + ve) * p.v_ld + s] = run[t];
          }
        }
      }
    } else {
#pragma unroll
      for (int r = 0; r < NS; ++r) {
        const int row = r * ROWS_PER + lane / CPR;
        segment[r] = *reinterpret_cast<const u32x4*>(area + row * (CPR * 16) + slot(row, chunk) * 16);
      }
    }
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  }
  if (!v_seq) store_segments(NJ - 1);
}

// Tile `logical` of the launch: groups of group_m row tiles walked column by
// column, so the tiles an XCD works on at a time share both x rows and w rows
// in its L2.
__device__ __forceinline__ void tile_at(const LinearParams& p, int logical, int& tile_m, int& tile_n) {
  const int group_tiles = p.group_m * p.tiles_n;
  const int group = logical / group_tiles;
  const int first = group * p.group_m;
  const int height = p.tiles_m - first < p.group_m ? p.tiles_m - first : p.group_m;
  const int in_group = logical - group * group_tiles;
  tile_n = in_group / height;
  tile_m = first + in_group - tile_n * height;
}

template <int NI, int NJ>
__device__ __forceinline__ void clear(f32x16 (&acc)[NI][NJ]) {
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
}

// One tile per workgroup of 2 x 2 waves, a ring of R stages.
template <typename T, int EPI, int TM, int TN, int R>
__global__ __launch_bounds__(256, 1) void linear_ring_kernel(LinearParams p) {
  typedef GemmTile<T, TM, TN, 2, 2> Tile;
  constexpr uint32_t kStageBytes = R * (Tile::XSTAGE + Tile::WSTAGE);
  constexpr uint32_t kAreaBytes = 32 * Tile::COLS * sizeof(T);
  __shared__ __attribute__((aligned(16))) unsigned char smem[kStageBytes + Tile::WAVES * kAreaBytes];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  // contiguous runs of tiles per XCD (ids are dealt round-robin over the 8)
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int per = p.num_tiles >> 3, rem = p.num_tiles & 7;
  int tile_m, tile_n;
  tile_at(p, xcd * per + (xcd < rem ? xcd : rem) + local, tile_m, tile_n);
  const int64_t m0 = (int64_t)tile_m * TM;
  const int n0 = tile_n * TN;
  Tile tile;
  tile.init(smem, R * Tile::XSTAGE);
  const int64_t left = p.rows - m0;
  tile.operands(static_cast<const T*>(p.x) + m0 * p.x_ld, p.x_ld, left < TM ? (int)left : TM,
                static_cast<const T*>(p.w) + (int64_t)n0 * p.k, p.k);
  const int n_wave = n0 + wave % 2 * Tile::COLS;
  WaveBias<T, Tile::NI> bias;
  bias.load(static_cast<const T*>(p.bias), n_wave);
  f32x16 acc[Tile::NI][Tile::NJ];
  clear(acc);
  tile.template ring<R>(smem, p.k / kTileK, acc);
  store_wave<T, EPI>(p, smem + kStageBytes + wave * kAreaBytes, m0 + wave / 2 * Tile::ROWS, n_wave, bias,
                     acc, [](int) {});
}

// Persistent workgroups of four waves, one per CU, each walking tiles of its
// XCD's contiguous run.  The next tile's first loads are issued before the
// epilogue (between its blocks on the 128 x 256 tile, which has the registers),
// and the wait for them counts the epilogue's stores behind them instead of
// waiting for those too.  The epilogue itself ends before the next tile's
// products begin.
template <typename T, int EPI, int TM, int TN>
__global__ __launch_bounds__(256, 1) void linear_deep_kernel(LinearParams p) {
  typedef GemmTile<T, TM, TN, 2, 2> Tile;
  constexpr uint32_t kStageBytes = 2 * (Tile::XSTAGE + Tile::WSTAGE);
  constexpr uint32_t kAreaBytes = 32 * Tile::COLS * sizeof(T);
  // Stores of a wave's full epilogue, all issued after the last of the next
  // tile's loads.
  constexpr int kBehind = 2 * Tile::NI * Tile::NJ;
  __shared__ __attribute__((aligned(16))) unsigned char smem[kStageBytes + 4 * kAreaBytes];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int per = p.num_tiles >> 3, rem = p.num_tiles & 7;
  const int run = xcd * per + (xcd < rem ? xcd : rem);  // the XCD's first tile
  const int end = run + per + (xcd < rem ? 1 : 0);
  const int stride = (gridDim.x + 7 - xcd) >> 3;        // workgroups of this XCD
  const int steps = p.k / kTileK;

  Tile tile;
  tile.init(smem, 2 * Tile::XSTAGE);
  int64_t m0 = 0;
  int n0 = 0;
  auto begin = [&](int logical) {
    int tile_m, tile_n;
    tile_at(p, logical, tile_m, tile_n);
    m0 = (int64_t)tile_m * TM;
    n0 = tile_n * TN;
    const int64_t left = p.rows - m0;
    tile.operands(static_cast<const T*>(p.x) + m0 * p.x_ld, p.x_ld, left < TM ? (int)left : TM,
                  static_cast<const T*>(p.w) + (int64_t)n0 * p.k, p.k);
  };
  int logical = run + local;
  if (logical >= end) return;
  begin(logical);
  tile.template deep_prefetch<0, 1>(steps);
  // The number of stores issued after the loads of step 0 is known (kBehind
  // or more), so those loads can be waited for without waiting for the stores.
  bool stores_behind = false;
  while (true) {
    if (stores_behind)
      wait_loads<kBehind>();
    else
      wait_loads<0>();
    tile_barrier();
    const int64_t m_wave = m0 + wave / 2 * Tile::ROWS;
    const int n_wave = n0 + wave % 2 * Tile::COLS;
    const bool full = m0 + TM <= p.rows && EPI != kEpiHeadsSeqValue;
    WaveBias<T, Tile::NI> bias;
    bias.load(static_cast<const T*>(p.bias), n_wave);
    f32x16 acc[Tile::NI][Tile::NJ];
    clear(acc);
    tile.deep(smem, steps, acc);
    logical += stride;
    const bool more = logical < end;
    if (more) begin(logical);
    // TN 256 x TM 256 has no registers to spare for loads between the blocks
    if (Tile::NJ > 2 && more) tile.template deep_prefetch<0, 1>(steps);
    store_wave<T, EPI>(p, smem + kStageBytes + wave * kAreaBytes, m_wave, n_wave, bias, acc, [&](int j) {
      if (Tile::NJ > 2 || !more) return;
      if (j == 0) tile.template deep_prefetch<0, 2>(steps);
      if (j == 1) tile.template deep_prefetch<1, 2>(steps);
    });
    if (!more) return;
    stores_behind = full;
  }
}

// The current device's compute units, asked once per device (every Linear call needs them).
int compute_units() {
  static std::atomic<int> known[64];
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0) return 256;
  int count = device < 64 ? known[device].load(std::memory_order_relaxed) : 0;
  if (count > 0) return count;
  if (hipDeviceGetAttribute(&count, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || count <= 0)
    return 256;
  if (device < 64) known[device].store(count, std::memory_order_relaxed);
  return count;
}

template <int TM, int TN>
void set_tiles(LinearParams& prm) {
  prm.tiles_m = (int)((prm.rows + TM - 1) / TM);
  prm.tiles_n = prm.n / TN;
  prm.num_tiles = prm.tiles_m * prm.tiles_n;
  prm.group_m = 4;
}

template <typename T, int EPI, int TM, int TN>
int launch_deep(LinearParams prm, hipStream_t stream) {
  set_tiles<TM, TN>(prm);
  const int cus = compute_units();
  hipLaunchKernelGGL((linear_deep_kernel<T, EPI, TM, TN>), dim3(prm.num_tiles < cus ? prm.num_tiles : cus),
                     dim3(256), 0, stream, prm);
  return check_hip(hipGetLastError(), "linear kernel launch");
}

template <typename T, int EPI, int TM, int TN, int R>
int launch_ring(LinearParams prm, hipStream_t stream) {
  set_tiles<TM, TN>(prm);
  hipLaunchKernelGGL((linear_ring_kernel<T, EPI, TM, TN, R>), dim3(prm.num_tiles), dim3(256), 0, stream, prm);
  return check_hip(hipGetLastError(), "linear kernel launch");
}

}  // namespace

LinearKernel linear_kernel_for(const LinearParams& prm, int epilogue) {
  // The tile by an estimate of its time in us: rounds of its grid on the CUs,
  // each of K / 64 steps and an epilogue.  A step costs what one CU loads
  // ((TM + TN) rows of 128 bytes) or multiplies; two 64 x 64 workgroups share a
  // CU.  Measured (bf16, us, plain Linear / with GELU), 64 x 64, 128 x 128,
  // 128 x 256 and 256 x 256:
  //   64 x 4096 -> 1024     19.7         37.4           43.8           68.0
  //   800 x 2048 -> 512     12.0         20.7           25.1           38.4
  //   777 x 1024 -> 4096    17.1         12.9 / 15.1    16.6 / 20.7    24.7 / 33.0
  //   2000 x 1024 -> 3072   24.2         23.7           18.8           25.9
  //   2000 x 1024 -> 4096                24.5 / 28.9    21.9 / 25.8    26.9 / 35.0
  //   6000 x 1024 -> 4096   89.1         72.0           57.5           55.6
  //   16384 x 2048 -> 512                42.3 / 45.8    35.8 / 40.2    43.3 / 51.1
  //   16384 x 512 -> 2048                57.4 / 71.7    47.6 / 66.8    44.2 / 59.2
  //   20002 x 1024 -> 3072               170 / 203      144 / 182      118 / 157
  // The estimates rank the tiles; they are not times: of one clock for all
  // loads, without GELU, they are up to a third low where the power limit holds
  // the clock down (20002 x 1024 -> 3072: 94 for 118).  At 6000 x 1024 -> 4096
  // they take 128 x 256 (43.7 against 47.0) where 256 x 256 is 3% faster.
  const int64_t cus = compute_units();
  const double steps = (double)(prm.k / kTileK);
  auto tiles = [&](int64_t tm, int64_t tn) { return ceil_div(prm.rows, tm) * (prm.n / tn); };
  auto rounds = [&](int64_t tm, int64_t tn) { return (double)ceil_div(tiles(tm, tn), cus); };
  const double t64 = (double)tiles(64, 64) / (double)(2 * cus);
  const double ring64 = t64 <= 0.5 ? steps * 0.28 + 1.0 : (t64 < 1.0 ? 1.0 : t64) * (steps * 0.39 + 1.5);
  const double ring128 = rounds(128, 128) * (steps * 0.54 + 2.5);
  const double deep128 = rounds(128, 256) * (steps * 0.66 + 4.0);
  const double deep256 = rounds(256, 256) * (steps * 1.03 + 7.0);
  if (ring64 <= ring128 && ring64 <= deep128 && ring64 <= deep256) return kRing64;
  if (ring128 <= deep128 && ring128 <= deep256) return kRing128;
  if (deep128 <= deep256) return kDeep128;
  // Up to three K steps leave the 256 x 256 tile little but its load latency
  // and its epilogue, which the register-staged kernel's eight waves pass
  // faster than four, until (five rounds and more) the chip is busy storing.
  // Measured (bf16 us, register-staged / 256 x 256; equal bits):
  //   20002 x 128 -> 512  11.0 / 12.2, GELU 19.3 / 20.9   10000 x 64 -> 1024   9.4 / 10.5
  //   50000 x 128 -> 512  21.2 / 22.2, GELU 37.6 / 39.5   16384 x 128 -> 1024 13.5 / 13.9
  //   12000 x 192 -> 768  12.5 / 13.1, GELU 20.8 / 22.0  131072 x 64 -> 1024  76.1 / 67.0
  // A fourth step only in one round and without GELU, whose arithmetic covers the stores:
  //   16384 x 256 -> 1024 17.6 / 22.3, GELU 27.0 / 26.3   32768 x 256 -> 512  17.7 / 21.3
  //   20002 x 256 -> 512  14.6 / 14.5, GELU 22.8 / 23.3   70000 x 256 -> 1024 72.5 / 70.1
  // Head-major (K is 256 or more there) always, but a seq-contiguous value only up to six rounds
  // and where its 8-token runs are aligned, as that kernel wants them (us at D 256, register-staged /
  // 256 x 256, then with such a value):
  //   B2 S8192   15.7 / 16.9, 18.9 / 22.9   B16 S4096  48.2 / 51.9, 52.8 / 49.7
  //   B1 S12000  15.3 / 16.3, 17.8 / 22.5   B20 S4000  58.2 / 65.8, 60.7 / 68.3
  //   B3 S5001   15.9 / 16.8, 51.3 / 23.3   B64 S1600  73.0 / 83.0, 76.1 / 83.0
  //                                         B1 S300000  233 / 243,   252 / 233
  int64_t most = 0;
  if (prm.k <= 3 * kTileK)
    most = 5 * cus;
  else if (prm.k == 4 * kTileK && epilogue == kEpiRows)
    most = cus;
  else if (prm.k == 4 * kTileK && epilogue == kEpiHeads)
    most = !prm.v_seq_major ? INT64_MAX : prm.seq_aligned ? 6 * cus : 0;
  if (tiles(256, 256) <= most) return kRegisterStaged;
  return kDeep256;
}

template <typename T, int EPI>
int launch_linear_tiles(LinearParams prm, LinearKernel kernel, hipStream_t stream) {
  if (prm.seq_len > 1) {
    // row / seq_len = (row * magic) >> (31 + l), 2^l >= seq_len, for rows below 2^31
    int l = 1;
    while ((1ull << l) < (unsigned long long)prm.seq_len) ++l;
    prm.seq_magic = (uint32_t)((1ull << (31 + l)) / (uint32_t)prm.seq_len + 1);
    prm.seq_shift = (uint32_t)(l - 1);
  }
  switch (kernel) {
    case kRing64: return launch_ring<T, EPI, 64, 64, 4>(prm, stream);
    case kRing128: return launch_ring<T, EPI, 128, 128, 4>(prm, stream);
    case kDeep128: return launch_deep<T, EPI, 128, 256>(prm, stream);
    default: return launch_deep<T, EPI, 256, 256>(prm, stream);
  }
}

template int launch_linear_tiles<bf16, kEpiRows>(LinearParams, LinearKernel, hipStream_t);
template int launch_linear_tiles<bf16, kEpiRowsGelu>(LinearParams, LinearKernel, hipStream_t);
template int launch_linear_tiles<bf16, kEpiHeads>(LinearParams, LinearKernel, hipStream_t);
template int launch_linear_tiles<bf16, kEpiHeadsSeqValue>(LinearParams, LinearKernel, hipStream_t);
template int launch_linear_tiles<f16, kEpiRows>(LinearParams, LinearKernel, hipStream_t);
template int launch_linear_tiles<f16, kEpiRowsGelu>(LinearParams, LinearKernel, hipStream_t);
template int launch_linear_tiles<f16, kEpiHeads>(LinearParams, LinearKernel, hipStream_t);
template int launch_linear_tiles<f16, kEpiHeadsSeqValue>(LinearParams, LinearKernel, hipStream_t);

}  // namespace sah
