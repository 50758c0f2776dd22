// fp32 causal attention, head_dim 64, for gfx950 (CDNA4): the reference's fp32
// portable path.  Scores, softmax and PV all in fp32, P kept in fp32 (the
// input dtype, so the reference's rounding of P is the identity).
//
// What bounds it: the fp32 matrix cores (157 TFLOP/s; v_mfma_f32_32x32x2 is a
// full-precision fp32 multiply-add).  A 32-query x 32-key block takes 64 of
// them, 4096 cycles, against about 150 other VALU instructions.
//  * One wavefront owns a block of 32 queries and walks 32-key blocks, S^T =
//    K Q^T then O^T = V^T P^T: a lane holds one query's scores (16 of the 32
//    keys; its partner in the other half wave the rest), so the row maximum
//    is in-lane plus one half-wave exchange, and the score registers are the
//    B operand of the PV products as they stand: register r of half h is key
//    8 (r / 4) + 4 h + r % 4, and V is read in that order.
//  * K and V go from global memory (L2) straight to registers: each block is
//    read by one wave only, K as 16-byte chunks of 32 rows, V as whole rows
//    (8 bytes a lane; dims 2 i and 2 i + 1 are rows i of the two output
//    blocks).  The next K block is loaded before the PV products, the next V
//    block between them: no LDS, no barrier in the loop.
//  * The softmax of a block runs between the score products of the next one
//    (two waves on a SIMD otherwise fall into step and neither hides the
//    other's: B1 H8 S8192 811 -> 614 us with it).
//  * The four waves of a workgroup split the keys of the same 32 queries
//    (block j goes to wave j mod 4) and merge their maxima, sums and outputs
//    through LDS once: short sequences have few query blocks, and the longest
//    one sets the time.
// Measured (us a call on one box; before it a VALU kernel, four lanes per query
// over 64-key LDS tiles, 193 VGPRs):
//   B4 H8 S777    318 -> 38.7     B2 H12 S1500   807 ->  76
//   B4 H12 S2500 3031 -> 368      B1 H8 S8192   5956 -> 614 (112 TFLOP/s)
#include <cfloat>
#include <cmath>

#include "attention_f32.hpp"

namespace sah {
namespace {

constexpr int kQ = 32;       // queries per workgroup
constexpr int kKeys = 32;    // keys per block
constexpr int kDim = 64;
constexpr int kSplit = 4;    // waves sharing the keys
constexpr int kORow = kDim + 4;

__device__ __forceinline__ f32x16 mfma32x2(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

__global__ __launch_bounds__(kSplit * 64, 2) void attn_fwd_f32_kernel(AttnF32Params p, int num_q) {
  __shared__ __attribute__((aligned(16))) float o_lds[kSplit][kQ][kORow];
  __shared__ float m_lds[kSplit][kQ], l_lds[kSplit][kQ];
  // longest query blocks first; heads on the fast axis, so with a multiple of
  // 8 of them a head stays in one XCD's L2
  const int64_t from_end = (int64_t)blockIdx.z * gridDim.y + blockIdx.y;
  if (from_end >= num_q) return;
  const int qt = num_q - 1 - (int)from_end;
  const int bh = blockIdx.x;
  const int b = bh / p.heads;
  const int h = bh - b * p.heads;
  const int S = p.seq_len;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31;
  const int half = lane >> 5;
  const float c = p.c;

  // q[4 u + i]: dim 8 u + 4 half + i of query l32 (rows past the end read the
  // last row; they are not stored)
  const int qi = qt * kQ + l32;
  const float* qrow = p.q + b * p.q_sb + h * p.q_sh + (int64_t)min(qi, S - 1) * p.q_ss + 4 * half;
  const float* kbase = p.k + b * p.k_sb + h * p.k_sh + 4 * half;
  const float* vbase = p.v + b * p.v_sb + h * p.v_sh + 2 * l32;
  f32x4 q[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    u32x4 raw = load16(qrow + 8 * u);
    raw = (raw & p.q_and) ^ p.q_xor;
    q[u] = __builtin_bit_cast(f32x4, raw);
  }

  // K block: chunk u is dims 8 u + 4 half .. + 3 of key k0 + l32.  V block:
  // v[r] is dims 2 l32, 2 l32 + 1 of the key of score register r.  Only the
  // last block can reach past the sequence; its rows past the end read the
  // last row (masked).
  f32x4 kf[8];
  f32x2 vf[16];
  auto k_row = [&](int j) { return kbase + (int64_t)min(j * kKeys + l32, S - 1) * p.k_ss; };
  auto load_v = [&](int j) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int key = min(j * kKeys + 8 * (r / 4) + 4 * half + r % 4, S - 1);
      vf[r] = *reinterpret_cast<const f32x2*>(vbase + (int64_t)key * p.v_ss);
    }
  };

  f32x16 o0, o1;
#pragma unroll
  for (int r = 0; r < 16; ++r) o0[r] = o1[r] = 0.0f;
  // Of this wave's keys; l_run of this half's.  The maximum starts at the
  // lowest shift instead of -inf: keys that all score -inf (or too low for the
  // shift) then weigh exp2(-inf) = 0, and nothing forms -inf + inf.
  float m_run = p.floor, mc_run = p.floor * c, l_run = 0.0f;
  auto load_k = [&](const float* row) {
#pragma unroll
    for (int u = 0; u < 8; ++u) kf[u] = *reinterpret_cast<const f32x4*>(row + 8 * u);
  };
  auto scores = [&]() {
    f32x16 s;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0.0f;
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) s = mfma32x2(kf[u][i], q[u][i], s);
    return s;
  };
  // The shift c m as one rounded number, the same for P, the rescaling and the
  // merge (the assembly keeps it from being formed again inside an fma there):
  // its rounding then cancels, where exp2(c (m_run - m_new)) beside it is off by
  // half an ulp of c m (error against float64, relative to the 64-key-tile
  // kernel's, over S 31-2500: 0.98-1.02 -> 0.97-1.01; with scores about 77000
  // 1.4e-4 -> 2.4e-7).
  auto shift = [&](float m) {
    float mc = m * c;
    asm("" : "+v"(mc));
    return mc;
  };
  // P = exp2(c (s - m)) in place, the row sums and the outputs rescaled.
  auto softmax = [&](f32x16& s) {
    float mx = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float m_new = fmaxf(m_run, mx);
    const float mc = shift(m_new);
    const float alpha = __builtin_amdgcn_exp2f(mc_run - mc);
    m_run = m_new;
    mc_run = mc;
    float sum = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = __builtin_amdgcn_exp2f(fmaf(s[r], c, -mc));
      sum += s[r];
    }
    l_run = l_run * alpha + sum;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      o0[r] *= alpha;
      o1[r] *= alpha;
    }
  };
  if (wave <= qt) {
    load_k(k_row(wave));
    load_v(wave);
    f32x16 s = scores();
    load_k(k_row(min(wave + kSplit, qt)));
    int j = wave;
    for (; j + kSplit <= qt; j += kSplit) {
      // The next block's score products with this block's softmax between
      // them, in the order of its dependences: the maximum after products
      // 0-6, the half-wave exchange after 7, the new shift after 13, then one
      // exponential and one rescaled output register pair per product.
      const float* row = k_row(min(j + 2 * kSplit, qt));
      f32x16 s_next;
#pragma unroll
      for (int r = 0; r < 16; ++r) s_next[r] = 0.0f;
      float mx = fmaxf(s[0], s[1]), other = 0.0f, alpha = 0.0f, mc = 0.0f, sum = 0.0f;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = 0; n < 32; ++n) {
        s_next = mfma32x2(kf[n / 4][n % 4], q[n / 4][n % 4], s_next);
        if (n < 7) mx = fmaxf(fmaxf(mx, s[2 * n + 2]), s[2 * n + 3]);
        if (n == 7) other = __shfl_xor(mx, 32);
        if (n == 13) {
          const float m_new = fmaxf(m_run, fmaxf(mx, other));
          mc = shift(m_new);
          alpha = __builtin_amdgcn_exp2f(mc_run - mc);
          m_run = m_new;
          mc_run = mc;
        }
        if (n >= 14 && n < 30) {
          const int r = n - 14;
          s[r] = __builtin_amdgcn_exp2f(fmaf(s[r], c, -mc));
          sum += s[r];
          o0[r] *= alpha;
          o1[r] *= alpha;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      l_run = l_run * alpha + sum;
      load_k(row);
      __builtin_amdgcn_sched_barrier(0);
      // The output products, each V row pair refilled once it has been used.
      if ((j + kSplit + 1) * kKeys <= S) {
        const float* first = vbase + (int64_t)((j + kSplit) * kKeys + 4 * half) * p.v_ss;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          o0 = mfma32x2(vf[r][0], s[r], o0);
          o1 = mfma32x2(vf[r][1], s[r], o1);
          vf[r] = *reinterpret_cast<const f32x2*>(first + (8 * (r / 4) + r % 4) * p.v_ss);
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          o0 = mfma32x2(vf[r][0], s[r], o0);
          o1 = mfma32x2(vf[r][1], s[r], o1);
        }
        load_v(j + kSplit);
      }
      s = s_next;
    }
    if (j == qt) {  // the diagonal block: keys past the query
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (8 * (r / 4) + 4 * half + r % 4 > l32) s[r] = -INFINITY;
    }
    softmax(s);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      o0 = mfma32x2(vf[r][0], s[r], o0);
      o1 = mfma32x2(vf[r][1], s[r], o1);
    }
  }

  // Register r of o0 / o1 is dim 2 i / 2 i + 1 with i = 8 (r / 4) + 4 half + r % 4.
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    float* dst = &o_lds[wave][l32][16 * g + 8 * half];
    *reinterpret_cast<f32x4*>(dst) = f32x4{o0[4 * g], o1[4 * g], o0[4 * g + 1], o1[4 * g + 1]};
    *reinterpret_cast<f32x4*>(dst + 4) = f32x4{o0[4 * g + 2], o1[4 * g + 2], o0[4 * g + 3], o1[4 * g + 3]};
  }
  l_run += __shfl_xor(l_run, 32);
  if (half == 0) {
    m_lds[wave][l32] = mc_run;
    l_lds[wave][l32] = l_run;
  }
  __syncthreads();

  // Merge: eight threads per query, 8 dims each.  A wave without a block, or
  // with no key above -inf, has the lowest shift, sum 0 and output 0.
  const int row = tid >> 3;
  const int d0 = (tid & 7) * 8;
  if (qt * kQ + row >= S) return;
  float m_all = m_lds[0][row];  // shifts c m
#pragma unroll
  for (int w = 1; w < kSplit; ++w) m_all = fmaxf(m_all, m_lds[w][row]);
  float l_all = 0.0f;
  f32x4 lo = {0.0f, 0.0f, 0.0f, 0.0f}, hi = lo;
#pragma unroll
  for (int w = 0; w < kSplit; ++w) {
    const float scale = __builtin_amdgcn_exp2f(m_lds[w][row] - m_all);
    l_all = fmaf(l_lds[w][row], scale, l_all);
    const f32x4 a = *reinterpret_cast<const f32x4*>(&o_lds[w][row][d0]);
    const f32x4 d = *reinterpret_cast<const f32x4*>(&o_lds[w][row][d0 + 4]);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      lo[e] = fmaf(a[e], scale, lo[e]);
      hi[e] = fmaf(d[e], scale, hi[e]);
    }
  }
  const float inv = 1.0f / l_all;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    lo[e] *= inv;
    hi[e] *= inv;
  }
  float* out = p.o + b * p.o_sb + (int64_t)(qt * kQ + row) * p.o_ss + (int64_t)h * kDim + d0;
  store16(out, __builtin_bit_cast(u32x4, lo));
  store16(out + 4, __builtin_bit_cast(u32x4, hi));
}

}  // namespace

int launch_attention_f32(AttnF32Params p, int batch, hipStream_t stream) {
  // -FLT_MAX where its product with c stays finite, else a little above -FLT_MAX / c
  p.floor = p.c > 1.0f ? -FLT_MAX / p.c * 0.999999f : -FLT_MAX;
  const int64_t num_q = ceil_div(p.seq_len, kQ);
  const int64_t rows = num_q < 32768 ? num_q : 32768;  // grid y, and z beyond it
  hipLaunchKernelGGL(attn_fwd_f32_kernel,
                     dim3((unsigned)(batch * p.heads), (unsigned)rows, (unsigned)ceil_div(num_q, rows)),
                     dim3(kSplit * 64), 0, stream, p, (int)num_q);
  return check_hip(hipGetLastError(), "fp32 attention launch");
}

}  // namespace sah
