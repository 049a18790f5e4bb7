// Plain FP32 demag rows, shared by the per-state mat-vec (demag.hip) and the
// fused small-problem kernel (llg.hip), so that both form the same sums in the
// same order.
#pragma once

#include "mt_common.h"

namespace mt {

template <bool NT>
__device__ inline float4 ld4(const float* p) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  const f32x4* q = reinterpret_cast<const f32x4*>(p);
  const f32x4 v = NT ? __builtin_nontemporal_load(q) : *q;
  return make_float4(v.x, v.y, v.z, v.w);
}

// The contribution of QC columns to the three components of one row, added to
// acc: one sum over the columns from the first product on, then one addition.
// Every product and addition is written out (no contraction by the compiler),
// so that all kernels that form these sums round alike.  k4: xx, xy, yy, zz,
// k2: xz, yz of each column.
template <int QC, typename K4, typename K2>
__device__ __forceinline__ void matvec_full(const K4 (&k4)[QC], const K2 (&k2)[QC], const float (&vx)[QC], const float (&vy)[QC],
                                   const float (&vz)[QC], float (&acc)[3]) {
#pragma clang fp contract(off)
  float x = k4[0].y * vy[0], y = k4[0].z * vy[0], z = k2[0].y * vy[0];
  x = __builtin_fmaf(k4[0].x, vx[0], x);
  y = __builtin_fmaf(k4[0].y, vx[0], y);
  z = __builtin_fmaf(k2[0].x, vx[0], z);
  x = __builtin_fmaf(k2[0].x, vz[0], x);
  y = __builtin_fmaf(k2[0].y, vz[0], y);
  z = __builtin_fmaf(k4[0].w, vz[0], z);
#pragma unroll
  for (int q = 1; q < QC; ++q) {
    x = __builtin_fmaf(k4[q].x, vx[q], x);
    y = __builtin_fmaf(k4[q].y, vx[q], y);
    z = __builtin_fmaf(k2[q].x, vx[q], z);
    x = __builtin_fmaf(k4[q].y, vy[q], x);
    y = __builtin_fmaf(k4[q].z, vy[q], y);
    z = __builtin_fmaf(k2[q].y, vy[q], z);
    x = __builtin_fmaf(k2[q].x, vz[q], x);
    y = __builtin_fmaf(k2[q].y, vz[q], y);
    z = __builtin_fmaf(k4[q].w, vz[q], z);
  }
  acc[0] += x;
  acc[1] += y;
  acc[2] += z;
}
// The same where xz and yz are +-0 and the states finite: their products are
// +-0, which leaves every sum but the sign of a zero as it is, and acc, which
// starts at +0, is never -0.
template <int QC, typename K4>
__device__ __forceinline__ void matvec_flat(const K4 (&k4)[QC], const float (&vx)[QC], const float (&vy)[QC],
                                   const float (&vz)[QC], float (&acc)[3]) {
#pragma clang fp contract(off)
  float x = k4[0].y * vy[0], y = k4[0].z * vy[0], z = k4[0].w * vz[0];
  x = __builtin_fmaf(k4[0].x, vx[0], x);
  y = __builtin_fmaf(k4[0].y, vx[0], y);
#pragma unroll
  for (int q = 1; q < QC; ++q) {
    x = __builtin_fmaf(k4[q].x, vx[q], x);
    y = __builtin_fmaf(k4[q].y, vx[q], y);
    z = __builtin_fmaf(k4[q].w, vz[q], z);
    x = __builtin_fmaf(k4[q].y, vy[q], x);
    y = __builtin_fmaf(k4[q].z, vy[q], y);
  }
  acc[0] += x;
  acc[1] += y;
  acc[2] += z;
}

template <int ROR>
__device__ __forceinline__ float add_row_ror(float v) {
  const int x = __builtin_bit_cast(int, v);
  return v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(x, x, 0x120 | ROR, 0xF, 0xF, false));
}
// Sum over the 64 lanes, v + v(lane xor 32), then xor 16, 8, 4, 2, 1; every lane
// gets it.  Half and row exchanges and row rotations (once lanes xor 8 are
// equal, a rotation by 4 in a row of 16 brings the value of lane xor 4) stay
// in the vector pipe: 2 swaps and 6 additions instead of six LDS permutes.
__device__ __forceinline__ float wave_tree_sum(float v) {
  unsigned x = __builtin_bit_cast(unsigned, v);
  const auto h = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  v = __uint_as_float(h[0]) + __uint_as_float(h[1]);
  x = __builtin_bit_cast(unsigned, v);
  const auto w = __builtin_amdgcn_permlane16_swap(x, x, false, false);
  v = __uint_as_float(w[0]) + __uint_as_float(w[1]);
  v = add_row_ror<8>(v);
  v = add_row_ror<4>(v);
  v = add_row_ror<2>(v);
  return add_row_ror<1>(v);
}

constexpr int kRowThreads = 256;  // of matvec_rows_f32

// Rows i0 .. i0 + RB - 1 of (K m) for S states m + s * m_stride (x, then y, then
// z of all cells) with a block of 256 threads: every thread sums its columns
// over the six receiver-major planes, then a tree per wave and the four waves
// in order; the tensor is read once for the S states, each of which sums as it
// would alone.  On return (after a barrier) sums[(s * RB + r) * 3 + c] holds
// component c of row i0 + r; red is the block's scratch.  Two barriers, which
// further waves of the block meet by themselves.  States from `have` on
// repeat the last one.
// NT: non-temporal tensor loads, for a tensor that the launch reads once, so that
// it does not displace the state vectors from L2.
template <int RB, bool VEC4, int S, bool NT = true>
__device__ __forceinline__ void matvec_rows_f32(const float* __restrict__ K, int n, const float* __restrict__ m,
                                       int64_t m_stride, int have, int i0, float (&red)[4][RB * S * 3],
                                       float (&sums)[RB * S * 3]) {
  const size_t nn = (size_t)n * n;
  constexpr int QC = VEC4 ? 4 : 1;
  float acc[RB][S][3];
#pragma unroll
  for (int r = 0; r < RB; ++r)
#pragma unroll
    for (int s = 0; s < S; ++s) acc[r][s][0] = acc[r][s][1] = acc[r][s][2] = 0.0f;
  for (int j = threadIdx.x * QC; j < n; j += 256 * QC) {
    float x[S][QC], y[S][QC], z[S][QC];
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const float* p = m + (s < have ? s : have - 1) * m_stride + j;
      if constexpr (VEC4) {
        const float4 vx = *reinterpret_cast<const float4*>(p), vy = *reinterpret_cast<const float4*>(p + n),
                     vz = *reinterpret_cast<const float4*>(p + 2 * (size_t)n);
        x[s][0] = vx.x; x[s][1] = vx.y; x[s][2] = vx.z; x[s][3] = vx.w;
        y[s][0] = vy.x; y[s][1] = vy.y; y[s][2] = vy.z; y[s][3] = vy.w;
        z[s][0] = vz.x; z[s][1] = vz.y; z[s][2] = vz.z; z[s][3] = vz.w;
      } else {
        x[s][0] = p[0];
        y[s][0] = p[n];
        z[s][0] = p[2 * (size_t)n];
      }
    }
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      const int i = i0 + r;
      if (i >= n) break;
      const float* row = K + (size_t)i * n + j;
      float4 k4[QC];
      float2 k2[QC];
      if constexpr (VEC4) {
        const float4 kxx = ld4<NT>(row), kxy = ld4<NT>(row + nn), kxz = ld4<NT>(row + 2 * nn),
                     kyy = ld4<NT>(row + 3 * nn), kyz = ld4<NT>(row + 4 * nn), kzz = ld4<NT>(row + 5 * nn);
        k4[0] = make_float4(kxx.x, kxy.x, kyy.x, kzz.x); k2[0] = make_float2(kxz.x, kyz.x);
        k4[1] = make_float4(kxx.y, kxy.y, kyy.y, kzz.y); k2[1] = make_float2(kxz.y, kyz.y);
        k4[2] = make_float4(kxx.z, kxy.z, kyy.z, kzz.z); k2[2] = make_float2(kxz.z, kyz.z);
        k4[3] = make_float4(kxx.w, kxy.w, kyy.w, kzz.w); k2[3] = make_float2(kxz.w, kyz.w);
      } else {
        k4[0] = make_float4(row[0], row[nn], row[3 * nn], row[5 * nn]);
        k2[0] = make_float2(row[2 * nn], row[4 * nn]);
      }
#pragma unroll
      for (int s = 0; s < S; ++s) matvec_full<QC>(k4, k2, x[s], y[s], z[s], acc[r][s]);
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const float v = wave_tree_sum(acc[r][s][c]);
        if (lane == 0) red[wave][(s * RB + r) * 3 + c] = v;
      }
  __syncthreads();
  if (threadIdx.x < RB * S * 3)
    sums[threadIdx.x] = red[0][threadIdx.x] + red[1][threadIdx.x] + red[2][threadIdx.x] + red[3][threadIdx.x];
  __syncthreads();
}

// Rows and states of block b, for G state groups (G > 1): the groups of one row
// block run one after the other on one XCD (b % 8), so that the tensor rows
// come from HBM once and from that XCD's L2 for the other groups.  A row block
// past the last one has no work.
__device__ inline void matvec_block(int b, int G, int& rows, int& group) {
  const int q = b / 8;
  group = q % G;
  rows = q / G * 8 + b % 8;
}
inline unsigned matvec_blocks(int row_blocks, int G) {
  return (unsigned)(G == 1 ? row_blocks : (row_blocks + 7) / 8 * 8 * G);
}

// States per block for the next `left` states: the narrowest kernel that takes
// them in one pass, some of its states idle (90 x 70 cells: 1 / 2 / 4 / 8 states
// 0.165 / 0.171 / 0.185 / 0.255 ms a pass, all HBM).
inline int matvec_group(int left) { return left > 4 ? 8 : (left > 2 ? 4 : left); }
// Receiver rows of its blocks: four (402.7 MB tensor, one state: 2 / 4 / 8 rows
// -> 72.2 / 66.8 / 114.4 us per launch); two beside eight states, whose sums and
// values take the registers.
constexpr int matvec_block_rows(int S) { return S >= 8 ? 2 : 4; }

}  // namespace mt
