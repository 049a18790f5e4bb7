// Plain FP32 demag rows, shared by the per-state mat-vec (demag.hip) and the
// fused small-problem kernel (llg.hip), so that both form the same sums in the
// same order.
#pragma once

#include <algorithm>

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

// Sums over the 64 lanes of N values, each by v + v(lane xor 32), then xor 16,
// 8, 4, 2, 1, to dst[0 .. N-1].  The lanes that a step leaves with copies of a
// sum take the next value's instead: two registers become one at every step, in
// the vector pipe throughout.  144 values: 0.4 thousand instructions where a
// tree to every lane for each takes 1.4, and 3 LDS writes for 144 (12 states of
// 45 x 17 x 2: 29.8 us a right-hand side, 37.3 with trees; 8 of 90 x 70: 0.227 ms
// a product, 0.234).
template <int CTRL, int BANKS>
__device__ __forceinline__ float dpp_into(float old, float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, old), __builtin_bit_cast(int, v),
                                                               CTRL, 0xF, BANKS, false));
}
// a + a(lane xor BIT) where lane & BIT is 0, b + b(lane xor BIT) where it is not
template <int BIT>
__device__ __forceinline__ float fold_lanes(float a, float b, int lane) {
  if constexpr (BIT == 32 || BIT == 16) {
    const unsigned x = __float_as_uint(a), y = __float_as_uint(b);
    const auto h = BIT == 32 ? __builtin_amdgcn_permlane32_swap(x, y, false, false)
                             : __builtin_amdgcn_permlane16_swap(x, y, false, false);
    return __uint_as_float(h[0]) + __uint_as_float(h[1]);
  } else if constexpr (BIT == 4) {  // rows of 16 lanes shifted left and right by 4, into alternate banks of 4
    float o = dpp_into<0x104, 0x5>(0.0f, a);
    o = dpp_into<0x114, 0xA>(o, b);
    return (lane & 4 ? b : a) + o;
  } else {  // row rotation by 8; quad permutations
    const float keep = lane & BIT ? b : a, send = lane & BIT ? a : b;
    return keep + dpp_into<BIT == 8 ? 0x128 : (BIT == 2 ? 0x4E : 0xB1), 0xF>(0.0f, send);
  }
}
template <int TOTAL, int BIT = 32, int N>
__device__ __forceinline__ void wave_tree_sums(const float (&v)[N], int lane, float* dst) {
  constexpr int M = (N + 1) / 2;
  float o[M];
#pragma unroll
  for (int i = 0; i < M; ++i) o[i] = fold_lanes<BIT>(v[2 * i], v[2 * i + 1 < N ? 2 * i + 1 : 2 * i], lane);
  if constexpr (BIT > 1) {
    wave_tree_sums<TOTAL, BIT / 2>(o, lane, dst);
  } else {
    const int first = (int)(__brev((unsigned)lane) >> 26);  // lane bit 5 chose value bit 0, and so on
#pragma unroll
    for (int i = 0; i < M; ++i)
      if (first + 64 * i < TOTAL) dst[first + 64 * i] = o[i];
  }
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
// it does not displace the state vectors from L2.  Where the tensor fits in L2 they
// cost nothing (32 x 8 cells, one state: 8.6 us a launch either way; 32 x 32: 10.1
// either way; 44 x 40: 21.8, cached loads 22.5).
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
  float v[RB * S * 3];
#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int c = 0; c < 3; ++c) v[(s * RB + r) * 3 + c] = acc[r][s][c];
  wave_tree_sums<RB * S * 3>(v, lane, red[wave]);
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
// 0.164 / 0.170 / 0.182 / 0.227 ms a pass, HBM up to four).  With single columns
// (n % 4 != 0) a thread holds a quarter of the values, and twelve states fit in one pass,
// which reads a large tensor once for nine to twelve.  us by twelves / by eights: twelve
// states 1530 cells 38/34 a product, 38/40 a right-hand side, 2001 46/48 a product, 3465
// 122/124 a right-hand side, 6461 348/386 a product; beyond twelve states eights are as
// good or better (13 16 24 64 states, 6461 cells: 534/386 557/386 598/509 1575/1185).
inline int matvec_group(int left, bool vec4) {
  if (left > 8 && left <= 12 && !vec4) return 12;
  return left > 4 ? 8 : (left > 2 ? 4 : left);
}
// Groups of S states of one launch, the last of them partly idle: its tensor rows come
// from L2, where a launch of its own for the states left over reads them from HBM (6300
// cells, 9 / 13 / 17 / 30 states 380 / 426 / 484 / 629 -> 306 / 327 / 414 / 540 us a
// product), and a launch takes 3 us (64 cells, 9 states 20 -> 17).
inline int matvec_groups(int left, int S) { return S == 8 ? std::min((left + 7) / 8, 64) : 1; }
// Receiver rows of its blocks: a value of a state is read from L2 once per block,
// so that more rows are less traffic, until the sums take a wave's registers.
// One state, 2 / 4 rows, us a launch: 32 x 8 8.2 / 8.6, 30 x 18 12.3 / 9.4, 32 x 32
// 14.1 / 10.1, 44 x 40 29.2 / 21.8, 77 x 33 44.2 / 38.5 (a tensor of 402.7 MB 72.2 /
// 66.8, 8 rows 114.4);
// 8 states of 90 x 70: 2 / 3 rows -> 0.254 / 0.234 ms (4: 299 registers, one wave
// per SIMD).
constexpr int matvec_block_rows(int S, bool vec4) { return S >= 8 && vec4 ? 3 : 4; }

}  // namespace mt
