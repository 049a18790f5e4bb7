// (c) Fused Landau-Lifshitz right-hand side and (d) the batched vector
// operations of the RKSUITE 'M' stepper.
//
// LL right-hand side, per cell and state, in FP64 (demag term FP32):
//   reference dmdt_fct and helpers, LandauLifshitzEquationSolver.f90:220-273,
//   exchange :440-474 (Laplacian with the Neumann rows of :1194-1522),
//   external field :485-514, anisotropy :523-548, demag scaling :749-754.
// All effective fields are kept negated as in the reference; the API's alpha
// is alpha_LL * gamma.
//
// Vector operations: one generic kernel forms linear combinations of state
// vectors (stage arguments, interpolants, copies) and, in the same pass,
// the weighted max-norms / inner products the step control needs
// (RKSuitef90.f90 step :1790-1874, stepa :1876-1955, stepb :1957-1976,
// step_integrate :1262-1270, stiff :2047-2357).  Reductions are two-pass
// (per-block partials, then a fixed-order combine), so sums are deterministic.

#include <hip/hip_bf16.h>

#include <algorithm>
#include <cfloat>
#include <type_traits>

#include "llg_cell.h"
#include "matvec_rows.h"
#include "mt_common.h"
#include "mt_kernels.h"

namespace mt {

namespace {

__device__ inline uint16_t bf16_bits(float v) {
  __hip_bfloat16 h = __float2bfloat16(v);
  return *reinterpret_cast<uint16_t*>(&h);
}
__device__ inline float bf16_value(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// One thread per (cell, state).  The grid is 1-D with a multiple of 8 blocks;
// block b runs on XCD b % 8, and XCD x takes the contiguous x-th eighth of the
// (state, cell block) range, so the exchange stencil's neighbour rows and
// planes are read through the L2 that already holds them.  INL: descriptors
// by value (inl) instead of from descs.  NEXT: also the next stage argument.
template <bool INL, bool NEXT>
__global__ void __launch_bounds__(256) llg_kernel(const LlgGrid g, const LlgDesc* __restrict__ descs,
                                                  LlgDescsInline inl, int cell_blocks, int nstates,
                                                  const StageDesc* __restrict__ nexts, StageDescsInline inext,
                                                  PackSpec pack) {
  const int total = cell_blocks * nstates;
  const int per_xcd = (int)(gridDim.x / 8);
  const int w = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
  if (w >= total) return;
  const int st = w / cell_blocks;
  const LlgDesc& D = INL ? inl.d[st] : descs[st];
  const int i = (w % cell_blocks) * blockDim.x + threadIdx.x;
  if (i >= g.n) return;
  // every read of the cell before the first sum waits for one
  const StageDesc& N = INL ? inext.d[st] : nexts[st];
  StageReads nr;
  if (NEXT) nr = stage_reads(N, D, g.n, i);
  const CellReads r = cell_reads(g, D, i);
  constexpr int kAhead = 4;  // partial sums read at once (four of the lattice product, two to eight of the GEMM's)
  float part[kAhead][3];
  const bool sums = !D.hpart64;
#pragma unroll
  for (int k = 0; k < kAhead; ++k)
    if (sums && k < D.nsplit) {
#pragma unroll
      for (int c = 0; c < 3; ++c) part[k][c] = D.hpart[(int64_t)k * D.split_stride + (int64_t)c * g.n + i];
    }
  double dm[3];
  llg_cell(
      g, D, i, r,
      [&](int c) {
        float s = 0.0f;
#pragma unroll
        for (int k = 0; k < kAhead; ++k)
          if (k < D.nsplit) s += part[k][c];
        for (int k = kAhead; k < D.nsplit; ++k) s += D.hpart[(int64_t)k * D.split_stride + (int64_t)c * g.n + i];
        if (D.sum_out) D.sum_out[(int64_t)c * g.n + i] = s;
        return s;
      },
      dm);
  if (NEXT) next_stage_cell(N, D, g.n, i, nr, dm, pack, st);
}

// The FP32 dense path's demag rows and LL right-hand side in one launch:
// block = RB receiver rows of S states, from s0 on (the sums of matvec_rows_f32),
// then one thread per row and state evaluates llg_cell with them (NEXT: and the
// next stage argument of the cell).
//
// AHEAD (one state): waves 0-3 sum the rows; wave 4 reads what the cells'
// right-hand sides need meanwhile and evaluates them after the rows' two
// barriers (44 x 40 x 1: 16.8 us a launch, 17.7 with the reads after the rows).
// With more states to a block its registers are worth more as waves in flight (2
// states, 44 x 40 x 1: 23.3 us with wave 4, 19.5 without; 8 states, 30 x 30 x 2:
// 53 and 38).
template <int S>
constexpr bool kAheadWave = S == 1;
template <int S>
constexpr int kDemagLlgThreads = kRowThreads + (kAheadWave<S> ? 64 : 0);

template <bool INL, bool VEC4, int RB, int S, bool ONE, bool NEXT>
__global__ void __launch_bounds__(kDemagLlgThreads<S>) demag_llg_f32_kernel(
    const float* __restrict__ K, const LlgGrid g, const LlgDesc* __restrict__ descs, LlgDescsInline inl,
    const float* __restrict__ m32, int64_t m_stride, int s0, int nstates, int groups,
    const StageDesc* __restrict__ nexts, StageDescsInline inext, PackSpec pack) {
  static_assert(RB * S <= 64, "a lane per cell");
  int rows = blockIdx.x, group = 0;
  if (!ONE) matvec_block(blockIdx.x, groups, rows, group);
  const int sb = s0 + group * S;
  const int i0 = rows * RB;
  if (i0 >= g.n) return;
  __shared__ float red[4][RB * S * 3];
  __shared__ float sums[RB * S * 3];
  constexpr bool AHEAD = kAheadWave<S>;
  constexpr int first = AHEAD ? kRowThreads : 0;  // thread of the first cell
  if (!AHEAD || __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) < kRowThreads / 64) {  // uniform: barriers inside
    matvec_rows_f32<RB, VEC4, S, ONE>(K, g.n, m32 + sb * m_stride, m_stride, nstates - sb, i0, red, sums);
    if (AHEAD) return;
  }
  const int r = threadIdx.x % RB, s = ((int)threadIdx.x - first) / RB;
  if (!AHEAD && s >= S) return;
  const bool active = s < S && sb + s < nstates && i0 + r < g.n;
  const int i = active ? i0 + r : i0, st = active ? sb + s : sb;
  const LlgDesc& D = INL ? inl.d[st] : descs[st];
  const StageDesc& N = INL ? inext.d[st] : nexts[st];
  StageReads nr;
  if (NEXT) nr = stage_reads(N, D, g.n, i);
  const CellReads cr = cell_reads(g, D, i);
  if (AHEAD) {
    __syncthreads();
    __syncthreads();
  }
  if (!active) return;
  // one partial-sum slot: S = 0 + row sum, as the LL kernel forms it
  double dm[3];
  llg_cell(
      g, D, i, cr,
      [&](int c) {
        float v = 0.0f;
        v += sums[(s * RB + r) * 3 + c];
        return v;
      },
      dm);
  if (NEXT) next_stage_cell(N, D, g.n, i, nr, dm, pack, st);
}

// Stage argument + FP32 demag rows + LL right-hand side (launch_stage_demag_llg_f32).
// Block = RB receiver rows of state blockIdx.y.  The whole stage vector goes to
// LDS (3n FP64, then its FP32 rounding); each element sums bconst, bcoef*base
// and the terms in the vector kernel's order, all operands of three elements
// loaded before their sums.
// Wave 4 reads the next stage's operands meanwhile (as in demag_llg_f32_kernel).
template <bool VEC4, int RB, bool NEXT>
__global__ void __launch_bounds__(kRowThreads + 64) stage_demag_llg_f32_kernel(const float* __restrict__ K,
                                                                               const LlgGrid g, StageDescsInline sd,
                                                                               LlgDescsInline inl,
                                                                               StageDescsInline inext, PackSpec pack) {
  extern __shared__ double stage_lds[];
  const int n = g.n, n3 = 3 * n;
  const int s = blockIdx.y;
  const int i0 = blockIdx.x * RB;
  double* m64 = stage_lds;
  float* m32 = reinterpret_cast<float*>(stage_lds + n3);
  __shared__ float red[4][RB * 3];
  __shared__ float sums[RB * 3];
  if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) < kRowThreads / 64) {  // uniform: both sides hold barriers
    const StageDesc& S = sd.d[s];
    const int nt = S.nterm;
    constexpr int E = 3;  // elements of a thread whose operands are read at once
    for (int e0 = threadIdx.x; e0 < n3; e0 += E * kRowThreads) {
      double x[kMaxTerms][E], b[E];
      int at[E];
#pragma unroll
      for (int q = 0; q < E; ++q) at[q] = std::min(e0 + q * kRowThreads, n3 - 1);
      if (S.base) {
#pragma unroll
        for (int q = 0; q < E; ++q) b[q] = S.base[at[q]];
      }
#pragma unroll
      for (int k = 0; k < kMaxTerms; ++k)
        if (k < nt) {
#pragma unroll
          for (int q = 0; q < E; ++q) x[k][q] = S.src[k][at[q]];
        }
      double v[E];
#pragma unroll
      for (int q = 0; q < E; ++q) v[q] = S.bconst;
      if (S.base) {
#pragma unroll
        for (int q = 0; q < E; ++q) v[q] += S.bcoef * b[q];
      }
#pragma unroll
      for (int k = 0; k < kMaxTerms; ++k)
        if (k < nt) {
#pragma unroll
          for (int q = 0; q < E; ++q) v[q] += S.coef[k] * x[k][q];
        }
#pragma unroll
      for (int q = 0; q < E; ++q) {
        v[q] = S.post_scale * v[q];
        m64[at[q]] = v[q];  // past the end: the last element's value once more
        m32[at[q]] = (float)v[q];
      }
    }
    __syncthreads();
    if (threadIdx.x < 3 * RB) {  // this block's cells of the stage argument
      const int c = threadIdx.x / RB, i = i0 + threadIdx.x % RB;
      if (i < n) S.dst[(int64_t)c * n + i] = m64[c * n + i];
    }
    matvec_rows_f32<RB, VEC4, 1>(K, n, m32, 0, 1, i0, red, sums);
    return;
  }
  const int r = threadIdx.x - kRowThreads;
  const bool active = r < RB && i0 + r < n;
  const int i = active ? i0 + r : i0;
  LlgDesc D = inl.d[s];
  D.m = m64;  // the stage argument from LDS (other blocks write its global copy)
  StageReads nr;
  if (NEXT) nr = stage_reads(inext.d[s], D, n, i);
  __syncthreads();
  const CellReads cr = cell_reads(g, D, i);
  __syncthreads();
  __syncthreads();
  if (!active) return;
  double dm[3];
  llg_cell(
      g, D, i, cr,
      [&](int c) {
        float v = 0.0f;
        v += sums[r * 3 + c];
        return v;
      },
      dm);
  if (NEXT) next_stage_cell(inext.d[s], D, n, i, nr, dm, pack, s);
}

__device__ inline double nan_to_inf(double v) { return isnan(v) ? INFINITY : v; }

// Generic vector op.  A block covers 2048 consecutive elements of one state;
// thread t of T handles elements t + T q (q < E), so every load and store of the
// combination and the reductions is coalesced.  Per element the arithmetic (and
// its order) is that of the scalar form
//   v = post_scale * (bconst + bcoef*base + sum_k coef[k]*src[k]).
// The BF16 pack needs eight consecutive elements per 16-byte store and goes
// through LDS.
// T, E = 256, 8: enough blocks to fill the chip.  Each operand vector is loaded
// for all eight elements before any of them is used: a wave keeps eight
// 512-byte loads in flight per operand instead of waiting on one at a time.
// T, E = 1024, 2: few blocks, whose time is their round trips to memory.  All
// operands of a combination (a reduction) are loaded before the first is used.
template <int T, int E>
__device__ __forceinline__ void load_e(const double* p, int e0, int n3, double (&x)[E]) {
#pragma unroll
  for (int q = 0; q < E; ++q) {
    const int e = e0 + T * q;
    x[q] = e < n3 ? p[e] : 0.0;
  }
}

// acc[q] += coef(k) * ptr(k)[e_q] for k = 0 .. cnt-1, in k order, cnt <= MOST.
// E = 8: operand k+1's loads are issued before operand k is accumulated, so two
// operands' loads are in flight; the last iteration reloads its own operand
// (cached) to keep the loop body free of branches, so the wait before each
// accumulation leaves exactly the next operand's eight loads outstanding.
template <int T, int E, int MOST, typename PF, typename CF>
__device__ __forceinline__ void accumulate(double (&acc)[E], int cnt, PF ptr, CF coef, int e0, int n3) {
  if (cnt <= 0) return;
  if constexpr (E <= 2) {
    double x[MOST][E];
#pragma unroll
    for (int k = 0; k < MOST; ++k)
      if (k < cnt) load_e<T>(ptr(k), e0, n3, x[k]);
#pragma unroll
    for (int k = 0; k < MOST; ++k)
      if (k < cnt) {
        const double c = coef(k);
#pragma unroll
        for (int q = 0; q < E; ++q) acc[q] += c * x[k][q];
      }
  } else {
    double x[E], y[E];
    load_e<T>(ptr(0), e0, n3, x);
    for (int k = 0; k < cnt; ++k) {
      load_e<T>(ptr(k + 1 < cnt ? k + 1 : k), e0, n3, y);
      const double c = coef(k);
#pragma unroll
      for (int q = 0; q < E; ++q) acc[q] += c * x[q];
#pragma unroll
      for (int q = 0; q < E; ++q) x[q] = y[q];
    }
  }
}

// INL: descriptors by value (inl) instead of from descs.  A block's reduction
// goes to the host (lines), or to partials; with one block per state it is the
// result (written to results).
template <bool INL, int T, int E>
__global__ void __launch_bounds__(T) vec_kernel(const VecDesc* __restrict__ descs, VecDescsInline inl, int n, int n3,
                                                int blocks_per_state, double* __restrict__ partials,
                                                double* __restrict__ results, ResultLines lines, PackSpec pack) {
  static_assert(T * E == 2048, "a block's elements");
  const VecDesc& D = INL ? inl.d[blockIdx.y] : descs[blockIdx.y];
  const int t0 = blockIdx.x * 2048;
  const int e0 = t0 + threadIdx.x;
  double r0 = 0.0, r1 = 0.0, r2 = 0.0, r3 = 0.0;
  const int kind = D.rkind;
  const bool do_pack = D.pack_col >= 0 && pack.mode != kPackNone && D.dst;
  __shared__ float tile[2048];
  bool ok[E];
#pragma unroll
  for (int q = 0; q < E; ++q) ok[q] = e0 + T * q < n3;
  double v[E], x[E];
#pragma unroll
  for (int q = 0; q < E; ++q) v[q] = 0.0;
  if (D.dst) {
#pragma unroll
    for (int q = 0; q < E; ++q) v[q] = D.bconst;
    // base first, then the terms in order
    const int nb = D.base ? 1 : 0;
    accumulate<T, E, kMaxTerms + 1>(
        v, nb + D.nterm, [&](int k) { return k < nb ? D.base : D.src[k - nb]; },
        [&](int k) { return k < nb ? D.bcoef : D.coef[k - nb]; }, e0, n3);
    const double ps = D.post_scale;
#pragma unroll
    for (int q = 0; q < E; ++q) {
      v[q] = ps * v[q];
      if (ok[q]) D.dst[e0 + T * q] = v[q];
    }
  }
  if (do_pack) {
    if (pack.mode == kPackF32) {
#pragma unroll
      for (int q = 0; q < E; ++q)
        if (ok[q]) pack.f32[(int64_t)D.pack_col * pack.col_stride + e0 + T * q] = (float)v[q];
    } else if (pack.mode == kPackLattice) {
      bool bad = false;
#pragma unroll
      for (int q = 0; q < E; ++q)
        if (ok[q]) {
          const int e = e0 + T * q, c = e / n;
          const float f = (float)v[q];
          pack.f32[lattice_state_offset(n, (int)pack.col_stride, D.pack_col, c, e - c * n)] = f;
          bad |= !(fabsf(f) <= FLT_MAX);
        }
      if (bad) *pack.nonfinite = 1;
    } else if (pack.mode == kPackF32Frag) {
#pragma unroll
      for (int q = 0; q < E; ++q)
        if (ok[q]) {
          const int e = e0 + T * q, c = e / n, j = e - c * n;
          *reinterpret_cast<float*>(pack.bf16 + f32_frag_offset(D.pack_col, c, j)) = (float)v[q];
        }
    } else {
      bool bad = false;
#pragma unroll
      for (int q = 0; q < E; ++q) {
        const float f = (float)v[q];
        tile[threadIdx.x + T * q] = f;
        bad |= !(fabsf(f) <= kBf16Max);
      }
      if (bad && pack.nonfinite) *pack.nonfinite = 1;
    }
  }
  switch (kind) {
    case kRedNone:
      break;
    case kRedStepB:    // max |sum c_k s_k| / max(0.5(|y|+|ynew|), thresh)
    case kRedFinal: {  // errest = scale * sum c_k s_k; w = max(0.5(|y|+|ynew|), thresh)
      double s[E], a[E];
#pragma unroll
      for (int q = 0; q < E; ++q) s[q] = 0.0;
      if constexpr (E <= 2) {
        load_e<T>(D.ra, e0, n3, a);
        load_e<T>(D.rb, e0, n3, x);
      }
      accumulate<T, E, 8>(
          s, D.rn, [&](int k) { return D.rsrc[k]; }, [&](int k) { return D.rcoef[k]; }, e0, n3);
      if constexpr (E > 2) {
        load_e<T>(D.ra, e0, n3, a);
        load_e<T>(D.rb, e0, n3, x);
      }
      const double th = D.thresh, sc = D.rscale;
#pragma unroll
      for (int q = 0; q < E; ++q) {
        if (!ok[q]) continue;
        const double w = fmax(0.5 * (fabs(a[q]) + fabs(x[q])), th);
        if (kind == kRedStepB) {
          r0 = fmax(r0, nan_to_inf(fabs(s[q]) / w));
        } else {
          const double sv = sc * s[q];
          const int e = e0 + T * q;
          if (D.rd) D.rd[e] = sv;
          if (D.rw) D.rw[e] = w;
          r0 = fmax(r0, nan_to_inf(fabs(sv / w)));
        }
      }
      break;
    }
    case kRedStepA: {  // w = max(w, |ynew|); max |y|/w, |ynew|/w, |ynew-y|/w, |f-yp|/w
      double ya[E], yn[E], wo[E], fc[E];
      load_e<T>(D.ra, e0, n3, ya);
      load_e<T>(D.rb, e0, n3, yn);
      load_e<T>(D.rw, e0, n3, wo);
      load_e<T>(D.rc, e0, n3, fc);
      load_e<T>(D.rd, e0, n3, x);
#pragma unroll
      for (int q = 0; q < E; ++q) {
        if (!ok[q]) continue;
        const double w = fmax(wo[q], fabs(yn[q]));
        D.rw[e0 + T * q] = w;
        r0 = fmax(r0, nan_to_inf(fabs(ya[q]) / w));
        r1 = fmax(r1, nan_to_inf(fabs(yn[q]) / w));
        r2 = fmax(r2, nan_to_inf(fabs(yn[q] - ya[q]) / w));
        r3 = fmax(r3, nan_to_inf(fabs(fc[q] - x[q]) / w));
      }
      break;
    }
    case kRedYpNorm: {  // w = max(|y|, thresh); max over y != 0 of |yp|/w
      double ya[E];
      load_e<T>(D.ra, e0, n3, ya);
      load_e<T>(D.rb, e0, n3, x);
#pragma unroll
      for (int q = 0; q < E; ++q) {
        if (!ok[q]) continue;
        const double w = fmax(fabs(ya[q]), D.thresh);
        D.rw[e0 + T * q] = w;
        if (ya[q] != 0.0) r0 = fmax(r0, nan_to_inf(fabs(x[q]) / w));
      }
      break;
    }
    case kRedWeightsAvg: {  // w = max(0.5(|a|+|b|), thresh)
      double a[E];
      load_e<T>(D.ra, e0, n3, a);
      load_e<T>(D.rb, e0, n3, x);
#pragma unroll
      for (int q = 0; q < E; ++q)
        if (ok[q]) D.rw[e0 + T * q] = fmax(0.5 * (fabs(a[q]) + fabs(x[q])), D.thresh);
      break;
    }
    case kRedWdot: {  // sums of (p/w)(q/w) for up to three pairs (rsrc[2k], rsrc[2k+1])
      double w[E], p[E];
      load_e<T>(D.rw, e0, n3, w);
      for (int k = 0; k < D.rn && k < 3; ++k) {
        load_e<T>(D.rsrc[2 * k], e0, n3, p);
        load_e<T>(D.rsrc[2 * k + 1], e0, n3, x);
        double r = 0.0;
#pragma unroll
        for (int q = 0; q < E; ++q)
          if (ok[q]) r += (p[q] / w[q]) * (x[q] / w[q]);
        if (k == 0) r0 = r;
        else if (k == 1) r1 = r;
        else r2 = r;
      }
      break;
    }
    case kRedMaxDiff: {
      double a[E];
      load_e<T>(D.ra, e0, n3, a);
      load_e<T>(D.rb, e0, n3, x);
#pragma unroll
      for (int q = 0; q < E; ++q)
        if (ok[q]) r0 = fmax(r0, nan_to_inf(fabs(a[q] - x[q])));
      break;
    }
    default:
      break;
  }
  if (do_pack && pack.mode == kPackBf16) {
    __syncthreads();
    const int l0 = threadIdx.x * 8;  // eight consecutive elements of this block's tile
    const int p0 = t0 + l0;
    if (l0 < 2048 && p0 < n3) {
      if ((n & 7) == 0 && p0 + 8 <= n3) {
        const int c = p0 / n, j0 = p0 - c * n;
        uint32_t hw[4], lw[4];
        for (int q = 0; q < 4; ++q) {
          float f0 = tile[l0 + 2 * q], f1 = tile[l0 + 2 * q + 1];
          uint16_t h0 = bf16_bits(f0), h1 = bf16_bits(f1);
          uint16_t g0 = bf16_bits(f0 - bf16_value(h0)), g1 = bf16_bits(f1 - bf16_value(h1));
          hw[q] = h0 | ((uint32_t)h1 << 16);
          lw[q] = g0 | ((uint32_t)g1 << 16);
        }
        int J = j0 / kTileK, half = (j0 % kTileK) / 8;
        int lane = (D.pack_col & 31) + 32 * half;
        int sb = D.pack_col / 32;
        int64_t frag = (((int64_t)J * 3 + c) * 2 + sb) * 2;
        uint4* p = reinterpret_cast<uint4*>(pack.bf16 + frag * kFragBytes + lane * 16);
        p[0] = make_uint4(hw[0], hw[1], hw[2], hw[3]);
        p[kFragBytes / 16] = make_uint4(lw[0], lw[1], lw[2], lw[3]);
      } else {
        for (int q = 0; q < 8 && p0 + q < n3; ++q) {
          int e = p0 + q;
          int c = e / n, j = e - c * n;
          float f = tile[l0 + q];
          uint16_t hi = bf16_bits(f);
          uint16_t lo = bf16_bits(f - bf16_value(hi));
          int J = j / kTileK, half = (j % kTileK) / 8;
          int lane = (D.pack_col & 31) + 32 * half;
          int sb = D.pack_col / 32;
          int64_t frag = (((int64_t)J * 3 + c) * 2 + sb) * 2;
          uint16_t* p = reinterpret_cast<uint16_t*>(pack.bf16 + frag * kFragBytes + lane * 16) + (j % 8);
          p[0] = hi;
          p[kFragBytes / 2] = lo;
        }
      }
    }
  }
  if (kind == kRedNone || kind == kRedWeightsAvg) return;
  const bool is_sum = kind == kRedWdot;
  // block reduction of four values
  __shared__ double red[T / 64][4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const double rv[4] = {r0, r1, r2, r3};
  for (int k = 0; k < 4; ++k) {
    double x = rv[k];
    for (int off = 32; off > 0; off >>= 1) {
      double o = __shfl_xor(x, off, 64);
      x = is_sum ? x + o : fmax(x, o);
    }
    if (lane == 0) red[wave][k] = x;
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    int k = threadIdx.x;
    double x = red[0][k];
    for (int w = 1; w < T / 64; ++w) x = is_sum ? x + red[w][k] : fmax(x, red[w][k]);
    if (lines.base) {
      ResultLine* l = lines.base + (int64_t)D.rslot * lines.stride + blockIdx.x;
      l->v[k] = x;
      __threadfence_system();  // the four lanes' values before the number
      if (k == 0) __hip_atomic_store(&l->seq, lines.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    } else if (blocks_per_state == 1 && results) results[D.rslot * 4 + k] = x;
    else partials[((int64_t)blockIdx.y * blocks_per_state + blockIdx.x) * 4 + k] = x;
  }
}

// One thread per (state, value): fixed-order combine of the block partials.
template <bool INL>
__global__ void finalize_kernel(const VecDesc* __restrict__ descs, VecDescsInline inl, int nstates,
                                int blocks_per_state, const double* __restrict__ partials,
                                double* __restrict__ results) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nstates * 4) return;
  int s = t / 4, k = t % 4;
  const VecDesc& D = INL ? inl.d[s] : descs[s];
  int kind = D.rkind;
  // a descriptor without a reduction leaves its slot alone: a result written
  // by an earlier launch may still be waiting to be read
  if (kind == kRedNone || kind == kRedWeightsAvg) return;
  bool is_sum = kind == kRedWdot;
  double x = partials[((int64_t)s * blocks_per_state) * 4 + k];
  for (int b = 1; b < blocks_per_state; ++b) {
    double o = partials[((int64_t)s * blocks_per_state + b) * 4 + k];
    x = is_sum ? x + o : fmax(x, o);
  }
  results[D.rslot * 4 + k] = x;
}

}  // namespace

// kernel arguments are limited to 4 KiB
static_assert(sizeof(VecDescsInline) + 256 <= 4096, "vector kernel arguments exceed 4 KiB");
static_assert(sizeof(LlgDescsInline) + sizeof(StageDescsInline) + sizeof(LlgGrid) + 256 <= 4096,
              "LL kernel arguments exceed 4 KiB");

namespace {
StageDescsInline inline_next(const NextStage& next, int nstates) {
  StageDescsInline d{};
  if (next.h_descs)
    for (int s = 0; s < nstates; ++s) d.d[s] = next.h_descs[s];
  return d;
}

template <bool INL>
int launch_llg_t(const LlgGrid& g, const LlgDesc* descs, const LlgDescsInline& inl, int nstates,
                 const NextStage& next, hipStream_t stream) {
  const int cell_blocks = (g.n + 255) / 256;
  const int64_t total = (int64_t)cell_blocks * nstates;
  const int64_t blocks = (total + 7) / 8 * 8;
  if (blocks > INT32_MAX) {
    set_error("LL kernel: too many cells x states for one launch");
    return kErrArg;
  }
  const StageDescsInline nx = inline_next(next, INL ? nstates : 0);
  if (next.on())
    hipLaunchKernelGGL((llg_kernel<INL, true>), dim3((unsigned)blocks), dim3(256), 0, stream, g, descs, inl,
                       cell_blocks, nstates, next.d_descs, nx, next.pack);
  else
    hipLaunchKernelGGL((llg_kernel<INL, false>), dim3((unsigned)blocks), dim3(256), 0, stream, g, descs, inl,
                       cell_blocks, nstates, next.d_descs, nx, next.pack);
  MT_HIP(hipGetLastError());
  return kOk;
}

// blocks up to which the vector kernel takes wide blocks: one to a CU
constexpr int kVecWideBlocks = 256;

template <bool INL>
int launch_vec_t(const VecDesc* descs, const VecDescsInline& inl, int nstates, int n, double* partials,
                 double* results, const PackSpec& pack, bool reduce, hipStream_t stream, const ResultLines& lines) {
  int n3 = 3 * n;
  int bps = vec_blocks_per_state(n3);
  dim3 grid((unsigned)bps, (unsigned)nstates);
  if ((int64_t)bps * nstates <= kVecWideBlocks)
    hipLaunchKernelGGL((vec_kernel<INL, 1024, 2>), grid, dim3(1024), 0, stream, descs, inl, n, n3, bps, partials,
                       results, lines, pack);
  else
    hipLaunchKernelGGL((vec_kernel<INL, 256, 8>), grid, dim3(256), 0, stream, descs, inl, n, n3, bps, partials, results,
                       lines, pack);
  MT_HIP(hipGetLastError());
  if (reduce && bps > 1 && !lines.base) {
    int t = nstates * 4;
    hipLaunchKernelGGL(finalize_kernel<INL>, dim3((unsigned)((t + 127) / 128)), dim3(128), 0, stream, descs, inl,
                       nstates, bps, partials, results);
    MT_HIP(hipGetLastError());
  }
  return kOk;
}
}  // namespace

int launch_llg(const LlgGrid& g, const LlgDesc* d_descs, int nstates, hipStream_t stream, const NextStage& next) {
  return launch_llg_t<false>(g, d_descs, LlgDescsInline{}, nstates, next, stream);
}

int launch_llg_inline(const LlgGrid& g, const LlgDesc* h_descs, int nstates, hipStream_t stream,
                      const NextStage& next) {
  if (nstates < 1 || nstates > kInlineStates) {
    set_error("LL kernel: descriptors by value hold at most kInlineStates states");
    return kErrArg;
  }
  LlgDescsInline inl{};
  for (int s = 0; s < nstates; ++s) inl.d[s] = h_descs[s];
  return launch_llg_t<true>(g, nullptr, inl, nstates, next, stream);
}

namespace {
template <int S>
int launch_demag_llg_s(const float* K, const LlgGrid& g, const LlgDesc* d_descs, const LlgDescsInline& inl,
                       const float* m32, int64_t m_stride, int s0, int nstates, int groups, const NextStage& next,
                       hipStream_t stream) {
  const bool vec4 = (g.n % 4) == 0 && (m_stride % 4) == 0;
  const StageDescsInline nx = inline_next(next, d_descs ? 0 : nstates);
  auto launch = [&](auto by_value, auto v4, auto one, auto with_next) {
    constexpr int RB = matvec_block_rows(S, decltype(v4)::value);
    const dim3 grid(matvec_blocks((g.n + RB - 1) / RB, groups));
    hipLaunchKernelGGL((demag_llg_f32_kernel<decltype(by_value)::value, decltype(v4)::value, RB, S,
                                             decltype(one)::value, decltype(with_next)::value>),
                       grid, dim3(kDemagLlgThreads<S>), 0, stream, K, g, d_descs, inl, m32, m_stride, s0, nstates, groups,
                       next.d_descs, nx, next.pack);
  };
  auto go = [&](auto by_value, auto v4, auto one) {
    next.on() ? launch(by_value, v4, one, std::true_type{}) : launch(by_value, v4, one, std::false_type{});
  };
  const std::true_type yes;
  const std::false_type no;
  auto by_columns = [&](auto v4) {
    if constexpr (S == 12) return go(no, v4, yes);  // matvec_group: one group
    if constexpr (S <= kInlineStates) {
      if (!d_descs) return go(yes, v4, yes);  // by value: one group
    }
    groups == 1 ? go(no, v4, yes) : go(no, v4, no);
  };
  if constexpr (S == 12) by_columns(no);  // matvec_group: single columns
  else vec4 ? by_columns(yes) : by_columns(no);
  MT_HIP(hipGetLastError());
  return kOk;
}
}  // namespace

int launch_demag_llg_f32(const float* K, const LlgGrid& g, const LlgDesc* d_descs, const LlgDesc* h_descs,
                         const float* m32, int64_t m_stride, int nstates, hipStream_t stream, const NextStage& next) {
  LlgDescsInline inl{};
  if (!d_descs) {
    if (nstates < 1 || nstates > kInlineStates) {
      set_error("demag + LL kernel: descriptors by value hold at most kInlineStates states");
      return kErrArg;
    }
    for (int s = 0; s < nstates; ++s) inl.d[s] = h_descs[s];
  }
  for (int s0 = 0; s0 < nstates;) {
    const int S = matvec_group(nstates - s0, g.n % 4 == 0 && m_stride % 4 == 0);
    const int groups = matvec_groups(nstates - s0, S);
    int rc = kOk;
    if (S == 12) rc = launch_demag_llg_s<12>(K, g, d_descs, inl, m32, m_stride, s0, nstates, groups, next, stream);
    else if (S == 8) rc = launch_demag_llg_s<8>(K, g, d_descs, inl, m32, m_stride, s0, nstates, groups, next, stream);
    else if (S == 4) rc = launch_demag_llg_s<4>(K, g, d_descs, inl, m32, m_stride, s0, nstates, 1, next, stream);
    else if (S == 2) rc = launch_demag_llg_s<2>(K, g, d_descs, inl, m32, m_stride, s0, nstates, 1, next, stream);
    else rc = launch_demag_llg_s<1>(K, g, d_descs, inl, m32, m_stride, s0, nstates, 1, next, stream);
    if (rc) return rc;
    s0 += S * groups;
  }
  return kOk;
}

bool next_stage_in_rows_pays(int n, int nstates) {
  if (n <= kStageFusedMaxCells) return true;
  if (matvec_group(nstates, n % 4 == 0) == 12) return n <= 3500;
  return n <= 2000 && nstates >= 2 && nstates <= 4;
}

static_assert(2 * sizeof(StageDescsInline) + sizeof(LlgDescsInline) + sizeof(LlgGrid) + 256 <= 4096,
              "stage + demag + LL kernel arguments exceed 4 KiB");

int launch_stage_demag_llg_f32(const float* K, const LlgGrid& g, const VecDesc* h_pre, const LlgDesc* h_descs,
                               int nstates, hipStream_t stream, const NextStage& next) {
  if (nstates < 1 || nstates > kInlineStates || g.n < 1 || g.n > kStageFusedMaxCells) {
    set_error("stage + demag + LL kernel: 1..kInlineStates states, 1..kStageFusedMaxCells cells");
    return kErrArg;
  }
  StageDescsInline sd{};
  LlgDescsInline inl{};
  for (int s = 0; s < nstates; ++s) {
    if (!stage_of(h_pre[s], sd.d[s])) {
      set_error("stage + demag + LL kernel: a stage combination with a destination and no reduction");
      return kErrArg;
    }
    inl.d[s] = h_descs[s];
  }
  constexpr int RB = 4;
  const dim3 grid((unsigned)((g.n + RB - 1) / RB), (unsigned)nstates);
  const size_t lds = (size_t)3 * g.n * (sizeof(double) + sizeof(float));
  const StageDescsInline nx = inline_next(next, nstates);
  auto go = [&](auto v4, auto with_next) {
    hipLaunchKernelGGL((stage_demag_llg_f32_kernel<decltype(v4)::value, RB, decltype(with_next)::value>), grid,
                       dim3(kRowThreads + 64), lds, stream, K, g, sd, inl, nx, next.pack);
  };
  if (g.n % 4 == 0) next.on() ? go(std::true_type{}, std::true_type{}) : go(std::true_type{}, std::false_type{});
  else next.on() ? go(std::false_type{}, std::true_type{}) : go(std::false_type{}, std::false_type{});
  MT_HIP(hipGetLastError());
  return kOk;
}

int vec_blocks_per_state(int n3) { return (n3 + 256 * 8 - 1) / (256 * 8); }

int launch_vec(const VecDesc* d_descs, int nstates, int n, double* partials, double* results, const PackSpec& pack,
               bool reduce, hipStream_t stream, const ResultLines& lines) {
  return launch_vec_t<false>(d_descs, VecDescsInline{}, nstates, n, partials, results, pack, reduce, stream, lines);
}

int launch_vec_inline(const VecDesc* h_descs, int nstates, int n, double* partials, double* results,
                      const PackSpec& pack, bool reduce, hipStream_t stream, const ResultLines& lines) {
  if (nstates < 1 || nstates > kInlineStates) {
    set_error("vector kernel: descriptors by value hold at most kInlineStates states");
    return kErrArg;
  }
  VecDescsInline inl{};
  for (int s = 0; s < nstates; ++s) inl.d[s] = h_descs[s];
  return launch_vec_t<true>(nullptr, inl, nstates, n, partials, results, pack, reduce, stream, lines);
}

}  // namespace mt
