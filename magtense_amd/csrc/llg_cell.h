// The Landau-Lifshitz right-hand side of one cell, shared by the LL kernel and
// the kernels that fuse it (llg.hip: FP32 demag rows + LL; demag.hip: the
// split product's near-band correction + LL), so that all of them form dm/dt
// with the same arithmetic in the same order.
//
// Reference: dmdt_fct, LandauLifshitzEquationSolver.f90:220-273; exchange
// :440-474 (Laplacian with the Neumann rows of :1194-1522); external field
// :485-514; anisotropy :523-548; demag scaling :749-754.  All effective fields
// are kept negated as in the reference; the API's alpha is alpha_LL * gamma.
#pragma once

#include <cfloat>

#include "mt_common.h"
#include "mt_kernels.h"

namespace mt {

// What the right-hand side of a cell reads, apart from the demag sums.  The
// kernels issue these reads (and the next stage's, below) before anything waits
// for another: a launch of a small problem is little more than its round trips
// to memory.  (The near-band kernel reads each value where it is used: 63 registers
// and eight waves per SIMD, 88 and five with all of them in flight, 123 and 171 us a
// launch of 64 states at 256 x 64 x 2.)
struct CellReads {
  double c0[3], xm[3], xp[3], ym[3], yp[3], zm[3], zp[3];
  double jf, kf, ms64, aniso[6];  // aniso: xx xy xz yy yz zz
  float ms32;
  int kb, ke;
};

__device__ __forceinline__ CellReads cell_reads(const LlgGrid& g, const LlgDesc& D, int i) {
  CellReads r;
  const int n = g.n;
  const double* m = D.m;
#pragma unroll
  for (int c = 0; c < 3; ++c) r.c0[c] = m[(size_t)c * n + i];
  r.jf = g.jfact[i];
  r.kb = r.ke = 0;
  if (g.xs) {
    r.kb = g.xs[i];
    r.ke = g.xe[i];
  } else {
    // the neighbour indices are clamped to the cell itself at a boundary, so
    // that every load is issued before the per-row formula is selected
    const int ix = i % g.nx, iy = (i / g.nx) % g.ny, iz = i / (g.nx * g.ny);
    const int sy = g.nx, sz = g.nx * g.ny;
    const int xm = ix > 0 ? i - 1 : i, xp = ix < g.nx - 1 ? i + 1 : i;
    const int ym = iy > 0 ? i - sy : i, yp = iy < g.ny - 1 ? i + sy : i;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double* v = m + (size_t)c * n;
      r.xm[c] = v[xm]; r.xp[c] = v[xp];
      r.ym[c] = v[ym]; r.yp[c] = v[yp];
    }
    if (g.nz > 1) {
      const int zm = iz > 0 ? i - sz : i, zp = iz < g.nz - 1 ? i + sz : i;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double* v = m + (size_t)c * n;
        r.zm[c] = v[zm]; r.zp[c] = v[zp];
      }
    }
  }
  if (D.hpart64) r.ms64 = g.ms64[i];
  else r.ms32 = g.ms32[i];
  if (g.aniso) {
    r.kf = g.kfact[i];
#pragma unroll
    for (int k = 0; k < 6; ++k) r.aniso[k] = g.aniso[(size_t)i * 6 + k];
  }
  return r;
}

// LL right-hand side of cell i for the state of descriptor D, from its reads.
// hsum(c) returns the FP32 demag sum S_c = sum of the partials of (K m)_c at i
// (used unless D.hpart64 holds FP64 sums).  dm: dm/dt, which goes to D.out as
// well.
template <bool AHEAD = true, typename HS>
__device__ __forceinline__ void llg_cell(const LlgGrid& g, const LlgDesc& D, int i, const CellReads& r, HS hsum,
                                         double (&dm)[3]) {
  const int n = g.n;
  const double* m = D.m;
  double mc[3], hj[3], hm[3], hk[3];
  if constexpr (AHEAD) {
    if (g.xs) {
      // loaded operator: alpha = -2 times the row's stored entries in order
      // (updateExchangeTerms, LandauLifshitzEquationSolver.f90:440-474)
      for (int c = 0; c < 3; ++c) {
        const double* v = m + (size_t)c * n;
        mc[c] = r.c0[c];
        double sum = 0.0;
        for (int k = r.kb; k < r.ke; ++k) sum += g.xv[k] * v[g.xc[k]];
        hj[c] = (-2.0 * sum) * r.jf;
      }
    } else {
      // Laplacian with the reference's boundary rows: (-1, 1) and (1, -1)
      const int ix = i % g.nx, iy = (i / g.nx) % g.ny, iz = i / (g.nx * g.ny);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double vi = r.c0[c];
        mc[c] = vi;
        double lx = ix == 0 ? (r.xp[c] - vi) : (ix == g.nx - 1 ? (r.xm[c] - vi) : (r.xm[c] - 2.0 * vi + r.xp[c]));
        double ly = iy == 0 ? (r.yp[c] - vi) : (iy == g.ny - 1 ? (r.ym[c] - vi) : (r.ym[c] - 2.0 * vi + r.yp[c]));
        double lap = lx * g.idx2 + ly * g.idy2;
        if (g.nz > 1) {
          double lz = iz == 0 ? (r.zp[c] - vi) : (iz == g.nz - 1 ? (r.zm[c] - vi) : (r.zm[c] - 2.0 * vi + r.zp[c]));
          lap += lz * g.idz2;
        }
        hj[c] = (-2.0 * lap) * r.jf;
      }
    }
  } else {
    const int ix = i % g.nx;
    const int iy = (i / g.nx) % g.ny;
    const int iz = i / (g.nx * g.ny);
    const int sy = g.nx, sz = g.nx * g.ny;
    if (g.xs) {
      // loaded operator: alpha = -2 times the row's stored entries in order
      // (updateExchangeTerms, LandauLifshitzEquationSolver.f90:440-474)
      const int kb = g.xs[i], ke = g.xe[i];
      for (int c = 0; c < 3; ++c) {
        const double* v = m + (size_t)c * n;
        mc[c] = v[i];
        double sum = 0.0;
        for (int k = kb; k < ke; ++k) sum += g.xv[k] * v[g.xc[k]];
        hj[c] = (-2.0 * sum) * g.jfact[i];
      }
    } else {
      // Laplacian with the reference's boundary rows: (-1, 1) and (1, -1).  The
      // neighbour indices are clamped to the cell itself at a boundary, so every
      // load is issued unconditionally before the per-row formula is selected.
      const int xm = ix > 0 ? i - 1 : i, xp = ix < g.nx - 1 ? i + 1 : i;
      const int ym = iy > 0 ? i - sy : i, yp = iy < g.ny - 1 ? i + sy : i;
      const bool z3 = g.nz > 1;
      const int zm = z3 && iz > 0 ? i - sz : i, zp = z3 && iz < g.nz - 1 ? i + sz : i;
      double c0[3], cxm[3], cxp[3], cym[3], cyp[3], czm[3], czp[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double* v = m + (size_t)c * n;
        c0[c] = v[i];
        cxm[c] = v[xm]; cxp[c] = v[xp];
        cym[c] = v[ym]; cyp[c] = v[yp];
        czm[c] = v[zm]; czp[c] = v[zp];
      }
      const double jf = g.jfact[i];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double vi = c0[c];
        mc[c] = vi;
        double lx = ix == 0 ? (cxp[c] - vi) : (ix == g.nx - 1 ? (cxm[c] - vi) : (cxm[c] - 2.0 * vi + cxp[c]));
        double ly = iy == 0 ? (cyp[c] - vi) : (iy == g.ny - 1 ? (cym[c] - vi) : (cym[c] - 2.0 * vi + cyp[c]));
        double lap = lx * g.idx2 + ly * g.idy2;
        if (z3) {
          double lz = iz == 0 ? (czp[c] - vi) : (iz == g.nz - 1 ? (czm[c] - vi) : (czm[c] - 2.0 * vi + czp[c]));
          lap += lz * g.idz2;
        }
        hj[c] = (-2.0 * lap) * jf;
      }
    }
  }
  // demag: S = sum_k partial (K m); field = fl32(fl32(-S) * Ms_i)
  if (D.hpart64) {
    for (int c = 0; c < 3; ++c) hm[c] = (-D.hpart64[(int64_t)c * n + i]) * (AHEAD ? r.ms64 : g.ms64[i]);
  } else {
    for (int c = 0; c < 3; ++c) {
      const float s = hsum(c);
      if (D.sum_out) D.sum_out[(int64_t)c * n + i] = s;
      float h = (-s) * (AHEAD ? r.ms32 : g.ms32[i]);
      hm[c] = (double)h;
    }
  }
  if (g.aniso) {
    auto axes = [&](const auto& A, double f) {  // xx xy xz yy yz zz
      hk[0] = f * (A[0] * mc[0] + A[1] * mc[1] + A[2] * mc[2]);
      hk[1] = f * (A[1] * mc[0] + A[3] * mc[1] + A[4] * mc[2]);
      hk[2] = f * (A[2] * mc[0] + A[4] * mc[1] + A[5] * mc[2]);
    };
    if constexpr (AHEAD) axes(r.aniso, -2.0 * r.kf);
    else axes(g.aniso + (size_t)i * 6, -2.0 * g.kfact[i]);
  } else {
    hk[0] = hk[1] = hk[2] = 0.0;
  }
  double hh[3] = {-D.hext[0], -D.hext[1], -D.hext[2]};
  double H[3];
  for (int c = 0; c < 3; ++c) H[c] = hh[c] + hj[c] + hm[c] + hk[c];
  double cx = -1.0 * (mc[1] * H[2] - mc[2] * H[1]);
  double cy = -1.0 * (mc[2] * H[0] - mc[0] * H[2]);
  double cz = -1.0 * (mc[0] * H[1] - mc[1] * H[0]);
  double dx = mc[1] * cz - mc[2] * cy;
  double dy = mc[2] * cx - mc[0] * cz;
  double dz = mc[0] * cy - mc[1] * cx;
  dm[0] = -D.gamma * cx - D.alpha * dx;
  dm[1] = -D.gamma * cy - D.alpha * dy;
  dm[2] = -D.gamma * cz - D.alpha * dz;
  if (D.out) {
    D.out[i] = dm[0];
    D.out[n + i] = dm[1];
    D.out[2 * n + i] = dm[2];
  }
  if (D.fields) {
    double* F = D.fields;
    for (int c = 0; c < 3; ++c) {
      F[(size_t)c * n + i] = hj[c];
      F[(size_t)(3 + c) * n + i] = hh[c];
      F[(size_t)(6 + c) * n + i] = hm[c];
      F[(size_t)(9 + c) * n + i] = hk[c];
    }
  }
}

// The next stage argument at cell i, straight after its right-hand side: the
// vector kernel's combination (same order, same roundings) over the cell's
// three components, with dm/dt taken from registers, and its demag input
// packed into column col.  Only the cell's own values are read, so the launch
// that evaluates dm/dt can write the next stage's argument as long as that is
// not a vector it reads at other cells.
struct StageReads {
  double base[3], x[kMaxTerms][3];
};
__device__ __forceinline__ StageReads stage_reads(const StageDesc& S, const LlgDesc& D, int n, int i) {
  StageReads r;
  const size_t at[3] = {(size_t)i, (size_t)n + i, 2 * (size_t)n + i};
  if (S.base) {
#pragma unroll
    for (int c = 0; c < 3; ++c) r.base[c] = S.base[at[c]];
  }
#pragma unroll
  for (int k = 0; k < kMaxTerms; ++k)
    if (k < S.nterm && S.src[k] != D.out) {
#pragma unroll
      for (int c = 0; c < 3; ++c) r.x[k][c] = S.src[k][at[c]];
    }
  return r;
}
__device__ __forceinline__ void next_stage_cell(const StageDesc& S, const LlgDesc& D, int n, int i,
                                                const StageReads& r, const double (&dm)[3], const PackSpec& pack,
                                                int col) {
  const size_t at[3] = {(size_t)i, (size_t)n + i, 2 * (size_t)n + i};
  double v[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) v[c] = S.bconst;
  if (S.base) {
#pragma unroll
    for (int c = 0; c < 3; ++c) v[c] = __builtin_fma(S.bcoef, r.base[c], v[c]);
  }
#pragma unroll
  for (int k = 0; k < kMaxTerms; ++k)
    if (k < S.nterm) {
#pragma unroll
      for (int c = 0; c < 3; ++c) v[c] = __builtin_fma(S.coef[k], S.src[k] != D.out ? r.x[k][c] : dm[c], v[c]);
    }
  bool bad = false;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    v[c] = S.post_scale * v[c];
    S.dst[at[c]] = v[c];
    const float f = (float)v[c];
    if (pack.mode == kPackF32) pack.f32[(int64_t)col * pack.col_stride + (int64_t)at[c]] = f;
    else if (pack.mode == kPackLattice) pack.f32[lattice_state_offset(n, (int)pack.col_stride, col, c, i)] = f;
    else if (pack.mode == kPackF32Frag) *reinterpret_cast<float*>(pack.bf16 + f32_frag_offset(col, c, i)) = f;
    bad |= !(fabsf(f) <= FLT_MAX);
  }
  if (bad && pack.nonfinite) *pack.nonfinite = 1;
}

}  // namespace mt
