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

// A cell and its neighbours on the uniform grid.  The neighbour indices are clamped
// to the cell itself at a boundary, so that every load is issued before the per-row
// formula is selected.
struct Stencil {
  double c0[3], xm[3], xp[3], ym[3], yp[3], zm[3], zp[3];
};

__device__ __forceinline__ Stencil stencil_reads(const LlgGrid& g, const LlgDesc& D, int i) {
  Stencil r;
  const int n = g.n;
  const int ix = i % g.nx, iy = (i / g.nx) % g.ny, iz = i / (g.nx * g.ny);
  const int sy = g.nx, sz = g.nx * g.ny;
  const int xm = ix > 0 ? i - 1 : i, xp = ix < g.nx - 1 ? i + 1 : i;
  const int ym = iy > 0 ? i - sy : i, yp = iy < g.ny - 1 ? i + sy : i;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const double* v = D.m + (size_t)c * n;
    r.c0[c] = v[i];
    r.xm[c] = v[xm]; r.xp[c] = v[xp];
    r.ym[c] = v[ym]; r.yp[c] = v[yp];
  }
  if (g.nz > 1) {
    const int zm = iz > 0 ? i - sz : i, zp = iz < g.nz - 1 ? i + sz : i;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double* v = D.m + (size_t)c * n;
      r.zm[c] = v[zm]; r.zp[c] = v[zp];
    }
  }
  return r;
}

// The operands of a cell, apart from the demag sums, read before anything waits
// for another (and with the next stage's, below): a launch of a small problem is
// little more than its round trips to memory.
struct CellReads {
  Stencil s;  // with a loaded exchange operator only s.c0
  double jf, kf, ms64, a[6];  // a: xx xy xz yy yz zz
  float ms32;
  int kb, ke;
  __device__ __forceinline__ const Stencil& stencil() const { return s; }
  __device__ __forceinline__ double centre(int c) const { return s.c0[c]; }
  __device__ __forceinline__ int row_begin() const { return kb; }
  __device__ __forceinline__ int row_end() const { return ke; }
  __device__ __forceinline__ double jfact() const { return jf; }
  __device__ __forceinline__ float ms_f32() const { return ms32; }
  __device__ __forceinline__ double ms_f64() const { return ms64; }
  __device__ __forceinline__ double kfact() const { return kf; }
  __device__ __forceinline__ double aniso(int k) const { return a[k]; }
};

__device__ __forceinline__ CellReads cell_reads(const LlgGrid& g, const LlgDesc& D, int i) {
  CellReads r;
  r.jf = g.jfact[i];
  r.kb = r.ke = 0;
  if (g.xs) {
#pragma unroll
    for (int c = 0; c < 3; ++c) r.s.c0[c] = D.m[(size_t)c * g.n + i];
    r.kb = g.xs[i];
    r.ke = g.xe[i];
  } else {
    r.s = stencil_reads(g, D, i);
  }
  if (D.hpart64) r.ms64 = g.ms64[i];
  else r.ms32 = g.ms32[i];
  if (g.aniso) {
    r.kf = g.kfact[i];
#pragma unroll
    for (int k = 0; k < 6; ++k) r.a[k] = g.aniso[(size_t)i * 6 + k];
  }
  return r;
}

// The same operands, each read where it is used.  The near-band kernel takes them
// like this: 62 registers and eight waves per SIMD, 88 and five with all of them in
// flight, 123 and 171 us a launch of 64 states at 256 x 64 x 2.
struct CellAtUse {
  const LlgGrid& g;
  const LlgDesc& D;
  int i;
  __device__ __forceinline__ Stencil stencil() const { return stencil_reads(g, D, i); }
  __device__ __forceinline__ double centre(int c) const { return D.m[(size_t)c * g.n + i]; }
  __device__ __forceinline__ int row_begin() const { return g.xs[i]; }
  __device__ __forceinline__ int row_end() const { return g.xe[i]; }
  __device__ __forceinline__ double jfact() const { return g.jfact[i]; }
  __device__ __forceinline__ float ms_f32() const { return g.ms32[i]; }
  __device__ __forceinline__ double ms_f64() const { return g.ms64[i]; }
  __device__ __forceinline__ double kfact() const { return g.kfact[i]; }
  __device__ __forceinline__ double aniso(int k) const { return g.aniso[(size_t)i * 6 + k]; }
};

// LL right-hand side of cell i for the state of descriptor D, from its operands
// (CellReads or CellAtUse).  hsum(c) returns the FP32 demag sum S_c = sum of the
// partials of (K m)_c at i (used unless D.hpart64 holds FP64 sums).  dm: dm/dt,
// which goes to D.out as well.  Every fused operation is written out, and the
// compiler fuses none by itself: what it would choose depends on the kernel around
// the cell, and a state's bits must not.
template <typename Operands, typename HS>
__device__ __forceinline__ void llg_cell(const LlgGrid& g, const LlgDesc& D, int i, const Operands& r, HS hsum,
                                         double (&dm)[3]) {
#pragma clang fp contract(off)
  const int n = g.n;
  const double* m = D.m;
  double mc[3], hj[3], hm[3], hk[3];
  if (g.xs) {
    // loaded operator: alpha = -2 times the row's stored entries in order
    // (updateExchangeTerms, LandauLifshitzEquationSolver.f90:440-474)
    const int kb = r.row_begin(), ke = r.row_end();
    for (int c = 0; c < 3; ++c) {
      const double* v = m + (size_t)c * n;
      mc[c] = r.centre(c);
      double sum = 0.0;
      for (int k = kb; k < ke; ++k) sum = __builtin_fma(g.xv[k], v[g.xc[k]], sum);
      hj[c] = (-2.0 * sum) * r.jfact();
    }
  } else {
    // Laplacian with the reference's boundary rows: (-1, 1) and (1, -1)
    const Stencil& x = r.stencil();
    const double jf = r.jfact();
    const int ix = i % g.nx, iy = (i / g.nx) % g.ny, iz = i / (g.nx * g.ny);
    auto row = [](int k, int cells, double low, double mid, double high) {
      return k == 0 ? high - mid : (k == cells - 1 ? low - mid : __builtin_fma(-2.0, mid, low) + high);
    };
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double vi = x.c0[c];
      mc[c] = vi;
      const double lx = row(ix, g.nx, x.xm[c], vi, x.xp[c]), ly = row(iy, g.ny, x.ym[c], vi, x.yp[c]);
      double lap = __builtin_fma(lx, g.idx2, ly * g.idy2);
      if (g.nz > 1) lap = __builtin_fma(row(iz, g.nz, x.zm[c], vi, x.zp[c]), g.idz2, lap);
      hj[c] = (-2.0 * lap) * jf;
    }
  }
  // demag: S = sum_k partial (K m); field = fl32(fl32(-S) * Ms_i)
  if (D.hpart64) {
    for (int c = 0; c < 3; ++c) hm[c] = (-D.hpart64[(int64_t)c * n + i]) * r.ms_f64();
  } else {
    const float ms = r.ms_f32();
    for (int c = 0; c < 3; ++c) {
      float h = (-hsum(c)) * ms;
      hm[c] = (double)h;
    }
  }
  if (g.aniso) {
    const double f = -2.0 * r.kfact();
    auto axis = [&](int x, int y, int z) {
      return f * __builtin_fma(r.aniso(z), mc[2], __builtin_fma(r.aniso(y), mc[1], r.aniso(x) * mc[0]));
    };
    hk[0] = axis(0, 1, 2);
    hk[1] = axis(1, 3, 4);
    hk[2] = axis(2, 4, 5);
  } else {
    hk[0] = hk[1] = hk[2] = 0.0;
  }
  double hh[3] = {-D.hext[0], -D.hext[1], -D.hext[2]};
  double H[3];
  for (int c = 0; c < 3; ++c) H[c] = hh[c] + hj[c] + hm[c] + hk[c];
  // t = m x H (the fields are negated: c = -t is m x H of the equation), d = m x c
  const double tx = __builtin_fma(mc[1], H[2], -(mc[2] * H[1]));
  const double ty = __builtin_fma(mc[2], H[0], -(mc[0] * H[2]));
  const double tz = __builtin_fma(mc[0], H[1], -(mc[1] * H[0]));
  const double dx = __builtin_fma(mc[2], ty, -(mc[1] * tz));
  const double dy = __builtin_fma(mc[0], tz, -(mc[2] * tx));
  const double dz = __builtin_fma(mc[1], tx, -(mc[0] * ty));
  dm[0] = __builtin_fma(D.gamma, tx, -(D.alpha * dx));
  dm[1] = __builtin_fma(D.gamma, ty, -(D.alpha * dy));
  dm[2] = __builtin_fma(D.gamma, tz, -(D.alpha * dz));
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
// packed into column col (kPackF32, kPackLattice: the products whose right-hand
// sides wait for the next stage).  Only the cell's own values are read, so the launch
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
    bad |= !(fabsf(f) <= FLT_MAX);
  }
  if (bad && pack.nonfinite) *pack.nonfinite = 1;
}

}  // namespace mt
