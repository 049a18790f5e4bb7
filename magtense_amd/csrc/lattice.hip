// FP32 demag product of a uniform grid from its distinct tensor entries.
//
// The dense FP32 tensor of an nx x ny x nz grid holds K(p_i - p_j) for every
// pair of cells.  The differences repeat: along each axis there are 2n - 1
// cell offsets, and the rounding of the cell centres gives each of them a few
// FP64 values (4 on average on a 128-cell axis).  LatticeTable stores the
// tensor once per distinct triple of differences, evaluated from the same FP64
// arguments as the dense assembly, and index maps from cell pairs to entries.
// An entry takes 16 bytes in one plane (xx, xy, yy, zz), 24 in several, and
// columns of equal entries are stored once: the same FP32 entries in about 1 MB
// instead of 402.7 MB for 128 x 32 x 1 (326 columns of 183 entries in a film of
// 500 x 125 nm), 105 MB instead of 25.8 GB for 256 x 64 x 2 cells of 4 nm, where
// next to nothing is equal.
//
// Product: the sums of matvec_rows_f32 (matvec_rows.h), bit for bit.  There a
// receiver row is summed by 256 threads, thread T taking the column quads
// 4T + 1024 k in order of k ("chain" T; single columns T + 256 k when n % 4),
// then a shuffle tree over each wave's 64 chains and the four waves in order.
// Here a lane is a receiver and walks whole chains, so that the states' values
// are wave-uniform (scalar loads) and the entries come from LDS.

#include <algorithm>
#include <cfloat>
#include <type_traits>
#include <vector>

#include "matvec_rows.h"
#include "mt_common.h"
#include "mt_kernels.h"

namespace mt {

namespace {

constexpr int kLatThreads = 1024;
constexpr int kLatLds = 160 * 1024;   // LDS of a CU
constexpr int kLatMaxRows = 4096;     // source rows x receiver rows of a tile

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// Asynchronous 16-byte-per-lane copy global -> LDS, lane l's bytes at lds +
// 16 l (see the GEMM kernels, demag.hip); completion by vmcnt.
__device__ inline void lat_dma16(const void* src, uint32_t lds) {
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %2\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, off\n\t"
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0"
      : "=&s"(saved)
      : "v"(src), "s"(__builtin_amdgcn_readfirstlane(lds))
      : "memory");
}

// Receiver tile of a workgroup: 64 lanes over one grid row (nx >= 64), or over
// rr = 64 / nx whole rows.
struct LatTile {
  int rr, per_row, count;
};
__host__ __device__ inline LatTile lat_tiles(int nx, int rows) {
  LatTile t;
  t.rr = nx >= 64 ? 1 : 64 / nx;
  t.per_row = nx >= 64 ? (nx + 63) / 64 : 1;
  t.count = t.per_row * ((rows + t.rr - 1) / t.rr);
  return t;
}

// LDS of a workgroup: the x map of its receivers, the table row of every
// (receiver row, source row), nbuf buffers of table rows.  A step's columns
// are one run of 256 (QC 4) or four of 64 (QC 1).
struct LatLds {
  int pmap, rowidx, touched, slabs, buf_a, buf, total;
};
__host__ __device__ inline LatLds lat_lds(const LatticeView& v, int qc, int nbuf) {
  LatLds L;
  const int rows = v.ny * v.nz;
  const LatTile t = lat_tiles(v.nx, rows);
  const int run = 64 * qc;
  // grid rows that a run touches (it starts at a multiple of its length)
  const int most = run % v.nx == 0 ? run / v.nx : (v.nx % run == 0 ? 1 : (run + v.nx - 2) / v.nx + 1);
  L.touched = std::min(rows, most);
  L.slabs = t.rr * L.touched * (4 / qc);
  L.pmap = (v.nx + 3) / 4 * 512;
  L.rowidx = (rows * t.rr * 4 + 15) / 16 * 16;
  L.buf_a = L.slabs * v.ux * 16;
  L.buf = L.buf_a + (v.b ? L.slabs * v.ux * 8 : 0);
  L.total = L.pmap + L.rowidx + nbuf * L.buf;
  return L;
}

// Workgroup (tile, w, state group): the chains 64 w .. 64 w + 63 of the tile's
// receivers for SB states, lane = receiver.  Wave r takes the four chains r +
// 16 c, which the shuffle tree joins first (lane xor 32, 16).  The columns go
// in steps of 1024, four to a chain ("quad"): 4 T + q for chain T (QC 4), T +
// 256 q (QC 1); the states lie quad by quad (lattice_state_offset).  Per step
// the table rows of the workgroup's columns are copied to LDS one step ahead
// (nbuf 2); a pair then costs a lane 2 bytes of the x map and 16 bytes (xx,
// xy, yy, zz) of LDS reads, 8 more for (xz, yz) between planes.  Those are +-0
// within a plane, where their products, which add +-0 to sums that are never
// -0, are left out unless *nonfinite says that a state holds an infinity or a
// NaN.
//
// Bound by LDS reads (one state, 256 x 64 x 2: their cycles and bank conflicts are
// 0.6 of the launch's) and by what a wave waits for between them.  The next sums'
// reads are issued after the last ones have arrived, the x map's values of a step
// before its barrier, and a step's place in the grid is kept up by addition.
// Kernel alone, us a launch (in parentheses with a wait per read): one state 128 x 32
// x 1 14 (15), 90 x 70 x 1 68 (79), 91 x 71 x 1 84 (116), 256 x 64 x 2 893 (1023),
// there four states 1879 (1985).
template <int QC, bool HASB, bool ALIGNED, int SB>
__global__ void __launch_bounds__(kLatThreads)
    lattice_rows_kernel(const LatticeView v, const float* __restrict__ m, int cols, float* __restrict__ out,
                        int64_t split_stride, int64_t col_stride, int nstates, int nbuf,
                        const int* __restrict__ nonfinite) {
  extern __shared__ __align__(16) uint8_t lat_smem[];
  constexpr int kWaves = kLatThreads / 64, CH = 64 / kWaves;  // chains of a wave
  static_assert(kWaves == 16 && CH == 4, "the order of the final sums");
  constexpr bool AHEAD = QC == 4 || SB < 4;  // registers for the reads of the next sums
  const int lane = threadIdx.x & 63;
  const int r = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nx = v.nx, ny = v.ny, rows = v.ny * v.nz, n = nx * rows;
  const LatTile T = lat_tiles(nx, rows);
  const LatLds L = lat_lds(v, QC, nbuf);
  const int tile = blockIdx.x, w = blockIdx.y, s0 = blockIdx.z * SB;
  const int row0 = tile / T.per_row * T.rr, ix0 = tile % T.per_row * 64;
  const int rho = nx >= 64 ? 0 : std::min(lane / nx, T.rr - 1);
  const int ix = std::min(nx >= 64 ? ix0 + lane : lane - rho * nx, nx - 1);
  const bool lane_ok = (nx >= 64 ? ix0 + lane < nx : lane < T.rr * nx) && row0 + rho < rows;
  uint16_t* pmap = reinterpret_cast<uint16_t*>(lat_smem);  // [jx / 4][lane][jx % 4]
  int* rowidx = reinterpret_cast<int*>(lat_smem + L.pmap);
  uint8_t* bufs = lat_smem + L.pmap + L.rowidx;
  const bool all = *nonfinite != 0;  // no product is left out

  // source rows [plane_lo, plane_hi) lie in the one plane of the tile's receivers
  const int plane0 = row0 / ny, plane1 = (std::min(row0 + T.rr, rows) - 1) / ny;
  const int plane_lo = plane0 * ny, plane_hi = plane0 == plane1 ? plane_lo + ny : plane_lo;
  constexpr int RUN = 64 * QC, NRUN = 4 / QC;
  // first column of run g of the step at `base`
  auto run_at = [&](int base, int g) { return base + RUN * w + (NRUN == 1 ? 0 : 256 * g); };
  // The grid rows and x of a step's run starts, kept up from step to step (no
  // divisions by nx in the loop).
  struct Cursor {
    int row[NRUN], jx[NRUN];
  };
  const int step_rows = 1024 / nx, step_x = 1024 - step_rows * nx;
  const int run_rows = (RUN - 1) / nx, run_x = RUN - 1 - run_rows * nx;
  auto next_step = [&](Cursor& c) {
#pragma unroll
    for (int g = 0; g < NRUN; ++g) {
      c.row[g] += step_rows;
      c.jx[g] += step_x;
      if (c.jx[g] >= nx) {
        c.jx[g] -= nx;
        c.row[g] += 1;
      }
    }
  };
  // last grid row of run g of the step at `base`, at cursor c
  auto last_row = [&](const Cursor& c, int base, int g) {
    const int left = n - run_at(base, g);
    if (left < RUN) return rows - 1;
    return c.row[g] + run_rows + (c.jx[g] + run_x >= nx ? 1 : 0);
  };
  // every source row of the step against the tile: only xx, xy, yy, zz
  auto flat_step = [&](const Cursor& c, int base) {
    if (all) return false;
    if (!HASB) return true;
    int g = NRUN - 1;  // the last run that has columns
    while (g > 0 && run_at(base, g) >= n) --g;
    return c.row[0] >= plane_lo && last_row(c, base, g) < plane_hi;
  };
  // table row of receiver row q of the tile against source row j
  auto table_row = [&](int q, int j) {
    const int i = std::min(row0 + q, rows - 1);
    return v.zmap[i / ny * v.nz + j / ny] * v.uy + v.ymap[i % ny * ny + j % ny];
  };
  // table rows of the step at `base` (cursor cur) into buffer b; the first step
  // looks them up itself, so that its copies run while the maps are filled
  auto stage = [&](auto first, const Cursor& cur, int base, int b) {
    constexpr bool FIRST = decltype(first)::value;
    uint8_t* A = bufs + (size_t)b * L.buf;
    const uint32_t la = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)A;
    const int pa = (v.ux + 63) / 64;
    const int hx = v.ux / 2, pb = (hx + 63) / 64;  // (xz, yz): two entries per lane
    const bool with_b = HASB && !flat_step(cur, base);
#pragma unroll
    for (int g = 0; g < NRUN; ++g) {
      if (run_at(base, g) >= n) break;
      const int ra = cur.row[g], nr = last_row(cur, base, g) - ra + 1, slab0 = g * L.touched * T.rr;
      for (int p = r; p < nr * T.rr * pa; p += kWaves) {
        const int slab = p / pa, o = (p - slab * pa) * 64;  // slab = source row x rr + receiver row
        const int sr = T.rr == 1 ? slab : slab / T.rr, q = slab - sr * T.rr;
        const int64_t src =
            (int64_t)__builtin_amdgcn_readfirstlane(FIRST ? table_row(q, ra + sr) : rowidx[q * rows + ra + sr]) * v.ux +
            o + lane;
        if (o + lane < v.ux) lat_dma16(v.a + src * 4, la + (uint32_t)((slab0 + slab) * v.ux + o) * 16);
      }
      if (with_b)
        for (int p = r; p < nr * T.rr * pb; p += kWaves) {
          const int slab = p / pb, o = (p - slab * pb) * 64;
          const int sr = T.rr == 1 ? slab : slab / T.rr, q = slab - sr * T.rr;
          const int64_t src =
              (int64_t)__builtin_amdgcn_readfirstlane(FIRST ? table_row(q, ra + sr) : rowidx[q * rows + ra + sr]) * hx +
              o + lane;
          if (o + lane < hx)
            lat_dma16(v.b + src * 4, la + (uint32_t)L.buf_a + (uint32_t)((slab0 + slab) * hx + o) * 16);
        }
    }
  };

  float acc[CH][SB][3];
#pragma unroll
  for (int c = 0; c < CH; ++c)
#pragma unroll
    for (int s = 0; s < SB; ++s) acc[c][s][0] = acc[c][s][1] = acc[c][s][2] = 0.0f;
  // the states through the constant address space: uniform reads become scalar
  // loads whatever the copies' memory clobbers
  typedef const __attribute__((address_space(4))) float* const_floats;
  const const_floats ms = (const_floats)(m + (size_t)s0 * 12);

  struct Entries {
    f32x4 a[4];
    f32x2 b[4];
  };
  constexpr int SH = SB < 2 ? SB : 2;  // states in scalar registers at a time
  struct States {
    float x[SH][4], y[SH][4], z[SH][4];
  };
  Cursor here;  // of the step that is computed
  // Places of the wave's chains: the x map's values of their columns, read for
  // all of them before the step's barrier (the map does not change), and the first
  // entries of the columns' grid rows in the step's buffer.
  constexpr int COLS = ALIGNED && QC == 4 ? 1 : 4;  // columns of a chain in rows of their own
  typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
  struct Places {
    u16x4 x[CH];
    int row[CH][COLS];
  };
  auto places = [&](Places& P, const Cursor& cur, int base) {
    int jx[COLS], row[COLS];
#pragma unroll
    for (int q = 0; q < COLS; ++q) {
      jx[q] = cur.jx[QC == 4 ? 0 : q] + (QC == 4 ? 4 * r + q : r);
      row[q] = (QC == 4 ? 0 : q) * L.touched * T.rr * v.ux;
    }
#pragma unroll
    for (int c = 0; c < CH; ++c)
#pragma unroll
      for (int q = 0; q < COLS; ++q) {
        while (jx[q] >= nx) {
          jx[q] -= nx;
          row[q] += T.rr * v.ux;
        }
        const uint16_t* m4 = pmap + (jx[q] >> 2) * 256 + lane * 4;
        if constexpr (COLS == 1) P.x[c] = *reinterpret_cast<const u16x4*>(m4);
        else P.x[c][q] = m4[jx[q] & 3];
        P.row[c][q] = row[q];
        jx[q] += QC * kWaves;
      }
  };
  // the same one chain at a time (QC 1); jx, row: where the last call stopped
  auto place_of = [&](Places& P, int c, int (&jx)[4], int (&row)[4]) {
#pragma unroll
    for (int q = 0; q < COLS; ++q) {
      jx[q] = c == 0 ? here.jx[q % NRUN] + r : jx[q] + kWaves;
      if (c == 0) row[q] = q * L.touched * T.rr * v.ux;
      while (jx[q] >= nx) {
        jx[q] -= nx;
        row[q] += T.rr * v.ux;
      }
      P.x[c][q] = pmap[(jx[q] >> 2) * 256 + lane * 4 + (jx[q] & 3)];
      P.row[c][q] = row[q];
    }
  };
  auto read_entries = [&](auto flat, Entries& k, const uint8_t* A, const Places& P, int c, int have) {
    constexpr bool FLAT = decltype(flat)::value;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (QC == 1 && q >= have) continue;
      const int e = P.row[c][COLS == 1 ? 0 : q] + rho * v.ux + P.x[c][q];
      k.a[q] = *reinterpret_cast<const f32x4*>(A + (size_t)e * 16);
      if (!FLAT) k.b[q] = HASB ? *reinterpret_cast<const f32x2*>(A + L.buf_a + (size_t)e * 8) : f32x2{0.0f, 0.0f};
    }
  };
  auto read_states = [&](States& t, const_floats f) {
#pragma unroll
    for (int s = 0; s < SH; ++s)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        t.x[s][q] = f[s * 12 + q];
        t.y[s][q] = f[s * 12 + 4 + q];
        t.z[s][q] = f[s * 12 + 8 + q];
      }
  };
  // states SH h .. SH h + SH - 1
  auto add = [&](auto flat, float (&a)[SB][3], int h, const Entries& k, const States& t, int have) {
    constexpr bool FLAT = decltype(flat)::value;
#pragma unroll
    for (int s = 0; s < SH; ++s) {
      float(&as)[3] = a[SH * h + s];
      if (QC == 4) {
        if (FLAT) matvec_flat<4>(k.a, t.x[s], t.y[s], t.z[s], as);
        else matvec_full<4>(k.a, k.b, t.x[s], t.y[s], t.z[s], as);
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (q >= have) continue;
          const f32x4 ka[1] = {k.a[q]};
          const f32x2 kb[1] = {k.b[q]};
          const float x[1] = {t.x[s][q]}, y[1] = {t.y[s][q]}, z[1] = {t.z[s][q]};
          if (FLAT) matvec_flat<1>(ka, x, y, z, as);
          else matvec_full<1>(ka, kb, x, y, z, as);
        }
      }
    }
  };
  // the step at `base`: the entries of the next chain and the states of the next
  // sums are read before a chain's (state pair's) sums, and after everything read
  // before has arrived: scalar loads return in any order, so that a wait for one
  // is a wait for all that are out.
  const int64_t chain_floats = (int64_t)kWaves * cols * 12;
  auto states_at = [&](int base) { return ms + (int64_t)(base / 4 + 64 * w + r) * cols * 12; };
  auto arrived = [&] { __builtin_amdgcn_s_waitcnt(0xC07F); };  // lgkmcnt(0)
  States t[2];
  auto compute = [&](auto flat, auto whole, Places& P, int base, int b) {
    constexpr bool WHOLE = decltype(whole)::value;
    const uint8_t* A = bufs + (size_t)b * L.buf;
    const_floats f = states_at(base);
    if (WHOLE) {
      Entries k[2];
      read_entries(flat, k[0], A, P, 0, 4);
#pragma unroll
      for (int u = 0; u < CH * (SB / SH); ++u) {
        const int c = u / (SB / SH), h = u % (SB / SH);
        arrived();
        __builtin_amdgcn_sched_barrier(0);
        if (h == 0 && c + 1 < CH) read_entries(flat, k[(c + 1) & 1], A, P, c + 1, 4);
        if (u + 1 < CH * (SB / SH)) {
          if (h + 1 == SB / SH) f += chain_floats - 12 * SH * (SB / SH - 1);
          else f += 12 * SH;
          read_states(t[(u + 1) & 1], f);
        }
        __builtin_amdgcn_sched_barrier(0);
        add(flat, acc[c], h, k[c & 1], t[u & 1], 4);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      int jx[4], row[4];
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        if constexpr (!AHEAD) place_of(P, c, jx, row);
        // QC 4: all of the quad's columns exist or none; QC 1: the first `have`
        const int j = run_at(base, 0) + QC * (r + kWaves * c);
        const int have = QC == 4 ? (j < n ? 4 : 0) : (j < n ? std::min(4, (n - 1 - j) / 256 + 1) : 0);
        if (have > 0) {
          Entries k;
          read_entries(flat, k, A, P, c, have);
#pragma unroll
          for (int h = 0; h < SB / SH; ++h) {
            States t1;
            read_states(t1, f + 12 * SH * h);
            add(flat, acc[c], h, k, t1, have);
          }
        }
        f += chain_floats;
      }
    }
  };

  Cursor cur;
#pragma unroll
  for (int g = 0; g < NRUN; ++g) {
    cur.row[g] = run_at(0, g) / nx;
    cur.jx[g] = run_at(0, g) - cur.row[g] * nx;
  }
  if (run_at(0, 0) < n) stage(std::true_type{}, cur, 0, 0);
  for (int jx = r; jx < nx; jx += kWaves) pmap[(jx >> 2) * 256 + lane * 4 + (jx & 3)] = v.pmap[jx * nx + ix];
  for (int e = threadIdx.x; e < rows * T.rr; e += kLatThreads) {
    const int q = e / rows;
    rowidx[e] = table_row(q, e - q * rows);
  }
  __syncthreads();  // the maps
  int b = 0;
  for (int base = 0; run_at(base, 0) < n; base += 1024) {
    if (nbuf == 1 && base > 0) {
      __syncthreads();  // the previous step's reads
      stage(std::false_type{}, cur, base, 0);
    }
    const bool whole = AHEAD && run_at(base, NRUN - 1) + RUN <= n;
    Places P;
    if constexpr (AHEAD) places(P, cur, base);
    if (whole) read_states(t[0], states_at(base));
    __builtin_amdgcn_s_waitcnt(0);  // my copies, my reads of the other buffer
    __syncthreads();
    here = cur;
    next_step(cur);
    if (nbuf == 2 && run_at(base + 1024, 0) < n) stage(std::false_type{}, cur, base + 1024, b ^ 1);
    if (flat_step(here, base)) {
      if (whole) compute(std::true_type{}, std::bool_constant<AHEAD>{}, P, base, b);
      else compute(std::true_type{}, std::false_type{}, P, base, b);
    } else {
      if (whole) compute(std::false_type{}, std::bool_constant<AHEAD>{}, P, base, b);
      else compute(std::false_type{}, std::false_type{}, P, base, b);
    }
    b ^= nbuf - 1;
  }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();

  // chains r + 16 c of this wave in the shuffle tree's order (xor 32, 16), then
  // the waves (xor 8, 4, 2, 1)
  float* part = reinterpret_cast<float*>(bufs);  // [wave][s][component][lane]
#pragma unroll
  for (int s = 0; s < SB; ++s)
#pragma unroll
    for (int a = 0; a < 3; ++a)
      part[((r * SB + s) * 3 + a) * 64 + lane] =
          (acc[0][s][a] + acc[2][s][a]) + (acc[1][s][a] + acc[3][s][a]);
  __syncthreads();
  for (int e = r; e < SB * 3; e += kWaves) {
    const int s = e / 3, a = e - s * 3;
    if (!lane_ok || s0 + s >= nstates) continue;
    float t[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) t[q] = part[((q * SB + s) * 3 + a) * 64 + lane];
#pragma unroll
    for (int h = 8; h > 0; h >>= 1)
#pragma unroll
      for (int q = 0; q < h; ++q) t[q] += t[q + h];
    out[(int64_t)w * split_stride + (int64_t)(s0 + s) * col_stride + (int64_t)a * n + (int64_t)(row0 + rho) * nx + ix] =
        t[0];
  }
}

// same[k] = 0 where x difference W + k (of offset owner[k]) and the commonest
// one of its offset have different entries in some row: blocks (k, rows).
__global__ void __launch_bounds__(256) lattice_same_kernel(const uint4* __restrict__ a, const uint2* __restrict__ b,
                                                           int ux, int rows, int W, const int* __restrict__ owner,
                                                           int* __restrict__ same) {
  const int k = blockIdx.x, u = W + k, o = owner[k];
  bool eq = true;
  for (int r = threadIdx.x; r < rows; r += blockDim.x) {
    const uint4 p = a[(size_t)r * ux + u], q = a[(size_t)r * ux + o];
    eq = eq && p.x == q.x && p.y == q.y && p.z == q.z && p.w == q.w;
    if (b) {
      const uint2 e = b[(size_t)r * ux + u], f = b[(size_t)r * ux + o];
      eq = eq && e.x == f.x && e.y == f.y;
    }
  }
  if (!eq) same[k] = 0;
}

// Distinct values of c[i] - c[j], the commonest value of each offset first:
// value u < 2 m - 1 belongs to offset u - (m - 1), the others follow offset by
// offset, so that the lanes of a row read neighbouring entries.  map[j * m + i]
// is the value of the pair.
void distinct_differences(const std::vector<double>& c, std::vector<double>& values, std::vector<int>& map) {
  const int m = (int)c.size(), W = 2 * m - 1;
  values.assign(W, 0.0);
  map.assign((size_t)m * m, 0);
  std::vector<double> seen;
  std::vector<int> count, id;
  for (int o = 0; o < W; ++o) {
    const int d = o - (m - 1);  // i - j
    const int j0 = std::max(0, -d), j1 = std::min(m, m - d);
    seen.clear();
    count.clear();
    for (int j = j0; j < j1; ++j) {
      const double x = c[j + d] - c[j];
      size_t k = 0;
      while (k < seen.size() && seen[k] != x) ++k;
      if (k == seen.size()) {
        seen.push_back(x);
        count.push_back(0);
      }
      count[k] += 1;
      map[(size_t)j * m + j + d] = (int)k;
    }
    const int top = (int)(std::max_element(count.begin(), count.end()) - count.begin());
    id.assign(seen.size(), 0);
    for (size_t k = 0; k < seen.size(); ++k) {
      if ((int)k == top) {
        id[k] = o;
        values[o] = seen[k];
      } else {
        id[k] = (int)values.size();
        values.push_back(seen[k]);
      }
    }
    for (int j = j0; j < j1; ++j) map[(size_t)j * m + j + d] = id[map[(size_t)j * m + j + d]];
  }
}

template <int QC, bool HASB, bool ALIGNED>
int launch_rows(const LatticeView& v, const float* m, int cols, float* out, int64_t split_stride, int64_t col_stride,
                int nstates, const int* nonfinite, hipStream_t stream) {
  const int nbuf = lat_lds(v, QC, 2).total <= kLatLds ? 2 : 1;
  const LatTile T = lat_tiles(v.nx, v.ny * v.nz);
  const int nw = lattice_nsplit(v.nx * v.ny * v.nz);
  auto go = [&](auto sb) {
    constexpr int SB = decltype(sb)::value;
    const size_t lds = std::max<size_t>(lat_lds(v, QC, nbuf).total,
                                        lat_lds(v, QC, 0).total + (size_t)kLatThreads * SB * 3 * sizeof(float));
    const dim3 grid((unsigned)T.count, (unsigned)nw, (unsigned)((nstates + SB - 1) / SB));
    hipLaunchKernelGGL((lattice_rows_kernel<QC, HASB, ALIGNED, SB>), grid, dim3(kLatThreads), lds, stream, v, m, cols,
                       out, split_stride, col_stride, nstates, nbuf, nonfinite);
  };
  if (nstates == 1) go(std::integral_constant<int, 1>{});
  else if (nstates == 2) go(std::integral_constant<int, 2>{});
  else go(std::integral_constant<int, 4>{});
  MT_HIP(hipGetLastError());
  return kOk;
}

}  // namespace

// Whether the product from the table and the LL kernel behind it beat the launch over
// the dense tensor.  Time of the table's right-hand side over the dense one's:
//   n % 4 == 0, one plane, states      1     4     8     12    16    24    48
//     36 x 30   (1080 cells)          1.17  1.28  1.15  1.18  1.18  1.19  1.29
//     64 x 17   (1088)                1.12  1.26  1.13  0.90  1.05  0.96  0.98
//     44 x 40   (1760)                0.93  1.16  1.11  1.05  1.20  1.34  1.36
//     64 x 30   (1920)                0.82  1.02  0.82  0.97  0.96  0.99  1.05
//     20 x 110  (2200)                0.76  0.85  1.05  0.95  1.13  1.16  1.18
//     96 x 24   (2304)                0.67  0.82  0.99  1.03  1.17  1.21  1.26
//     128 x 20  (2560)                0.59  0.75  0.83  0.83  0.96  0.99  1.02
//     50 x 82   (4100)                0.53  0.73  0.83  0.78  1.01  1.08  1.18
//     128 x 64  (8192)                0.19  0.35  0.52  0.54        0.75
//   several planes, where (xz, yz) cost a second LDS read a pair
//     30 x 30 x 2   (1800)            1.25  1.52  1.15  1.47  1.46  1.59  1.72
//     32 x 33 x 2   (2112)            0.94  1.03  1.29  1.12  1.35  1.37  1.38
//     64 x 12 x 3   (2304)            0.79  0.98  1.25  1.13  1.38  1.36  1.35
//     48 x 16 x 4   (3072)            0.58  0.81  1.08  1.20  1.49  1.60  1.67
//     50 x 37 x 2   (3700)            0.69  1.13  1.42  1.31  1.57  1.70  1.88
//     64 x 16 x 4   (4096)            0.37  0.60  0.75  0.73  0.91  1.04  1.17
//     100 x 30 x 2  (6000)            0.41  0.66  0.96  0.96  1.20  1.34  1.48
//   n % 4 != 0: a chain's four columns lie in four places of the grid
//     77 x 33   (2541)                1.19  1.58  1.88  1.53  2.09  2.09  2.23
//     91 x 41   (3731, lanes 0.71)    0.67  0.91  1.12  1.03  1.30  1.46  1.56
//     63 x 57   (3591, lanes 0.98)    0.47  0.62  0.86  0.82  1.02  1.19  1.24
//     63 x 101  (6363, lanes 0.98)    0.35  0.56  0.82  0.73  0.98  1.07  1.14
//     91 x 71   (6461, lanes 0.71)    0.47  0.75  1.03  1.00  1.25  1.40  1.52
//     45 x 41 x 2   (3690)            1.40  1.57  1.99  1.88  2.50  2.74  2.94
//     17 x 17 x 13  (3757)            1.57  1.77  2.08  1.94  2.29  2.46  2.69
//     45 x 45 x 3   (6075)            1.18  1.48  2.06  2.08        2.60
//     65 x 49 x 3   (9555)            1.45  1.70  2.67  2.75        3.73
//     45 x 79 x 3   (10665)           1.00  1.25  1.91  2.06        2.59
//     49 x 49 x 5   (12005)           0.87  1.12  1.71  1.97        2.45
// (4096 cells of 128 x 32, one state: 22 us against 74.)
// From 8192 cells on, where the dense tensor takes 1.6 GB and its assembly 4 ms, the
// table is kept at any number of states except on odd layered grids, whose dense rows
// are twice as fast.
bool lattice_pays(int nx, int ny, int nz, int nstates) {
  const int64_t n = (int64_t)nx * ny * nz;
  const bool wide = nx >= 64;
  const bool full = n * 20 >= (int64_t)lat_tiles(nx, ny * nz).count * 64 * 19;  // lanes with a receiver
  if (n % 4 && nz > 1) return n > 10000 && nstates == 1 && !wide;
  if (n >= 8192) return true;
  if (n % 4) return n > 3500 && (nstates <= 4 || (nstates <= 12 && full));
  if (nz > 1) return nstates <= 4 ? n > 2000 : n > 4000 && wide && (nstates <= 8 || (nstates <= 12 && full));
  if (nstates <= 12 && n > 2000) return true;
  return n > 1024 && nstates > 8 && wide && full;
}

int lattice_wanted(int nx, int ny, int nz, int nstates, bool* wanted) {
  const double n = (double)nx * ny * nz, dense = 24.0 * n * n;
  *wanted = lattice_pays(nx, ny, nz, nstates);
  if (!*wanted && dense < (double)(1 << 30)) return kOk;
  size_t free_b = 0, total_b = 0;
  MT_HIP(hipMemGetInfo(&free_b, &total_b));
  if (dense > 0.9 * (double)free_b) *wanted = true;   // no room for the dense tensor
  if (dense >= (double)total_b) *wanted = false;      // a problem too large for the device stays refused
  return kOk;
}

int lattice_nsplit(int n) {
  const int width = n % 4 == 0 ? 256 : 64;
  return std::min(4, (n + width - 1) / width);
}

void LatticeTable::release() {
  auto f = [](void* p) {
    if (p) (void)hipFree(p);
  };
  f(a); f(b); f(pmap); f(ymap); f(zmap);
  a = b = nullptr;
  pmap = nullptr;
  ymap = zmap = nullptr;
  v = LatticeView{};
}

int LatticeTable::build(int nx, int ny, int nz, const std::vector<double>& cx, const std::vector<double>& cy,
                        const std::vector<double>& cz, const double d[3], hipStream_t stream, bool* fits) {
  release();
  *fits = false;
  if (nx < 16 || nx > 1024 || (int64_t)ny * nz * lat_tiles(nx, ny * nz).rr > kLatMaxRows) return kOk;
  std::vector<double> val[3];
  std::vector<int> map[3];
  distinct_differences(cx, val[0], map[0]);
  if (val[0].size() % 2) {  // rows of whole 16-byte pieces; an entry that no pair has
    val[0].push_back(val[0][0]);
  }
  if (val[0].size() > 65535) return kOk;
  LatticeView q{};
  q.nx = nx; q.ny = ny; q.nz = nz;
  q.ux = (int)val[0].size();
  if (nz > 1) q.b = reinterpret_cast<const float*>(sizeof(float));  // any non-null: the layout with (xz, yz)
  if (lat_lds(q, nx * ny * nz % 4 == 0 ? 4 : 1, 1).total > kLatLds) return kOk;
  distinct_differences(cy, val[1], map[1]);
  distinct_differences(cz, val[2], map[2]);
  q.uy = (int)val[1].size();
  const int64_t entries = (int64_t)val[0].size() * val[1].size() * val[2].size();
  const int64_t n = (int64_t)nx * ny * nz;
  if (entries > n * n / 8) return kOk;
  // the kernel looks rows up by receiver, then source
  auto by_receiver = [](const std::vector<int>& t, int m) {
    std::vector<int> o(t.size());
    for (int j = 0; j < m; ++j)
      for (int i = 0; i < m; ++i) o[(size_t)i * m + j] = t[(size_t)j * m + i];
    return o;
  };
  const std::vector<int> ym = by_receiver(map[1], ny), zm = by_receiver(map[2], nz);
  const int W = 2 * nx - 1, extra = (int)val[0].size() - W;
  DevArr<double> dv[3];
  for (int k = 0; k < 3; ++k) {
    MT_HIP(dv[k].alloc(val[k].size()));
    MT_HIP(hipMemcpyAsync(dv[k].p, val[k].data(), val[k].size() * sizeof(double), hipMemcpyHostToDevice, stream));
  }
  auto entries_of = [&](const std::vector<double>& x) -> int {
    const int64_t cnt = (int64_t)x.size() * val[1].size() * val[2].size();
    MT_HIP(hipMalloc(&a, (size_t)cnt * 4 * sizeof(float)));
    if (nz > 1) MT_HIP(hipMalloc(&b, (size_t)cnt * 2 * sizeof(float)));
    return launch_lattice_entries(dv[0].p, (int)x.size(), dv[1].p, (int)val[1].size(), dv[2].p, (int)val[2].size(), d,
                                  a, b, stream);
  };
  int rc = entries_of(val[0]);
  if (rc) return rc;
  // x differences whose entries all equal those of their offset's commonest
  // one are the same column of the table: 997 -> 326 columns at 128 x 32 x 1
  // (500 x 125 nm)
  std::vector<int> owner(std::max(extra, 1), 0), same(std::max(extra, 1), 1);
  for (int j = 0; j < nx; ++j)
    for (int i = 0; i < nx; ++i) {
      const int u = map[0][(size_t)j * nx + i];
      if (u >= W) owner[u - W] = i - j + nx - 1;
    }
  if (extra > 0) {
    DevArr<int> downer, dsame;
    MT_HIP(downer.alloc(extra));
    MT_HIP(dsame.alloc(extra));
    MT_HIP(hipMemcpyAsync(downer.p, owner.data(), extra * sizeof(int), hipMemcpyHostToDevice, stream));
    MT_HIP(hipMemcpyAsync(dsame.p, same.data(), extra * sizeof(int), hipMemcpyHostToDevice, stream));
    hipLaunchKernelGGL(lattice_same_kernel, dim3((unsigned)extra), dim3(256), 0, stream,
                       reinterpret_cast<const uint4*>(a), reinterpret_cast<const uint2*>(b), q.ux,
                       (int)(val[1].size() * val[2].size()), W, downer.p, dsame.p);
    MT_HIP(hipGetLastError());
    MT_HIP(hipMemcpyAsync(same.data(), dsame.p, extra * sizeof(int), hipMemcpyDeviceToHost, stream));
    MT_HIP(hipStreamSynchronize(stream));
    std::vector<double> x(val[0].begin(), val[0].begin() + W);
    std::vector<int> to(extra);
    for (int k = 0; k < extra; ++k) {
      to[k] = same[k] ? owner[k] : (int)x.size();
      if (!same[k]) x.push_back(val[0][W + k]);
    }
    if (x.size() % 2) x.push_back(x[0]);
    if (x.size() < val[0].size()) {
      for (int& u : map[0])
        if (u >= W) u = to[u - W];
      release();
      q.ux = (int)x.size();
      MT_HIP(hipMemcpyAsync(dv[0].p, x.data(), x.size() * sizeof(double), hipMemcpyHostToDevice, stream));
      rc = entries_of(x);
      if (rc) return rc;
      MT_HIP(hipStreamSynchronize(stream));  // x leaves scope
    }
  }
  const std::vector<uint16_t> pm(map[0].begin(), map[0].end());
  MT_HIP(hipMalloc(&pmap, pm.size() * sizeof(uint16_t)));
  MT_HIP(hipMalloc(&ymap, ym.size() * sizeof(int)));
  MT_HIP(hipMalloc(&zmap, zm.size() * sizeof(int)));
  MT_HIP(hipMemcpyAsync(pmap, pm.data(), pm.size() * sizeof(uint16_t), hipMemcpyHostToDevice, stream));
  MT_HIP(hipMemcpyAsync(ymap, ym.data(), ym.size() * sizeof(int), hipMemcpyHostToDevice, stream));
  MT_HIP(hipMemcpyAsync(zmap, zm.data(), zm.size() * sizeof(int), hipMemcpyHostToDevice, stream));
  MT_HIP(hipStreamSynchronize(stream));
  q.a = a; q.b = b; q.pmap = pmap; q.ymap = ymap; q.zmap = zmap;
  v = q;
  *fits = true;
  return kOk;
}

int launch_lattice_rows(const LatticeView& v, const float* m, int cols, float* out, int64_t split_stride,
                        int64_t col_stride, int nstates, const int* nonfinite, hipStream_t stream) {
  const int n = v.nx * v.ny * v.nz;
  if (nstates < 1 || nstates > 65535 || !v.a || cols % 4 || cols < nstates) {
    set_error("lattice product: no table, states outside 1..65535, or a state layout of the wrong width");
    return kErrArg;
  }
  auto by_b = [&](auto qc, auto aligned) {
    constexpr int QC = decltype(qc)::value;
    constexpr bool AL = decltype(aligned)::value;
    return v.b ? launch_rows<QC, true, AL>(v, m, cols, out, split_stride, col_stride, nstates, nonfinite, stream)
               : launch_rows<QC, false, AL>(v, m, cols, out, split_stride, col_stride, nstates, nonfinite, stream);
  };
  if (n % 4) return by_b(std::integral_constant<int, 1>{}, std::true_type{});
  if (v.nx % 4 == 0) return by_b(std::integral_constant<int, 4>{}, std::true_type{});
  return by_b(std::integral_constant<int, 4>{}, std::false_type{});
}

}  // namespace mt
