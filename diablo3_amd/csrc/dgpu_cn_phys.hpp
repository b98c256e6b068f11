// dgpu_cn_phys.hpp — the physical-space Crank–Nicolson solve of an LES substep.
#pragma once
#include "../../include/diablo_gpu.h"
#include "dgpu_kernels.hpp"

#include <type_traits>

namespace dgpu {

// ---------------------------------------------------------------------------
// Crank–Nicolson solve per physical (x, z) column with the eddy viscosity /
// diffusivity (rk_chan_1, for/solver.f90:875-903, 990-1233): the explicit half
// of the nu_t term is added to the right-hand side r (the inverse transform of
// the Fourier right-hand side, which already holds the molecular part), the
// matrix gets the implicit half, the BC rows of apply_BC_* are set for every
// column, and the system of rows 0..Nyp+1 is solved (the reference's
// thomas_forward/backward_real_mpi at one rank, for/solver.f90:1691-1761,
// 1816-1852).
//
// A block owns TC consecutive columns of one field (the fields' systems are
// independent) in P = NT / TC chunks of rows, RPT rows a thread at
// most, all loaded at once and kept in registers: the field, nu_t and the
// right-hand side are read once and the solution written once.  A thread
// eliminates its rows down to the last row of the chunk before (L) and its own
// last row (R); the last rows of all chunks form a tridiagonal system, reduced
// cyclically in LDS; back substitution finishes the rows between.  (One thread
// per column needed every row's 1/b' and g' in memory between its two sweeps:
// 72 bytes a point and field against 32, in float 40 against 16.)  With the rows
// of a column nx values apart (the [z][j][x] layout) a block stays within one or
// two pages; plane after plane (a 2 MB stride at 512x512) the same kernel took
// 2546 us.  Measured, one thread per column -> this: 512x257x512 FP64 3852 -> 1855 us,
// mixed 2038 -> 1207; 128x129x128 FP64 252 -> 60; 1024x385x1024 mixed 10.5-11.2 ->
// 11.9 ms.  FP64 moves 7.6 GB (nu_t is found in L2), 4.1 TB/s of the 5.7 of a large
// one-read-one-write pass, with waves waiting 41% of their cycles.  Mixed moves 6.5 GB
// where 4.3 would do, and that traffic (5.4 TB/s) bounds it: a block's 16 float columns
// are half a 128-byte line, and the block with the other half runs on another XCD.
//
// INC (the mixed-precision path): u is the state at the substep's start in
// float and r holds r - u (float).  The solve is then for the increment
// delta = u_new - u: right-hand side rhs - (l u_{j-1} + d u_j + c u_{j+1}) of the
// same rows, solved in FP64, and delta is written back to r (0 outside
// [wlo, whi]), so the state moves by a float transform of an O(dt) quantity.
// Otherwise the solution overwrites u on rows [wlo, whi].
// ---------------------------------------------------------------------------
template <typename TU, typename TV>
struct PhysCnArgs {
  Geo g;
  int nf;
  int field[MAXF];                    // slot -> field (0 u1, 1 u2, 2 u3, 3+n th_n)
  int blo[MAXF], bhi[MAXF], wlo[MAXF], whi[MAXF];
  int lo_kind[MAXF], hi_kind[MAXF];   // BC code at each wall (0 Dirichlet, 1 Neumann)
  double lo_c1[MAXF], hi_c1[MAXF];
  double tcn[MAXF];                   // temp1 nu_v_scale (/Pr for scalars)
  double temp2;
  const double* __restrict__ dy;
  const double* __restrict__ dyf;
  const double* __restrict__ rowc;    // [ny2][RC_COUNT] per-row grid coefficients
  TU* u[MAXF];                        // physical field
  TU* r[MAXF];                        // right-hand side (INC: r - u, then delta)
  const TV* visc[MAXF];               // nu_t (velocity) or kappa_t_n (scalar)
};

// One row of a field's system that does not depend on the column: the couplings
// of an equation row (w = d = 1), or a BC row l, d, c | rhs (ilo = ihi = w = 0).
struct alignas(16) CnRow {
  double ilo, ihi, l, d, c, rhs, w;
};
template <typename TU, typename TV>
__device__ __forceinline__ CnRow cn_row(const PhysCnArgs<TU, TV>& a, int e, int j) {
  const int ny = a.g.ny;
  const bool v2 = a.field[e] == 1;
  CnRow R{0.0, 0.0, 0.0, 1.0, 0.0, 0.0, 0.0};
  // The reference's rows (for/solver.f90:1136-1145 and the nu_t terms of
  // les_chan) divide T and temp2 nu by dy(j) dyf(j) and dy(j+1) dyf(j)
  // (GYF rows), dyf(j-1) dy(j) and dyf(j) dy(j) (u2's GY rows, nu_t averaged
  // to the faces); the host table holds those reciprocals.
  if (j >= a.blo[e] && j <= a.bhi[e]) {
    const double* k = a.rowc + (long long)j * RC_COUNT;
    R.ilo = k[v2 ? RC_GLO : RC_FLO];
    R.ihi = k[v2 ? RC_GHI : RC_FHI];
    R.w = 1.0;
  }
  // BC rows (apply_BC_* of the reference, for/solver.f90:1901-2232)
  const int klo = a.lo_kind[e], khi = a.hi_kind[e];
  if (!v2) {
    if (j == 0 || j == ny + 1) R = CnRow{0.0, 0.0, 0.0, 1.0, 0.0, 0.0, 0.0};
    if (j == 1) {
      if (klo == DGPU_BC_DIRICHLET) R = CnRow{0.0, 0.0, 0.0, 1.0, 0.0, a.lo_c1[e], 0.0};
      else R = CnRow{0.0, 0.0, 0.0, -1.0, 1.0, a.dy[2] * a.lo_c1[e], 0.0};
    }
    if (j == ny) {
      if (khi == DGPU_BC_DIRICHLET) R = CnRow{0.0, 0.0, 0.0, 1.0, 0.0, a.hi_c1[e], 0.0};
      else R = CnRow{0.0, 0.0, -1.0, 1.0, 0.0, a.dy[ny] * a.hi_c1[e], 0.0};
    }
  } else {
    if (klo == DGPU_BC_DIRICHLET) {
      if (j == 1 || j == 2) R = CnRow{0.0, 0.0, 0.0, 1.0, 0.0, a.lo_c1[e], 0.0};
    } else if (klo == DGPU_BC_NEUMANN) {
      if (j == 1) R = CnRow{0.0, 0.0, 0.0, -1.0, 1.0, a.dyf[1] * a.lo_c1[e], 0.0};
    }
    if (j == 0) R = CnRow{0.0, 0.0, 0.0, 1.0, 0.0, 0.0, 0.0};
    if (khi == DGPU_BC_DIRICHLET) {
      if (j == ny + 1 || j == ny) R = CnRow{0.0, 0.0, 0.0, 1.0, 0.0, a.hi_c1[e], 0.0};
    } else if (khi == DGPU_BC_NEUMANN) {
      if (j == ny + 1) R = CnRow{0.0, 0.0, -1.0, 1.0, 0.0, a.dyf[ny] * a.hi_c1[e], 0.0};
    }
  }
  return R;
}

constexpr int CN_PHYS_NT = 512;  // threads per block at most
template <typename TU, typename TV, bool INC, int TC, int RPT>
__global__ __launch_bounds__(CN_PHYS_NT) void k_cn_phys(PhysCnArgs<TU, TV> a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int NT = blockDim.x, P = NT / TC;
  CnRow* srow = (CnRow*)smem;               // [n2]
  double* sx = (double*)(srow + a.g.ny2);   // the chunks' exchange, two buffers of three
  const Geo& g = a.g;
  const int tid = threadIdx.x, cc = tid % TC, p = tid / TC;
  // block -> (column group, field): the fields of a group follow one another on one
  // XCD (blocks b, b + 8, ...), so that the velocity's systems find nu_t in its L2
  const int ng = (int)(g.pp / TC), b8 = blockIdx.x >> 3;
  const bool whole = ng % 8 == 0;
  const int e = whole ? b8 % a.nf : blockIdx.x % a.nf;
  const int gc = whole ? b8 / a.nf * 8 + (blockIdx.x & 7) : blockIdx.x / a.nf;
  const int n2 = g.ny2, last = g.ny + 1;
  const int j0 = chunk_start(n2, P, p), cnt = chunk_start(n2, P, p + 1) - j0;
  const bool full = cnt == RPT;  // else RPT - 1 rows
  // the columns lie in one z slab (TC divides nx): its base, and offsets within it
  const long long q0 = pcol(g, (long long)gc * TC), slab = q0 - (q0 & (g.nx - 1));
  const unsigned x0 = (unsigned)(q0 & (g.nx - 1)) + cc;
  TU* u = a.u[e] + slab;
  TU* r = a.r[e] + slab;
  const TV* nt = a.visc[e] + slab;
  // an element by its 32-bit byte offset (the base stays in scalar registers)
  auto ld = [](auto* base, unsigned o) {
    using E = typename std::remove_const<typename std::remove_pointer<decltype(base)>::type>::type;
    return *(const __attribute__((address_space(1))) E*)((const char*)base + o * (unsigned)sizeof(E));
  };
  // rows past the field are read in bounds and their values not used
  TU uu[RPT + 2], rr[RPT];
  TV vv[RPT + 2];
#pragma unroll
  for (int m = 0; m < RPT + 2; ++m) {
    const int j = j0 - 1 + m;
    const unsigned o = (unsigned)(j < 0 ? 0 : (j > last ? last : j)) * g.nx + x0;
    uu[m] = ld(u, o);
    vv[m] = ld(nt, o);
    if (m < RPT) rr[m] = ld(r, (unsigned)(j + 1 > last ? last : j + 1) * g.nx + x0);
  }
  for (int j = tid; j < n2; j += NT) srow[j] = cn_row(a, e, j);
  __syncthreads();
  const double T = a.tcn[e], t2 = a.temp2;
  const bool v2 = a.field[e] == 1;  // nu_t averaged to the faces
  const int wlo = a.wlo[e], whi = a.whi[e];
  // forward: x_m = G_m - A_m x_L - Q_m x_{m+1} for the thread's rows
  double A[RPT], Q[RPT], G[RPT];
#pragma unroll
  for (int m = 0; m < RPT; ++m) {
    const CnRow& R = srow[min(j0 + m, last)];
    const double um = (double)uu[m], uc = (double)uu[m + 1], up = (double)uu[m + 2];
    const double nm = (double)vv[m], nc = (double)vv[m + 1], np = (double)vv[m + 2];
    const double nlo = v2 ? 0.5 * (nc + nm) : nc, nhi = v2 ? 0.5 * (nc + np) : np;
    const double lo = (T + t2 * nlo) * R.ilo, hi = (T + t2 * nhi) * R.ihi;
    double l = R.l - lo, c = R.c - hi, d = R.d + lo + hi;
    double rhs = R.rhs + R.w * (INC ? (double)rr[m] + uc : (double)rr[m]);
    rhs = rhs + t2 * (nhi * (up - uc) * R.ihi - nlo * (uc - um) * R.ilo);
    if (INC) rhs = rhs - (l * um + d * uc + c * up);
    if (m > 0) {
      d = d - l * Q[m - 1];
      rhs = rhs - l * G[m - 1];
      l = -l * A[m - 1];
    }
    const double rb = 1.0 / d;
    A[m] = l * rb;
    Q[m] = c * rb;
    G[m] = rhs * rb;
    __builtin_amdgcn_sched_barrier(0);  // one row at a time: interleaved rows cost registers
  }
  // the chunk's last row, and its first row as x_0 = f - fa x_L - fe x_R
  static_assert(RPT >= 2, "every chunk has a row");
  constexpr int LS = RPT - 2;  // the last row of a chunk of RPT - 1
  const double sa = full ? A[RPT - 1] : A[LS], sq = full ? Q[RPT - 1] : Q[LS], sg = full ? G[RPT - 1] : G[LS];
  double fa = full ? A[LS] : 0.0, fe = full ? Q[LS] : 0.0, f = full ? G[LS] : 0.0;
#pragma unroll
  for (int m = RPT - 3; m >= 0; --m) {
    const bool first = m == RPT - 3 && !full;  // the row above a short chunk's last
    fa = first ? A[m] : A[m] - Q[m] * fa;
    f = first ? G[m] : G[m] - Q[m] * f;
    fe = first ? Q[m] : -(Q[m] * fe);
  }
  double *cur = sx, *nxt = sx + 3 * NT;
  auto put = [&](double* b, double x, double y, double z) { b[tid] = x; b[NT + tid] = y; b[2 * NT + tid] = z; };
  put(cur, fa, fe, f);
  __syncthreads();
  double al = sa, ga = sq, de = sg;  // x_R + al x_L + ga x_{next R} = de
  if (p + 1 < P) {
    const int cntn = chunk_start(n2, P, p + 2) - chunk_start(n2, P, p + 1);
    if (cntn > 1) {  // else the next chunk's first row is its last
      const int w = tid + TC;
      const double rb = 1.0 / (1.0 - sq * cur[w]);
      al = sa * rb;
      ga = -(sq * cur[NT + w]) * rb;
      de = (sg - sq * cur[2 * NT + w]) * rb;
    }
  }
  put(nxt, al, ga, de);
  __syncthreads();
  { double* t = cur; cur = nxt; nxt = t; }
  for (int s = 1; s < P; s <<= 1) {
    const bool dn = p >= s, up = p + s < P;
    const int wd = dn ? tid - s * TC : tid, wu = up ? tid + s * TC : tid;
    const double ad = dn ? al : 0.0, gu = up ? ga : 0.0;
    const double rb = 1.0 / (1.0 - ad * cur[NT + wd] - gu * cur[wu]);
    de = (de - ad * cur[2 * NT + wd] - gu * cur[2 * NT + wu]) * rb;
    al = -(ad * cur[wd]) * rb;
    ga = -(gu * cur[NT + wu]) * rb;
    put(nxt, al, ga, de);
    __syncthreads();
    double* t = cur; cur = nxt; nxt = t;
  }
  // back substitution
  const double xl = p > 0 ? cur[2 * NT + tid - TC] : 0.0;
  double x = de;
#pragma unroll
  for (int m = RPT - 1; m >= 0; --m) {
    const int j = j0 + m;
    const bool own = m + 1 < RPT || full;
    if (m == RPT - 2) x = full ? G[m] - A[m] * xl - Q[m] * x : x;
    else if (m < RPT - 2) x = G[m] - A[m] * xl - Q[m] * x;
    if (own) {
      const unsigned o = (unsigned)j * g.nx + x0;
      const bool in = j >= wlo && j <= whi;
      if (INC) r[o] = (TU)(in ? x : 0.0);
      else if (in) u[o] = (TU)x;
    }
  }
}

// ---- host side (dgpu_cn_phys.hip): FP64, FP64 with float nu_t, float increments
int launch_cn_phys(const PhysCnArgs<double, double>& a, hipStream_t st);
int launch_cn_phys(const PhysCnArgs<double, float>& a, hipStream_t st);
int launch_cn_phys(const PhysCnArgs<float, float>& a, hipStream_t st);

}  // namespace dgpu
