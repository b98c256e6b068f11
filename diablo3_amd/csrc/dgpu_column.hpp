// dgpu_column.hpp — the column kernels of a substep, register resident.
//
// k_column: per (kx, kz) column and all rows j = 0..Nyp+1
//  1. Fourier-space assembly of rk_chan_1 (for/solver.f90:385-838, 909-973, and
//     user_rhs_chan_fourier 35-111): new RK memory cf and the right-hand side cr,
//     including the explicit half of Crank–Nicolson (for/solver.f90:850-870,
//     981-1002) and the BC rows of apply_BC_* (for/solver.f90:1901-2232);
//  2. the Crank–Nicolson solves of every scalar, u2, u1, u3 (for/solver.f90:
//     1004-1233) in Fourier space (the DNS operator does not depend on x or z);
//  3. rem_div_chan (for/solver.f90:1302-1379, BC rows 2330-2371), the velocity
//     correction and the pressure update (for/solver.f90:1261-1267).
// k_project: step 3 alone on a state in memory (LES substeps, rem_div_chan,
// poisson_p_chan).
//
// A block owns TC columns; thread (p, cc) owns the rows of chunk p of column cc,
// RPT of them at most, and keeps them in registers from the assembly to the
// corrected velocity: with every state field read once and written once 632 MB a
// substep at 256x129x256 FP64.  Counted, it is 793 MB (516 in, 277 out): a chunk reads
// the rows next to it again, and a short chunk (29 of 32 there) the row it does not
// own.  (942 MB counted for an assembly + solve kernel that kept its right-hand sides
// in LDS and a projection kernel that read the velocity back.)  What crosses chunks is
// small and goes through shuffles (the chunks of
// one wave) and LDS (the waves of a block): the carries of the two Thomas sweeps,
// and the Poisson system of the chunks' last rows.
//
// Measured (MI355X, per substep, those two kernels -> k_column): 256x129x256 FP64
// 268 -> 179 us, mixed 269 -> 169; 64x65x64 FP64 23.5 -> 18.4; 128x97x64 mixed, two
// scalars 55 -> 37.  k_project alone (LES), 512x257x512: 709 -> 520 us.  What bounds
// k_column is that traffic (4.4 TB/s; a large one-read-one-write pass reaches 5.7) and
// the length of one block's chain (rows one after another, then the scans and log2 P
// exchange steps): waves wait 44% of their cycles, at 1.5 waves per SIMD, which 256
// registers a thread allow (5 rows and one scalar: all 256, and 12 bytes of scratch).
// On the smallest grids the chain is all of it: with 11 blocks (16 points in x and z) it
// takes up to 1 us longer than the two kernels, whose blocks were narrower (a step of
// 16x65x16 103 -> 105 us; 32x65x32 122 -> 119).
#pragma once
#include "dgpu_kernels.hpp"

#include <type_traits>

namespace dgpu {

constexpr int COLUMN_NT = 512;    // threads per block at most: 256 registers per thread
constexpr int COLUMN_ROWS = 320;  // rows whose tables fit LDS beside the exchange (8 columns, 5 rows a chunk)

// The tallest column a DNS step takes: 80 KiB of right-hand sides (16 bytes a row and
// field), a limit of the interface.  No kernel holds them any more; the projection and
// the LES step take every row count of a handle.
__host__ __device__ constexpr int column_max_rows(int nth) { return 80 * 1024 / (16 * (3 + nth)); }

// Columns per block, chunks per column (a power of two), rows per chunk: a chunk
// holds rpt or rpt - 1 rows.
struct ColShape {
  int tc, P, rpt;
  bool big;
};

// The row coefficients the column kernels take: the first RQ of RowCoef, staged in
// LDS, or in global memory on the tall columns (BIG).
template <int NTH>
constexpr int RQ = RC_TW0 + 4 * NTH;
__device__ __forceinline__ void stage_rows(double* __restrict__ s, const double* __restrict__ rowc, int n2, int rq,
                                           int tid, int NT) {
  for (int t = tid; t < n2 * rq; t += NT) {
    const int j = t / rq, k = t - j * rq;
    s[t] = rowc[(long long)j * RC_COUNT + k];
  }
}
// Complex values at a byte offset from a device-memory base.  A 32-bit offset that
// is formed where it is used leaves the base in scalar registers (pin keeps the
// compiler from carrying its 64-bit extension from an earlier use).
template <typename T, typename I>
__device__ __forceinline__ cx<T> gload(const void* base, I off) {
  typedef T v2 __attribute__((ext_vector_type(2)));
  const v2 v = *(const __attribute__((address_space(1))) v2*)((const char*)base + off);
  return {v.x, v.y};
}
template <typename I>
__device__ __forceinline__ void gstore(void* base, I off, cd z) {
  typedef double v2 __attribute__((ext_vector_type(2)));
  *(__attribute__((address_space(1))) v2*)((char*)base + off) = v2{z.x, z.y};
}
__device__ __forceinline__ unsigned pin(unsigned o) {
  asm("" : "+v"(o));
  return o;
}
__device__ __forceinline__ long long pin(long long o) { return o; }

// LDS of k_column, in doubles: the row coefficients; the CN factors with the wave
// totals of the scans behind them, later the Poisson exchange; the old pressures.
// On the tall columns (big) the coefficients and factors stay in global memory.
__host__ __device__ constexpr int column_part(int n2, int nth, int nt, bool big) {
  const int f = big ? 0 : 3 * (3 + nth) * n2, head = f > 6 * nt ? f : 6 * nt;
  return head + 4 * nt > 12 * nt ? head + 4 * nt : 12 * nt;
}
constexpr size_t column_lds(int n2, int nth, int nt, int rpt, bool big) {
  return 8 * ((size_t)(big ? 0 : n2 * (RC_TW0 + 4 * nth)) + column_part(n2, nth, nt, big) + (size_t)2 * rpt * nt);
}
constexpr size_t project_lds(int n2, int nt, int rpt, bool big) {
  return 8 * ((size_t)(big ? 0 : n2 * RC_TW0) + (size_t)(12 + 2 * rpt) * nt);
}

// The value computed here and not later (the compiler sinks arithmetic to its use,
// and holds the inputs in registers until then).
__device__ __forceinline__ cd here(cd v) {
  asm volatile("" : "+v"(v.x), "+v"(v.y));
  return v;
}
__device__ __forceinline__ cd pick(bool c, cd a, cd b) { return {c ? a.x : b.x, c ? a.y : b.y}; }

// ---------------------------------------------------------------------------
// The Poisson rows 1..Nyp of rem_div_chan by partition: the thread eliminates its
// chunk's rows down to a coupling with the last row of the chunk before (L) and
// its own last row (R); the last rows of all chunks form a tridiagonal system of P
// unknowns, solved by parallel cyclic reduction in LDS; the rows in between follow
// by back substitution.  (Whole-column cyclic reduction spends 8 levels on 129
// rows with two divisions per row and level; here a row costs two divisions and
// a chunk two per level of log2 P.)
//
// Every row is kept with off-diagonals a, c >= 0 and diagonal b <= 0 (the bottom
// BC row is negated), and by its row sum s = a + b + c instead of b: the interior
// rows sum to exactly -(kx^2 + kz^2) and the BC rows to 0 (or -1 for the
// Dirichlet row of the (0,0) mode).  Adding al times row i to row j (al >= 0) adds
// the row sums and couplings, all of one sign, and b = s - a - c follows without
// cancellation, where the textbook b + al c cancels almost all of b for the weakly
// dominant rows of small kx^2 + kz^2 (on a 257-row stretched grid plain cyclic
// reduction lost 3-4 digits there).  Rows 0 and Nyp+1 are decoupled (s = -1).
//
// d: right-hand sides in, the solution out; returns the solution of row j0 - 1.
// Caller: a barrier before the call if other threads still read sm.
// ---------------------------------------------------------------------------
template <int TC, int RPT, typename RL>
__device__ __forceinline__ cd poisson_chunk(const ColArgs& a, RL rl, double k2, int c, int j0, int cnt, int p, int P,
                                            int tid, double* __restrict__ sm, cd* d) {
  const int ny = a.g.ny, n2 = a.g.ny2, NT = P * TC;
  double A[RPT], S[RPT], rB[RPT], C[RPT];
#pragma unroll
  for (int m = 0; m < RPT; ++m) {
    const int j = j0 + m;
    const auto rc = rl(min(j, n2 - 1));
    const bool in = j > 1 && j < ny;
    double aj = in ? rc[RC_FLO] : 0.0, cj = in ? rc[RC_FHI] : 0.0, sj = in ? k2 : -1.0;
    if (j == 1) {
      // (1, -1) Neumann, or (1) for phi(1) = 0 in the (0,0) mode; negated
      cj = (c == 0) ? 0.0 : 1.0;
      sj = (c == 0) ? -1.0 : 0.0;
    }
    if (j == ny) { aj = 1.0; sj = 0.0; }  // (1, -1)
    C[m] = cj;
    if (m == 0) {
      A[0] = aj; S[0] = sj;
    } else {
      const double al = -aj * rB[m - 1];
      A[m] = al * A[m - 1];
      S[m] = sj + al * S[m - 1];
      d[m] = d[m] + al * d[m - 1];
    }
    rB[m] = 1.0 / (S[m] - A[m] - cj);
  }
  // the chunk's own last row, and its first row in terms of L and R (the rows
  // between eliminated upwards; E couples to R)
  const bool full = cnt == RPT;
  double sA = 0.0, sS = -1.0, sC = 0.0, fA = 0.0, fS = -1.0, fE = 0.0;
  cd sD = {0.0, 0.0}, fD = {0.0, 0.0};
  constexpr int LS = RPT >= 2 ? RPT - 2 : 0;  // the last row of a chunk of RPT - 1
  sA = full ? A[RPT - 1] : (RPT >= 2 ? A[LS] : sA);
  sS = full ? S[RPT - 1] : (RPT >= 2 ? S[LS] : sS);
  sC = full ? C[RPT - 1] : (RPT >= 2 ? C[LS] : sC);
  sD = pick(full, d[RPT - 1], RPT >= 2 ? d[LS] : sD);
  if constexpr (RPT >= 2) {
    fA = full ? A[LS] : fA;
    fS = full ? S[LS] : fS;
    fE = full ? C[LS] : fE;
    fD = pick(full, d[LS], fD);
#pragma unroll
    for (int m = RPT - 3; m >= 0; --m) {
      const bool first = m == RPT - 3 && !full;  // the row above a short chunk's last
      const double ga = first ? 0.0 : -C[m] / (fS - fA - fE);
      fA = A[m] + ga * fA;
      fS = S[m] + ga * fS;
      fE = first ? C[m] : ga * fE;
      fD = d[m] + ga * fD;
    }
  }
  // exchange rows of six values: a, s, c, 1/b and the right-hand side
  auto put = [&](double* b, double u, double v, double w, cd z) {
    b[tid] = u; b[NT + tid] = v; b[2 * NT + tid] = w; b[3 * NT + tid] = 1.0 / (v - u - w);
    b[4 * NT + tid] = z.x; b[5 * NT + tid] = z.y;
  };
  double *cur = sm + 6 * NT, *nxt = sm;
  put(nxt, fA, fS, fE, fD);
  __syncthreads();
  if (p + 1 < P) {
    const int q = tid + TC;
    const int cntn = chunk_start(n2, P, p + 2) - chunk_start(n2, P, p + 1);
    if (cntn > 1) {  // else the next chunk's first row is its last: C couples to it
      const double ga = -sC * nxt[3 * NT + q];
      sC = ga * nxt[2 * NT + q];
      sS = sS + ga * nxt[NT + q];
      sD = sD + ga * cd{nxt[4 * NT + q], nxt[5 * NT + q]};
    }
  }
  put(cur, sA, sS, sC, sD);
  __syncthreads();
  for (int s = 1; s < P; s <<= 1) {
    double a2 = 0.0, c2 = 0.0;
    if (p - s >= 0) {
      const int q = tid - s * TC;
      const double al = -sA * cur[3 * NT + q];
      a2 = al * cur[q];
      sS = sS + al * cur[NT + q];
      sD = sD + al * cd{cur[4 * NT + q], cur[5 * NT + q]};
    }
    if (p + s < P) {
      const int q = tid + s * TC;
      const double ga = -sC * cur[3 * NT + q];
      c2 = ga * cur[2 * NT + q];
      sS = sS + ga * cur[NT + q];
      sD = sD + ga * cd{cur[4 * NT + q], cur[5 * NT + q]};
    }
    sA = a2; sC = c2;
    put(nxt, sA, sS, sC, sD);
    __syncthreads();
    double* t = cur; cur = nxt; nxt = t;
  }
  // every unknown stands alone: the chunk's last row and the one before the chunk
  const cd R = cur[3 * NT + tid] * sD;
  cd Lv = {0.0, 0.0};
  if (p > 0) Lv = cur[3 * NT + tid - TC] * cd{cur[4 * NT + tid - TC], cur[5 * NT + tid - TC]};
  d[RPT - 1] = pick(full, R, d[RPT - 1]);
#pragma unroll
  for (int m = RPT - 2; m >= 0; --m) {
    const cd v = rB[m] * (d[m] - A[m] * Lv - C[m] * d[m + 1]);
    d[m] = (m == RPT - 2) ? pick(full, v, R) : v;
  }
  return Lv;
}

// project = 0 stops after the Crank–Nicolson solves (courant reads that velocity).
template <typename T, int NTH, int TC, int RPT, bool BIG>
__global__ __launch_bounds__(COLUMN_NT) void k_column(ColArgs a, int project) {
  constexpr int NF = 3 + NTH;
  using Ix = typename std::conditional<BIG, long long, unsigned>::type;
  extern __shared__ double smd[];
  const Geo& g = a.g;
  const int n2 = g.ny2, ny = g.ny, tid = threadIdx.x, NT = blockDim.x, P = NT / TC;
  const int cc = tid % TC, p = tid / TC;
  const int tile = xcd_tile(blockIdx.x, (int)(g.pc / TC));
  if (tile < 0) return;
  const int c = tile * TC + cc;  // column in the padded plane: c = k*kxp + i
  const int i = c % g.kxp, k = c / g.kxp;
  const bool active = i < g.kxr, mean = c == 0;
  const Ix pc16 = (Ix)g.pc * 16, c16 = (Ix)c * 16;  // bytes of a plane, of the columns before c
  const int j0 = chunk_start(n2, P, p), cnt = chunk_start(n2, P, p + 1) - j0;
  const bool full = cnt == RPT;  // else RPT - 1 rows
  const double kxi = active ? a.kx[i] : 0.0, kzk = a.kz[k];
  double* srow = smd;                                       // row coefficients
  double* sfac = srow + (BIG ? 0 : n2 * RQ<NTH>);           // CN factors [NF][3][n2], then the Poisson exchange
  double* spx = sfac + column_part(n2, NTH, NT, BIG);       // the thread's old pressures, [RPT][2][NT]
  auto rl = [&](int j) -> const double* {
    if constexpr (BIG) return a.rowc + (long long)j * RC_COUNT;
    else return srow + j * RQ<NTH>;
  };

  // ---- 1. assembly of cf and cr, row by row with a three-row window of the state;
  // the loads of row j + 1 are issued before row j is assembled.  Rows past the
  // field and the padding columns (zero) are read in bounds and dropped.
  cd x[NF][RPT];
  {
    const ColK K = col_k(a, kxi, kzk, mean);
    auto off = [&](int j) { return (Ix)(j < 0 ? 0 : (j >= n2 ? n2 - 1 : j)) * pc16 + c16; };
    RowIn<NTH> r, nx;
    // the RK memory's addresses and whether row 1 is an equation's own, held in
    // scalar registers (left to itself the compiler reads them again at each store,
    // one exposed scalar load after the other)
    cd* cfp[NF];
    int own1 = 0;
#pragma unroll
    for (int e = 0; e < NF; ++e) {
      cfp[e] = a.cf[e];
      asm volatile("" : "+s"(cfp[e]));
      own1 |= a.rows[e].blo <= 1 ? 1 << e : 0;
    }
    own1 = __builtin_amdgcn_readfirstlane(own1);
    auto fetch = [&](int j) {
      const Ix o = pin(off(j)), op = pin(off(j + 1));
#pragma unroll
      for (int e = 0; e < NF; ++e) nx.up[e] = gload<double>(a.u[e], op);
      nx.pc_ = gload<double>(a.p, o);
#pragma unroll
      for (int e = 0; e < NF; ++e) nx.nl[e] = cvt<double>(gload<T>(a.nl[e], sizeof(T) == 8 ? o : o / 2));
#pragma unroll
      for (int e = 0; e < NF; ++e) nx.cfo[e] = cd{0.0, 0.0};
      if (a.rk > 1) {
#pragma unroll
        for (int e = 0; e < NF; ++e) nx.cfo[e] = gload<double>(cfp[e], o);
      }
    };
    {
      const Ix o = off(j0), om = off(j0 - 1);
      r.pc_ = gload<double>(a.p, om);
#pragma unroll
      for (int e = 0; e < NF; ++e) { r.uc[e] = gload<double>(a.u[e], om); r.up[e] = gload<double>(a.u[e], o); }
    }
    fetch(j0);
    if constexpr (!BIG) {  // the tables, while the first rows are on their way
      stage_rows(srow, a.rowc, n2, RQ<NTH>, tid, NT);
      for (int t = tid; t < NF * 3 * n2; t += NT) sfac[t] = a.thc[t];
      __syncthreads();
    }
#pragma unroll
    for (int m = 0; m < RPT; ++m) {
      const int j = j0 + m;
      r.pm = r.pc_; r.pc_ = nx.pc_;
#pragma unroll
      for (int e = 0; e < NF; ++e) {
        r.um[e] = r.uc[e]; r.uc[e] = r.up[e]; r.up[e] = nx.up[e];
        r.nl[e] = nx.nl[e]; r.cfo[e] = nx.cfo[e];
      }
      if (m + 1 < RPT) fetch(j + 1);
      // one row of loads ahead and no more: the scheduler would hoist them all (spills)
      __builtin_amdgcn_sched_barrier(0);
      cd cf[NF], cr[NF];
      assemble_row<NTH>(a, r, rl(min(j, n2 - 1)), K, cf, cr);
#pragma unroll
      for (int e = 0; e < NF; ++e) x[e][m] = here(cr[e]);
      spx[2 * m * NT + tid] = r.pc_.x;
      spx[(2 * m + 1) * NT + tid] = r.pc_.y;
      const bool own = active && (m + 1 < RPT || full) && j <= ny;
      if (own && j >= 2) {
        const Ix o = pin(off(j));
#pragma unroll
        for (int e = 0; e < NF; ++e) gstore(cfp[e], o, cf[e]);
      } else if (own && j == 1) {
        const Ix o = pin(off(j));
#pragma unroll
        for (int e = 0; e < NF; ++e)
          if (own1 >> e & 1) gstore(cfp[e], o, cf[e]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (mean) {
      const double f = mean_dpdx(a);
#pragma unroll
      for (int m = 0; m < RPT; ++m) x[0][m].x = x[0][m].x - f;
    }
    // the BC rows (every row that no equation owns is one): zero, in the mean mode
    // the BC value
    if (j0 <= 2 || j0 + RPT > ny) {
#pragma unroll
      for (int m = 0; m < RPT; ++m) {
        const int j = j0 + m, sr = j <= 2 ? j : (j >= ny ? j - ny + 3 : 5);
        const unsigned bits = sr < 5 ? (unsigned)(a.bcmask >> (sr * MAXF)) : 0u;
#pragma unroll
        for (int e = 0; e < NF; ++e) {
          x[e][m] = pick(bits >> e & 1, cd{0.0, 0.0}, x[e][m]);
          if (mean && (bits >> e & 1)) x[e][m].x = a.rows[e].val[sr];
        }
      }
    }
  }

  // ---- 2. Thomas with the host's factorisation in chunks: local elimination from
  // zero, the chunk-boundary carries (the affine maps y -> A y + B compose) by a
  // shuffle scan over the chunks of a wave and a fold over the waves, and the
  // fix-up with the host's in-chunk products.  The same linear map as
  // thomas_forward/backward_real_mpi (for/solver.f90:1691-1761, 1816-1852); the
  // fields' systems are independent.
  constexpr int PW = 64 / TC;  // chunks per wave
  const int w = tid >> 6, NW = NT >> 6, pl = p % PW;
  auto fac = [&](int e, int q, int m) {
    const int t = (e * 3 + q) * n2 + min(j0 + m, n2 - 1);
    if constexpr (BIG) return a.thc[t];
    else return sfac[t];
  };
  double* swf = sfac + max(BIG ? 0 : NF * 3 * n2, 6 * NT);  // wave totals, [wave][NF][3][TC]
  double* swb = swf + 2 * NT;
  {
    double Ax[NF];
    cd Bx[NF];
#pragma unroll
    for (int e = 0; e < NF; ++e) {
      double Af = 1.0;
      cd Bf = {0.0, 0.0};
#pragma unroll
      for (int m = 0; m < RPT; ++m) {
        const double mu = fac(e, 0, m);
        x[e][m] = x[e][m] + mu * Bf;
        Bf = (m + 1 < RPT) ? x[e][m] : pick(full, x[e][m], Bf);
        Af = (m + 1 < RPT || full) ? Af * mu : Af;
      }
#pragma unroll
      for (int s = 1; s < PW; s <<= 1) {
        const double Au = __shfl_up(Af, s * TC);
        const cd Bu = {__shfl_up(Bf.x, s * TC), __shfl_up(Bf.y, s * TC)};
        if (pl >= s) {
          Bf = Af * Bu + Bf;
          Af = Af * Au;
        }
      }
      if (pl == PW - 1) {
        double* t = swf + ((w * NF + e) * 3) * TC + cc;
        t[0] = Af; t[TC] = Bf.x; t[2 * TC] = Bf.y;
      }
      Ax[e] = __shfl_up(Af, TC);
      Bx[e] = cd{__shfl_up(Bf.x, TC), __shfl_up(Bf.y, TC)};
      if (pl == 0) { Ax[e] = 1.0; Bx[e] = cd{0.0, 0.0}; }
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < NF; ++e) {
      cd y = {0.0, 0.0};
      for (int q = 0; q < w; ++q) {
        const double* t = swf + ((q * NF + e) * 3) * TC + cc;
        y = t[0] * y + cd{t[TC], t[2 * TC]};
      }
      y = Ax[e] * y + Bx[e];
#pragma unroll
      for (int m = 0; m < RPT; ++m) {
        y = fac(e, 0, m) * y;
        x[e][m] = x[e][m] + y;
      }
    }
  }
  {
    double Ax[NF];
    cd Bx[NF];
#pragma unroll
    for (int e = 0; e < NF; ++e) {
      double Ab = 1.0;
      cd Bb = {0.0, 0.0};
#pragma unroll
      for (int m = RPT - 1; m >= 0; --m) {
        const double ga = fac(e, 2, m);
        x[e][m] = fac(e, 1, m) * x[e][m] + ga * Bb;
        Bb = (m + 1 < RPT) ? x[e][m] : pick(full, x[e][m], Bb);
        Ab = (m + 1 < RPT || full) ? Ab * ga : Ab;
      }
#pragma unroll
      for (int s = 1; s < PW; s <<= 1) {
        const double Ad = __shfl_down(Ab, s * TC);
        const cd Bd = {__shfl_down(Bb.x, s * TC), __shfl_down(Bb.y, s * TC)};
        if (pl + s < PW) {
          Bb = Ab * Bd + Bb;
          Ab = Ab * Ad;
        }
      }
      if (pl == 0) {
        double* t = swb + ((w * NF + e) * 3) * TC + cc;
        t[0] = Ab; t[TC] = Bb.x; t[2 * TC] = Bb.y;
      }
      Ax[e] = __shfl_down(Ab, TC);
      Bx[e] = cd{__shfl_down(Bb.x, TC), __shfl_down(Bb.y, TC)};
      if (pl == PW - 1) { Ax[e] = 1.0; Bx[e] = cd{0.0, 0.0}; }
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < NF; ++e) {
      cd y = {0.0, 0.0};
      for (int q = NW - 1; q > w; --q) {
        const double* t = swb + ((q * NF + e) * 3) * TC + cc;
        y = t[0] * y + cd{t[TC], t[2 * TC]};
      }
      y = Ax[e] * y + Bx[e];
#pragma unroll
      for (int m = RPT - 1; m >= 0; --m) {
        const cd z = fac(e, 2, m) * y;
        x[e][m] = x[e][m] + z;
        y = (m + 1 < RPT) ? z : pick(full, z, y);
      }
    }
  }
  // the scalars are done; without the projection the velocity too
#pragma unroll
  for (int m = 0; m < RPT; ++m) {
    const int j = j0 + m;
    if ((m + 1 < RPT || full) && active) {
      const Ix o = pin((Ix)j * pc16 + c16);
#pragma unroll
      for (int e = 0; e < NF; ++e)
        if ((e >= 3 || !project) && j >= a.rows[e].wlo && j <= a.rows[e].whi) gstore(a.u[e], o, x[e][m]);
    }
  }
  if (!project) return;  // uniform over the grid

  // ---- 3. divergence, Poisson, velocity correction, pressure
  double* sx2 = swf;  // u2 of every chunk's first row
  sx2[tid] = x[1][0].x;
  sx2[NT + tid] = x[1][0].y;
  __syncthreads();
  cd up = {0.0, 0.0};
  if (p + 1 < P) up = cd{sx2[tid + TC], sx2[NT + tid + TC]};
  cd d[RPT];
#pragma unroll
  for (int m = RPT - 1; m >= 0; --m) {
    const int j = j0 + m;
    const cd v = ik(kxi, x[0][m]) + rl(min(j, n2 - 1))[RC_RDYF] * (up - x[1][m]) + ik(kzk, x[2][m]);
    d[m] = pick(j > 1 && j < ny, v, cd{0.0, 0.0});
    up = (m + 1 < RPT) ? x[1][m] : pick(full, x[1][m], up);
  }
  cd pl_ = poisson_chunk<TC, RPT>(a, rl, -(kxi * kxi) - kzk * kzk, c, j0, cnt, p, P, tid, sfac, d);
  if (!active) return;
  const double r4 = 1.0 / a.temp4;
#pragma unroll
  for (int m = 0; m < RPT; ++m) {
    const int j = j0 + m;
    if (m + 1 < RPT || full) {
      const Ix o = pin((Ix)j * pc16 + c16);
      if (j >= 1 && j <= ny) {
        const cd phi = d[m];
        gstore(a.u[0], o, x[0][m] - ik(kxi, phi));
        gstore(a.u[2], o, x[2][m] - ik(kzk, phi));
        gstore(a.u[1], o, j >= 2 ? x[1][m] - rl(j)[RC_RDY] * (phi - pl_) : x[1][m]);
        if (j >= a.jstart) gstore(a.p, o, cd{spx[2 * m * NT + tid], spx[(2 * m + 1) * NT + tid]} + r4 * phi);
        pl_ = phi;
      } else {  // the ghost rows the solves write
#pragma unroll
        for (int e = 0; e < 3; ++e)
          if (j >= a.rows[e].wlo && j <= a.rows[e].whi) gstore(a.u[e], o, x[e][m]);
      }
    }
  }
}

// Step 3 on a state in memory; update_p: also the pressure update.  With
// a.prhs it is poisson_p_chan's solve and the solution goes to p.
template <int TC, int RPT, bool BIG>
__global__ __launch_bounds__(COLUMN_NT) void k_project(ColArgs a, int update_p) {
  extern __shared__ double smd[];
  const Geo& g = a.g;
  const int n2 = g.ny2, ny = g.ny, tid = threadIdx.x, NT = blockDim.x, P = NT / TC;
  const int cc = tid % TC, p = tid / TC;
  const int tile = xcd_tile(blockIdx.x, (int)(g.pc / TC));
  if (tile < 0) return;
  const int c = tile * TC + cc;
  const int i = c % g.kxp, k = c / g.kxp;
  const bool active = i < g.kxr;
  const long long pc = g.pc;
  const int j0 = chunk_start(n2, P, p), cnt = chunk_start(n2, P, p + 1) - j0;
  cd* __restrict__ u1 = a.u[0];
  cd* __restrict__ u2 = a.u[1];
  cd* __restrict__ u3 = a.u[2];
  const double kxi = active ? a.kx[i] : 0.0, kzk = a.kz[k];
  const bool full = cnt == RPT;
  double* sex = smd + (BIG ? 0 : n2 * RQ<0>);  // the Poisson exchange
  double* spx = sex + 12 * NT;                 // the thread's old pressures, [RPT][2][NT]
  auto rl = [&](int j) -> const double* {
    if constexpr (BIG) return a.rowc + (long long)j * RC_COUNT;
    else return smd + j * RQ<0>;
  };
  if constexpr (!BIG) stage_rows(smd, a.rowc, n2, RQ<0>, tid, NT);
  cd v1[RPT], v2[RPT], v3[RPT], d[RPT];
  if (a.prhs) {
    // poisson_p_chan (for/solver.f90:1382-1560): vec = -(source + the scalars' y
    // gradient, except in the (0, 0) mode).  Rows past the chunk are read in bounds and
    // dropped, as below: loads under a row's own condition wait for one another
    // (poisson_p with its transforms, us: 64x65x64 58.8 -> 57.7, 256x129x256 665 -> 656,
    // 64x385x64 158.5 -> 152.1; the kernel of one row a thread before it 57.2, 657, 154)
    double yf[RPT + 2];
    auto row = [&](int m) { const int j = j0 - 1 + m; return j < 0 ? 0 : (j >= n2 ? n2 - 1 : j); };
#pragma unroll
    for (int m = 0; m < RPT; ++m) d[m] = a.prhs[(long long)row(m + 1) * pc + c];
#pragma unroll
    for (int m = 0; m < RPT + 2; ++m) yf[m] = a.gyf[row(m)];
    for (int n = 0; n < a.pnth; ++n) {
      cd t[RPT + 2];
#pragma unroll
      for (int m = 0; m < RPT + 2; ++m) t[m] = a.u[3 + n][(long long)row(m) * pc + c];
#pragma unroll
      for (int m = 0; m < RPT; ++m) {
        const cd dt = t[m + 2] - t[m];
        const double den = yf[m + 2] - yf[m];
        d[m] = pick(c != 0, d[m] + cd{dt.x / den, dt.y / den}, d[m]);
      }
    }
#pragma unroll
    for (int m = 0; m < RPT; ++m) {
      const int j = j0 + m;
      d[m] = pick((m + 1 < RPT || full) && j > 1 && j < ny && active, -1.0 * d[m], cd{0.0, 0.0});
    }
    __syncthreads();  // the row coefficients
  } else {
    // rows past the chunk and the padding columns (zero) are read in bounds and
    // dropped: the loads carry no condition, so all are in flight together
    cd up;
#pragma unroll
    for (int m = 0; m < RPT; ++m) {
      const long long o = (long long)min(j0 + m, n2 - 1) * pc + c;
      v1[m] = u1[o]; v2[m] = u2[o]; v3[m] = u3[o];
    }
    up = u2[(long long)min(j0 + cnt, n2 - 1) * pc + c];
    if (update_p) {  // the old pressures too, kept in LDS
#pragma unroll
      for (int m = 0; m < RPT; ++m) {
        const cd q = a.p[(long long)min(j0 + m, n2 - 1) * pc + c];
        spx[2 * m * NT + tid] = q.x;
        spx[(2 * m + 1) * NT + tid] = q.y;
      }
    }
    __syncthreads();  // the row coefficients
#pragma unroll
    for (int m = RPT - 1; m >= 0; --m) {
      const int j = j0 + m;
      const cd v = ik(kxi, v1[m]) + rl(min(j, n2 - 1))[RC_RDYF] * (up - v2[m]) + ik(kzk, v3[m]);
      d[m] = pick(j > 1 && j < ny, v, cd{0.0, 0.0});
      up = (m + 1 < RPT) ? v2[m] : pick(full, v2[m], up);
    }
  }
  cd pl_ = poisson_chunk<TC, RPT>(a, rl, -(kxi * kxi) - kzk * kzk, c, j0, cnt, p, P, tid, sex, d);
  if (!active) return;
  const double r4 = 1.0 / a.temp4;
#pragma unroll
  for (int m = 0; m < RPT; ++m) {
    const int j = j0 + m;
    if ((m + 1 < RPT || full) && j >= 1 && j <= ny) {
      const long long o = (long long)j * pc + c;
      const cd phi = d[m];
      if (a.prhs) {  // cp(j) = vec(j), j = 1..Nyp
        a.p[o] = phi;
        continue;
      }
      u1[o] = v1[m] - ik(kxi, phi);
      u3[o] = v3[m] - ik(kzk, phi);
      if (j >= 2) u2[o] = v2[m] - rl(j)[RC_RDY] * (phi - pl_);
      if (update_p && j >= a.jstart) a.p[o] = cd{spx[2 * m * NT + tid], spx[(2 * m + 1) * NT + tid]} + r4 * phi;
      pl_ = phi;
    }
  }
}


// ---- host side (dgpu_column.hip)
// the shape for a grid; false where no shape holds the column
bool column_shape(const Geo& g, ColShape* s);
int launch_column(const ColArgs& a, const ColShape& s, int nth, bool mixed, int project, hipStream_t st);
int launch_project(const ColArgs& a, const ColShape& s, int update_p, hipStream_t st);

}  // namespace dgpu
