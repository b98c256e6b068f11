// dgpu_kernels.hpp — HIP kernels of the RKW3 + CN channel step (gfx950).
//
// Device layouts (one rank, Nyp = ny):
//   Fourier  C[j][k][i]  complex double, i = 0..Nkx active (kxr of them) in rows of
//                        pitch kxp = kxr rounded up to 8 (128-byte rows for complex
//                        double), k = 0..2Nkz (kzr), j = 0..ny+1; pc = kxp*kzr.
//   x-spectra H[j][z][i] complex T: the x transform of physical line (j, z)
//                        restricted to i = 0..Nkx, same pitch kxp (ph = nz*kxp).
//   physical R[z][j][x]  T (pp = nz*nx points a plane): the y column of a point lies in
//                        one slab of ny2 nx values, rows nx apart.  The kernels
//                        that march or solve in y then stay within a page or two;
//                        with z inside j ([j][z][x]) the rows of a column are nz nx
//                        values apart, a page each.
// Padding columns i = kxr..kxp-1 are zero and never read as modes.
// Every kernel indexes only inside these extents; grids are sized by the host to
// the same extents (the host checks them before launch).
#pragma once
#include "dgpu_fft.hpp"

namespace dgpu {

constexpr int MAXTH = 4;
constexpr int MAXF = 3 + MAXTH;         // u1, u2, u3, th_1..th_n
constexpr int MAXO = 3 * MAXF;         // largest transform batch (LES: v, dv/dx, dv/dz)

struct Geo {
  int nx, nz, ny, ny2, nkx, nkz, kxr, kzr, kxp;
  long long pc, ph, pp;
  int lx;  // log2 nx
};
// first point of physical line (j, z); a point of plane 0 by its index z nx + x, and
// the distance from row to row
__host__ __device__ __forceinline__ long long pline(const Geo& g, int j, int z) {
  return ((long long)z * g.ny2 + j) * g.nx;
}
__device__ __forceinline__ long long pcol(const Geo& g, long long q) {
  return ((q >> g.lx) * g.ny2 << g.lx) + (q & (g.nx - 1));
}

// Rows 0..n-1 in P chunks: base rows each, one more for the last n mod P of them.
__host__ __device__ inline int chunk_start(int n, int P, int p) {
  const int base = n / P, rem = n - base * P, extra = p - (P - rem);
  return p * base + (extra > 0 ? extra : 0);
}

template <typename P, int M>
struct Ptrs {
  P p[M];
};

// packed kz index p -> row of the length-nz z transform (for/fft.f90:293-305, 316-333)
__device__ __forceinline__ int zpos(const Geo& g, int p) { return p <= g.nkz ? p : p + g.nz - g.kzr; }
// row z of the z transform -> packed index, or -1 for the de-aliased rows
__device__ __forceinline__ int zpack(const Geo& g, int z) {
  return z <= g.nkz ? z : (z >= g.nz - g.nkz ? z - g.nz + g.kzr : -1);
}

// Tile order for the 8 XCDs: the dispatcher deals blocks (in linear order) to
// the XCDs in turn, so within each group of 8 K consecutive blocks XCD x is
// given the K consecutive tiles x K .. x K + K - 1.  Neighbouring column blocks
// of a z transform each read half of the same 128-byte line of every z row;
// ordered this way they run on one XCD together and the second half comes from
// its L2.  Blocks past the last whole group keep their own index.
__device__ __forceinline__ int xcd_tile(int b, int total, int K) {
  const int C = 8 * K;
  if (b >= (total / C) * C) return b;
  return (b / C) * C + (b & 7) * K + (b % C) / 8;
}
constexpr int XCD_K = 16;

// Blocks of a batch of nf fields over ns places: XCD x (blocks x, x + 8, ...) takes
// runs of K consecutive places through all fields before its next run, so that
// fields with a common source (v and dv/dz) find it in its L2 (512x257x512 FP64, 8
// fields of 4 sources: 1234 -> 1066 us).  batch_grid
// blocks in all; false for those past the last place.
__host__ __device__ __forceinline__ int batch_grid(int ns, int nf, int K) { return (ns + 8 * K - 1) / (8 * K) * 8 * K * nf; }
__device__ __forceinline__ bool batch_place(int b, int ns, int nf, int K, int& place, int& f) {
  const int t = b >> 3, r = t / K;
  f = r % nf;
  place = (r / nf * 8 + (b & 7)) * K + t % K;
  return place < ns;
}

// ---------------------------------------------------------------------------
// z transforms: inverse (packed C -> H) and forward (H -> packed C)
// ---------------------------------------------------------------------------
// Places of a run on one XCD: neighbouring column tiles where a tile's rows are less
// than a 128-byte line (each line is then read by two of them), else one.
template <typename T, int TI>
constexpr int ZK = TI * sizeof(cx<T>) < 128 ? XCD_K : 1;
// Field f of a batch with bit f of dzmask set is multiplied by i kz before the
// transform (the x-spectrum of its z derivative).
template <typename T, int NZ, int TI, int NT>
__global__ __launch_bounds__(NT) void k_inv_z(Ptrs<const cd*, MAXO> src, Ptrs<cx<T>*, MAXO> dst,
                                              Geo g, int j0, int nj, int nf, const cx<T>* __restrict__ tw,
                                              const double* __restrict__ kz, unsigned dzmask) {
  constexpr int LD = NZ + 1;
  const int nib = (g.kxr + TI - 1) / TI;
  int tt, f;
  if (!batch_place(blockIdx.x, nib * nj, nf, ZK<T, TI>, tt, f)) return;
  __shared__ cx<T> s[TI * LD];
  __shared__ cx<T> stw[NZ];  // twiddles
  stage_twiddles<T, NZ, NT>(stw, tw, threadIdx.x);
  const int j = j0 + tt / nib, i0 = (tt % nib) * TI, tid = threadIdx.x;
  const cd* __restrict__ C = src.p[f] + (long long)j * g.pc;
  const bool dz = (dzmask >> f) & 1u;
  // every load of the thread first, then the LDS stores (the loads overlap)
  constexpr int PER = (TI * NZ + NT - 1) / NT;
  cx<T> v[PER];
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int idx = tid + q * NT;
    v[q] = {T(0), T(0)};
    if (PER * NT == TI * NZ || idx < TI * NZ) {
      const int ii = idx % TI, z = idx / TI, i = i0 + ii, p = zpack(g, z);
      if (i < g.kxr && p >= 0) {
        const cd c = C[(long long)p * g.kxp + i];
        v[q] = cvt<T>(dz ? ik(kz[p], c) : c);
      }
    }
  }
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int idx = tid + q * NT;
    if (PER * NT == TI * NZ || idx < TI * NZ) s[(idx % TI) * LD + swz<T>(idx / TI)] = v[q];
  }
  __syncthreads();
  fft_lds<T, NZ, TI, NT, +1>(s, LD, stw, tid);
  cx<T>* __restrict__ H = dst.p[f] + (long long)j * g.ph;
  for (int idx = tid; idx < TI * NZ; idx += NT) {
    const int ii = idx % TI, z = idx / TI, i = i0 + ii;
    if (i < g.kxr) H[(long long)z * g.kxp + i] = s[ii * LD + swz<T>(z)];
  }
}

// ACC: add the transform into the destination (an increment of the state).
// dj, dk: distance of the destination's planes and kz rows (the packed layout's, or
// a Fortran array's, whose columns kxr..izero-1 the plane's last block fills with zeros).
template <typename T, int NZ, int TI, int NT, bool ACC = false>
__global__ __launch_bounds__(NT) void k_fwd_z(Ptrs<const cx<T>*, MAXO> src, Ptrs<cd*, MAXO> dst, Geo g, int j0,
                                              const cx<T>* __restrict__ tw, long long dj, int dk, int izero) {
  constexpr int LD = NZ + 1;
  __shared__ cx<T> s[TI * LD];
  __shared__ cx<T> stw[NZ];  // twiddles
  stage_twiddles<T, NZ, NT>(stw, tw, threadIdx.x);
  // grid (column blocks, planes, fields), taken in xcd_tile order
  const int nib = gridDim.x, nj = gridDim.y;
  const int tt = xcd_tile(blockIdx.x + nib * (blockIdx.y + nj * blockIdx.z), nib * nj * gridDim.z, XCD_K);
  const int f = tt / (nib * nj), j = j0 + (tt / nib) % nj, i0 = (tt % nib) * TI, tid = threadIdx.x;
  const cx<T>* __restrict__ H = src.p[f] + (long long)j * g.ph;
  for (int idx = tid; idx < TI * NZ; idx += NT) {
    const int ii = idx % TI, z = idx / TI, i = i0 + ii;
    s[ii * LD + swz<T>(z)] = (i < g.kxr) ? H[(long long)z * g.kxp + i] : cx<T>{T(0), T(0)};
  }
  __syncthreads();
  fft_lds<T, NZ, TI, NT, -1>(s, LD, stw, tid);
  cd* __restrict__ C = dst.p[f] + j * dj;
  const double rnz = 1.0 / NZ;
  for (int idx = tid; idx < TI * g.kzr; idx += NT) {
    const int ii = idx % TI, p = idx / TI, i = i0 + ii;
    if (i < g.kxr) {
      cd v = cvt<double>(s[ii * LD + swz<T>(zpos(g, p))]);
      cd& c = C[(long long)p * dk + i];
      if constexpr (ACC) c = c + rnz * v;
      else c = rnz * v;
    }
  }
  if (i0 + TI >= g.kxr) {
    const int nzc = izero - g.kxr;
    for (int idx = tid; idx < nzc * g.kzr; idx += NT) C[(long long)(idx / nzc) * dk + g.kxr + idx % nzc] = cd{0.0, 0.0};
  }
}

// ---------------------------------------------------------------------------
// x transforms, two real lines (z, z+1) per complex transform
// ---------------------------------------------------------------------------
// split the spectrum Z of a + i b into the half spectra of a and b at bin i
template <typename T>
__device__ __forceinline__ void pair_split(const cx<T>* __restrict__ Zl, int i, int nx, cx<T>& A, cx<T>& B) {
  const cx<T> zk = Zl[swz<T>(i)], zm = conjg(Zl[swz<T>((nx - i) & (nx - 1))]);
  const cx<T> sm = zk + zm, df = zk - zm;
  A = {T(0.5) * sm.x, T(0.5) * sm.y};
  B = {T(0.5) * df.y, T(-0.5) * df.x};
}

// Field f of a batch with bit f of dxmask set yields its x derivative.
template <typename T, int NX, int ZP, int NT>
__global__ __launch_bounds__(NT) void k_inv_x(Ptrs<const cx<T>*, MAXO> src, Ptrs<T*, MAXO> dst,
                                              Geo g, int j0, const cx<T>* __restrict__ tw,
                                              const double* __restrict__ kx, unsigned dxmask) {
  __shared__ cx<T> s[ZP * NX];
  __shared__ cx<T> stw[NX];  // twiddles
  stage_twiddles<T, NX, NT>(stw, tw, threadIdx.x);
  const int f = blockIdx.z, j = j0 + blockIdx.y, tid = threadIdx.x;
  const int zb = blockIdx.x * ZP * 2;
  const cx<T>* __restrict__ H = src.p[f] + (long long)j * g.ph;
  const bool dx = (dxmask >> f) & 1u;
  // Each half-spectrum bin m = 0..NX/2 of the two lines is loaded once and gives
  // both bins m and NX - m of the pair spectrum (the hermitian completion of A + iB
  // written out for the two halves; for an x derivative the bins times i kx, DC zero);
  // bins i > Nkx are zero, and the imaginary part of each DC bin is dropped (a real
  // line's DC bin is real; FFTW's c2r ignores it).  Every load of the thread first,
  // then the LDS stores (the loads overlap).
  constexpr int HB = NX / 2 + 1;
  constexpr int PER = (ZP * HB + NT - 1) / NT;
  cx<T> lo[PER], hi[PER];
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int idx = tid + p * NT;
    if (idx < ZP * HB) {
      const int q = idx / HB, m = idx % HB, z = zb + 2 * q;
      const cx<T>* A = H + (long long)z * g.kxp;
      const cx<T>* B = H + (long long)(z + 1) * g.kxp;
      cx<T> l = {T(0), T(0)}, u = {T(0), T(0)};
      if (m == 0) {
        if (!dx) l = {A[0].x, B[0].x};  // DC: the imaginary parts dropped; d/dx of DC is 0
      } else if (m <= g.nkx) {
        cx<T> a = A[m], b = B[m];
        if (dx) {
          const T k = (T)kx[m];
          a = ik(k, a);
          b = ik(k, b);
        }
        l = {a.x - b.y, a.y + b.x};
        u = {a.x + b.y, b.x - a.y};
      }
      lo[p] = l;
      hi[p] = u;
    }
  }
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int idx = tid + p * NT;
    if (idx < ZP * HB) {
      const int q = idx / HB, m = idx % HB;
      s[q * NX + swz<T>(m)] = lo[p];
      if (m > 0 && m < NX / 2) s[q * NX + swz<T>(NX - m)] = hi[p];
    }
  }
  __syncthreads();
  fft_lds_sync<T, NX, ZP, NT, +1>(s, NX, stw, tid);
  T* __restrict__ R = dst.p[f];
  for (int idx = tid; idx < ZP * NX; idx += NT) {
    const int q = idx / NX, n = idx % NX, z = zb + 2 * q;
    const cx<T> v = s[q * NX + swz<T>(n)];
    R[pline(g, j, z) + n] = v.x;
    R[pline(g, j, z + 1) + n] = v.y;
  }
}

// sj, sz: distance of the physical lines of consecutive planes and rows (the device
// layout's, or a Fortran array's).
template <typename T, int NX, int ZP, int NT>
__global__ __launch_bounds__(NT) void k_fwd_x(Ptrs<const T*, MAXO> src, Ptrs<cx<T>*, MAXO> dst,
                                              Geo g, int j0, const cx<T>* __restrict__ tw, long long sj, long long sz) {
  __shared__ cx<T> s[ZP * NX];
  __shared__ cx<T> stw[NX];  // twiddles
  stage_twiddles<T, NX, NT>(stw, tw, threadIdx.x);
  const int f = blockIdx.z, j = j0 + blockIdx.y, tid = threadIdx.x;
  const int zb = blockIdx.x * ZP * 2;
  const T* __restrict__ R = src.p[f] + j * sj;
  for (int idx = tid; idx < ZP * NX; idx += NT) {
    const int q = idx / NX, n = idx % NX, z = zb + 2 * q;
    s[q * NX + swz<T>(n)] = {R[z * sz + n], R[(z + 1) * sz + n]};
  }
  __syncthreads();
  fft_lds_sync<T, NX, ZP, NT, -1>(s, NX, stw, tid);
  cx<T>* __restrict__ H = dst.p[f] + (long long)j * g.ph;
  const T rnx = T(1) / T(NX);
  for (int idx = tid; idx < ZP * g.kxr; idx += NT) {
    const int q = idx / g.kxr, i = idx % g.kxr, z = zb + 2 * q;
    cx<T> A, B;
    pair_split(s + q * NX, i, NX, A, B);
    H[(long long)z * g.kxp + i] = rnx * A;
    H[(long long)(z + 1) * g.kxp + i] = rnx * B;
  }
}

// ---------------------------------------------------------------------------
// Fused DNS x pass: inverse x transform of u1, u2, u3, th at planes j-1, j, j+1,
// the nonlinear products of rk_chan_1 (for/solver.f90:655-815, 914-964) with their
// y stencils, forward x transform, and the x-derivative factors applied in
// x-spectral space.  Outputs, per plane j, the x-spectra of
//   N1 = -ikx F(u1u1) - F(flux1)     Z1 = F(u3u1)
//   N2 = -ikx F(u1u2i) - F(flux2)    Z2 = F(u3u2i)
//   N3 = -ikx F(u3u1) - F(flux3)     Z3 = F(u3u3)
//   Nt = -ikx F(th u1) - F(fluxth)   Zt = F(th u3)       (per scalar)
// so that the nonlinear tendency of equation e is Fz(Ne) - ikz Fz(Ze).
// ---------------------------------------------------------------------------
// Per-row coefficients of the assembly, computed once on the host from the grid
// (the reference evaluates them inline; the host table holds the same quotients).
enum RowCoef {
  RC_RDY = 0,    // 1/dy(j)
  RC_RDYF,       // 1/dyf(j)
  RC_WTH,        // dyf(j-1)/(2 dy(j)): weight of th(j) in the GY interpolation
  RC_WTHM,       // dyf(j)/(2 dy(j)):   weight of th(j-1)
  RC_FLO,        // 1/(dy(j) dyf(j)):    lower coupling of a GYF row (u1, u3, scalars)
  RC_FHI,        // 1/(dy(j+1) dyf(j)):  upper coupling of a GYF row
  RC_GLO,        // 1/(dyf(j-1) dy(j)):  lower coupling of a GY row (u2)
  RC_GHI,        // 1/(dyf(j) dy(j)):    upper coupling of a GY row
  RC_TW0,        // per scalar n, 4 entries at RC_TW0 + 4n:
  // +0 dthdx (gyf-Ly/2) delta/Ro_inv, +1 -dthdz (gyf-Ly/2) delta/Ro_inv,
  // +2 dthdx (gy-Ly/2) delta/Ro_inv,  +3 -dthdz (gy-Ly/2) delta/Ro_inv
  RC_RDYFM = RC_TW0 + 4 * MAXTH,  // 1/dyf(j-1)
  RC_YX,         // 2 dy(j) / (dx beta_sgs):  the AMD closure's width ratios at GY j
  RC_XY,         // (dx beta_sgs) / (2 dy(j))
  RC_YZ,         // 2 dy(j) / (dz beta_sgs)
  RC_ZY,         // (dz beta_sgs) / (2 dy(j))
  RC_COUNT
};

struct XProdArgs {
  Geo g;
  int jlo;
  int jstart, jend, jstart_th[MAXTH], jend_th[MAXTH];
  const double* __restrict__ dyf;   // k_xmarch, as rowc and hin (the LES pass has AmdArgs)
  const double* __restrict__ rowc;  // [ny2][RC_COUNT] grid quotients
  const double* __restrict__ kx;
  const void* hin[MAXF];   // x-spectra of u1, u2, u3, th_n (all planes)
  void* hout[MAXO];        // N1, N2, N3, Z1, Z2, Z3, (Nt, Zt) per scalar
  const void* tw;
};

// The NP = 8 + 3 NTH product lines of one column x at plane j, from the physical
// fields of planes j-1, j, j+1 (index 0, 1, 2) of the line pair (the .x and .y
// components), with rk_chan_1's y stencils (for/solver.f90:655-815, 914-964):
//   0 u3u1, 1 u1u1, 2 u3u3 (GYF, rows jstart..jend), 3 u1u2i, 4 u3u2i (GY, rows
//   2..Nyp), 5 flux of u1, 6 flux of u3 (GYF), 7 the GY derivative of u2u2, and
//   per scalar n: 8+3n th u1, 9+3n th u3, 10+3n flux of th (rows jstart_th..jend_th).
template <typename T, int NTH>
__device__ __forceinline__ void xprod_products(const XProdArgs& a, int j, const cx<T>* U1, const cx<T>* U2,
                                               const cx<T>* U3, const cx<T> (*TH)[3], cx<T>* P) {
  const bool vrow = (j >= a.jstart && j <= a.jend);
  const bool v2row = (j >= 2 && j <= a.g.ny);
  const double* rc = a.rowc + (long long)j * RC_COUNT;
  const T rdy = (T)rc[RC_RDY], rdyf = (T)rc[RC_RDYF];
  const T dyfj = (T)a.dyf[j], dyfm = (T)a.dyf[j - 1];
  const T cint = T(0.5) * rdy;  // interpolation to GY(j): (dyf_j u_j + dyf_{j-1} u_{j-1})/(2 dy_j)
  // the two real lines of the pair are the .x and .y components
#define DG_PROD(expr_x, expr_y) cx<T>{expr_x, expr_y}
#define C(v, c) (v).c
  if (vrow) {
    P[0] = DG_PROD(C(U3[1], x) * C(U1[1], x), C(U3[1], y) * C(U1[1], y));
    P[1] = DG_PROD(C(U1[1], x) * C(U1[1], x), C(U1[1], y) * C(U1[1], y));
    P[2] = DG_PROD(C(U3[1], x) * C(U3[1], x), C(U3[1], y) * C(U3[1], y));
    const T r2f = T(0.5) * rdyf;
    P[5] = DG_PROD((C(U1[2], x) * C(U2[2], x) + C(U1[1], x) * C(U2[2], x) - C(U1[1], x) * C(U2[1], x) -
                    C(U1[0], x) * C(U2[1], x)) * r2f,
                   (C(U1[2], y) * C(U2[2], y) + C(U1[1], y) * C(U2[2], y) - C(U1[1], y) * C(U2[1], y) -
                    C(U1[0], y) * C(U2[1], y)) * r2f);
    P[6] = DG_PROD((C(U3[2], x) * C(U2[2], x) + C(U3[1], x) * C(U2[2], x) - C(U3[1], x) * C(U2[1], x) -
                    C(U3[0], x) * C(U2[1], x)) * r2f,
                   (C(U3[2], y) * C(U2[2], y) + C(U3[1], y) * C(U2[2], y) - C(U3[1], y) * C(U2[1], y) -
                    C(U3[0], y) * C(U2[1], y)) * r2f);
  } else {
    P[0] = P[1] = P[2] = P[5] = P[6] = cx<T>{T(0), T(0)};
  }
  if (v2row) {
    P[3] = DG_PROD(((dyfj * C(U1[1], x) + dyfm * C(U1[0], x)) * cint) * C(U2[1], x),
                   ((dyfj * C(U1[1], y) + dyfm * C(U1[0], y)) * cint) * C(U2[1], y));
    P[4] = DG_PROD(((dyfj * C(U3[1], x) + dyfm * C(U3[0], x)) * cint) * C(U2[1], x),
                   ((dyfj * C(U3[1], y) + dyfm * C(U3[0], y)) * cint) * C(U2[1], y));
    const T apx = C(U2[1], x) + C(U2[2], x), amx = C(U2[1], x) + C(U2[0], x);
    const T apy = C(U2[1], y) + C(U2[2], y), amy = C(U2[1], y) + C(U2[0], y);
    P[7] = DG_PROD((T(0.25) * (apx * apx) - T(0.25) * (amx * amx)) * rdy,
                   (T(0.25) * (apy * apy) - T(0.25) * (amy * amy)) * rdy);
  } else {
    P[3] = P[4] = P[7] = cx<T>{T(0), T(0)};
  }
#pragma unroll
  for (int n = 0; n < NTH; ++n) {
    const bool trow = (j >= a.jstart_th[n] && j <= a.jend_th[n]);
    if (trow) {
      const T r2f = T(0.5) * rdyf;
      P[8 + 3 * n] = DG_PROD(C(TH[n][1], x) * C(U1[1], x), C(TH[n][1], y) * C(U1[1], y));
      P[9 + 3 * n] = DG_PROD(C(TH[n][1], x) * C(U3[1], x), C(TH[n][1], y) * C(U3[1], y));
      P[10 + 3 * n] = DG_PROD(
          (C(TH[n][2], x) * C(U2[2], x) + C(TH[n][1], x) * C(U2[2], x) - C(TH[n][1], x) * C(U2[1], x) -
           C(TH[n][0], x) * C(U2[1], x)) * r2f,
          (C(TH[n][2], y) * C(U2[2], y) + C(TH[n][1], y) * C(U2[2], y) - C(TH[n][1], y) * C(U2[1], y) -
           C(TH[n][0], y) * C(U2[1], y)) * r2f);
    } else {
      P[8 + 3 * n] = P[9 + 3 * n] = P[10 + 3 * n] = cx<T>{T(0), T(0)};
    }
  }
#undef DG_PROD
#undef C
}

// The product lines of the pair, forward-transformed in LDS (line p at s + p NX),
// to the 6 + 2 NTH x-spectra of plane j: the two real lines split apart, the
// derivative lines times -ikx less the flux lines, 1/Nx.  hout: the output
// pointers, kxt: kx (either may be a copy in LDS).
template <typename T, int NX, int NT, int NTH, typename KT>
__device__ __forceinline__ void xprod_store(const cx<T>* __restrict__ s, const Geo& g, void* const* hout,
                                            const KT* __restrict__ kxt, int z, int j, int tid) {
  constexpr int NO = 6 + 2 * NTH;
  const T rnx = T(1) / T(NX);
  for (int idx = tid; idx < NO * g.kxr; idx += NT) {
    const int o = idx / g.kxr, i = idx % g.kxr;
    const T kxi = (T)kxt[i];
    cx<T> A0, B0, A1, B1;
    int pd, pf;  // derivative product (times -ikx) and flux product; pf < 0: plain copy of pd
    if (o == 0) { pd = 1; pf = 5; }
    else if (o == 1) { pd = 3; pf = 7; }
    else if (o == 2) { pd = 0; pf = 6; }
    else if (o == 3) { pd = 0; pf = -1; }
    else if (o == 4) { pd = 4; pf = -1; }
    else if (o == 5) { pd = 2; pf = -1; }
    else {
      const int n = (o - 6) >> 1;
      if (((o - 6) & 1) == 0) { pd = 8 + 3 * n; pf = 10 + 3 * n; }
      else { pd = 9 + 3 * n; pf = -1; }
    }
    pair_split(s + pd * NX, i, NX, A0, B0);
    cx<T> ra, rb;
    if (pf >= 0) {
      pair_split(s + pf * NX, i, NX, A1, B1);
      // -ikx F - Fflux
      ra = cx<T>{kxi * A0.y, -(kxi * A0.x)} - A1;
      rb = cx<T>{kxi * B0.y, -(kxi * B0.x)} - B1;
    } else {
      ra = A0;
      rb = B0;
    }
    // device memory (the pointer may come from LDS: say so, for global stores)
    typedef T v2 __attribute__((ext_vector_type(2)));
    typedef __attribute__((address_space(1))) v2 gv2;
    gv2* H = (gv2*)((cx<T>*)hout[o] + (long long)j * g.ph);
    H[(long long)z * g.kxp + i] = v2{rnx * ra.x, rnx * ra.y};
    H[(long long)(z + 1) * g.kxp + i] = v2{rnx * rb.x, rnx * rb.y};
  }
}

// The DNS x pass in one kernel, marching in y.  Block (z pair, segment) owns the
// line pair (z, z+1) over the planes j0..j1 of its segment and keeps the physical
// fields of planes j-1, j, j+1 at its columns in registers: each plane's
// x-spectra are read once (the segment's two halo planes aside), inverse-
// transformed, multiplied out and forward-transformed without the physical
// fields ever reaching HBM.  One LDS FFT per plane serves both directions: the
// NP product lines of plane j and, conjugated (the inverse transform is
// conj(F(conj(X))), the same arithmetic as the +i transform), the NF field lines
// of plane j+2; the raw spectra of plane j+3 are loaded into registers meanwhile
// (unconditional loads from per-thread addresses fixed for the whole block, so
// that nothing waits on them before they are used one plane later; the output
// pointers and kx sit in LDS, so the stores wait on no global load either).
template <typename T, int NX, int NT, int NTH>
__global__ __launch_bounds__(NT) void k_xmarch(XProdArgs a, int seg) {
  constexpr int NF = 3 + NTH, NP = 8 + 3 * NTH, NL = NP + NF, NO = 6 + 2 * NTH;
  static_assert(3 * NF <= NL, "the three first planes share one FFT batch");
  static_assert(NX <= NT, "one column per thread");
  constexpr int HB = NX / 2 + 1;                  // bins 0..NX/2 of a line pair
  constexpr int PREF = (NF * HB + NT - 1) / NT;   // loaded bins per thread
  constexpr bool ALLX = NX == NT;
  __shared__ cx<T> s[NL * NX];
  __shared__ cx<T> stw[NX];  // twiddles
  __shared__ T skx[NX / 2];
  __shared__ void* sout[NO];
  stage_twiddles<T, NX, NT>(stw, (const cx<T>*)a.tw, threadIdx.x);
  const Geo& g = a.g;
  const int tid = threadIdx.x, z = 2 * blockIdx.x, x = tid;
  for (int i = tid; i < g.kxr; i += NT) skx[i] = (T)a.kx[i];
  if (tid < NO) sout[tid] = a.hout[tid];
  const int j0 = a.jlo + blockIdx.y * seg;
  const int j1 = min(j0 + seg - 1, g.ny);
  // bin m of field f per prefetch slot; the slot reads bins min(m, Nkx) of the
  // two lines (in bounds for every slot; unused values are dropped at put time)
  const cx<T>* pb[PREF];
  int pm[PREF];
#pragma unroll
  for (int p = 0; p < PREF; ++p) {
    const int idx = tid + p * NT;
    const bool live = idx < NF * HB;
    const int f = live ? idx / HB : 0;
    const int m = live ? idx % HB : -1;
    pm[p] = m;
    pb[p] = (const cx<T>*)a.hin[f] + (long long)z * g.kxp + (m > 0 ? min(m, g.nkx) : 0);
  }
  cx<T> ra[PREF], rb[PREF];
  auto load_plane = [&](int jp) {
    const long long off = (long long)jp * g.ph;
#pragma unroll
    for (int p = 0; p < PREF; ++p) {
      ra[p] = pb[p][off];
      rb[p] = pb[p][off + g.kxp];
    }
  };
  // the pair spectrum (bins m and NX - m, as k_inv_x: i > Nkx zero, the DC bins'
  // imaginary parts dropped), conjugated, into lines line0 + f
  auto put_plane = [&](int line0) {
#pragma unroll
    for (int p = 0; p < PREF; ++p) {
      const int m = pm[p];
      if (m >= 0) {
        const int f = (tid + p * NT) / HB;
        const cx<T> u = ra[p], v = rb[p];
        cx<T> lo = {T(0), T(0)}, hi = {T(0), T(0)};
        if (m == 0) {
          lo = {u.x, v.x};
        } else if (m <= g.nkx) {
          lo = {u.x - v.y, u.y + v.x};
          hi = {u.x + v.y, v.x - u.y};
        }
        s[(line0 + f) * NX + swz<T>(m)] = conjg(lo);
        if (m > 0 && m < NX / 2) s[(line0 + f) * NX + swz<T>(NX - m)] = conjg(hi);
      }
    }
  };
  cx<T> W[3][NF];  // fields at column x, planes j-1, j, j+1
  auto get_plane = [&](int line0, cx<T>* w) {
#pragma unroll
    for (int f = 0; f < NF; ++f) w[f] = conjg(s[(line0 + f) * NX + swz<T>(x)]);
  };
  // the window's first three planes
  load_plane(j0 - 1);
  put_plane(0);
  load_plane(j0);
  put_plane(NF);
  load_plane(j0 + 1);
  put_plane(2 * NF);
  if (j0 + 2 <= j1 + 1) load_plane(j0 + 2);
  __syncthreads();
  fft_lds<T, NX, 3 * NF, NT, -1>(s, NX, stw, tid);
  if (ALLX || x < NX) {
    get_plane(0, W[0]);
    get_plane(NF, W[1]);
    get_plane(2 * NF, W[2]);
  }
  __syncthreads();
  for (int j = j0; j <= j1; ++j) {
    const bool next = j + 2 <= j1 + 1;  // plane j+2 enters the window
    if (ALLX || x < NX) {
      cx<T> U1[3] = {W[0][0], W[1][0], W[2][0]};
      cx<T> U2[3] = {W[0][1], W[1][1], W[2][1]};
      cx<T> U3[3] = {W[0][2], W[1][2], W[2][2]};
      cx<T> TH[NTH > 0 ? NTH : 1][3];
#pragma unroll
      for (int n = 0; n < NTH; ++n) {
        TH[n][0] = W[0][3 + n];
        TH[n][1] = W[1][3 + n];
        TH[n][2] = W[2][3 + n];
      }
      cx<T> P[NP];
      xprod_products<T, NTH>(a, j, U1, U2, U3, TH, P);
#pragma unroll
      for (int p = 0; p < NP; ++p) s[p * NX + swz<T>(x)] = P[p];
    }
    if (next) {
      put_plane(NP);
      if (j + 3 <= j1 + 1) load_plane(j + 3);
    }
    __syncthreads();
    fft_lds_sync<T, NX, NL, NT, -1>(s, NX, stw, tid);
    xprod_store<T, NX, NT, NTH>(s, g, sout, skx, z, j, tid);
    if (next && (ALLX || x < NX)) {
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        W[0][f] = W[1][f];
        W[1][f] = W[2][f];
      }
      get_plane(NP, W[2]);
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// z forward transform of the fused product spectra: the nonlinear tendency of
// every equation, NL_e = Fz(N_e) - ikz Fz(Z_e), scaled by 1/Nz, on the rows the
// equation owns (u1, u3: jstart..jend; u2: 2..Nyp; th_n: jstart_th..jend_th).
// ---------------------------------------------------------------------------
struct NlArgs {
  Geo g;
  int jlo;
  int jstart, jend, jstart_th[MAXTH], jend_th[MAXTH];
  const double* __restrict__ kz;
  const void* h[MAXO];
  void* nl[MAXF];
  const void* tw;
};

__device__ __forceinline__ void eq_rows(int e, int jstart, int jend, const int* jst, const int* jet,
                                        int ny, int& lo, int& hi) {
  if (e == 0 || e == 2) { lo = jstart; hi = jend; }
  else if (e == 1) { lo = 2; hi = ny; }
  else { lo = jst[e - 3]; hi = jet[e - 3]; }
}

// Persistent blocks: tile t = (column block, plane, equation) runs t = b,
// b + gridDim.x, ... with b the block's xcd_tile position (gridDim.x a multiple
// of 8: XCD x works on a contiguous range of each round's tiles); the next
// tile's spectra are loaded into registers while the current tile is
// transformed and stored, so the loads overlap the FFT and the stores (kz sits
// in LDS: a global load of kz in the store loop made every store wait for the
// whole prefetch).  One tile per block otherwise, in xcd_tile order.
template <typename T, int NZ, int TI, int NT, bool PERSIST>
__global__ __launch_bounds__(NT) void k_fwdz_nl(NlArgs a, int ntiles) {
  constexpr int LD = NZ + 1;
  constexpr int NE = 2 * TI * NZ;              // elements per tile
  constexpr int PER = (NE + NT - 1) / NT;      // per thread
  __shared__ cx<T> s[2 * TI * LD];
  __shared__ cx<T> stw[NZ];  // twiddles
  __shared__ T skz[NZ];      // kz of the packed rows (kzr < NZ)
  stage_twiddles<T, NZ, NT>(stw, (const cx<T>*)a.tw, threadIdx.x);
  const Geo& g = a.g;
  const int tid = threadIdx.x;
  for (int k = tid; k < g.kzr; k += NT) skz[k] = (T)a.kz[k];
  const int nib = (g.kxr + TI - 1) / TI, nj = g.ny - a.jlo + 1;
  const T rnz = T(1) / T(NZ);
  // tile -> (equation e, plane j, first column i0); live: j is one of e's rows
  auto coords = [&](int t, int& e, int& j, int& i0) -> bool {
    const int ib = t % nib, r = t / nib;
    j = a.jlo + r % nj;
    e = r / nj;
    i0 = ib * TI;
    int lo, hi;
    eq_rows(e, a.jstart, a.jend, a.jstart_th, a.jend_th, g.ny, lo, hi);
    return j >= lo && j <= hi;
  };
  cx<T> buf[PER];
  auto load = [&](int t) {
    if (t >= ntiles) return;
    int e, j, i0;
    const bool live = coords(t, e, j, i0);
    const int oN = e < 3 ? e : 6 + 2 * (e - 3);
    const int oZ = e < 3 ? 3 + e : 7 + 2 * (e - 3);
    const cx<T>* HN = (const cx<T>*)a.h[oN] + (long long)j * g.ph;
    const cx<T>* HZ = (const cx<T>*)a.h[oZ] + (long long)j * g.ph;
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int idx = tid + p * NT;
      const int ii = idx % TI, r = idx / TI, which = r / NZ, z = r - which * NZ, i = i0 + ii;
      const cx<T>* Hs = which ? HZ : HN;
      buf[p] = (live && idx < NE && i < g.kxr) ? Hs[(long long)z * g.kxp + i] : cx<T>{T(0), T(0)};
    }
  };
  const int step = PERSIST ? (int)gridDim.x : ntiles;  // one tile per block unless persistent
  int t = PERSIST ? ((gridDim.x & 7) ? (int)blockIdx.x : xcd_tile(blockIdx.x, gridDim.x, gridDim.x / 8))
                  : xcd_tile(blockIdx.x, ntiles, XCD_K);
  load(t);
  __syncthreads();  // the twiddle table
  for (; t < ntiles; t += step) {
    int e, j, i0;
    const bool live = coords(t, e, j, i0);
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int idx = tid + p * NT;
      if (idx < NE) {
        const int ii = idx % TI, r = idx / TI, which = r / NZ, z = r - which * NZ;
        s[(which * TI + ii) * LD + swz<T>(z)] = buf[p];
      }
    }
    __syncthreads();
    if (PERSIST) load(t + step);
    fft_lds_sync<T, NZ, 2 * TI, NT, -1>(s, LD, stw, tid);
    if (live) {
      cx<T>* NL = (cx<T>*)a.nl[e] + (long long)j * g.pc;
      for (int idx = tid; idx < TI * g.kzr; idx += NT) {
        const int ii = idx % TI, k = idx / TI, i = i0 + ii;
        if (i >= g.kxr) continue;
        const int zp = zpos(g, k);
        const cx<T> fn = s[ii * LD + swz<T>(zp)], fz = s[(TI + ii) * LD + swz<T>(zp)];
        NL[(long long)k * g.kxp + i] = rnz * (fn - ik(skz[k], fz));
      }
    }
    __syncthreads();  // s is rewritten by the next tile
  }
}

// ---------------------------------------------------------------------------
// Arguments and the Fourier-space assembly of the column kernels (dgpu_column.hpp)
// and of k_assemble.
// ---------------------------------------------------------------------------

struct SolveRows {
  int blo, bhi;      // build range: rows whose cr comes from the assembly
  int wlo, whi;      // rows written back
  int kind[5];       // rows 0, 1, 2, ny, ny+1: -1 = build-range rule, 0 = zero, 1 = BC value
  double val[5];     // BC value of the mean mode at those rows
};

struct ColArgs {
  Geo g;
  int rk;
  int cr_minus_u;   // k_assemble: write the right-hand side minus the state (increment solves)
  int jstart, f_type;
  double nu, beta, grav_x, grav_y, grav_z, px0, omega0, amp_omega0, time;
  double dthdx[MAXTH], dthdz[MAXTH];
  double temp3, temp4, temp5;
  // host-precomputed scalars: Ro_inv/delta; the scalars' sums of dthdx delta/Ro_inv
  // and -dthdz delta/Ro_inv (0 without the thermal wind); per scalar nu/Pr,
  // temp1 nu_v_scale/Pr; temp1 nu_v_scale
  double cori, twu_x, twu_z, nupr[MAXTH], t1pr[MAXTH], t1v;
  double twon;   // 1 with the front's thermal-wind terms, else 0
  const double* __restrict__ rowc;  // [ny2][RC_COUNT]
  const double *__restrict__ gyf, *__restrict__ kx, *__restrict__ kz;
  SolveRows rows[MAXF];
  unsigned long long bcmask;  // bit MAXF s + e: row s of SolveRows::kind is a BC row of field e
  // Thomas factorisation of the CN systems, [field][3][ny2]: mu_j (forward
  // multiplier), beta_j = 1/b'_j, gamma_j = -c_j/b'_j
  const double* __restrict__ thc;
  cd* u[MAXF];
  cd* p;
  cd* cf[MAXF];
  const void* nl[MAXF];
  cd* crout[MAXF];  // k_assemble: right-hand side rows [blo, bhi] of the physical-space solve
  // k_project in its poisson_p_chan form: the transformed source (else null), the
  // scalar count for its buoyancy term; the solution goes to p
  const cd* prhs;
  int pnth;
};

// Workgroups are dispatched round-robin over the 8 XCDs (each with its own L2).
// The grid is padded to a multiple of 8 and block b takes tile
// (b % 8) * (grid / 8) + b / 8, so that every XCD works on one contiguous range of
// tiles and neighbouring tiles, which share cache lines, meet in one L2.
__device__ __forceinline__ int xcd_tile(int b, int nb) {
  const int per = (int)gridDim.x / 8;
  const int t = (b % 8) * per + b / 8;
  return t < nb ? t : -1;
}

// Inputs of the assembly at one (row j, column) point, fields u1, u2, u3, th_n:
// the state on rows j-1, j, j+1, the pressure on j-1, j, the old RK memory and
// the nonlinear terms.
template <int NTH>
struct RowIn {
  cd um[3 + NTH], uc[3 + NTH], up[3 + NTH], pm, pc_, cfo[3 + NTH], nl[3 + NTH];
};

// Per-column constants of the assembly: the wavenumbers, (kx^2 + kz^2)^beta, and
// the wavenumbers that the thermal wind's advection takes (0 without it).
struct ColK {
  double kx, kz, kk, kxt, kzt, gyb;
};
__device__ __forceinline__ ColK col_k(const ColArgs& a, double kx, double kz, bool mean) {
  const double k2 = kx * kx + kz * kz;
  return {kx, kz, (a.beta == 1.0) ? k2 : pow(k2, a.beta), a.twon * kx, a.twon * kz, mean ? 0.0 : a.grav_y};
}

// cf and cr of every equation at one point (for/solver.f90:385-838, 850-870,
// 981-1002 and user_rhs_chan_fourier 35-111); rc[RowCoef] the row's coefficients.
// The linear terms of one field share a form: -damp u - i s u, with the thermal
// wind's advection in s.
template <int NTH, typename RC>
__device__ __forceinline__ void assemble_row(const ColArgs& a, const RowIn<NTH>& r, const RC rc, const ColK& K, cd* cf,
                                             cd* cr) {
  double sf[NTH > 0 ? NTH : 1], sft = 0.0, sgt = 0.0;
#pragma unroll
  for (int n = 0; n < NTH; ++n) {
    sf[n] = rc[RC_TW0 + 4 * n] * K.kzt + rc[RC_TW0 + 4 * n + 1] * K.kxt;
    sft = sft + sf[n];
    sgt = sgt + (rc[RC_TW0 + 4 * n + 2] * K.kzt + rc[RC_TW0 + 4 * n + 3] * K.kxt);
  }
  const double damp = a.nu * K.kk;
  auto lin = [](cd u, double d, double s) { return cd{s * u.y - d * u.x, -(s * u.x) - d * u.y}; };
  // u1 and u3
  const cd u2m = 0.5 * (r.uc[1] + r.up[1]);
  cf[0] = lin(r.uc[0], damp, sft) + a.cori * r.uc[2] - a.twu_z * u2m + r.nl[0];
  cf[2] = lin(r.uc[2], damp, sft) - a.cori * r.uc[0] - a.twu_x * u2m + r.nl[2];
  // u2 (the buoyancy not in the mean mode)
  cf[1] = lin(r.uc[1], damp, sgt) + r.nl[1];
#pragma unroll
  for (int n = 0; n < NTH; ++n) {
    const cd t = r.uc[3 + n];
    cf[0] = cf[0] + a.grav_x * t;
    cf[2] = cf[2] + a.grav_z * t;
    cf[1] = cf[1] + (K.gyb * rc[RC_WTH]) * t + (K.gyb * rc[RC_WTHM]) * r.um[3 + n];
    cf[3 + n] = lin(t, a.nupr[n] * K.kk, sf[n]) - a.dthdx[n] * r.uc[0] - a.dthdz[n] * r.uc[2] + r.nl[3 + n];
  }
  const double flo = rc[RC_FLO], fhi = rc[RC_FHI];
  const double px = a.temp4 * K.kx, pz = a.temp4 * K.kz;
#pragma unroll
  for (int e = 0; e < 3 + NTH; ++e) {
    const double t1 = e < 3 ? a.t1v : a.t1pr[e < 3 ? 0 : e - 3];
    const double lo = t1 * (e == 1 ? rc[RC_GLO] : flo), hi = t1 * (e == 1 ? rc[RC_GHI] : fhi);
    cd v = r.uc[e] + a.temp3 * r.cfo[e];
    if (e == 0) v = v - ik(px, r.pc_);
    if (e == 1) v = v - (a.temp4 * rc[RC_RDY]) * (r.pc_ - r.pm);
    if (e == 2) v = v - ik(pz, r.pc_);
    v = v + a.temp5 * cf[e];
    cr[e] = v + hi * (r.up[e] - r.uc[e]) - lo * (r.uc[e] - r.um[e]);
  }
}

// The mean pressure gradient of f_type 1 and 2 in u1's (0, 0) mode.
__device__ __forceinline__ double mean_dpdx(const ColArgs& a) {
  if (a.f_type == 1) return a.temp4 * a.px0;
  if (a.f_type == 2) return a.temp4 * (a.px0 + a.amp_omega0 * cos(a.omega0 * a.time));
  return 0.0;
}

// The assembly of k_column alone (the LES branch, whose CN solve runs per physical
// column): cf and the right-hand side (or the right-hand side minus the state,
// cr_minus_u) of every equation at one point per thread.  The columns of a row
// are consecutive threads, so every load and store of a wave is one contiguous
// run of the plane.
template <typename T, int NTH>
__global__ __launch_bounds__(256) void k_assemble(ColArgs a) {
  constexpr int NF = 3 + NTH;
  const Geo& g = a.g;
  const long long c = (long long)blockIdx.x * 256 + threadIdx.x;
  const int j = blockIdx.y;
  if (c >= g.pc) return;
  const int i = (int)(c % g.kxp), k = (int)(c / g.kxp);
  if (i >= g.kxr) return;  // padding columns: k_column writes nothing there either
  const long long pc = g.pc;
  const ColK K = col_k(a, a.kx[i], a.kz[k], c == 0);
  const long long o = (long long)j * pc + c;
  const bool inner = j >= 1 && j <= g.ny;
  RowIn<NTH> r;
  cd cf[NF], cr[NF];
  if (inner) {
#pragma unroll
    for (int e = 0; e < NF; ++e) {
      const cd* __restrict__ u = a.u[e];
      r.um[e] = u[o - pc]; r.uc[e] = u[o]; r.up[e] = u[o + pc];
    }
    r.pm = a.p[o - pc]; r.pc_ = a.p[o];
#pragma unroll
    for (int e = 0; e < NF; ++e) {
      r.cfo[e] = (a.rk > 1) ? ((const cd* __restrict__)a.cf[e])[o] : cd{0.0, 0.0};
      r.nl[e] = cvt<double>(((const cx<T>* __restrict__)a.nl[e])[o]);
    }
    assemble_row<NTH>(a, r, a.rowc + (long long)j * RC_COUNT, K, cf, cr);
    if (c == 0) cr[0].x = cr[0].x - mean_dpdx(a);
  }
#pragma unroll
  for (int e = 0; e < NF; ++e) {
    const SolveRows& SR = a.rows[e];
    cd v = {0.0, 0.0};
    if (inner && j >= SR.blo && j <= SR.bhi) {
      v = cr[e];
      a.cf[e][o] = cf[e];
      if (a.cr_minus_u) v = v - r.uc[e];
    }
    a.crout[e][o] = v;
  }
}

}  // namespace dgpu
