// dgpu_les.hpp — kernels of the LES branch of rk_chan_1 (use_LES after the
// spin-up gate of for/solver.f90:615), les_model_type 5: the anisotropic
// minimum-dissipation (AMD) closure of les_chan / les_chan_th (for/les.f90).
//
// The reference forms 27 spectral gradient fields, transforms each to physical
// space, evaluates the model, and transforms 9 stress fields back (for/les.f90:
// 551-901, 1201-1395).  Here:
//  * the state's ghost planes get the BC posts of les_chan (k_bc_post);
//  * x-spectra of u, du/dz (k_inv_z with the ikz option) give, by one inverse x
//    transform each, u, du/dx (ikx option) and du/dz in physical space: 3 fields
//    per transported variable instead of 27 transforms (every strain, rotation
//    and invariant tensor entry is a pointwise combination of these, and
//    d/dy is the reference's own difference stencil applied in physical space);
//  * k_les_products evaluates nu_t, kappa_t and the SGS stresses per point and adds
//    the stresses to the nonlinear products whose spectral derivatives the
//    reference applies to the stress (tau_11 joins u1u1, tau_13 joins u1u3, ...),
//    so the stress divergence rides on the products' x transforms, which follow in
//    the same kernel;
//  * the Crank–Nicolson solve with nu_t runs per physical (x, z) column
//    (k_cn_phys), as in the reference, since nu_t varies in x and z.
// Transforms are linear, so moving a linear operation across one changes only
// round-off; the placement of every non-linear operation is the reference's.
#pragma once
#include "dgpu_kernels.hpp"

#include <type_traits>

namespace dgpu {

constexpr double C_AMD = 0.2887;     // for/les.f90:25
constexpr double C_SMAG = 0.17;      // for/les.f90:24
constexpr double BETA_SGS = 3.0;     // for/les.f90:43

// ---------------------------------------------------------------------------
// apply_BC_vel_mpi_post + apply_BC_th_mpi_post at one rank (for/flow.f90:
// 1161-1360, 1596-1732), then apply_BC_les / apply_BC_th_les (for/les.f90:
// 1980-2079), on the Fourier state.  One thread per (kx, kz) column; the mean
// mode is column 0.
// ---------------------------------------------------------------------------
struct BcArgs {
  Geo g;
  int nth, les;  // les: also apply_BC_les / apply_BC_th_les
  int u_lo, v_lo, w_lo, u_hi, v_hi, w_hi, th_lo[MAXTH], th_hi[MAXTH];
  double u_lo_c1, v_lo_c1, w_lo_c1, u_hi_c1, v_hi_c1, w_hi_c1, w_hi_tr, th_lo_c1[MAXTH], th_hi_c1[MAXTH];
  double dy1, dy2, dyny, dyf1;
  cd* u[MAXF];
};

__global__ __launch_bounds__(256) void k_bc_post(BcArgs a) {
  const Geo& g = a.g;
  const long long c = (long long)blockIdx.x * 256 + threadIdx.x;
  if (c >= g.pc) return;
  if (c % g.kxp >= g.kxr) return;
  const bool mean = (c == 0);
  const int ny = g.ny;
  auto at = [&](cd* f, int j) -> cd& { return f[(long long)j * g.pc + c]; };
  const cd z0 = {0.0, 0.0};
  // GYF fields u1, u3 and every scalar share the form of the lower/upper posts
  auto gyf_lo = [&](cd* f, int bc, double c1) {
    if (bc == DGPU_BC_DIRICHLET) {
      at(f, 0) = z0; at(f, 1) = z0;
      if (mean) { at(f, 1) = cd{c1, 0.0}; at(f, 0) = cd{c1, 0.0}; }
    } else {
      at(f, 1) = at(f, 2); at(f, 0) = at(f, 1);
      if (mean) { at(f, 1) = at(f, 2) - cd{a.dy2 * c1, 0.0}; at(f, 0) = at(f, 1) - cd{a.dy1 * c1, 0.0}; }
    }
  };
  auto gyf_hi = [&](cd* f, int bc, double c1d, double c1n, bool w) {
    if (bc == DGPU_BC_DIRICHLET) {
      at(f, ny) = z0; at(f, ny + 1) = z0;
      if (mean) { at(f, ny) = cd{c1d, 0.0}; at(f, ny + 1) = cd{c1d, 0.0}; }
      if (w && mean) at(f, ny + 1) = z0;  // for/flow.f90:1311
    } else {
      at(f, ny) = at(f, ny - 1); at(f, ny + 1) = at(f, ny);
      if (mean) {
        at(f, ny) = at(f, ny - 1) + cd{a.dyny * c1n, 0.0};
        at(f, ny + 1) = at(f, ny) + cd{a.dyny * c1n, 0.0};
      }
    }
  };
  cd *u1 = a.u[0], *u2 = a.u[1], *u3 = a.u[2];
  // lower: u1, u3, then u2
  gyf_lo(u1, a.u_lo, a.u_lo_c1);
  gyf_lo(u3, a.w_lo, a.w_lo_c1);
  if (a.v_lo == DGPU_BC_DIRICHLET) {
    at(u2, 1) = cd{2.0 * a.v_lo_c1, 0.0} - at(u2, 2);
    at(u2, 0) = at(u2, 1);
  } else {
    at(u2, 1) = at(u2, 2); at(u2, 0) = at(u2, 1);
    if (mean) {
      at(u2, 1) = at(u2, 2) - cd{a.dyf1 * a.v_lo_c1, 0.0};
      at(u2, 0) = at(u2, 1) - cd{a.dyf1 * a.v_lo_c1, 0.0};
    }
  }
  // upper: u1, u3, then u2
  gyf_hi(u1, a.u_hi, a.u_hi_c1, a.u_hi_c1, false);
  gyf_hi(u3, a.w_hi, a.w_hi_c1, a.w_hi_tr, true);
  if (a.v_hi == DGPU_BC_DIRICHLET) {
    if (mean) at(u2, ny + 1) = cd{2.0 * a.v_hi_c1, 0.0} - at(u2, ny);
  } else {
    at(u2, ny) = at(u2, ny - 1); at(u2, ny + 1) = at(u2, ny);
    if (mean) at(u2, ny + 1) = at(u2, ny) + cd{a.dyny * a.v_hi_c1, 0.0};
  }
  for (int n = 0; n < a.nth; ++n) {
    gyf_lo(a.u[3 + n], a.th_lo[n], a.th_lo_c1[n]);
    gyf_hi(a.u[3 + n], a.th_hi[n], a.th_hi_c1[n], a.th_hi_c1[n], false);
  }
  if (!a.les) return;
  // apply_BC_les: Neumann ghosts copy the first interior plane, mean included
  if (a.u_hi == DGPU_BC_NEUMANN) { at(u1, ny) = at(u1, ny - 1); at(u1, ny + 1) = at(u1, ny); }
  if (a.w_hi == DGPU_BC_NEUMANN) { at(u3, ny) = at(u3, ny - 1); at(u3, ny + 1) = at(u3, ny); }
  if (a.u_lo == DGPU_BC_NEUMANN) { at(u1, 1) = at(u1, 2); at(u1, 0) = at(u1, 1); }
  if (a.w_lo == DGPU_BC_NEUMANN) { at(u3, 1) = at(u3, 2); at(u3, 0) = at(u3, 1); }
  for (int n = 0; n < a.nth; ++n) {
    cd* t = a.u[3 + n];
    if (a.th_hi[n] == DGPU_BC_NEUMANN) { at(t, ny) = at(t, ny - 1); at(t, ny + 1) = at(t, ny); }
    if (a.th_lo[n] == DGPU_BC_NEUMANN) { at(t, 1) = at(t, 2); at(t, 0) = at(t, 1); }
  }
}

// ---------------------------------------------------------------------------
// AMD model per point (for/les.f90:571-797, 1213-1346).
// Inputs (physical, [z][j][x], all planes): for each transported field v in
// (u1, u2, u3, th_n): v, dv/dx, dv/dz.  Outputs (zero where the reference adds
// nothing):
//   nu_t, kappa_t_n            at GY points, zero at j = 0, 1, 2, Nyp, Nyp+1 (written on
//                              the planes the products have; zero from the start on the others)
//   A0 = tau_11  (joins u1u1)       A1 = tau_13 (joins u1u3)   rows jstart..Nyp-1
//   A2 = tau_33  (joins u3u3)       A3 = (tau_12(j+1)-tau_12(j))/dyf(j)  (u1 flux)
//   A4 = (tau_23(j+1)-tau_23(j))/dyf(j)  (u3 flux)                        rows jstart..Nyp-1
//   A5 = tau_12 - nu_t du1/dy (joins u1 u2 at GY)   A6 = tau_23 - nu_t du3/dy   rows 2..Nyp
//   A7+2n = flux_x of th_n (joins th u1)  A8+2n = flux_z (joins th u3)  rows jstart_th..jend_th
// with tau including the filter-width factor delta(j) of the reference.
// ---------------------------------------------------------------------------
struct AmdArgs {
  Geo g;
  int nth, jstart, jend, jstart_th[MAXTH], jend_th[MAXTH];
  double dxs, dzs;                      // dx * beta_sgs, dz * beta_sgs
  double zx, xz;                        // dzs / dxs, dxs / dzs
  const double* __restrict__ rowc;      // [ny2][RC_COUNT] per-row grid quotients
  const double* __restrict__ dy;
  const double* __restrict__ dyf;
  const double* __restrict__ dlt;       // [2][ny2]: delta_yf(j), delta_y(j)
  const void* f[3 * MAXF];              // v, dv/dx, dv/dz per transported field
  void* nut;
  void* kap[MAXTH];
  // les_model_type 6: the learned closure's coefficients at GY (k_closure), in
  // the transform precision T, sign bit set where the point took the AMD value
  const void* cgy;   // velocity
  const void* kgy;   // scalar
};

// the invariant-scaled strain/rotation entries of one GYF plane
template <typename R>
struct Gyf {
  R a1, a2, a3, a5, o5;
};
// ... and of one GY plane
template <typename R>
struct Gy {
  R a4, o4, a6, o6;
};

// What the model takes from the grid at one row: the quotients of the row table
// (RowCoef), the filter widths and the spacings.  The reference divides by dy(j),
// dyf(j) and the widths at every point; the kernels multiply (the results agree to
// rounding).
enum RowK { K_RDY, K_RDYF, K_WTH, K_WTHM, K_RDYFM, K_YX, K_XY, K_YZ, K_ZY, K_DLT, K_DLTY, K_DY, K_DYF, K_N };

// The inputs one point reads: every slot on rows j - 1 .. j + 2, loaded into
// registers before any arithmetic (the reads of the model's branches and of the
// neighbour rows are then all in flight at once instead of in dependent groups), and
// the grid's rows j - 1 .. j + 1 in the model's precision.  at() and rc() are called
// with rows j + const, so the window index folds to a constant.
template <typename T>
struct AmdIn {
  T (*w)[4];         // the kernel's arrays (apart from j0, so that they can be split into registers)
  const T (*k)[K_N];
  int j0;            // j - 1
  int nx;            // from row to row
  __device__ T at(int f, int row, long long) const { return w[f][row - j0]; }
  __device__ T rc(int row, int c) const { return k[row - j0][c]; }
};
// rows outside 0..Nyp+1 are clamped (no caller uses such a row's value)
__device__ __forceinline__ int clamp_row(int row, int last) { return row < 0 ? 0 : (row > last ? last : row); }
template <typename T>
__device__ __forceinline__ void load_rows(T (*k)[K_N], const AmdArgs& a, int j) {
  constexpr int rc[9] = {RC_RDY, RC_RDYF, RC_WTH, RC_WTHM, RC_RDYFM, RC_YX, RC_XY, RC_YZ, RC_ZY};
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const int row = clamp_row(j - 1 + r, a.g.ny + 1);
    const double* t = a.rowc + (long long)row * RC_COUNT;
#pragma unroll
    for (int c = 0; c < 9; ++c) k[r][c] = T(t[rc[c]]);
    k[r][K_DLT] = T(a.dlt[row]);
    k[r][K_DLTY] = T(a.dlt[a.g.ny2 + row]);
    k[r][K_DY] = T(a.dy[row]);
    k[r][K_DYF] = T(a.dyf[row]);
  }
}
// NS slots
template <typename T, int NS>
__device__ __forceinline__ void load_window(AmdIn<T>& in, const AmdArgs& a, int j, long long q) {
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      in.w[s][r] = ((const T*)a.f[s])[(long long)clamp_row(j - 1 + r, a.g.ny + 1) * a.g.nx + q];
}

// the GY interpolation of GYF values c (row j) and m (row j-1):
// (c dyf(j-1) + m dyf(j)) / (2 dy(j))
template <typename T>
__device__ __forceinline__ T gy_interp(const AmdIn<T>& in, int j, T c, T m) {
  return c * in.rc(j, K_WTH) + m * in.rc(j, K_WTHM);
}

// field slots: 3*f + {0: v, 1: dv/dx, 2: dv/dz}, f = 0 u1, 1 u2, 2 u3, 3+n th_n
template <typename T>
__device__ __forceinline__ Gyf<T> gyf_plane(const AmdIn<T>& in, const AmdArgs& a, int j, long long q) {
  using R = T;
  Gyf<T> r;
  const R du1dz = in.at(2, j, q), du3dx = in.at(7, j, q);
  r.a1 = in.at(1, j, q);                                              // SI11 = du1/dx
  r.a2 = (in.at(3, j + 1, q) - in.at(3, j, q)) * in.rc(j, K_RDYF);    // SI22 = du2/dy
  r.a3 = in.at(8, j, q);                                              // SI33 = du3/dz
  r.a5 = R(0.5) * (du1dz * R(a.zx) + du3dx * R(a.xz));                // SI13
  r.o5 = R(0.5) * (du1dz * R(a.zx) - du3dx * R(a.xz));                // O13
  return r;
}
template <typename T>
__device__ __forceinline__ Gy<T> gy_plane(const AmdIn<T>& in, const AmdArgs& a, int j, long long q) {
  using R = T;
  Gy<T> r;
  // the width ratios 2 dy / (dx beta), ... of the scaled gradient, from the row table
  const R rdy = in.rc(j, K_RDY), yx = in.rc(j, K_YX), xy = in.rc(j, K_XY), yz = in.rc(j, K_YZ), zy = in.rc(j, K_ZY);
  const R du1dy = (in.at(0, j, q) - in.at(0, j - 1, q)) * rdy;
  const R du3dy = (in.at(6, j, q) - in.at(6, j - 1, q)) * rdy;
  const R du2dx = in.at(4, j, q), du2dz = in.at(5, j, q);
  r.a4 = R(0.5) * (du1dy * yx + du2dx * xy);
  r.o4 = R(0.5) * (du1dy * yx - du2dx * xy);
  r.a6 = R(0.5) * (du2dz * zy + du3dy * yz);
  r.o6 = R(0.5) * (du2dz * zy - du3dy * yz);
  return r;
}

// max{0, -(I3 - I4)} / (I1 - I2) from the six strain and three rotation entries
template <typename R>
__device__ __forceinline__ R amd_coef(R a1, R a2, R a3, R a4, R a5, R a6,
                                           R o4, R o5, R o6) {
  R v = a1 * a1 * a1 + a2 * a2 * a2 + a3 * a3 * a3 + R(3.0) * a1 * (a4 * a4) + R(3.0) * a1 * (a5 * a5) +
             R(3.0) * a2 * (a4 * a4) + R(3.0) * a2 * (a6 * a6) + R(3.0) * a3 * (a5 * a5) + R(3.0) * a3 * (a6 * a6) +
             R(6.0) * a4 * a5 * a6;
  v = -v - a1 * (o4 * o4) - a1 * (o5 * o5) - a2 * (o4 * o4) - a2 * (o6 * o6) - a3 * (o5 * o5) -
      a3 * (o6 * o6) - R(2.0) * a4 * o5 * o6 + R(2.0) * a5 * o4 * o6 - R(2.0) * a6 * o4 * o5;
  const R d = a1 * a1 + a2 * a2 + a3 * a3 + R(2.0) * (a4 * a4) + R(2.0) * (o4 * o4) + R(2.0) * (a5 * a5) +
              R(2.0) * (o5 * o5) + R(2.0) * (a6 * a6) + R(2.0) * (o6 * o6);
  return v <= R(0.0) ? R(0.0) : v / d;
}

// coefficient at GYF j (GY entries averaged from j and j+1)
template <typename T>
__device__ __forceinline__ T coef_gyf(const AmdIn<T>& in, const AmdArgs& a, int j, long long q) {
  using R = T;
  const Gyf<T> f = gyf_plane(in, a, j, q);
  const Gy<T> p = gy_plane(in, a, j + 1, q), m = gy_plane(in, a, j, q);
  return amd_coef(f.a1, f.a2, f.a3, R(0.5) * (p.a4 + m.a4), f.a5, R(0.5) * (p.a6 + m.a6), R(0.5) * (p.o4 + m.o4), f.o5,
                  R(0.5) * (p.o6 + m.o6));
}
// coefficient at GY j (GYF entries interpolated from j-1 and j)
template <typename T>
__device__ __forceinline__ T coef_gy(const AmdIn<T>& in, const AmdArgs& a, int j, long long q) {
  using R = T;
  const Gyf<T> f = gyf_plane(in, a, j, q), fm = gyf_plane(in, a, j - 1, q);
  const Gy<T> p = gy_plane(in, a, j, q);
  auto w = [&](R c, R m) { return gy_interp(in, j, c, m); };
  return amd_coef(w(f.a1, fm.a1), w(f.a2, fm.a2), w(f.a3, fm.a3), p.a4, w(f.a5, fm.a5), p.a6, p.o4,
                  w(f.o5, fm.o5), p.o6);
}

// The strain S and rotation O of the unscaled gradient (compute_strain_chan,
// compute_rotation_chan, for/les.f90:1443-1596), per GYF and GY plane, for types 1, 4
template <typename R>
struct Sgyf {
  R s1, s2, s3, s5, o5;
};
template <typename R>
struct Sgy {
  R s4, s6, o4, o6;
};
template <typename T>
__device__ __forceinline__ Sgyf<T> sgyf_plane(const AmdIn<T>& in, const AmdArgs& a, int j, long long q) {
  using R = T;
  const R du1dz = in.at(2, j, q), du3dx = in.at(7, j, q);
  return {in.at(1, j, q), (in.at(3, j + 1, q) - in.at(3, j, q)) * in.rc(j, K_RDYF), in.at(8, j, q),
          R(0.5) * (du1dz + du3dx), R(0.5) * (du1dz - du3dx)};
}
template <typename T>
__device__ __forceinline__ Sgy<T> sgy_plane(const AmdIn<T>& in, const AmdArgs& a, int j, long long q) {
  using R = T;
  const R rdy = in.rc(j, K_RDY);
  const R du1dy = (in.at(0, j, q) - in.at(0, j - 1, q)) * rdy;
  const R du3dy = (in.at(6, j, q) - in.at(6, j - 1, q)) * rdy;
  const R du2dx = in.at(4, j, q), du2dz = in.at(5, j, q);
  return {R(0.5) * (du1dy + du2dx), R(0.5) * (du2dz + du3dy), R(0.5) * (du1dy - du2dx), R(0.5) * (du2dz - du3dy)};
}
// type 4 (for/les.f90:276-440): the AMD polynomial with the squared filter widths
// dX, dY, dZ as weights; at GYF (g6 = false) the last cubic term multiplies
// a4 a5 a6, at GY a4 a6 a5 (the reference's operand orders)
template <typename R>
__device__ __forceinline__ R amd4_coef(R dX, R dY, R dZ, R a1, R a2, R a3,
                                            R a4, R a5, R a6, R o4, R o5, R o6,
                                            bool gy) {
  R v = dX * (a1 * a1 * a1) + dY * (a2 * a2 * a2) + dZ * (a3 * a3 * a3) + (R(2.0) * dX + dY) * a1 * (a4 * a4) +
             (R(2.0) * dX + dZ) * a1 * (a5 * a5) + (R(2.0) * dY + dX) * a2 * (a4 * a4) + (R(2.0) * dY + dZ) * a2 * (a6 * a6) +
             (R(2.0) * dZ + dX) * a3 * (a5 * a5) + (R(2.0) * dZ + dY) * a3 * (a6 * a6) +
             (gy ? R(2.0) * (dX + dY + dZ) * a4 * a6 * a5 : R(2.0) * (dX + dY + dZ) * a4 * a5 * a6);
  v = -v - dY * a1 * (o4 * o4) - dZ * a1 * (o5 * o5) - dX * a2 * (o4 * o4) - dZ * a2 * (o6 * o6) -
      dX * a3 * (o5 * o5) - dY * a3 * (o6 * o6) - R(2.0) * dZ * a4 * o5 * o6 + R(2.0) * dY * a5 * o4 * o6 -
      R(2.0) * dX * a6 * o4 * o5;
  const R d = a1 * a1 + a2 * a2 + a3 * a3 + R(2.0) * (a4 * a4) + R(2.0) * (o4 * o4) + R(2.0) * (a5 * a5) +
              R(2.0) * (o5 * o5) + R(2.0) * (a6 * a6) + R(2.0) * (o6 * o6);
  return v <= R(0.0) ? R(0.0) : v / d;
}

// the model coefficient at GYF j (s1 of les_chan) and at GY j (temp)
template <int MODEL, typename T>
__device__ __forceinline__ T model_gyf(const AmdIn<T>& in, const AmdArgs& a, int j, long long q) {
  using R = T;
  if constexpr (MODEL == 5) {
    return coef_gyf(in, a, j, q);
  } else if constexpr (MODEL == 6) {
    // the mean of the network's GY j and j+1 values, else the type-5 GYF coefficient
    const R c0 = (R)((const T*)a.cgy)[(long long)j * in.nx + q];
    const R c1 = (R)((const T*)a.cgy)[(long long)(j + 1) * in.nx + q];
    return (!signbit(c0) && !signbit(c1)) ? R(0.5) * (c0 + c1) : coef_gyf(in, a, j, q);
  } else {
    const Sgyf<T> f = sgyf_plane(in, a, j, q);
    const Sgy<T> p = sgy_plane(in, a, j + 1, q), m = sgy_plane(in, a, j, q);
    const R s4 = R(0.5) * (p.s4 + m.s4), s6 = R(0.5) * (p.s6 + m.s6);
    if constexpr (MODEL == 1) {  // |S| (for/les.f90:99-112)
      return sqrt(R(2.0) * (f.s1 * f.s1) + R(4.0) * (s4 * s4) + R(4.0) * (f.s5 * f.s5) + R(2.0) * (f.s2 * f.s2) +
                  R(4.0) * (s6 * s6) + R(2.0) * (f.s3 * f.s3));
    } else {
      const R dY = (in.rc(j, K_DY) * R(2.0)) * (in.rc(j, K_DY) * R(2.0));
      return amd4_coef(R(a.dxs) * R(a.dxs), dY, R(a.dzs) * R(a.dzs), f.s1, f.s2, f.s3, s4, f.s5, s6, R(0.5) * (p.o4 + m.o4),
                       f.o5, R(0.5) * (p.o6 + m.o6), false);
    }
  }
}
template <int MODEL, typename T>
__device__ __forceinline__ T model_gy(const AmdIn<T>& in, const AmdArgs& a, int j, long long q) {
  using R = T;
  if constexpr (MODEL == 5) {
    return coef_gy(in, a, j, q);
  } else if constexpr (MODEL == 6) {
    return fabs((R)((const T*)a.cgy)[(long long)j * in.nx + q]);
  } else {
    const Sgyf<T> f = sgyf_plane(in, a, j, q), fm = sgyf_plane(in, a, j - 1, q);
    const Sgy<T> p = sgy_plane(in, a, j, q);
    auto w = [&](R c, R m) { return gy_interp(in, j, c, m); };
    const R s1 = w(f.s1, fm.s1), s2 = w(f.s2, fm.s2), s3 = w(f.s3, fm.s3), s5 = w(f.s5, fm.s5);
    if constexpr (MODEL == 1) {  // (for/les.f90:114-132)
      return sqrt(R(2.0) * (s1 * s1) + R(4.0) * (p.s4 * p.s4) + R(4.0) * (s5 * s5) + R(2.0) * (s2 * s2) + R(4.0) * (p.s6 * p.s6) +
                  R(2.0) * (s3 * s3));
    } else {
      const R dY = (in.rc(j, K_DY) * R(2.0)) * (in.rc(j, K_DY) * R(2.0));
      return amd4_coef(R(a.dxs) * R(a.dxs), dY, R(a.dzs) * R(a.dzs), s1, s2, s3, p.s4, s5, p.s6, p.o4, w(f.o5, fm.o5), p.o6,
                       true);
    }
  }
}

// The type-5 scalar coefficient max{0, v}/|b'|^2 (les_chan_th), with the scaled
// scalar gradient b' = (delta_x th_x, delta_y th_y, delta_z th_z) and the
// unscaled th_y it was formed from
template <typename R>
struct ThCoef {
  R c, bx, by, bz, ty;
};
// at GY j (for/les.f90:1259-1306)
template <typename T>
__device__ __forceinline__ ThCoef<T> amd_th_gy(const AmdIn<T>& in, const AmdArgs& a, int ft, int j, long long q) {
  using R = T;
  const R dxs2 = R(a.dxs) * R(a.dxs), dzs2 = R(a.dzs) * R(a.dzs);
  const R dyl = in.rc(j, K_DY) * R(2.0), dyl2 = dyl * dyl;
  const R rdy = in.rc(j, K_RDY);
  auto w = [&](int s) { return gy_interp(in, j, in.at(s, j, q), in.at(s, j - 1, q)); };
  const R du1dx = w(1), du3dz = w(8), du1dz = w(2), du3dx = w(7);
  const R du2dy = gy_interp(in, j, (in.at(3, j + 1, q) - in.at(3, j, q)) * in.rc(j, K_RDYF),
                            (in.at(3, j, q) - in.at(3, j - 1, q)) * in.rc(j, K_RDYFM));
  const R tx = w(ft + 1), tz = w(ft + 2);
  const R ty = (in.at(ft, j, q) - in.at(ft, j - 1, q)) * rdy;
  const R du1dy = (in.at(0, j, q) - in.at(0, j - 1, q)) * rdy;
  const R du3dy = (in.at(6, j, q) - in.at(6, j - 1, q)) * rdy;
  const R du2dx = in.at(4, j, q), du2dz = in.at(5, j, q);
  const R v = -(dxs2 * du1dx * (tx * tx) + dyl2 * du2dy * (ty * ty) + dzs2 * du3dz * (tz * tz) +
                     (dyl2 * du1dy + dxs2 * du2dx) * tx * ty + (dzs2 * du1dz + dxs2 * du3dx) * tx * tz +
                     (dzs2 * du2dz + dyl2 * du3dy) * ty * tz);
  const R ax = R(a.dxs) * tx, ay = dyl * ty, az = R(a.dzs) * tz;
  return {v > R(0.0) ? v / (ax * ax + ay * ay + az * az) : R(0.0), ax, ay, az, ty};
}
// at GYF j (for/les.f90:1221-1256, 1310-1318)
template <typename T>
__device__ __forceinline__ ThCoef<T> amd_th_gyf(const AmdIn<T>& in, const AmdArgs& a, int ft, int j, long long q) {
  using R = T;
  const R dxs2 = R(a.dxs) * R(a.dxs), dzs2 = R(a.dzs) * R(a.dzs);
  const R dyl = in.rc(j, K_DYF) * R(2.0), dyl2 = dyl * dyl;
  auto gyv = [&](int s, int jj) { return (in.at(s, jj, q) - in.at(s, jj - 1, q)) * in.rc(jj, K_RDY); };
  const R tx = in.at(ft + 1, j, q), tz = in.at(ft + 2, j, q);
  const R ty = R(0.5) * (gyv(ft, j + 1) + gyv(ft, j));
  const R du1dx = in.at(1, j, q), du3dz = in.at(8, j, q);
  const R du2dy = (in.at(3, j + 1, q) - in.at(3, j, q)) * in.rc(j, K_RDYF);
  const R du1dy = R(0.5) * (gyv(0, j + 1) + gyv(0, j)), du3dy = R(0.5) * (gyv(6, j + 1) + gyv(6, j));
  const R du2dx = R(0.5) * (in.at(4, j + 1, q) + in.at(4, j, q));
  const R du2dz = R(0.5) * (in.at(5, j + 1, q) + in.at(5, j, q));
  const R du1dz = in.at(2, j, q), du3dx = in.at(7, j, q);
  const R v = -(dxs2 * du1dx * (tx * tx) + dyl2 * du2dy * (ty * ty) + dzs2 * du3dz * (tz * tz) +
                     (dyl2 * du1dy + dxs2 * du2dx) * tx * ty + (dzs2 * du1dz + dxs2 * du3dx) * tx * tz +
                     (dzs2 * du2dz + dyl2 * du3dy) * ty * tz);
  const R ax = R(a.dxs) * tx, ay = dyl * ty, az = R(a.dzs) * tz;
  return {v > R(0.0) ? v / (ax * ax + ay * ay + az * az) : R(0.0), ax, ay, az, ty};
}

// tau_12 (e = 0) or tau_23 (e = 1) at GY j: delta_y(j) coef(j) (S - du/dy / 2).
// At j = 1 types 4 and 5 scale the strain itself (their coefficient loops start
// at j = 2, for/les.f90:454, 762), type 1 multiplies it (for/les.f90:145); that
// row feeds only rows the BC rows overwrite.
// coef: model_gy at row j (unused on the row-1 special case).
template <int MODEL, bool INNER, typename T>
__device__ __forceinline__ T tau_gy(const AmdIn<T>& in, const AmdArgs& a, int e, int j, long long q, T coef) {
  using R = T;
  const R dlt = in.rc(j, K_DLTY);
  const R half = R(0.5) * in.at(e ? 5 : 4, j, q);
  if constexpr (MODEL == 1 || INNER) return dlt * (coef * half);
  // the row asked for through a copy of j: where the compiler knows that j is 1 it
  // addresses the window by 2 - j, in memory
  int jc = j;
  asm("" : "+s"(jc));
  const R dvdy = (in.at(e ? 6 : 0, j, q) - in.at(e ? 6 : 0, j - 1, q)) * in.rc(j, K_RDY);
  return jc == 1 ? dlt * R(0.5) * (dvdy + in.at(e ? 5 : 4, j, q)) : dlt * (coef * half);
}

// Block b of a 1D grid over (256-point block qb, row j) pairs.  The dispatcher
// deals blocks to the 8 XCDs in turn, so with nqb a multiple of 8 XCD b % 8
// takes q-blocks 8 g + b % 8 (its pass g) through the rows in order, and the
// neighbour rows j - 1 .. j + 2 a block reads are in that XCD's L2 from the
// blocks of the rows around it.
__device__ __forceinline__ void xcd_rows(int b, int nqb, int nj, int& qb, int& j) {
  if (nqb % 8) {
    qb = b % nqb;
    j = b / nqb;
    return;
  }
  const int t = b >> 3;
  j = t % nj;
  qb = (t / nj) * 8 + (b & 7);
}

// The model at one point of row j: nu_t and kappa_t (GY), and the additions to the
// products.  INNER: a row on which every term is present (les_inner), without the
// tests, so that the strains three coefficients share are formed once.
template <typename T, int NTH>
struct AmdOut {
  T nut, kap[NTH > 0 ? NTH : 1], A[7 + 2 * NTH];
};
template <typename T, int NTH, int MODEL, bool INNER>
__device__ __forceinline__ void amd_point(const AmdIn<T>& in, const AmdArgs& a, int j, long long q, AmdOut<T, NTH>& r) {
  using R = T;
  const Geo& g = a.g;
  const int ny = g.ny;
  const long long o = (long long)j * g.nx + q;
  // the model coefficient at GY j and j + 1, each evaluated once: nu_t, the two
  // stresses at GY j and the GYF flux differences take them (row 1 of types 4
  // and 5 needs none)
  const bool need_j = INNER || (j <= ny && (j >= 2 || (MODEL == 1 && j == 1)));
  const R cj = need_j ? model_gy<MODEL>(in, a, j, q) : R(0.0);
  const R cj1 = (INNER || (j >= a.jstart && j <= ny - 1)) ? model_gy<MODEL>(in, a, j + 1, q) : R(0.0);
  // nu_t at GY j (zero on the wall rows of ghost_les_mpi)
  r.nut = R(0.0);
  if (INNER || (j >= 3 && j <= ny - 1)) r.nut = -R(0.5) * in.rc(j, K_DLTY) * cj;
#pragma unroll
  for (int m = 0; m < 7 + 2 * NTH; ++m) r.A[m] = R(0.0);
  // GYF stresses, rows j1..j2 = jstart..Nyp-1
  if (INNER || (j >= a.jstart && j <= ny - 1)) {
    const R dyf = in.rc(j, K_DLT) * model_gyf<MODEL>(in, a, j, q);
    const R du1dz = in.at(2, j, q), du3dx = in.at(7, j, q);
    r.A[0] = dyf * in.at(1, j, q);
    r.A[1] = dyf * (R(0.5) * (du1dz + du3dx));
    r.A[2] = dyf * in.at(8, j, q);
    const R rdyf = in.rc(j, K_RDYF);
    r.A[3] = (tau_gy<MODEL, INNER>(in, a, 0, j + 1, q, cj1) - tau_gy<MODEL, INNER>(in, a, 0, j, q, cj)) * rdyf;
    r.A[4] = (tau_gy<MODEL, INNER>(in, a, 1, j + 1, q, cj1) - tau_gy<MODEL, INNER>(in, a, 1, j, q, cj)) * rdyf;
  }
  // GY stresses and the explicit cross terms, rows 2..Nyp
  if (INNER || (j >= 2 && j <= ny)) {
    const R rdy = in.rc(j, K_RDY);
    r.A[5] = tau_gy<MODEL, INNER>(in, a, 0, j, q, cj) - r.nut * ((in.at(0, j, q) - in.at(0, j - 1, q)) * rdy);
    r.A[6] = tau_gy<MODEL, INNER>(in, a, 1, j, q, cj) - r.nut * ((in.at(6, j, q) - in.at(6, j - 1, q)) * rdy);
  }
#pragma unroll
  for (int n = 0; n < NTH; ++n) {
    const int ft = 3 * (3 + n);
    const bool row = INNER || (j >= a.jstart_th[n] && j <= a.jend_th[n]);
    r.kap[n] = R(0.0);
    if constexpr (MODEL == 1 || MODEL == 4) {
      // les_chan_th types 1 and 4 (for/les.f90:1118-1193): kappa_t = nu_t (GY), and
      // cfth += ikx F(kappa_t dth/dx) + ikz F(kappa_t dth/dz) on rows jstart_th..jend_th
      r.kap[n] = r.nut;
      r.A[7 + 2 * n] = row ? -(r.nut * in.at(ft + 1, j, q)) : R(0.0);
      r.A[8 + 2 * n] = row ? -(r.nut * in.at(ft + 2, j, q)) : R(0.0);
    } else {
      // les_chan_th type 5; type 6 reads the learned coefficients.
      // kappa_t at GY j (for/les.f90:1259-1306, 1344-1348)
      if (INNER || (j >= 3 && j <= ny - 1)) {
        R c;
        if constexpr (MODEL == 6) c = fabs((R)((const T*)a.kgy)[o]);
        else c = amd_th_gy(in, a, ft, j, q).c;
        r.kap[n] = -R(0.5) * in.rc(j, K_DLTY) * c;
      }
      // SGS flux at GYF j (for/les.f90:1221-1256, 1310-1318, 1372-1393)
      if (row) {
        R s1;
        if constexpr (MODEL == 6) {
          const R k0 = (R)((const T*)a.kgy)[o], k1 = (R)((const T*)a.kgy)[o + g.nx];
          s1 = (!signbit(k0) && !signbit(k1)) ? R(0.5) * (k0 + k1) : amd_th_gyf(in, a, ft, j, q).c;
        } else {
          s1 = amd_th_gyf(in, a, ft, j, q).c;
        }
        const R f = R(0.5) * in.rc(j, K_DLT) * s1;
        r.A[7 + 2 * n] = f * in.at(ft + 1, j, q);
        r.A[8 + 2 * n] = f * in.at(ft + 2, j, q);
      }
    }
  }
}

// whether row j has every term of amd_point and les_products (all rows but those at
// the walls)
template <int NTH>
__device__ __forceinline__ bool les_inner(const XProdArgs& x, const AmdArgs& a, int j) {
  bool in = j >= 3 && j >= a.jstart && j >= x.jstart && j <= a.g.ny - 1 && j <= x.jend;
#pragma unroll
  for (int n = 0; n < NTH; ++n)
    in = in && j >= a.jstart_th[n] && j <= a.jend_th[n] && j >= x.jstart_th[n] && j <= x.jend_th[n];
  return in;
}

// The products of xprod_products at one point, plus the SGS additions.
template <typename T, int NTH, bool INNER>
__device__ __forceinline__ void les_products(const XProdArgs& x, const AmdIn<T>& in, int j, const AmdOut<T, NTH>& r,
                                             T* P) {
  const int ny = x.g.ny;
  // rows j-1, j, j+1 of u1, u2, u3
  const T u0 = in.w[0][0], u = in.w[0][1], up = in.w[0][2];
  const T v0 = in.w[3][0], v = in.w[3][1], vp = in.w[3][2];
  const T w0 = in.w[6][0], w = in.w[6][1], wp = in.w[6][2];
  const T rdy = in.rc(j, K_RDY), r2f = T(0.5) * in.rc(j, K_RDYF);
  const T dyfj = in.rc(j, K_DYF), dyfm = in.rc(j - 1, K_DYF);
  const T cint = T(0.5) * rdy;
#pragma unroll
  for (int p = 0; p < 8 + 3 * NTH; ++p) P[p] = T(0);
  if (INNER || (j >= x.jstart && j <= x.jend)) {
    P[0] = w * u + r.A[1];
    P[1] = u * u + r.A[0];
    P[2] = w * w + r.A[2];
    P[5] = (up * vp + u * vp - u * v - u0 * v) * r2f + r.A[3];
    P[6] = (wp * vp + w * vp - w * v - w0 * v) * r2f + r.A[4];
  }
  if (INNER || (j >= 2 && j <= ny)) {
    P[3] = ((dyfj * u + dyfm * u0) * cint) * v + r.A[5];
    P[4] = ((dyfj * w + dyfm * w0) * cint) * v + r.A[6];
    const T ap = v + vp, am = v + v0;
    P[7] = (T(0.25) * (ap * ap) - T(0.25) * (am * am)) * rdy;
  }
#pragma unroll
  for (int n = 0; n < NTH; ++n) {
    const T t0 = in.w[9 + 3 * n][0], t = in.w[9 + 3 * n][1], tp = in.w[9 + 3 * n][2];
    if (INNER || (j >= x.jstart_th[n] && j <= x.jend_th[n])) {
      P[8 + 3 * n] = t * u + r.A[7 + 2 * n];
      P[9 + 3 * n] = t * w + r.A[8 + 2 * n];
      P[10 + 3 * n] = (tp * vp + t * vp - t * v - t0 * v) * r2f;
    }
  }
}

// b in scalar registers and opaque.  In float the bases are formed one after another
// (volatile): all at once they spill to memory with two scalars.  In FP64 the order
// costs registers the other way (one block per CU at 512 lines).
template <typename T>
__device__ __forceinline__ void scalar_base(const char*& b) {
  if constexpr (sizeof(T) == 4) asm volatile("" : "+s"(b));
  else asm("" : "+s"(b));
}

// SPLIT: the order of the product lines, u1's and u3's equations (u1u1, flux of u1,
// u3u1, flux of u3, u3u3), then u2's and the scalars' (u1u2i, flux, u3u2i; th u1,
// flux, th u3).
template <int NTH>
constexpr int les_line(int p) {
  constexpr int first[8] = {1, 5, 0, 6, 2, 3, 7, 4};
  if (p < 8) return first[p];
  const int n = (p - 8) / 3, r = (p - 8) % 3;
  return 8 + 3 * n + (r == 0 ? 0 : (r == 1 ? 2 : 1));
}
// xprod_store for the lines of one half.
template <typename T, int NX, int NT, int NTH, int HALF>
__device__ __forceinline__ void les_store(const cx<T>* __restrict__ s, const Geo& g, void* const* hout,
                                          const double* __restrict__ kxt, int z, int j, int tid) {
  constexpr int NO = HALF == 0 ? 4 : 2 + 2 * NTH;
  const T rnx = T(1) / T(NX);
#pragma unroll
  for (int t = 0; t < NO; ++t) {
    // output, derivative line (times -ikx) and flux line of the half; no flux: a copy
    const int o = HALF == 0 ? (t == 0 ? 0 : t == 1 ? 2 : t == 2 ? 3 : 5) : (t == 0 ? 1 : t == 1 ? 4 : 4 + t);
    const int pd = HALF == 0 ? (t == 0 ? 0 : t == 3 ? 4 : 2) : (t < 2 ? 2 * t : 3 + 3 * ((t - 2) / 2) + 2 * (t % 2));
    const int pf = HALF == 0 ? (t == 0 ? 1 : t == 1 ? 3 : -1)
                             : (t == 0 ? 1 : t == 1 || t % 2 == 1 ? -1 : 4 + 3 * ((t - 2) / 2));
    cx<T>* H = (cx<T>*)hout[o] + (long long)j * g.ph;
    for (int i = tid; i < g.kxr; i += NT) {
      cx<T> A0, B0;
      pair_split(s + pd * NX, i, NX, A0, B0);
      if (pf >= 0) {
        const T k = (T)kxt[i];
        cx<T> A1, B1;
        pair_split(s + (pf >= 0 ? pf : 0) * NX, i, NX, A1, B1);
        A0 = cx<T>{k * A0.y, -(k * A0.x)} - A1;
        B0 = cx<T>{k * B0.y, -(k * B0.x)} - B1;
      }
      H[(long long)z * g.kxp + i] = rnx * A0;
      H[(long long)(z + 1) * g.kxp + i] = rnx * B0;
    }
  }
}

// The LES x pass: the closure, the products and their forward x transforms in one
// kernel.  Block (z pair, plane j): every thread evaluates the model at its columns
// of the two lines, one point after another, writes nu_t and kappa_t, and puts the
// products with the SGS stresses added into the LDS lines (the pair's first line in
// the real parts, the second in the imaginary ones).  The gradient fields are read
// once; the 7 + 2 N_th SGS fields a separate model kernel wrote and the product
// kernel read back never reach memory.  Planes follow one another on an XCD
// (blocks b, b + 8, ...), so that the rows j - 1 .. j + 2 a block reads are in its L2.
// In float the vector instructions bound it (845 per 64 points, 90% of the issue slots;
// 5.3 GB, the bytes of its fields, at 2.9 TB/s); in FP64 the two waves per SIMD that
// 255 registers leave (54% of the issue slots, 10.5 GB at 3.3 TB/s).
//
// SPLIT: the lines of u1's and u3's equations are transformed first, those of u2's
// and the scalars' held in registers meanwhile, so that the tile is half the size
// and two or more blocks share a CU (where the whole tile leaves room for one, a
// CU's loads, arithmetic and transforms run one after another).
//
// The model takes more instructions than the transforms, so a point's are kept down:
// the rows' grid quotients are read and converted once per block, addresses are a
// scalar base and 32 bits per lane, and rows away from the walls run without tests
// (with all three in the point's code: 4370 us FP64, 2080 float).  512 threads per
// block in float, 4 waves per SIMD instead of 3: 1846 against 1825 us.
//
// One launch, against the model and product kernels it replaces: 512x257x512 FP64
// 6350 -> 3220 us, float 2796 -> 1825; 128x129x128 FP64 (in one piece) 213 -> 116.
// (two blocks of 256 threads, where LDS has room for them, leave 256 registers each)
template <typename T, int NX, int NTH, bool SPLIT>
constexpr int les_waves() {
  return SPLIT && 2 * sizeof(cx<T>) * (NTH == 2 ? 10 : 6 + NTH) * NX <= 163840 ? 2 : 1;
}
template <typename T, int NX, int NT, int NTH, int MODEL, bool SPLIT>
__global__ __launch_bounds__(NT, (les_waves<T, NX, NTH, SPLIT>())) void k_les_products(XProdArgs x, AmdArgs a, int nj) {
  constexpr int NP = 8 + 3 * NTH, NA = 5, NB = NP - NA;
  constexpr int NL = SPLIT ? (NA > NB ? NA : NB) : NP;
  constexpr int K = (2 * NX + NT - 1) / NT;  // points per thread
  __shared__ cx<T> s[NL * NX];
  __shared__ cx<T> stw[NX];  // twiddles
  stage_twiddles<T, NX, NT>(stw, (const cx<T>*)x.tw, threadIdx.x);
  const Geo& g = x.g;
  const int tid = threadIdx.x, pairs = g.nz / 2;
  int zp, jj;
  xcd_rows(blockIdx.x, pairs, nj, zp, jj);
  const int z = 2 * zp;
  // one value to the compiler: the window's row differences fold to constants
  const int j = __builtin_amdgcn_readfirstlane(x.jlo + jj);
  T PB[SPLIT ? K : 1][NB];
  T rows[3][K_N];
  load_rows<T>(rows, a, j);
  // Point k of the thread: column xc of line `line`, c = tid + k NT = line NX + xc.  The
  // plane's first column is the same for the block, and the line too where a line is
  // NT points or more, so that base addresses are scalar and a lane adds 32 bits.
  auto point = [&](auto inner, int k, T* pb) __attribute__((always_inline)) {
    constexpr bool INNER = decltype(inner)::value;
    const int kl = NX >= NT ? k * NT / NX : 0;  // line, the lane's part of it
    const int c = NX >= NT ? tid + k * NT % NX : tid;
    const int xc = c & (NX - 1), ll = NX >= NT ? 0 : c / NX, line = kl + ll;
    unsigned lane = (unsigned)(ll * g.ny2 * NX + xc) * (unsigned)sizeof(T);
    asm("" : "+v"(lane));  // formed here: a 64-bit copy made before the loop would be added to each base
    const long long q = (long long)(z + kl) * g.ny2 * NX;  // lane apart
    auto addr = [&](const void* f, int row) { return (const char*)f + (q + (long long)row * NX) * (long long)sizeof(T); };
    T win[3 * (3 + NTH)][4];
    AmdIn<T> in;
    in.w = win;
    in.k = rows;
    in.j0 = j - 1;
    in.nx = NX;
    // one scalar base for the rows a load's immediate offset (+-4 KiB) reaches
    constexpr int RB = NX * (int)sizeof(T), G = 2 * RB <= 4096 ? 4 : (RB <= 4096 ? 2 : 1);
#pragma unroll
    for (int f = 0; f < 3 * (3 + NTH); ++f)
#pragma unroll
      for (int r0 = 0; r0 < 4; r0 += INNER ? G : 1) {
        const char* b = addr(a.f[f], INNER ? j - 1 + r0 + G / 2 : clamp_row(j - 1 + r0, g.ny + 1));
        scalar_base<T>(b);
#pragma unroll
        for (int r = 0; r < (INNER ? G : 1); ++r)
          win[f][r0 + r] =
              *(const __attribute__((address_space(1))) T*)(b + (INNER ? (r - G / 2) * RB : 0) + lane);
      }
    AmdOut<T, NTH> r;
    amd_point<T, NTH, MODEL, INNER>(in, a, j, q + lane / (unsigned)sizeof(T), r);
    auto out = [&](void* f, T v) { 
      const char* b = addr(f, j);
      scalar_base<T>(b);
      *(__attribute__((address_space(1))) T*)((char*)b + lane) = v;
    };
    out(a.nut, r.nut);
#pragma unroll
    for (int n = 0; n < NTH; ++n) out(a.kap[n], r.kap[n]);
    T P[NP];
    les_products<T, NTH, INNER>(x, in, j, r, P);
    auto put = [&](int slot, T v) { ((T*)&s[slot * NX + swz<T>(xc)])[line] = v; };
    if constexpr (SPLIT) {
#pragma unroll
      for (int p = 0; p < NA; ++p) put(p, P[les_line<NTH>(p)]);
#pragma unroll
      for (int p = 0; p < NB; ++p) pb[p] = P[les_line<NTH>(NA + p)];
    } else {
#pragma unroll
      for (int p = 0; p < NP; ++p) put(p, P[p]);
    }
  };
  auto points = [&](auto inner) __attribute__((always_inline)) {
    if constexpr (SPLIT) {
      static_assert(2 * NX == K * NT, "whole points");
#pragma unroll
      for (int k = 0; k < K; ++k) point(inner, k, PB[k]);
    } else {
#pragma unroll 1
      for (int k = 0; k < K; ++k)
        if (2 * NX >= NT || tid < 2 * NX) point(inner, k, PB[0]);
    }
  };
  // (two scalars in halves hold 9 lines of every point in registers: there the rows
  // without tests spill, 417 us against 342 at 512x65x128 FP64;
  // the constant-coefficient model does not)
  if (!(SPLIT && NTH == 2 && MODEL != 1) && les_inner<NTH>(x, a, j)) points(std::true_type{});
  else points(std::false_type{});
  __syncthreads();
  if constexpr (SPLIT) {
    fft_lds_sync<T, NX, NA, NT, -1>(s, NX, stw, tid);
    les_store<T, NX, NT, NTH, 0>(s, g, x.hout, x.kx, z, j, tid);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int c = tid + k * NT, xc = c & (NX - 1), line = c / NX;
#pragma unroll
      for (int p = 0; p < NB; ++p) ((T*)&s[p * NX + swz<T>(xc)])[line] = PB[k][p];
    }
    __syncthreads();
    fft_lds_sync<T, NX, NB, NT, -1>(s, NX, stw, tid);
    les_store<T, NX, NT, NTH, 1>(s, g, x.hout, x.kx, z, j, tid);
  } else {
    fft_lds_sync<T, NX, NP, NT, -1>(s, NX, stw, tid);
    xprod_store<T, NX, NT, NTH>(s, g, x.hout, x.kx, z, j, tid);
  }
}

}  // namespace dgpu
