// dgpu_column_launch.hpp — the launch of k_column for one precision of the nonlinear
// terms; dgpu_column.hip and dgpu_column_f32.hip instantiate it (two translation
// units, so that they compile side by side).
#pragma once
#include "dgpu_column.hpp"
#include "dgpu_error.hpp"

#include <string>

namespace dgpu {

// TC, RPT, BIG
#define DG_COLUMN_SHAPES(X)                                                            \
  X(8, 1, false) X(8, 2, false) X(8, 3, false) X(8, 4, false) X(8, 5, false)           \
  X(4, 3, true) X(4, 4, true) X(4, 5, true)                                            \
  X(2, 3, true) X(2, 4, true) X(2, 5, true) X(2, 6, true) X(2, 7, true) X(2, 8, true)

template <typename T>
int launch_column_t(const ColArgs& a, const ColShape& s, int nth, int project, hipStream_t st);

#ifdef DG_COLUMN_T
template <typename T, int NTH, int TC, int RPT, bool BIG>
int run_column(const ColArgs& a, int P, int project, hipStream_t st) {
  const int nt = P * TC;
  const size_t lds = column_lds(a.g.ny2, NTH, nt, RPT, BIG);
  hipError_t e = hipFuncSetAttribute((const void*)&k_column<T, NTH, TC, RPT, BIG>,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e == hipSuccess) {
    k_column<T, NTH, TC, RPT, BIG><<<(unsigned)((a.g.pc / TC + 7) / 8 * 8), nt, lds, st>>>(a, project);
    e = hipGetLastError();
  }
  return e == hipSuccess ? 0 : set_error(10, std::string("k_column: ") + hipGetErrorString(e));
}

// whether a column of the rows that k_column takes can have RPT rows a chunk (two
// columns a block run with 256 chunks)
template <int NTH, int TC, int RPT>
constexpr bool column_reaches = TC > 2 || (RPT - 1) * 256 < column_max_rows(NTH);

template <typename T>
int launch_column_t(const ColArgs& a, const ColShape& s, int nth, int project, hipStream_t st) {
#define DG_N(NTH_, TC_, RPT_, BIG_)                                                     \
  if constexpr (column_reaches<NTH_, TC_, RPT_>)                                        \
    if (nth == NTH_) return run_column<T, NTH_, TC_, RPT_, BIG_>(a, s.P, project, st);
#define DG_X(TC_, RPT_, BIG_)                                                           \
  if (s.tc == TC_ && s.rpt == RPT_ && s.big == BIG_) {                                  \
    DG_N(0, TC_, RPT_, BIG_) DG_N(1, TC_, RPT_, BIG_) DG_N(2, TC_, RPT_, BIG_)          \
  }
  DG_COLUMN_SHAPES(DG_X)
#undef DG_X
#undef DG_N
  return set_error(2, "ny too large for the column kernels");
}
#endif

}  // namespace dgpu
