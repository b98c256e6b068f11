// dgpu_column.hip — shapes and launches of the column kernels (dgpu_column.hpp).
#define DG_COLUMN_T
#include "dgpu_column_launch.hpp"

#include <string>
#include <type_traits>

using namespace dgpu;

namespace {

template <int TC, int RPT, bool BIG>
int run_project(const ColArgs& a, int P, int update_p, hipStream_t st) {
  const int nt = P * TC;
  const size_t lds = project_lds(a.g.ny2, nt, RPT, BIG);
  hipError_t e = hipFuncSetAttribute((const void*)&k_project<TC, RPT, BIG>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)lds);
  if (e == hipSuccess) {
    k_project<TC, RPT, BIG><<<(unsigned)((a.g.pc / TC + 7) / 8 * 8), nt, lds, st>>>(a, update_p);
    e = hipGetLastError();
  }
  return e == hipSuccess ? 0 : set_error(10, std::string("k_project: ") + hipGetErrorString(e));
}

}  // namespace

namespace dgpu {

extern template int launch_column_t<float>(const ColArgs&, const ColShape&, int, int, hipStream_t);
template int launch_column_t<double>(const ColArgs&, const ColShape&, int, int, hipStream_t);

// 8 columns a block: a wave's load then takes whole 128-byte lines, and narrower
// blocks were slower even on the grids that leave CUs idle (one comparison, k_column
// alone: 64x65x64, 129 blocks, 20.7 us; 4 columns, 258 blocks, 23.6; 2 columns 27.4.
// 256x129x256: 179, 232, 382).  32 chunks (256 threads, two blocks per CU) up to 5 rows each (5 rows:
// 179 us; 64 chunks of 3: 249; a step of 32x65x32 119 us, with 64 chunks 130, with 16 125;
// of 16x33x16, two scalars, 104, 114, 104), then 64 chunks up to the 320 rows whose tables fit
// LDS (512x257x512 DNS mixed, 64 chunks of 5: 1449 us; 4 columns 1648).  Taller
// columns take narrower blocks with the tables in global memory, and 64-bit offsets (up
// to 320 rows the widest field is below 4 GiB).
static_assert(344ll * 683 * COLUMN_ROWS * 16 < (1ll << 32), "kxp kzr of 1024 x 1024 points");
bool column_shape(const Geo& g, ColShape* s) {
  const int n2 = g.ny2;
  int tc = 8, P = n2 <= 160 ? 32 : 64;
  const bool big = n2 > COLUMN_ROWS;
  if (big) {
    tc = n2 <= 640 ? 4 : 2;
    P = n2 <= 640 ? 128 : 256;
  }
  *s = {tc, P, (n2 + P - 1) / P, big};
  return s->rpt <= (big ? 8 : 5);
}

int launch_column(const ColArgs& a, const ColShape& s, int nth, bool mixed, int project, hipStream_t st) {
  return mixed ? launch_column_t<float>(a, s, nth, project, st) : launch_column_t<double>(a, s, nth, project, st);
}

int launch_project(const ColArgs& a, const ColShape& s, int update_p, hipStream_t st) {
#define DG_X(TC_, RPT_, BIG_) \
  if (s.tc == TC_ && s.rpt == RPT_ && s.big == BIG_) return run_project<TC_, RPT_, BIG_>(a, s.P, update_p, st);
  DG_COLUMN_SHAPES(DG_X)
#undef DG_X
  return set_error(2, "ny too large for the column kernels");
}

}  // namespace dgpu
