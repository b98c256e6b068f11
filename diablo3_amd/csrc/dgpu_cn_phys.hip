// dgpu_cn_phys.hip — shapes and launches of k_cn_phys (dgpu_cn_phys.hpp).
#include "dgpu_cn_phys.hpp"
#include "dgpu_error.hpp"

#include <string>

namespace dgpu {
namespace {

// TC columns in chunks of RPT or RPT - 1 rows, if the grid fits that
template <typename TU, typename TV, bool INC, int TC, int RPT>
bool run(const PhysCnArgs<TU, TV>& a, hipStream_t st, int* rc) {
  const int n2 = a.g.ny2, P = (n2 + RPT - 1) / RPT, nt = TC * P;
  if (a.g.nx % TC || nt > CN_PHYS_NT || n2 / P < RPT - 1) return false;
  const size_t lds = sizeof(CnRow) * n2 + sizeof(double) * 6 * nt;
  hipError_t e = hipFuncSetAttribute((const void*)&k_cn_phys<TU, TV, INC, TC, RPT>,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e == hipSuccess) {
    k_cn_phys<TU, TV, INC, TC, RPT><<<(unsigned)(a.g.pp / TC * a.nf), nt, lds, st>>>(a);
    e = hipGetLastError();
  }
  *rc = e == hipSuccess ? 0 : set_error(10, std::string("k_cn_phys: ") + hipGetErrorString(e));
  return true;
}

template <typename TU, typename TV, bool INC>
int launch(const PhysCnArgs<TU, TV>& a, hipStream_t st) {
  // Chunks of 9 rows on 32 columns (whole 256-byte row segments in FP64) while 512
  // threads hold the column, else on 16; the float increments take 17 rows on 16
  // then (fewer exchange steps; a float row costs half the bytes but the same
  // arithmetic).  Measured, us: 128x129x128 FP64 32 columns x 9 rows 60, 16 x 9 66,
  // 16 x 17 71; mixed 45, 56, 58; 512x257x512 FP64 16 x 9 1855, 16 x 17 2007; mixed
  // 16 x 9 1484, 16 x 17 1210, 32 x 17 1447.  The rest serves the tallest columns, the
  // shortest, and nx = 16.
  int rc = 0;
  if (run<TU, TV, INC, 32, 9>(a, st, &rc)) return rc;
  if (!INC && run<TU, TV, INC, 16, 9>(a, st, &rc)) return rc;
  if (run<TU, TV, INC, 16, 17>(a, st, &rc)) return rc;
  if (run<TU, TV, INC, 8, 17>(a, st, &rc)) return rc;
  if (run<TU, TV, INC, 4, 17>(a, st, &rc)) return rc;
  if (run<TU, TV, INC, 16, 9>(a, st, &rc)) return rc;
  if (run<TU, TV, INC, 16, 5>(a, st, &rc)) return rc;
  if (run<TU, TV, INC, 16, 2>(a, st, &rc)) return rc;
  return set_error(2, "ny too large for the column kernels");
}

}  // namespace

int launch_cn_phys(const PhysCnArgs<double, double>& a, hipStream_t st) { return launch<double, double, false>(a, st); }
int launch_cn_phys(const PhysCnArgs<double, float>& a, hipStream_t st) { return launch<double, float, false>(a, st); }
int launch_cn_phys(const PhysCnArgs<float, float>& a, hipStream_t st) { return launch<float, float, true>(a, st); }

}  // namespace dgpu
