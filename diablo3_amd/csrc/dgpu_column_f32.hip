// dgpu_column_f32.hip — k_column with float nonlinear terms (the mixed mode).
#define DG_COLUMN_T
#include "dgpu_column_launch.hpp"

namespace dgpu {
template int launch_column_t<float>(const ColArgs&, const ColShape&, int, int, hipStream_t);
}
