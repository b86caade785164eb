// The general row-gather kernel, f16 elements.
#include "rows_launch.h"

namespace amoe {

int launch_rows_f16(const RowsParams& p, bool w_kc, int mode, int grid, hipStream_t st) {
  return w_kc ? launch_rows_of<f16_t, true>(p, mode, grid, st) : launch_rows_of<f16_t, false>(p, mode, grid, st);
}

}  // namespace amoe
