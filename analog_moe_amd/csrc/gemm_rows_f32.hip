// The general row-gather kernel, f32 elements.
#include "rows_launch.h"

namespace amoe {

int launch_rows_f32(const RowsParams& p, bool w_kc, int mode, int grid, hipStream_t st) {
  return w_kc ? launch_rows_of<float, true>(p, mode, grid, st) : launch_rows_of<float, false>(p, mode, grid, st);
}

}  // namespace amoe
