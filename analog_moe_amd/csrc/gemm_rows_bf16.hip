// The general row-gather kernel, bf16 elements.
#include "rows_launch.h"

namespace amoe {

int launch_rows_bf16(const RowsParams& p, bool w_kc, int mode, int grid, hipStream_t st) {
  return w_kc ? launch_rows_of<uint16_t, true>(p, mode, grid, st) : launch_rows_of<uint16_t, false>(p, mode, grid, st);
}

}  // namespace amoe
