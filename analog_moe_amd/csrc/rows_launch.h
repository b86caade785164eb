// Launches of the general row-gather kernel, instantiated per element type by gemm_rows_<type>.hip.
#pragma once
#include "host_util.h"

namespace amoe {

template <typename T, bool W_KC, bool FAST>
int launch_rows_mode(const RowsParams& p, int mode, int grid, hipStream_t st) {
  if (mode == MODE_FWD) {
    auto k = &gemm_rows_kernel<T, W_KC, MODE_FWD, FAST>;
    hipLaunchKernelGGL(k, dim3(grid), dim3(kThreads), 0, st, p);
  } else if (mode == MODE_FWD_SPLIT) {
    auto k = &gemm_rows_kernel<T, W_KC, MODE_FWD_SPLIT, FAST>;
    hipLaunchKernelGGL(k, dim3(grid), dim3(kThreads), 0, st, p);
  } else {
    auto k = &gemm_rows_kernel<T, W_KC, MODE_BWDX, FAST>;
    hipLaunchKernelGGL(k, dim3(grid), dim3(kThreads), 0, st, p);
  }
  return launch_rc();
}

template <typename T, bool W_KC>
int launch_rows_of(const RowsParams& p, int mode, int grid, hipStream_t st) {
  return rows_all_interior(p, mode, Elem<T>::kBK) ? launch_rows_mode<T, W_KC, true>(p, mode, grid, st)
                                            : launch_rows_mode<T, W_KC, false>(p, mode, grid, st);
}

}  // namespace amoe
