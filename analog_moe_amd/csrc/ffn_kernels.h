// Small kernels of the layer calls (ffn.hip).
#pragma once
#include "common.h"

namespace amoe {

// fp32 input-range tables of the two projections from the layer's parameter ir [2, E, ir_cols] of element type T:
// ir_up [E, n_up] = ir[0, :, :n_up], ir_dn [E, n_dn] = ir[1, :, :n_dn].
template <typename T>
__global__ __launch_bounds__(kThreads) void ir_tables_kernel(const T* __restrict__ ir, int ir_cols, int E, int n_up,
                                                              float* __restrict__ ir_up, int n_dn, float* __restrict__ ir_dn) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i < E * n_up) ir_up[i] = Elem<T>::to_f32(ir[(long long)(i / n_up) * ir_cols + i % n_up]);
  if (i < E * n_dn) ir_dn[i] = Elem<T>::to_f32(ir[(long long)(E + i / n_dn) * ir_cols + i % n_dn]);
}

inline int launch_ir_tables(int dtype, const void* ir, int ir_cols, int E, int n_up, float* ir_up, int n_dn, float* ir_dn,
                            hipStream_t st) {
  const dim3 grid((unsigned)((E * (n_up > n_dn ? n_up : n_dn) + kThreads - 1) / kThreads));
  if (dtype == AMOE_F32)
    hipLaunchKernelGGL((&ir_tables_kernel<float>), grid, dim3(kThreads), 0, st, static_cast<const float*>(ir), ir_cols, E, n_up, ir_up, n_dn, ir_dn);
  else if (dtype == AMOE_BF16)
    hipLaunchKernelGGL((&ir_tables_kernel<uint16_t>), grid, dim3(kThreads), 0, st, static_cast<const uint16_t*>(ir), ir_cols, E, n_up, ir_up, n_dn, ir_dn);
  else
    hipLaunchKernelGGL((&ir_tables_kernel<f16_t>), grid, dim3(kThreads), 0, st, static_cast<const f16_t*>(ir), ir_cols, E, n_up, ir_up, n_dn, ir_dn);
  return launch_rc();
}

}  // namespace amoe
