// Launches of the forward kernel for few rows per expert or few output columns.
#include "host_util.h"
#include "gemm_direct.h"

namespace amoe {

int launch_direct(const RowsParams& p0, bool w_kc, const amoe_fwd_args* a, bool split_waves, hipStream_t st) {
  RowsParams p = p0;
  const int64_t es = (int64_t)esize(a->dtype);
  // the stages the kernel has: ranges with the input quantiser or neither, one max |W| per expert, generated noise
  if (a->abs_max || a->noise || a->code_out || (a->ir != nullptr) != (a->inp_res > 0.f)) return AMOE_EUNSUPPORTED;
  if ((a->out_bound > 0.f || a->noise_std > 0.f) && a->wmax_cols != 1) return AMOE_EUNSUPPORTED;
  // 4-byte aligned rows and K-tiles; column pairs; weights within 32-bit byte offsets
  if (!aligned(a->x, 4) || !aligned(a->w, 4) || (a->ldx * es) % 4 || (a->w_stride_e * es) % 4) return AMOE_EUNSUPPORTED;
  for (int t = 0; t < a->n_tiles; t++)
    if ((a->tile_bounds[t] * es) % 4) return AMOE_EUNSUPPORTED;
  if (w_kc ? (a->w_stride_n * es) % 4 != 0 : ((a->w_stride_k * es) % 4 != 0 || a->N % 2 != 0)) return AMOE_EUNSUPPORTED;
  if (((int64_t)a->K * a->w_stride_k + (int64_t)a->N * a->w_stride_n) * es >= (1LL << 31)) return AMOE_EUNSUPPORTED;
  p.n_col_blocks = (a->N + kDirCols - 1) / kDirCols;
  // (a tile for every 32 rows and one more per expert that can have any)
  const int64_t tiles = (int64_t)a->M / kDirRows + (a->E < a->M ? a->E : a->M);
  if (tiles * p.n_col_blocks > 0x7fffffffLL) return AMOE_EUNSUPPORTED;
  const int64_t work = tiles * p.n_col_blocks;
  if (split_waves) {
    const dim3 grid((unsigned)work), block(kDirThreads);
#define AMOE_DIRECT(T)                                                                  \
  do {                                                                                  \
    if (w_kc) hipLaunchKernelGGL((&direct_fwd_kernel<T, true>), grid, block, 0, st, p); \
    else hipLaunchKernelGGL((&direct_fwd_kernel<T, false>), grid, block, 0, st, p);     \
  } while (0)
    if (a->dtype == AMOE_F32) AMOE_DIRECT(float);
    else if (a->dtype == AMOE_F16) AMOE_DIRECT(f16_t);
    else AMOE_DIRECT(uint16_t);
#undef AMOE_DIRECT
    return launch_rc();
  }
  constexpr int kWaves = kDirWaveThreads / 64;
  const dim3 grid((unsigned)((work + kWaves - 1) / kWaves)), block(kDirWaveThreads);
#define AMOE_DIRECT(T, SPLIT)                                                                   \
  do {                                                                                          \
    if (w_kc) hipLaunchKernelGGL((&direct_wave_kernel<T, true, SPLIT>), grid, block, 0, st, p); \
    else hipLaunchKernelGGL((&direct_wave_kernel<T, false, SPLIT>), grid, block, 0, st, p);     \
  } while (0)
#define AMOE_DIRECT_T(T)                    \
  do {                                      \
    if (a->n_tiles > 1) AMOE_DIRECT(T, true); \
    else AMOE_DIRECT(T, false);             \
  } while (0)
  if (a->dtype == AMOE_F32) AMOE_DIRECT_T(float);
  else if (a->dtype == AMOE_F16) AMOE_DIRECT_T(f16_t);
  else AMOE_DIRECT_T(uint16_t);
#undef AMOE_DIRECT_T
#undef AMOE_DIRECT
  return launch_rc();
}

}  // namespace amoe
