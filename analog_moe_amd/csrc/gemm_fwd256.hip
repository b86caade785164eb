// Forward launches of the training shapes (bf16 and fp16): 128 x 256 tiles, or the weights in registers.
#include "host_util.h"
#include "gemm_fwd256.h"

namespace amoe {
namespace {

// The 128 x 256 forward kernel for the usual training shapes (bf16 or fp16, every tile interior, per-expert input
// ranges, one max |W| per expert).  AMOE_EUNSUPPORTED: this launch is not one of them; the general kernel runs.
template <typename T, int A_MODE, bool ANALOG, bool NOISE, bool SPLIT2, bool ZCODES = false>
int launch_fwd256_as(const RowsParams& p, int grid, hipStream_t st) {
  auto k = &fwd256_kernel<T, A_MODE, ANALOG, NOISE, SPLIT2, ZCODES>;
  hipLaunchKernelGGL(k, dim3(grid), dim3(kThreads), 0, st, p);
  return launch_rc();
}

template <typename T>
int launch_fwd256_of(RowsParams p, int mode, const amoe_fwd_args* a, hipStream_t st) {
  if (!rows_all_interior(p, mode, kFBK) || a->N % kFCols) return AMOE_EUNSUPPORTED;
  if (a->noise != nullptr || a->n_tiles > 2) return AMOE_EUNSUPPORTED;
  const bool dac = a->ir != nullptr;                 // (interior launches have the range and the quantiser, or neither)
  if (dac && !a->ir_by_expert) return AMOE_EUNSUPPORTED;
  const bool adc = a->out_bound > 0.f, noisy = a->noise_std > 0.f;
  const bool analog = adc && a->out_res > 0.f && a->wmax_cols == 1 && dac;
  if ((adc || noisy) && !analog) return AMOE_EUNSUPPORTED;
  if (a->n_tiles == 2 && !(analog && !a->x_is_quantized)) return AMOE_EUNSUPPORTED;
  // the two-K-tile variant parks the first tile's ADC codes as bytes (code + 128): a finer output quantiser than
  // 254 states does not fit them, and the general kernel (fp32 partial results) serves the launch
  if (a->n_tiles == 2 && !(p.out_half_states <= 127.f)) return AMOE_EUNSUPPORTED;
  if (a->code_out && !analog) return AMOE_EUNSUPPORTED;
  if (a->code_out && (!amoe_fwd_codes_supported(a) || !aligned(a->code_out, 16))) return AMOE_EUNSUPPORTED;
  if (a->n_tiles == 1 && !a->relu && !a->xq_out && (a->x_is_quantized || !dac) && (a->code_out || !analog)) {
    // one K-tile of 256, the operand plain or already coded, the result plain, rescaled or as ADC codes: the
    // weights stay in registers and the rows stream past them
    RowsParams q = p;
    const int grid = a->code_out ? ws256_plan(q, a->n_out_rows, a->ldcode) : ws256_plan(q, a->n_out_rows, a->ldo * 2);
    if (grid > 0) {
      if (a->code_out) {
        if (noisy) hipLaunchKernelGGL((&ws256_kernel<T, false, 64, WS_ZCODES, true>), dim3(grid), dim3(kThreads), 0, st, q);
        else hipLaunchKernelGGL((&ws256_kernel<T, false, 64, WS_ZCODES, false>), dim3(grid), dim3(kThreads), 0, st, q);
      } else if (dac) {
        hipLaunchKernelGGL((&ws256_kernel<T, false, 64, WS_SCALE, false>), dim3(grid), dim3(kThreads), 0, st, q);
      } else {
        hipLaunchKernelGGL((&ws256_kernel<T, false, 64, WS_PLAIN, false>), dim3(grid), dim3(kThreads), 0, st, q);
      }
      return launch_rc();
    }
  }
  p.n_col_blocks = a->N / kFCols;
  const int grid = persistent_grid(max_row_tiles(a->M, a->E), p.n_col_blocks);
  if (!dac) return launch_fwd256_as<T, FA_PLAIN, false, false, false>(p, grid, st);
  if (!analog)
    return a->x_is_quantized ? launch_fwd256_as<T, FA_CODES, false, false, false>(p, grid, st)
                             : launch_fwd256_as<T, FA_DAC, false, false, false>(p, grid, st);
  if (a->code_out) {
    // codes leave instead of values: one output quantiser whose half range fits a byte, no second output
    if (a->x_is_quantized)
      return noisy ? launch_fwd256_as<T, FA_CODES, true, true, false, true>(p, grid, st)
                   : launch_fwd256_as<T, FA_CODES, true, false, false, true>(p, grid, st);
    return noisy ? launch_fwd256_as<T, FA_DAC, true, true, false, true>(p, grid, st)
                 : launch_fwd256_as<T, FA_DAC, true, false, false, true>(p, grid, st);
  }
  if (a->x_is_quantized)
    return noisy ? launch_fwd256_as<T, FA_CODES, true, true, false>(p, grid, st)
                 : launch_fwd256_as<T, FA_CODES, true, false, false>(p, grid, st);
  if (a->n_tiles == 2)
    return noisy ? launch_fwd256_as<T, FA_DAC, true, true, true>(p, grid, st)
                 : launch_fwd256_as<T, FA_DAC, true, false, true>(p, grid, st);
  return noisy ? launch_fwd256_as<T, FA_DAC, true, true, false>(p, grid, st)
               : launch_fwd256_as<T, FA_DAC, true, false, false>(p, grid, st);
}

}  // namespace

int launch_fwd256(const RowsParams& p, int mode, const amoe_fwd_args* a, hipStream_t st) {
  return a->dtype == AMOE_F16 ? launch_fwd256_of<f16_t>(p, mode, a, st) : launch_fwd256_of<uint16_t>(p, mode, a, st);
}

}  // namespace amoe
