// Input-gradient launches of the training shapes (bf16 and fp16): 128 x 256 tiles, or the weights in registers.
#include "host_util.h"
#include "gemm_bwdx256.h"

namespace amoe {
namespace {

// The 128 x 256 input-gradient kernel, for the same launches (and column tiles that are multiples of 256).  The
// partial sums of the input-range gradient then cover 256 columns each; *n_count_blocks is the grid that ran.
template <typename T, int COLS>
int launch_bwdx256_cols(RowsParams p, const amoe_bwd_x_args* a, hipStream_t st, int* n_count_blocks) {
  p.n_col_blocks = count_col_blocks(p.col_bounds, p.n_col_tiles, COLS);
  const int grid = persistent_grid(max_row_tiles(a->M, a->E), p.n_col_blocks, COLS == 128 ? 3 : 2);
  *n_count_blocks = grid;
  const bool relu = a->relu_mask != 0, xc = a->xc_out != nullptr;
  if (!bwdx_reads_x(a)) {
    hipLaunchKernelGGL((&bwdx256_kernel<T, false, false, false, COLS>), dim3(grid), dim3(kThreads), 0, st, p);
  } else if (!relu) {
    if (xc) hipLaunchKernelGGL((&bwdx256_kernel<T, true, false, true, COLS>), dim3(grid), dim3(kThreads), 0, st, p);
    else hipLaunchKernelGGL((&bwdx256_kernel<T, true, false, false, COLS>), dim3(grid), dim3(kThreads), 0, st, p);
  } else {
    if (xc) hipLaunchKernelGGL((&bwdx256_kernel<T, true, true, true, COLS>), dim3(grid), dim3(kThreads), 0, st, p);
    else hipLaunchKernelGGL((&bwdx256_kernel<T, true, true, false, COLS>), dim3(grid), dim3(kThreads), 0, st, p);
  }
  return launch_rc();
}

template <typename T>
int launch_bwdx256_of(RowsParams p, const amoe_bwd_x_args* a, hipStream_t st, int* n_count_blocks, int* block_cols) {
  if (!rows_all_interior(p, MODE_BWDX, kFBK)) return AMOE_EUNSUPPORTED;
  if (!bwdx_reads_x(a) && a->ir == nullptr && a->gate == nullptr && p.out_stage) {
    // a plain product with a contraction of 256: the weights stay in registers and the rows stream past them
    RowsParams q = p;
    if (const int grid = ws256_plan(q, a->M, a->ldo * 2)) {
      hipLaunchKernelGGL((&ws256_kernel<T, true, 64, WS_PLAIN, false>), dim3(grid), dim3(kThreads), 0, st, q);
      return launch_rc();
    }
  }
  if (a->ir != nullptr && !a->ir_by_expert) return AMOE_EUNSUPPORTED;
  if (a->x != nullptr && (!aligned(a->x, 16) || a->ldx % 8)) return AMOE_EUNSUPPORTED;   // 16-byte pieces of x rows
  // With a short contraction an item is mostly its mask stage: 128-column tiles at three workgroups per CU then
  // hide more of it (C3's up-projection, contraction 256: 0.197 vs 0.212 ms; at 512 the wide tile wins again).
  const bool narrow = bwdx_reads_x(a) && a->N <= 256;
  const int cols = narrow ? 128 : kFCols;
  for (int t = 0; t < a->n_tiles; t++)
    if ((a->tile_bounds[t + 1] - a->tile_bounds[t]) % cols) return AMOE_EUNSUPPORTED;
  *block_cols = cols;
  return narrow ? launch_bwdx256_cols<T, 128>(p, a, st, n_count_blocks)
                : launch_bwdx256_cols<T, kFCols>(p, a, st, n_count_blocks);
}

}  // namespace

int launch_bwdx256(const RowsParams& p, const amoe_bwd_x_args* a, hipStream_t st, int* n_count_blocks, int* block_cols) {
  return a->dtype == AMOE_F16 ? launch_bwdx256_of<f16_t>(p, a, st, n_count_blocks, block_cols)
                              : launch_bwdx256_of<uint16_t>(p, a, st, n_count_blocks, block_cols);
}

}  // namespace amoe
