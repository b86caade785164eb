// Host-side helpers shared by the launchers: argument checks, grid sizes, and the launch functions of the GEMM
// families, one translation unit each (they take minutes to compile as one).
#pragma once
#include <amoe.h>
#include "gemm_rows.h"
#include "gemm_ws256.h"

namespace amoe {

inline bool aligned(const void* p, size_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }
inline int launch_rc() {
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? AMOE_OK : (int)e;
}
inline int check_bounds(int n_tiles, const int32_t* b, int K) {
  if (n_tiles < 1 || n_tiles > AMOE_MAX_TILES) return AMOE_EINVAL;
  if (b[0] != 0 || b[n_tiles] != K) return AMOE_ESHAPE;
  for (int t = 0; t < n_tiles; t++)
    if (b[t + 1] <= b[t]) return AMOE_ESHAPE;
  return AMOE_OK;
}
inline bool bounds_multiple_of(int n_tiles, const int32_t* b, int m) {
  for (int t = 0; t <= n_tiles; t++)
    if (b[t] % m) return false;
  return true;
}
inline size_t esize(int dtype) { return dtype == AMOE_F32 ? 4 : 2; }
// Whether every DAC code of a quantiser with step inp_res (codes -1/inp_res .. 1/inp_res) is exact in the type.
inline bool dac_codes_fit(int dtype, float inp_res) {
  if (dtype == AMOE_F32 || !(inp_res > 0.f)) return true;
  return 1.0f / inp_res <= (dtype == AMOE_BF16 ? 256.f : 2048.f) * (1.0f + 1e-6f);
}
constexpr int kDirRows = 32, kDirCols = 64;   // output tile of gemm_direct.h
inline int max_row_tiles(int64_t M, int E) { return (int)(M / kTileRows) + E; }

// Compute units of the current device (read once; the value cannot change while the process lives).
inline int num_compute_units() {
  static const int n = [] {
    int dev = 0, cu = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 256;
    if (hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cu <= 0) return 256;
    return cu;
  }();
  return n;
}

// Persistent grid of the row-gather GEMM: two workgroups per compute unit, more if a workgroup
// would otherwise get more work items than its descriptor table holds, rounded up to a multiple
// of the column-block count (so that the column blocks of one row tile run side by side), never
// more than there are work items.
inline int persistent_grid(int row_tiles, int col_blocks, int per_cu = 2) {
  const long long work = (long long)row_tiles * col_blocks;
  long long g = (long long)per_cu * num_compute_units();
  const long long need = (work + kMaxDesc - 1) / kMaxDesc;
  if (need > g) g = need;
  if (g % col_blocks) g += col_blocks - g % col_blocks;
  if (g > work) g = work;
  return g < 1 ? 1 : (int)g;
}

// Every tile of the launch is interior: the FAST instantiation applies.
inline bool rows_all_interior(const RowsParams& p, int mode, int bk) {
  if (!p.a_vec || !p.w_vec || !p.out_stage || !p.buf_ok || p.abs_max != nullptr) return false;
  if (p.xq_out != nullptr && !p.xq_stage) return false;
  if (p.xc_out != nullptr && !p.xc_vec) return false;
  // forward: the edge-free code has the clip-and-quantise input stage or none at all
  if (mode != MODE_BWDX && (p.ir != nullptr) != (p.inp_res > 0.f)) return false;
  if (p.noise != nullptr && !p.noise_vec) return false;
  if (p.xf != nullptr && !p.xf_vec) return false;
  for (int t = 0; t < p.n_col_tiles; t++)
    if ((p.col_bounds[t + 1] - p.col_bounds[t]) % kTileCols) return false;
  for (int t = 0; t < p.n_kd_tiles; t++)
    if ((p.kd_bounds[t + 1] - p.kd_bounds[t]) % bk) return false;
  return true;
}

// The input gradient reads the forward input x (through xf_index) only for the features that need it: the
// input-range clip, the ReLU mask, the clipped-input output.  A caller that passes x without any of them has not
// been asked for xf_index, and its launch is a plain product.
inline bool bwdx_reads_x(const amoe_bwd_x_args* a) {
  return a->x != nullptr && a->xf_index != nullptr && (a->ir != nullptr || a->relu_mask != 0 || a->xc_out != nullptr);
}

// The kernel that keeps the weights in registers (gemm_ws256.h): a contraction of exactly 256, output columns in
// groups of 256, interior launches.  Two workgroups per CU, in equal shares per column group, and more if a
// workgroup's run of 32-row blocks would not fit its descriptor table; returns the grid, or 0 when the launch is not
// one of these.
inline int ws256_plan(RowsParams& p, int64_t out_rows, int64_t out_row_bytes) {
  if (p.KD != kWsK || p.ND % 256 || !p.a_vec || !p.w_vec || !p.buf_ok || p.abs_max != nullptr) return 0;
  if (out_rows * out_row_bytes >= (int64_t)kWsOutLimit || (int64_t)p.M * 4 >= (1LL << 31)) return 0;
  p.n_col_blocks = p.ND / 256;
  const long long blocks = (long long)p.M / kWsRows + p.E;                 // bound on the 32-row blocks
  long long runs = 2LL * num_compute_units() / p.n_col_blocks;
  if (runs < 1) runs = 1;
  if (runs * kMaxDesc < blocks) runs = (blocks + kMaxDesc - 1) / kMaxDesc;
  if (runs > blocks) runs = blocks;
  return (int)(runs * p.n_col_blocks);
}

// gemm_rows_<type>.hip: the general kernel
int launch_rows_f32(const RowsParams& p, bool w_kc, int mode, int grid, hipStream_t st);
int launch_rows_bf16(const RowsParams& p, bool w_kc, int mode, int grid, hipStream_t st);
int launch_rows_f16(const RowsParams& p, bool w_kc, int mode, int grid, hipStream_t st);
inline int launch_rows(int dtype, const RowsParams& p, bool w_kc, int mode, int grid, hipStream_t st) {
  return dtype == AMOE_F32   ? launch_rows_f32(p, w_kc, mode, grid, st)
         : dtype == AMOE_F16 ? launch_rows_f16(p, w_kc, mode, grid, st)
                             : launch_rows_bf16(p, w_kc, mode, grid, st);
}
// gemm_fwd256.hip, gemm_bwdx256.hip: the tiled kernels of the training shapes and the weights-in-registers kernel
// (16-bit types).  AMOE_EUNSUPPORTED: not one of their launches, the general kernel runs it.
int launch_fwd256(const RowsParams& p, int mode, const amoe_fwd_args* a, hipStream_t st);
// gemm_direct.hip: small tiles; split_waves: a tile's contraction over the waves of a workgroup, else one wave per tile
int launch_direct(const RowsParams& p, bool w_kc, const amoe_fwd_args* a, bool split_waves, hipStream_t st);
int launch_bwdx256(const RowsParams& p, const amoe_bwd_x_args* a, hipStream_t st, int* n_count_blocks, int* block_cols);

}  // namespace amoe
