// Input-range gradient: from the partial row sums of the kernels that clip to one value per sorted position.
#pragma once
#include "common.h"

namespace amoe {

// Sum the column-block partials into ir_grad[M, n_tiles] and apply the scaling and decay rules.
struct IrFinalizeParams {
  int M, n_tiles, KD_total;      // KD_total = columns of x (for the un-clipped fraction)
  int block_cols;                // width of the column blocks the partial sums were made over
  int col_bounds[kMaxTiles + 1];
  const float* irg_partial; const int32_t* notclip_count; int n_blocks;
  const int32_t* row_index;      // optional: the partial sums of sorted position r lie at row row_index[r]
  const float* ir; int ir_by_expert; const int32_t* offsets; int E; float* ir_grad;
  int relative; float scale, decay, min_pct;
};

__global__ __launch_bounds__(kThreads) void ir_grad_finalize_kernel(const IrFinalizeParams p) {
  __shared__ long long sTot[4];
  __shared__ int sOff[kSelMaxExperts];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // the segment starts come to LDS in the same round trip as the counts: the search below then runs on LDS
  // instead of on a chain of dependent global loads (E <= kSelMaxExperts: the entry points check it)
  if (p.ir_by_expert)
    for (int i = tid; i < p.E; i += kThreads) sOff[i] = p.offsets[i];
  long long c = 0;
  if (p.decay > 0.f)
    for (int i = tid; i < p.n_blocks; i += kThreads) c += p.notclip_count[i];
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) c += wave_shfl_xor(c, d);
  if (lane == 0) sTot[wave] = c;
  __syncthreads();
  float flag = 0.f;
  if (p.decay > 0.f) {
    const long long tot = sTot[0] + sTot[1] + sTot[2] + sTot[3];
    const float pct = (float)tot / (float)((long long)p.M * (long long)p.KD_total);
    flag = pct > p.min_pct ? 1.f : 0.f;
  }
  const int r = blockIdx.x * kThreads + tid;
  if (r >= p.M) return;
  int ir_row = r;
  if (p.ir_by_expert) {  // expert of sorted position r: last e with offsets[e] <= r
    int lo = 0, hi = p.E - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (sOff[mid] <= r) lo = mid; else hi = mid - 1;
    }
    ir_row = lo;
  }
  const int pr = p.row_index ? p.row_index[r] : r;
  int cb = 0;
  for (int t = 0; t < p.n_tiles; t++) {
    const int nb = (p.col_bounds[t + 1] - p.col_bounds[t] + p.block_cols - 1) / p.block_cols;
    float s = 0.f;
    for (int b = 0; b < nb; b++) s += p.irg_partial[(int64_t)(cb + b) * p.M + pr];
    cb += nb;
    const float irv = p.ir[(int64_t)ir_row * p.n_tiles + t];
    if (p.relative) s = s * irv * p.scale;
    if (p.decay > 0.f) s = s + p.decay * irv * flag;
    p.ir_grad[(int64_t)r * p.n_tiles + t] = s;
  }
}

}  // namespace amoe
