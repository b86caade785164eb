// The analog router at inference as one launch (router_kernel.h).
#include <amoe.h>

#include "host_util.h"
#include "router_kernel.h"

using namespace amoe;

extern "C" int amoe_router_fwd(int32_t dtype, const void* x, int64_t ldx, int64_t T, int32_t D, const void* w, int64_t ldw, int32_t E,
                               int32_t k, const void* ir, int32_t n_tiles, const int32_t* bounds, float inp_res, float out_bound,
                               float out_res, void* sel_val, int64_t* sel_idx, void* stream) {
  if (dtype != AMOE_F32 && dtype != AMOE_BF16 && dtype != AMOE_F16) return AMOE_EINVAL;
  if (T < 0 || D < 1 || E < 1 || k < 1 || k > E) return AMOE_EINVAL;
  if (T == 0) return AMOE_OK;
  if (!x || !w || !ir || !bounds || !sel_val || !sel_idx) return AMOE_ENULL;
  if (int rc = check_bounds(n_tiles, bounds, D)) return rc;
  if (ldx < D || ldw < D) return AMOE_ESHAPE;
  const int64_t es = (int64_t)esize(dtype);
  if (!aligned(x, es) || !aligned(w, es) || !aligned(ir, es) || !aligned(sel_val, es) || !aligned(sel_idx, 8)) return AMOE_EALIGN;
  // a workgroup holds the logits of all experts; a K-tile has a whole number of its waves; 4-byte aligned rows
  if (E > 128 || T > 0x7fffffffLL || kDirWaves % n_tiles != 0) return AMOE_EUNSUPPORTED;
  if (!(inp_res > 0.f) || !dac_codes_fit(dtype, inp_res)) return AMOE_EUNSUPPORTED;
  if (!aligned(x, 4) || !aligned(w, 4) || (ldx * es) % 4 || (ldw * es) % 4) return AMOE_EUNSUPPORTED;
  RouterParams p{};
  for (int t = 0; t <= n_tiles; t++) {
    if (t < n_tiles && (bounds[t] * es) % 4) return AMOE_EUNSUPPORTED;
    p.bounds[t] = bounds[t];
  }
  p.x = x; p.ldx = ldx; p.w = w; p.ldw = ldw;
  p.T = (int)T; p.K = D; p.E = E; p.k = k;
  p.n_tiles = n_tiles; p.ir = ir;
  p.inp_res = inp_res; p.out_bound = out_bound;
  p.out_half_states = (out_bound > 0.f && out_res > 0.f) ? 0.5f * fmaxf(out_res, 1.0f / out_res) : 0.f;
  p.sel_val = sel_val; p.sel_idx = sel_idx;
  // A wave's rows go through the top-k one after the other and every workgroup reads all of W: as few rows per workgroup
  // as one workgroup per CU allows.
  p.rows_per_block = 8;
  while (p.rows_per_block < kDirRows && (T + p.rows_per_block - 1) / p.rows_per_block > num_compute_units()) p.rows_per_block *= 2;
  const dim3 grid((unsigned)((T + p.rows_per_block - 1) / p.rows_per_block)), block(kDirThreads);
  hipStream_t st = static_cast<hipStream_t>(stream);
#define AMOE_ROUTER(TYPE)                                                             \
  do {                                                                                \
    if (E <= 64) hipLaunchKernelGGL((&router_kernel<TYPE, 2>), grid, block, 0, st, p); \
    else hipLaunchKernelGGL((&router_kernel<TYPE, 4>), grid, block, 0, st, p);         \
  } while (0)
  if (dtype == AMOE_F32) AMOE_ROUTER(float);
  else if (dtype == AMOE_F16) AMOE_ROUTER(f16_t);
  else AMOE_ROUTER(uint16_t);
#undef AMOE_ROUTER
  return launch_rc();
}
