// Weight gradient: argument checks and launches.
#include "host_util.h"
#include "gemm_wgrad256.h"
#include "gemm_wgrad.h"

using namespace amoe;

extern "C" {

namespace {
// Rows per chunk of the weight gradient: enough (expert, chunk, tile) workgroups to fill the chip
// twice over, chunks of 256 .. 4096 rows; 0 when one chunk per expert already does that.
struct WgradSplit { int rows_per_chunk; long long slots; int tiles; };
WgradSplit wgrad_split(const amoe_bwd_w_args* a) {
  WgradSplit s{0, 0, 0};
  const int kb = count_col_blocks(a->tile_bounds, a->n_tiles);
  const int nb = (a->N + kTileCols - 1) / kTileCols;
  s.tiles = kb * nb;
  long long R;
  if (a->rows_per_chunk > 0) {
    R = ((long long)a->rows_per_chunk + 63) / 64 * 64;
  } else {
    const long long target = 4LL * num_compute_units();
    const long long chunks = (target + s.tiles - 1) / s.tiles;
    R = chunks > 0 ? (a->M + chunks - 1) / chunks : a->M;
    R = (R + 255) / 256 * 256;
    R = R < 256 ? 256 : (R > 4096 ? 4096 : R);
  }
  if (R >= a->M) return s;                 // a single chunk everywhere
  s.rows_per_chunk = (int)R;
  s.slots = 2LL * a->M / R + 1;            // bound on the chunks of the experts that are cut
  return s;
}
}  // namespace

size_t amoe_bwd_w_workspace(const amoe_bwd_w_args* a) {
  if (!a || a->M < 1 || a->N < 1 || a->K < 1 || a->E < 1) return 0;
  if (check_bounds(a->n_tiles, a->tile_bounds, a->K)) return 0;
  const WgradSplit s = wgrad_split(a);
  if (s.rows_per_chunk == 0) return 0;
  return (size_t)s.slots * s.tiles * kWgradTileElems * sizeof(float);
}

int amoe_cvmm_bwd_w(const amoe_bwd_w_args* a, void* stream) {
  if (!a) return AMOE_ENULL;
  if (a->dtype != AMOE_F32 && a->dtype != AMOE_BF16 && a->dtype != AMOE_F16) return AMOE_EINVAL;
  if (a->M < 0 || a->N < 1 || a->K < 1 || a->E < 1 || a->n_x_rows < 0 || a->n_g_rows < 0) return AMOE_EINVAL;
  if (!a->grad_w || !a->offsets) return AMOE_ENULL;
  if (a->M > 0 && (!a->x || !a->g || !a->in_index)) return AMOE_ENULL;
  if (int rc = check_bounds(a->n_tiles, a->tile_bounds, a->K)) return rc;
  if (a->M > 0 && (a->ldx < a->K || a->ldg < a->N)) return AMOE_ESHAPE;
  const size_t es = esize(a->dtype);
  if (!aligned(a->x, es) || !aligned(a->g, es) || !aligned(a->grad_w, es) || !aligned(a->offsets, 4) ||
      !aligned(a->in_index, 4) || !aligned(a->g_index, 4) || !aligned(a->ir, 4) || !aligned(a->g_scale, es))
    return AMOE_EALIGN;
  const int CH = a->dtype == AMOE_F32 ? 4 : 8;
  WgradParams p{};
  p.M = a->M; p.N = a->N; p.K = a->K; p.E = a->E;
  p.x = a->x; p.ldx = a->ldx; p.g = a->g; p.ldg = a->ldg; p.grad_w = a->grad_w;
  p.offsets = a->offsets; p.in_index = a->in_index; p.g_index = a->g_index;
  p.ir = a->ir; p.ir_by_expert = a->ir_by_expert; p.g_scale = a->g_scale; p.n_tiles = a->n_tiles;
  for (int t = 0; t <= a->n_tiles; t++) p.bounds[t] = a->tile_bounds[t];
  p.n_k_blocks = count_col_blocks(p.bounds, p.n_tiles);
  p.n_n_blocks = (a->N + kTileCols - 1) / kTileCols;
  p.x_vec = aligned(a->x, 16) && (a->ldx % CH == 0) && bounds_multiple_of(a->n_tiles, a->tile_bounds, CH);
  p.g_vec = aligned(a->g, 16) && (a->ldg % CH == 0);
  p.out_vec = aligned(a->grad_w, 16) && (a->N % 4 == 0);
  p.out_stage = aligned(a->grad_w, 16) && (a->N % CH == 0);
  p.buf_ok = a->n_x_rows > 0 && a->n_g_rows > 0 && a->n_x_rows * a->ldx * (long long)es < (1LL << 31) &&
             a->n_g_rows * a->ldg * (long long)es < (1LL << 31);
  hipStream_t st = static_cast<hipStream_t>(stream);
  long long pairs = a->E;                  // (expert, chunk) pairs, worst case
  if (a->workspace != nullptr && a->M > 0) {
    const WgradSplit s = wgrad_split(a);
    if (s.rows_per_chunk > 0) {
      if (!aligned(a->workspace, 16)) return AMOE_EALIGN;
      if (a->workspace_bytes < amoe_bwd_w_workspace(a)) return AMOE_EWORKSPACE;
      if (a->E > kSelMaxExperts) return AMOE_EUNSUPPORTED;
      p.rows_per_chunk = s.rows_per_chunk;
      p.partial = static_cast<float*>(a->workspace);
      pairs = a->M / s.rows_per_chunk + a->E;
    }
  }
  const long long grid = 8LL * ((pairs + 7) / 8) * p.n_k_blocks * p.n_n_blocks;   // see the id mapping in the kernel
  if (grid > 0x7fffffffLL) return AMOE_EUNSUPPORTED;
  const long long rgrid = (long long)a->E * p.n_k_blocks * p.n_n_blocks * kWgradReduceSplit;
  if (rgrid > 0x7fffffffLL) return AMOE_EUNSUPPORTED;
  // the 256 x 256 kernel for the training shapes (16-bit elements, interior tiles, per-expert ranges)
  bool wide = a->dtype != AMOE_F32 && p.x_vec && p.g_vec && p.out_stage && p.buf_ok && a->N % kW256Tile == 0 &&
              (a->ir == nullptr || a->ir_by_expert);
  for (int t = 0; t < a->n_tiles && wide; t++) wide = (a->tile_bounds[t + 1] - a->tile_bounds[t]) % kW256Tile == 0;
  if (wide) {
    const long long grid256 = 8LL * ((pairs + 7) / 8) * (p.n_k_blocks / 2) * (p.n_n_blocks / 2);
    if (a->dtype == AMOE_BF16) {
      hipLaunchKernelGGL((&wgrad256_kernel<uint16_t>), dim3((unsigned)grid256), dim3(kW256Threads), 0, st, p);
    } else {
      hipLaunchKernelGGL((&wgrad256_kernel<f16_t>), dim3((unsigned)grid256), dim3(kW256Threads), 0, st, p);
    }
    if (int rc = launch_rc()) return rc;
    if (p.rows_per_chunk > 0) {
      if (a->dtype == AMOE_BF16) {
        hipLaunchKernelGGL((&wgrad_reduce_kernel<uint16_t>), dim3((unsigned)rgrid), dim3(kThreads), 0, st, p);
      } else {
        hipLaunchKernelGGL((&wgrad_reduce_kernel<f16_t>), dim3((unsigned)rgrid), dim3(kThreads), 0, st, p);
      }
    }
    return launch_rc();
  }
  if (a->dtype == AMOE_F32) {
    auto k = &gemm_wgrad_kernel<float>;
    hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(kThreads), 0, st, p);
    if (int rc = launch_rc()) return rc;
    if (p.rows_per_chunk > 0) {
      auto r = &wgrad_reduce_kernel<float>;
      hipLaunchKernelGGL(r, dim3((unsigned)rgrid), dim3(kThreads), 0, st, p);
    }
  } else if (a->dtype == AMOE_BF16) {
    auto k = &gemm_wgrad_kernel<uint16_t>;
    hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(kThreads), 0, st, p);
    if (int rc = launch_rc()) return rc;
    if (p.rows_per_chunk > 0) {
      auto r = &wgrad_reduce_kernel<uint16_t>;
      hipLaunchKernelGGL(r, dim3((unsigned)rgrid), dim3(kThreads), 0, st, p);
    }
  } else {
    auto k = &gemm_wgrad_kernel<f16_t>;
    hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(kThreads), 0, st, p);
    if (int rc = launch_rc()) return rc;
    if (p.rows_per_chunk > 0) {
      auto r = &wgrad_reduce_kernel<f16_t>;
      hipLaunchKernelGGL(r, dim3((unsigned)rgrid), dim3(kThreads), 0, st, p);
    }
  }
  return launch_rc();
}

}  // extern "C"
