// C ABI of libamoe: argument checks on the host, then kernel launches on the caller's stream.
#include <amoe.h>

#include <atomic>

#include "host_util.h"
#include "ir_grad.h"
#include "misc_kernels.h"
#include "weight_kernels.h"
#include "select_kernels.h"
#include "prepare_sel.h"

using namespace amoe;

extern "C" {

int amoe_version(void) { return AMOE_VERSION; }

const char* amoe_strerror(int rc) {
  switch (rc) {
    case AMOE_OK: return "ok";
    case AMOE_EINVAL: return "invalid size, stride or scalar";
    case AMOE_ENULL: return "required pointer is NULL";
    case AMOE_ESHAPE: return "inconsistent sizes";
    case AMOE_EALIGN: return "pointer not aligned to 4 bytes";
    case AMOE_EWORKSPACE: return "workspace too small (or the call exceeds the library's own scratch array)";
    case AMOE_EUNSUPPORTED: return "not supported by this build";
    default: return rc > 0 ? "HIP launch error" : "unknown error";
  }
}

// ------------------------------------------------------------------------------ selection
size_t amoe_prepare_sel_workspace(int64_t M, int32_t E) {
  if (M < 0 || E < 1) return 0;
  const int64_t per = sel_by_groups(M, E) ? sel_span(M, E) : sel_unit(M);
  const int64_t units = (M + per - 1) / per;
  return (size_t)(units > 0 ? units : 1) * (size_t)E * sizeof(int32_t);
}

int amoe_prepare_sel(const void* sel, int32_t sel_is_i64, int64_t M, int32_t E, int32_t k,
                     int32_t* sel_sorted, int32_t* perm, int32_t* in_index, int32_t* offsets,
                     int32_t* bad_flag, void* workspace, size_t workspace_bytes, void* stream) {
  if (M < 0 || M > 0x7fffffffLL || E < 1 || k < 1) return AMOE_EINVAL;
  if (E > kSelMaxExperts) return AMOE_EUNSUPPORTED;
  if (!offsets || !workspace || (M > 0 && (!sel || !sel_sorted || !perm || !in_index))) return AMOE_ENULL;
  if (!aligned(sel, sel_is_i64 ? 8 : 4) || !aligned(sel_sorted, 4) || !aligned(perm, 4) ||
      !aligned(in_index, 4) || !aligned(offsets, 4) || !aligned(workspace, 4) || !aligned(bad_flag, 4))
    return AMOE_EALIGN;
  if (workspace_bytes < amoe_prepare_sel_workspace(M, E)) return AMOE_EWORKSPACE;
  SelParams p;
  p.sel = sel; p.sel_is_i64 = sel_is_i64; p.M = M; p.E = E; p.k = k;
  const bool by_groups = sel_by_groups(M, E);
  p.unit = by_groups ? sel_span(M, E) : sel_unit(M);
  p.n_units = (int)((M + p.unit - 1) / p.unit);
  p.key_bits = 0;
  while ((1 << p.key_bits) < E) p.key_bits++;
  p.sel_sorted = sel_sorted; p.perm = perm; p.in_index = in_index; p.offsets = offsets;
  p.bad_flag = bad_flag; p.unit_hist = static_cast<int32_t*>(workspace);
  p.table_vec = aligned(workspace, 16) && E % 4 == 0;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (by_groups) {
    const int groups = p.n_units > 0 ? p.n_units : 1;        // (no elements: the offsets are still written)
    if (M <= kSelSmall) {
      hipLaunchKernelGGL((&sel_group_scatter_kernel<true>), dim3(groups), dim3(kThreads), 0, st, p);
      return launch_rc();
    }
    hipLaunchKernelGGL(sel_group_hist_kernel, dim3(groups), dim3(kThreads), 0, st, p);
    if (int rc = launch_rc()) return rc;
    hipLaunchKernelGGL((&sel_group_scatter_kernel<false>), dim3(groups), dim3(kThreads), 0, st, p);
    return launch_rc();
  }
  const int blocks = (p.n_units + 3) / 4;
  if (blocks > 0) {
    hipLaunchKernelGGL(sel_hist_kernel, dim3(blocks), dim3(kThreads), 0, st, p);
    if (int rc = launch_rc()) return rc;
  }
  hipLaunchKernelGGL(sel_unit_scan_kernel, dim3((E + 3) / 4), dim3(kThreads), 0, st, p);
  if (int rc = launch_rc()) return rc;
  hipLaunchKernelGGL(sel_offsets_kernel, dim3(1), dim3(kThreads), 0, st, p);
  if (int rc = launch_rc()) return rc;
  if (blocks > 0) {
    hipLaunchKernelGGL(sel_scatter_kernel, dim3(blocks), dim3(kThreads), 0, st, p);
    if (int rc = launch_rc()) return rc;
  }
  return AMOE_OK;
}

// ---- selection without any allocation: the unit histograms live in a device array of the library ----------
}  // extern "C"

// One copy per GPU the library runs on, held until the process ends.  In host code the array's NAME is only a
// stand-in for the symbol, not a device address: the device address is asked for once per device and kept.
static __device__ __align__(256) unsigned char scratch[AMOE_NOALLOC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::atomic<void*> g_scratch_ptr[kMaxDevices];

// Device address of `scratch` on the current device (looked up on the first call per device).
int scratch_address(void** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= kMaxDevices) return AMOE_EUNSUPPORTED;
  void* ptr = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (ptr == nullptr) {
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    if (ptr == nullptr) return AMOE_EUNSUPPORTED;
    g_scratch_ptr[dev].store(ptr, std::memory_order_release);   // every thread would store the same address
  }
  *out = ptr;
  return AMOE_OK;
}
}  // namespace

extern "C" {

size_t amoe_noalloc_scratch_bytes(void) { return AMOE_NOALLOC_SCRATCH_BYTES; }

int amoe_prepare_sel_noalloc(const void* sel, int32_t sel_is_i64, int64_t M, int32_t E, int32_t k,
                             int32_t* sel_sorted, int32_t* perm, int32_t* in_index, int32_t* offsets,
                             int32_t* bad_flag, void* stream) {
  if (M < 0 || M > 0x7fffffffLL || E < 1 || k < 1) return AMOE_EINVAL;
  if (E > kSelMaxExperts) return AMOE_EUNSUPPORTED;
  // the histograms of this call must fit the library's array; nothing is allocated to make room
  if (amoe_prepare_sel_workspace(M, E) > (size_t)AMOE_NOALLOC_SCRATCH_BYTES) return AMOE_EWORKSPACE;
  void* ws = nullptr;
  if (int rc = scratch_address(&ws)) return rc;
  // every unit's histogram row is written by the first pass before anything reads it, so what the previous
  // call left in the array does not matter and nothing has to be cleared
  return amoe_prepare_sel(sel, sel_is_i64, M, E, k, sel_sorted, perm, in_index, offsets, bad_flag, ws,
                          (size_t)AMOE_NOALLOC_SCRATCH_BYTES, stream);
}

int amoe_offsets_from_sorted(const int32_t* sel_sorted, int64_t M, int32_t E, int32_t* offsets, void* stream) {
  if (M < 0 || M > 0x7fffffffLL || E < 1) return AMOE_EINVAL;
  if (!offsets || (M > 0 && !sel_sorted)) return AMOE_ENULL;
  if (!aligned(sel_sorted, 4) || !aligned(offsets, 4)) return AMOE_EALIGN;
  const int blocks = (int)((M + 1 + kThreads - 1) / kThreads);
  hipLaunchKernelGGL(offsets_from_sorted_kernel, dim3(blocks), dim3(kThreads), 0, static_cast<hipStream_t>(stream),
                     sel_sorted, (long long)M, (int)E, offsets);
  return launch_rc();
}

// ------------------------------------------------------------------------------ forward
int amoe_fwd_codes_supported(const amoe_fwd_args* a) {
  if (!a || (a->dtype != AMOE_BF16 && a->dtype != AMOE_F16)) return 0;
  if (a->N < 1 || a->K < 1 || a->E < 1 || a->n_tiles != 1 || a->w_stride_n != 1) return 0;
  // every tile interior, 16-byte pieces everywhere, 32-bit byte offsets
  if (a->N % kFCols || a->K % kFBK || a->ldx % 8 || a->w_stride_e % 8 || a->w_stride_k % 8 || a->ldcode % 16) return 0;
  if (a->ldx < a->K || a->w_stride_k < a->N || a->ldcode < a->N) return 0;
  const long long lim = 1LL << 31;
  if (a->n_in_rows <= 0 || (long long)a->n_in_rows * a->ldx * 2 >= lim ||
      ((long long)a->K * a->w_stride_k + (long long)a->N) * 2 >= lim)
    return 0;
  // the analog stages the kernel is built for: per-expert input ranges with an input quantiser whose codes the type
  // holds, one max |W| per expert, generated noise or none, an output quantiser whose codes fit a byte
  if (!a->ir || !a->ir_by_expert || !(a->inp_res > 0.f) || !dac_codes_fit(a->dtype, a->inp_res) || a->abs_max) return 0;
  if (a->noise || !a->wmax || a->wmax_cols != 1 || !(a->out_bound > 0.f) || !(a->out_res > 0.f)) return 0;
  if (!(0.5f * fmaxf(a->out_res, 1.0f / a->out_res) <= 127.f)) return 0;
  if (a->xq_out || a->relu) return 0;
  return 1;
}

// Which kernel of gemm_direct.h takes the launch: one wave per 32 x 64 tile, eight waves per tile, or none.
//
// Against the tiled kernels: these re-read weights per 32 rows and rows per 64 columns.  What one wave per tile gains it gains
// by overlapping the stages around the product, so it is taken in fp32, and where the tiled kernel would run its element-wise
// edge code, but not
//   in fp32 without an input stage past a wave per SIMD: 2048 -> 512, 1096 tiles 195 against 157 us, 64 -> 512, 3344 tiles
//   23.3 against 20.1 (at 1 tile per SIMD and less 1.4 to 2 times faster);
//   in fp32 with an input but no output stage in many whole column blocks: 64 -> 256, 32788 tiles 178 against 160 us, 128 ->
//   256 257 against 235; up to 64 tiles per CU it is 1.15 to 1.3 times faster (128 -> 512, 4168 tiles 40.8 against 45.4), and
//   with the ADC or noise at any size (32 768 tokens 412 -> 128, 8210 tiles 174 against 187; 224 -> 512, 9808 tiles 116
//   against 168).  Loads that are exactly even over 8 experts can be tiled without a remainder, and lose up to a fifth
//   (8192 rows 256 -> 1024 63.5 against 52.3 us);
//   in 16 bits over a long contraction with many tiles, where the edge code is a small part: 1800 -> 512, 32904 tiles 853
//   against 771 us, 2044 -> 512 944 against 916 (1500 -> 256, 16452 tiles 379 against 403, 1004 -> 512, 32904 tiles 522
//   against 544).
// bf16 with edges, 8192 tokens 128 -> 412: 38 against 73 us, 1024 -> 320 in two K-tiles 112 against 284.  Edge-free 16-bit
// launches go there only while they are small: 512 -> 128 with 544 tiles 18.7 against 21.7 us, with 2176 tiles 39.5 against
// 28.1.  A contraction of 256 with columns in groups of 256 stays with the weights-in-registers kernel and its twins.
//
// One wave or eight: a wave walks its contraction in 5 us + 45 ns (fp32) or 22 ns (16-bit) per element of K; eight waves
// need 5 us + 12 ns or 6 ns, but fill a CU by themselves, so they do it once per 256 tiles (fp32 412 -> 128, 146 tiles 13.4
// against 25.0 us, 544 tiles 37.1 against 26.8; bf16 1024 -> 320, 400 tiles 20.3 against 29.9, 1360 tiles 61 against 41.5).
enum { DIRECT_NO = 0, DIRECT_WAVE = 1, DIRECT_SPLIT = 2 };
static int direct_choice(const amoe_fwd_args* a, const RowsParams& p, bool w_kc, int mode) {
  const bool f32 = a->dtype == AMOE_F32;
  if (!f32 && !w_kc && a->K == kWsK && a->N % 256 == 0) return DIRECT_NO;
  const int64_t rows = a->M / kDirRows + (a->E < a->M ? a->E : a->M) / 2 + 1;     // an expert's last tile is half full
  const int64_t tiles = rows * ((a->N + kDirCols - 1) / kDirCols), cus = num_compute_units();
  const bool edge_free = !f32 && rows_all_interior(p, mode, a->N % kFCols == 0 && !w_kc ? kFBK : Elem<uint16_t>::kBK);
  if (edge_free && tiles > 3 * cus) return DIRECT_NO;
  if (f32 && a->ir == nullptr && tiles > 4 * cus) return DIRECT_NO;
  if (a->N % kTileCols == 0) {
    if (f32 && !(a->out_bound > 0.f) && !(a->noise_std > 0.f) && tiles > 64 * cus) return DIRECT_NO;
    if (!f32 && a->K >= 1400 && tiles * a->K > 28000000LL) return DIRECT_NO;
  }
  const int64_t rounds = (tiles + cus - 1) / cus, K = a->K;
  const bool split = f32 ? rounds * (400 + K) * 5 < 2000 + 18 * K : rounds * (900 + K) < 800 + 4 * K;
  return split ? DIRECT_SPLIT : DIRECT_WAVE;
}

int amoe_cvmm_fwd(const amoe_fwd_args* a, void* stream) {
  if (!a) return AMOE_ENULL;
  if (a->dtype != AMOE_F32 && a->dtype != AMOE_BF16 && a->dtype != AMOE_F16) return AMOE_EINVAL;
  if (a->M < 0 || a->N < 1 || a->K < 1 || a->E < 1 || a->n_in_rows < 0 || a->n_out_rows < 0) return AMOE_EINVAL;
  if (a->M == 0) return AMOE_OK;
  if (!a->x || !a->w || (!a->out && !a->code_out) || !a->offsets || !a->in_index) return AMOE_ENULL;
  if (a->code_out && (!a->code_scale_out || a->ldcode < a->N)) return AMOE_EINVAL;
  if (int rc = check_bounds(a->n_tiles, a->tile_bounds, a->K)) return rc;
  if (a->ldx < a->K || (a->out && a->ldo < a->N)) return AMOE_ESHAPE;
  if (a->w_stride_n != 1 && a->w_stride_k != 1) return AMOE_EUNSUPPORTED;
  const bool gen_noise = a->noise == nullptr && a->noise_std > 0.f;
  const bool adc = a->out_bound > 0.f;
  if ((gen_noise || adc) && (!a->wmax || (a->wmax_cols != 1 && a->wmax_cols != a->N))) return AMOE_ESHAPE;
  if (a->noise && (a->ldnoise < a->N)) return AMOE_ESHAPE;
  if (a->xq_out && (!a->xq_ir || !(a->xq_inp_res > 0.f))) return AMOE_EINVAL;
  if (a->xq_out && a->ldxq < a->N) return AMOE_ESHAPE;
  if (a->x_is_quantized && (!a->ir || !(a->inp_res > 0.f) || a->abs_max || a->n_tiles != 1)) return AMOE_EINVAL;
  // 16-bit element types carry the DAC codes themselves to the matrix unit (and in xq_out): integers are exact up
  // to 256 in bf16 and 2048 in fp16, so a finer input quantiser needs fp32 tensors
  if (!dac_codes_fit(a->dtype, a->inp_res) || (a->xq_out && !dac_codes_fit(a->dtype, a->xq_inp_res)))
    return AMOE_EUNSUPPORTED;
  const size_t es = esize(a->dtype);
  if (!aligned(a->x, es) || !aligned(a->w, es) || !aligned(a->out, es) || !aligned(a->offsets, 4) ||
      !aligned(a->in_index, 4) || !aligned(a->out_index, 4) || !aligned(a->ir, 4) || !aligned(a->abs_max, 4) ||
      !aligned(a->noise, 4) || !aligned(a->wmax, 4) || !aligned(a->range_flag, 4) || !aligned(a->noise_seed_dev, 8) ||
      !aligned(a->xq_out, es) || !aligned(a->xq_ir, 4))
    return AMOE_EALIGN;

  const int CH = a->dtype == AMOE_F32 ? 4 : 8;
  RowsParams p{};
  p.M = a->M; p.E = a->E; p.KD = a->K; p.ND = a->N;
  p.a = a->x; p.lda = a->ldx;
  p.w = a->w; p.w_se = a->w_stride_e; p.w_skd = a->w_stride_k; p.w_snd = a->w_stride_n;
  p.out = a->out; p.ldo = a->ldo;
  p.offsets = a->offsets; p.a_index = a->in_index; p.out_index = a->out_index;
  p.n_kd_tiles = a->n_tiles;
  for (int t = 0; t <= a->n_tiles; t++) p.kd_bounds[t] = a->tile_bounds[t];
  p.n_col_tiles = 1; p.col_bounds[0] = 0; p.col_bounds[1] = a->N;
  p.n_col_blocks = count_col_blocks(p.col_bounds, 1);
  p.ir = a->ir; p.ir_cols = a->n_tiles; p.ir_by_expert = a->ir_by_expert; p.abs_max = a->abs_max;
  p.inp_res = a->inp_res;
  p.noise = a->noise; p.noise_ts = a->noise_tile_stride; p.ldnoise = a->ldnoise;
  p.noise_std = a->noise_std; p.seed = a->noise_seed; p.seed_dev = a->noise_seed_dev;
  p.wmax = a->wmax; p.wmax_cols = a->wmax_cols;
  p.out_bound = a->out_bound;
  p.out_half_states = (adc && a->out_res > 0.f) ? 0.5f * fmaxf(a->out_res, 1.0f / a->out_res) : 0.f;
  p.relu = a->relu; p.range_flag = a->range_flag;
  p.xq_out = a->xq_out; p.ldxq = a->ldxq; p.xq_ir = a->xq_ir; p.xq_inp_res = a->xq_inp_res;
  p.xq_vec = a->xq_out && aligned(a->xq_out, 16) && (a->ldxq % 4 == 0);
  p.xq_stage = a->xq_out && aligned(a->xq_out, 16) && (a->ldxq % CH == 0);
  p.a_prequant = a->x_is_quantized;
  p.code_out = a->code_out; p.ldcode = a->ldcode; p.code_scale_out = a->code_scale_out;
  const bool w_kc = a->w_stride_n != 1;
  p.a_vec = aligned(a->x, 16) && (a->ldx % CH == 0) && bounds_multiple_of(a->n_tiles, a->tile_bounds, CH);
  p.w_vec = aligned(a->w, 16) && (a->w_stride_e % CH == 0) &&
            (w_kc ? (a->w_stride_n % CH == 0 && bounds_multiple_of(a->n_tiles, a->tile_bounds, CH))
                  : (a->w_stride_k % CH == 0));
  p.out_vec = aligned(a->out, 16) && (a->ldo % 4 == 0);
  p.out_stage = aligned(a->out, 16) && (a->ldo % CH == 0);
  p.noise_vec = a->noise && aligned(a->noise, 16) && (a->ldnoise % 4 == 0) && (a->noise_tile_stride % 4 == 0);
  const long long lim = 1LL << 31;
  // (n_in_rows == 0: the caller does not state the rows of x, so nothing bounds its extent)
  p.buf_ok = a->n_in_rows > 0 && (long long)a->n_in_rows * a->ldx * (long long)es < lim &&
             ((long long)a->K * a->w_stride_k + (long long)a->N * a->w_stride_n) * (long long)es < lim;
  const int mode = a->n_tiles > 1 ? MODE_FWD_SPLIT : MODE_FWD;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (const int direct = direct_choice(a, p, w_kc, mode)) {
    const int rc = launch_direct(p, w_kc, a, direct == DIRECT_SPLIT, st);
    if (rc != AMOE_EUNSUPPORTED) return rc;
  }
  if (a->dtype != AMOE_F32 && !w_kc) {
    const int rc = launch_fwd256(p, mode, a, st);
    if (rc != AMOE_EUNSUPPORTED) return rc;
  }
  if (a->code_out) return AMOE_EUNSUPPORTED;      // only the kernel above writes codes
  const int grid = persistent_grid(max_row_tiles(a->M, a->E), p.n_col_blocks);
  return launch_rows(a->dtype, p, w_kc, mode, grid, st);
}

// ------------------------------------------------------------------------------ input gradient
size_t amoe_bwd_x_workspace(int64_t M, int32_t K, int32_t n_tiles) {
  if (M < 0 || K < 1 || n_tiles < 1) return 0;
  // worst case: every K-tile adds one partial column block
  const int64_t col_blocks = (K + kTileCols - 1) / kTileCols + n_tiles;
  const int64_t row_tiles = M / kTileRows + kSelMaxExperts;
  return (size_t)(col_blocks * (M > 0 ? M : 1)) * sizeof(float) + (size_t)(row_tiles * col_blocks) * sizeof(int32_t);
}

// Plain input gradients (no mask, gate or range) in fp32 or with edges, up to a wave per SIMD: the forward product with
// contraction-contiguous weights, one wave per 32 x 64 tile.  Always one wave: it adds in the tiled kernel's order, so
// that the clip applied by the sum over the heads gives the masked launch's result bit for bit.  With more tiles the
// tiled kernel's shared operands win.  us per launch, tiled and direct, contraction -> columns:
//   fp32  64 -> 132, 963 tiles 16.5 / 13.0; 128 -> 412, 483 tiles 16.4 / 12.1; 256 -> 1028, 629 tiles 28.4 / 19.5;
//         516 -> 2044, 672 tiles 51.5 / 31.8; but 128 -> 412, 2247 tiles 27.5 / 29.1; 516 -> 2044, 1184 tiles 53.2 / 53.8
//   bf16  64 -> 132, 579 tiles 7.0 / 6.1; 516 -> 2044, 672 tiles 24.8 / 16.6; 256 -> 1028, 629 tiles 11.0 / 10.8; but
//         1173 tiles 12.0 / 17.3; 128 -> 412, 1351 tiles 11.1 / 12.7
static bool bwdx_direct(const amoe_bwd_x_args* a, const RowsParams& p) {
  if (bwdx_reads_x(a) || a->ir || a->relu_mask || a->gate || a->xc_out) return false;
  const int64_t rows = a->M / kDirRows + (a->E < a->M ? a->E : a->M) / 2 + 1;     // an expert's last tile is half full
  if (rows * ((a->K + kDirCols - 1) / kDirCols) > 4 * num_compute_units()) return false;
  return a->dtype == AMOE_F32 || !rows_all_interior(p, MODE_BWDX, Elem<uint16_t>::kBK);
}

static int launch_bwdx_direct(const amoe_bwd_x_args* a, const RowsParams& p, hipStream_t st) {
  amoe_fwd_args f{};
  f.dtype = a->dtype;
  f.M = a->M; f.K = a->N; f.N = a->K; f.E = a->E;
  f.x = a->g; f.ldx = a->ldg;
  f.w = a->w; f.w_stride_e = a->w_stride_e; f.w_stride_k = 1; f.w_stride_n = a->w_stride_k;
  f.n_tiles = 1; f.tile_bounds[1] = a->N;
  f.inp_res = -1.f;
  return launch_direct(p, true, &f, false, st);
}

int amoe_cvmm_bwd_x(const amoe_bwd_x_args* a, void* stream) {
  if (!a) return AMOE_ENULL;
  if (a->dtype != AMOE_F32 && a->dtype != AMOE_BF16 && a->dtype != AMOE_F16) return AMOE_EINVAL;
  if (a->M < 0 || a->N < 1 || a->K < 1 || a->E < 1 || a->E > kSelMaxExperts || a->n_g_rows < 0) return AMOE_EINVAL;
  if (a->M == 0) return AMOE_OK;
  if (!a->g || !a->w || !a->grad_x_full || !a->offsets || !a->g_index || !a->out_index) return AMOE_ENULL;
  if (int rc = check_bounds(a->n_tiles, a->tile_bounds, a->K)) return rc;
  const bool use_ir = a->ir != nullptr;
  if ((use_ir || a->relu_mask) && (!a->x || !a->xf_index)) return AMOE_ENULL;
  if (use_ir && (!a->ir_grad || !a->workspace)) return AMOE_ENULL;
  if (a->xc_out && (!a->x || !a->xf_index)) return AMOE_ENULL;
  if (a->xc_out && a->ldxc < a->K) return AMOE_ESHAPE;
  if (a->ldg < a->N || a->ldo < a->K || (a->x && a->ldx < a->K) || a->w_stride_k < a->N) return AMOE_ESHAPE;
  const size_t es = esize(a->dtype);
  if (!aligned(a->g, es) || !aligned(a->w, es) || !aligned(a->grad_x_full, es) || !aligned(a->x, es) ||
      !aligned(a->gate, es) || !aligned(a->offsets, 4) || !aligned(a->g_index, 4) || !aligned(a->out_index, 4) ||
      !aligned(a->xf_index, 4) || !aligned(a->ir, 4) || !aligned(a->ir_grad, 4) || !aligned(a->workspace, 4))
    return AMOE_EALIGN;
  const int CH = a->dtype == AMOE_F32 ? 4 : 8;
  RowsParams p{};
  p.M = a->M; p.E = a->E; p.KD = a->N; p.ND = a->K;
  p.a = a->g; p.lda = a->ldg;
  p.w = a->w; p.w_se = a->w_stride_e; p.w_skd = 1; p.w_snd = a->w_stride_k;
  p.out = a->grad_x_full; p.ldo = a->ldo;
  p.offsets = a->offsets; p.a_index = a->g_index; p.out_index = a->out_index;
  p.n_kd_tiles = 1; p.kd_bounds[0] = 0; p.kd_bounds[1] = a->N;
  p.n_col_tiles = a->n_tiles;
  for (int t = 0; t <= a->n_tiles; t++) p.col_bounds[t] = a->tile_bounds[t];
  p.n_col_blocks = count_col_blocks(p.col_bounds, p.n_col_tiles);
  p.ir = a->ir; p.ir_cols = a->n_tiles; p.ir_by_expert = a->ir_by_expert; p.inp_res = -1.f;
  p.xf = a->x; p.ldxf = a->ldx; p.xf_index = a->xf_index; p.gate = a->gate; p.relu_mask = a->relu_mask;
  p.xc_out = a->xc_out; p.ldxc = a->ldxc;
  p.xc_vec = a->xc_out && aligned(a->xc_out, 16) && (a->ldxc % CH == 0) && bounds_multiple_of(a->n_tiles, a->tile_bounds, CH);
  const int grid = persistent_grid(max_row_tiles(a->M, a->E), p.n_col_blocks);
  if (use_ir) {
    // (one count per workgroup; no grid is larger than the number of work items)
    const size_t need = (size_t)p.n_col_blocks * a->M * sizeof(float) +
                        (size_t)max_row_tiles(a->M, a->E) * p.n_col_blocks * sizeof(int32_t);
    if (a->workspace_bytes < need) return AMOE_EWORKSPACE;
    p.irg_partial = static_cast<float*>(a->workspace);
    p.notclip_count = reinterpret_cast<int32_t*>(p.irg_partial + (size_t)p.n_col_blocks * a->M);
  }
  p.a_vec = aligned(a->g, 16) && (a->ldg % CH == 0);
  p.w_vec = aligned(a->w, 16) && (a->w_stride_e % CH == 0) && (a->w_stride_k % CH == 0);
  p.buf_ok = a->n_g_rows > 0 && (long long)a->n_g_rows * a->ldg * (long long)es < (1LL << 31) &&
             (long long)a->K * a->w_stride_k * (long long)es < (1LL << 31);
  p.out_vec = aligned(a->grad_x_full, 16) && (a->ldo % 4 == 0) && bounds_multiple_of(a->n_tiles, a->tile_bounds, 4);
  p.out_stage = aligned(a->grad_x_full, 16) && (a->ldo % CH == 0) && bounds_multiple_of(a->n_tiles, a->tile_bounds, CH);
  p.xf_vec = a->x && aligned(a->x, 16) && (a->ldx % 4 == 0) && bounds_multiple_of(a->n_tiles, a->tile_bounds, 4);
  hipStream_t st = static_cast<hipStream_t>(stream);
  int block_cols = kTileCols, n_count_blocks = grid;
  int rc = bwdx_direct(a, p) ? launch_bwdx_direct(a, p, st) : AMOE_EUNSUPPORTED;
  if (rc == AMOE_EUNSUPPORTED && a->dtype != AMOE_F32) {
    int cols = kTileCols;
    rc = launch_bwdx256(p, a, st, &n_count_blocks, &cols);
    if (rc == AMOE_OK) block_cols = cols;
  }
  if (rc == AMOE_EUNSUPPORTED)
    rc = launch_rows(a->dtype, p, true, MODE_BWDX, grid, st);
  if (rc) return rc;
  if (use_ir) {
    IrFinalizeParams f{};
    f.M = a->M; f.n_tiles = a->n_tiles; f.KD_total = a->K; f.block_cols = block_cols;
    for (int t = 0; t <= a->n_tiles; t++) f.col_bounds[t] = a->tile_bounds[t];
    f.irg_partial = p.irg_partial; f.notclip_count = p.notclip_count; f.n_blocks = n_count_blocks;
    f.ir = a->ir; f.ir_by_expert = a->ir_by_expert; f.offsets = a->offsets; f.E = a->E; f.ir_grad = a->ir_grad;
    f.relative = a->gradient_relative; f.scale = a->gradient_scale; f.decay = a->decay;
    f.min_pct = a->input_min_percentage;
    hipLaunchKernelGGL(ir_grad_finalize_kernel, dim3((a->M + kThreads - 1) / kThreads), dim3(kThreads), 0, st, f);
    rc = launch_rc();
  }
  return rc;
}

// ------------------------------------------------------------------------------ row-wise companions
static int bump_only(int64_t* counter, int64_t counter_add, void* stream);

static int head_reduce(int32_t dtype, const void* z, const void* gate, void* y, int64_t T, int32_t k, int32_t D,
                       void* stream, int64_t* counter_ = nullptr, int64_t counter_add_ = 0) {
  if (dtype != AMOE_F32 && dtype != AMOE_BF16 && dtype != AMOE_F16) return AMOE_EINVAL;
  if (T < 0 || k < 1 || D < 1) return AMOE_EINVAL;
  if (!aligned(counter_, 8)) return AMOE_EALIGN;
  if (T == 0) return bump_only(counter_, counter_add_, stream);
  long long* counter = reinterpret_cast<long long*>(counter_);
  const long long counter_add = counter_add_;
  if (!z || !y) return AMOE_ENULL;
  const size_t es = esize(dtype);
  if (!aligned(z, es) || !aligned(y, es) || !aligned(gate, es)) return AMOE_EALIGN;
  const int CH = dtype == AMOE_F32 ? 4 : 8;
  const int vec = aligned(z, 16) && aligned(y, 16) && (D % CH == 0);
  const long long work = (long long)T * ((D + CH - 1) / CH);
  const long long blocks = (work + kThreads - 1) / kThreads;
  if (blocks > 0x7fffffffLL) return AMOE_EUNSUPPORTED;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == AMOE_F32) {
    auto kf = &head_reduce_kernel<float>;
    hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, static_cast<const float*>(z),
                       static_cast<const float*>(gate), static_cast<float*>(y), (long long)T, (int)k, (int)D, vec,
                       counter, counter_add);
  } else if (dtype == AMOE_BF16) {
    auto kf = &head_reduce_kernel<uint16_t>;
    hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, static_cast<const uint16_t*>(z),
                       static_cast<const uint16_t*>(gate), static_cast<uint16_t*>(y), (long long)T, (int)k, (int)D,
                       vec, counter, counter_add);
  } else {
    auto kf = &head_reduce_kernel<f16_t>;
    hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, static_cast<const f16_t*>(z),
                       static_cast<const f16_t*>(gate), static_cast<f16_t*>(y), (long long)T, (int)k, (int)D,
                       vec, counter, counter_add);
  }
  return launch_rc();
}

// the counter still moves when a call has no rows to reduce
__global__ void bump_kernel(long long* counter, long long add) { bump_counter(counter, add); }
static int bump_only(int64_t* counter, int64_t counter_add, void* stream) {
  if (!counter) return AMOE_OK;
  hipLaunchKernelGGL(bump_kernel, dim3(1), dim3(64), 0, static_cast<hipStream_t>(stream),
                     reinterpret_cast<long long*>(counter), (long long)counter_add);
  return launch_rc();
}

int amoe_gate_reduce(int32_t dtype, const void* z, const void* gate, void* y, int64_t T, int32_t k, int32_t D,
                     int64_t* counter, int64_t counter_add, void* stream) {
  if (T > 0 && !gate) return AMOE_ENULL;
  return head_reduce(dtype, z, gate, y, T, k, D, stream, counter, counter_add);
}

int amoe_ksum(int32_t dtype, const void* full, void* out, int64_t T, int32_t k, int32_t D, void* stream) {
  return head_reduce(dtype, full, nullptr, out, T, k, D, stream);
}

constexpr int kHeadClipBlocks = 1024;      // workgroups of the head sum with the clip: four per CU, all resident

size_t amoe_ksum_clip_workspace(int64_t T, int32_t k, int32_t n_tiles) {
  if (T < 0 || k < 1 || n_tiles < 1) return 0;
  return (size_t)n_tiles * (size_t)(T > 0 ? T * k : 1) * sizeof(float) + (size_t)kHeadClipBlocks * sizeof(int32_t);
}

int amoe_ksum_clip(const amoe_ksum_clip_args* a, void* stream) {
  if (!a) return AMOE_ENULL;
  if (a->dtype != AMOE_F32 && a->dtype != AMOE_BF16 && a->dtype != AMOE_F16) return AMOE_EINVAL;
  if (a->T < 0 || a->k < 1 || a->D < 1 || a->E < 1 || a->E > kSelMaxExperts) return AMOE_EINVAL;
  if (int rc = check_bounds(a->n_tiles, a->tile_bounds, a->D)) return rc;
  const long long M = (long long)a->T * a->k;
  if (M > 0x7fffffffLL) return AMOE_EUNSUPPORTED;
  if (a->T == 0) return AMOE_OK;
  if (!a->full || !a->x || !a->sel || !a->perm || !a->offsets || !a->ir || !a->grad_x || !a->ir_grad || !a->workspace)
    return AMOE_ENULL;
  if (a->ldx < a->D) return AMOE_ESHAPE;
  const int CH = a->dtype == AMOE_F32 ? 4 : 8;
  if (!aligned(a->full, 16) || !aligned(a->x, 16) || !aligned(a->grad_x, 16) || !aligned(a->sel, a->sel_is_i64 ? 8 : 4) ||
      !aligned(a->perm, 4) || !aligned(a->offsets, 4) || !aligned(a->ir, 4) || !aligned(a->ir_grad, 4) ||
      !aligned(a->workspace, 4))
    return AMOE_EALIGN;
  if (a->k > 8 || a->D % CH || a->ldx % CH || !bounds_multiple_of(a->n_tiles, a->tile_bounds, CH)) return AMOE_EUNSUPPORTED;
  if (a->workspace_bytes < amoe_ksum_clip_workspace(a->T, a->k, a->n_tiles)) return AMOE_EWORKSPACE;
  HeadClipParams p{};
  p.full = a->full; p.x = a->x; p.ldx = a->ldx; p.out = a->grad_x;
  p.sel = a->sel; p.sel_is_i64 = a->sel_is_i64;
  p.ir = a->ir; p.n_tiles = a->n_tiles;
  for (int t = 0; t <= a->n_tiles; t++) p.bounds[t] = a->tile_bounds[t];
  p.row_part = static_cast<float*>(a->workspace);
  p.count = reinterpret_cast<int32_t*>(p.row_part + (size_t)a->n_tiles * M);
  p.tokens = a->T; p.k = a->k; p.D = a->D;
  const long long want = (a->T + 3) / 4;
  const int blocks = (int)(want < kHeadClipBlocks ? want : kHeadClipBlocks);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (a->dtype == AMOE_F32) hipLaunchKernelGGL((&head_sum_clip_kernel<float>), dim3(blocks), dim3(kThreads), 0, st, p);
  else if (a->dtype == AMOE_BF16) hipLaunchKernelGGL((&head_sum_clip_kernel<uint16_t>), dim3(blocks), dim3(kThreads), 0, st, p);
  else hipLaunchKernelGGL((&head_sum_clip_kernel<f16_t>), dim3(blocks), dim3(kThreads), 0, st, p);
  if (int rc = launch_rc()) return rc;
  IrFinalizeParams f{};
  f.M = (int)M; f.n_tiles = a->n_tiles; f.KD_total = a->D; f.block_cols = a->D;     // one partial sum per K-tile
  for (int t = 0; t <= a->n_tiles; t++) f.col_bounds[t] = a->tile_bounds[t];
  f.irg_partial = p.row_part; f.notclip_count = p.count; f.n_blocks = blocks; f.row_index = a->perm;
  f.ir = a->ir; f.ir_by_expert = 1; f.offsets = a->offsets; f.E = a->E; f.ir_grad = a->ir_grad;
  f.relative = a->gradient_relative; f.scale = a->gradient_scale; f.decay = a->decay;
  f.min_pct = a->input_min_percentage;
  hipLaunchKernelGGL(ir_grad_finalize_kernel, dim3((unsigned)((M + kThreads - 1) / kThreads)), dim3(kThreads), 0, st, f);
  return launch_rc();
}

int amoe_gate_grad(int32_t dtype, const void* z, const void* dy, void* grad_gate, int64_t T, int32_t k, int32_t D,
                   void* stream) {
  if (dtype != AMOE_F32 && dtype != AMOE_BF16 && dtype != AMOE_F16) return AMOE_EINVAL;
  if (T < 0 || k < 1 || D < 1) return AMOE_EINVAL;
  if (T == 0) return AMOE_OK;
  if (!z || !dy || !grad_gate) return AMOE_ENULL;
  const size_t es = esize(dtype);
  if (!aligned(z, es) || !aligned(dy, es) || !aligned(grad_gate, es)) return AMOE_EALIGN;
  const long long blocks = ((long long)T + 3) / 4;            // one wave per token
  if (blocks > 0x7fffffffLL) return AMOE_EUNSUPPORTED;
  const int vec = aligned(z, 16) && aligned(dy, 16) && (D % (dtype == AMOE_F32 ? 4 : 8) == 0);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == AMOE_F32) {
    auto kf = &gate_grad_kernel<float>;
    hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, static_cast<const float*>(z),
                       static_cast<const float*>(dy), static_cast<float*>(grad_gate), (long long)T, (int)k, (int)D, vec);
  } else if (dtype == AMOE_BF16) {
    auto kf = &gate_grad_kernel<uint16_t>;
    hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, static_cast<const uint16_t*>(z),
                       static_cast<const uint16_t*>(dy), static_cast<uint16_t*>(grad_gate), (long long)T, (int)k, (int)D, vec);
  } else {
    auto kf = &gate_grad_kernel<f16_t>;
    hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, static_cast<const f16_t*>(z),
                       static_cast<const f16_t*>(dy), static_cast<f16_t*>(grad_gate), (long long)T, (int)k, (int)D, vec);
  }
  return launch_rc();
}

static int codes_args_ok(int32_t dtype, const uint8_t* codes, const float* scale, const void* sel, int32_t sel_is_i64,
                         const void* a, const void* b, int64_t T, int32_t k, int32_t D) {
  if (dtype != AMOE_F32 && dtype != AMOE_BF16 && dtype != AMOE_F16) return AMOE_EINVAL;
  if (T < 0 || k < 1 || D < 1) return AMOE_EINVAL;
  if (D % 16) return AMOE_EUNSUPPORTED;
  if (T == 0) return AMOE_OK;
  if (!codes || !scale || !sel || !a || !b) return AMOE_ENULL;
  if (!aligned(codes, 16) || !aligned(scale, 4) || !aligned(sel, sel_is_i64 ? 8 : 4) || !aligned(a, esize(dtype)) ||
      !aligned(b, 16))
    return AMOE_EALIGN;
  return AMOE_OK;
}

int amoe_gate_reduce_codes(int32_t dtype, const uint8_t* codes, const float* scale, const void* sel, int32_t sel_is_i64,
                           const void* gate, void* y, int64_t T, int32_t k, int32_t D, int64_t* counter_,
                           int64_t counter_add_, void* stream) {
  if (int rc = codes_args_ok(dtype, codes, scale, sel, sel_is_i64, gate, y, T, k, D)) return rc;
  if (!aligned(counter_, 8)) return AMOE_EALIGN;
  if (T == 0) return bump_only(counter_, counter_add_, stream);
  long long* counter = reinterpret_cast<long long*>(counter_);
  const long long counter_add = counter_add_;
  const long long blocks = ((long long)T * (D / 16) + kThreads - 1) / kThreads;
  if (blocks > 0x7fffffffLL) return AMOE_EUNSUPPORTED;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == AMOE_F32) {
    auto kf = &head_reduce_codes_kernel<float>;
    hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, codes, scale, sel, (int)sel_is_i64,
                       static_cast<const float*>(gate), static_cast<float*>(y), (long long)T, (int)k, (int)D,
                       counter, counter_add);
  } else if (dtype == AMOE_BF16) {
    auto kf = &head_reduce_codes_kernel<uint16_t>;
    hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, codes, scale, sel, (int)sel_is_i64,
                       static_cast<const uint16_t*>(gate), static_cast<uint16_t*>(y), (long long)T, (int)k, (int)D,
                       counter, counter_add);
  } else {
    auto kf = &head_reduce_codes_kernel<f16_t>;
    hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, codes, scale, sel, (int)sel_is_i64,
                       static_cast<const f16_t*>(gate), static_cast<f16_t*>(y), (long long)T, (int)k, (int)D,
                       counter, counter_add);
  }
  return launch_rc();
}

int amoe_gate_grad_codes(int32_t dtype, const uint8_t* codes, const float* scale, const void* sel, int32_t sel_is_i64,
                         const void* dy, void* grad_gate, int64_t T, int32_t k, int32_t D, void* stream) {
  if (int rc = codes_args_ok(dtype, codes, scale, sel, sel_is_i64, grad_gate, dy, T, k, D)) return rc;
  if (T == 0) return AMOE_OK;
  const long long blocks = ((long long)T + 4 * kCodeTokens - 1) / (4 * kCodeTokens);
  if (blocks > 0x7fffffffLL) return AMOE_EUNSUPPORTED;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == AMOE_F32) {
    auto kf = &gate_grad_codes_kernel<float>;
    hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, codes, scale, sel, (int)sel_is_i64,
                       static_cast<const float*>(dy), static_cast<float*>(grad_gate), (long long)T, (int)k, (int)D);
  } else if (dtype == AMOE_BF16) {
    auto kf = &gate_grad_codes_kernel<uint16_t>;
    hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, codes, scale, sel, (int)sel_is_i64,
                       static_cast<const uint16_t*>(dy), static_cast<uint16_t*>(grad_gate), (long long)T, (int)k, (int)D);
  } else {
    auto kf = &gate_grad_codes_kernel<f16_t>;
    hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, codes, scale, sel, (int)sel_is_i64,
                       static_cast<const f16_t*>(dy), static_cast<f16_t*>(grad_gate), (long long)T, (int)k, (int)D);
  }
  return launch_rc();
}

int amoe_row_abs_max(int32_t dtype, const void* x, int64_t ldx, int64_t rows, int32_t K, float* abs_max,
                     void* stream) {
  if (dtype != AMOE_F32 && dtype != AMOE_BF16 && dtype != AMOE_F16) return AMOE_EINVAL;
  if (rows < 0 || K < 1 || ldx < K) return AMOE_EINVAL;
  if (rows == 0) return AMOE_OK;
  if (!x || !abs_max) return AMOE_ENULL;
  if (!aligned(x, esize(dtype)) || !aligned(abs_max, 4)) return AMOE_EALIGN;
  const long long blocks = (rows + 3) / 4;
  if (blocks > 0x7fffffffLL) return AMOE_EUNSUPPORTED;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == AMOE_F32) {
    auto kf = &row_abs_max_kernel<float>;
    hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, static_cast<const float*>(x),
                       (long long)ldx, (long long)rows, (int)K, abs_max);
  } else if (dtype == AMOE_BF16) {
    auto kf = &row_abs_max_kernel<uint16_t>;
    hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, static_cast<const uint16_t*>(x),
                       (long long)ldx, (long long)rows, (int)K, abs_max);
  } else {
    auto kf = &row_abs_max_kernel<f16_t>;
    hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, static_cast<const f16_t*>(x),
                       (long long)ldx, (long long)rows, (int)K, abs_max);
  }
  return launch_rc();
}

// Work split of the per-channel reductions over w [E, K, N]: lanes per row (a power of two covering the row's
// 16-byte chunks, at most 64) and K slices (at least eight loads per lane, about four workgroups per CU overall).
struct ColSplit { int width, slices, col_blocks; };
static ColSplit col_split(int dtype, int E, int K, int N) {
  const int CH = 16 / (int)esize(dtype);
  const int chunks = (N + CH - 1) / CH;
  ColSplit c;
  c.width = 64;
  while (c.width / 2 >= chunks) c.width /= 2;
  const int rows_per_block = 4 * (64 / c.width);
  const int most = (K + 8 * rows_per_block - 1) / (8 * rows_per_block);
  const int want = (1024 + E - 1) / E;
  c.slices = most < 1 ? 1 : (most > want ? want : most);
  c.col_blocks = (chunks + 63) / 64;
  return c;
}

int amoe_weight_abs_max_pair(int32_t dtype, const void* w_a, int32_t K_a, int32_t N_a, float* wmax_a,
                             const void* w_b, int32_t K_b, int32_t N_b, float* wmax_b, int32_t E, void* stream) {
  return amoe_layer_tables(dtype, w_a, K_a, N_a, wmax_a, w_b, K_b, N_b, wmax_b, E, AMOE_F32, nullptr, 0, 0, nullptr, 0,
                           nullptr, stream);
}

int amoe_layer_tables(int32_t dtype, const void* w_a, int32_t K_a, int32_t N_a, float* wmax_a, const void* w_b,
                      int32_t K_b, int32_t N_b, float* wmax_b, int32_t E, int32_t ir_dtype, const void* input_range,
                      int32_t ir_cols, int32_t n_up, float* ir_up, int32_t n_dn, float* ir_dn, void* stream) {
  if (dtype != AMOE_F32 && dtype != AMOE_BF16 && dtype != AMOE_F16) return AMOE_EINVAL;
  if (E < 1 || K_a < 1 || N_a < 1 || K_b < 1 || N_b < 1) return AMOE_EINVAL;
  if (!w_a || !w_b || !wmax_a || !wmax_b) return AMOE_ENULL;
  if (!aligned(w_a, esize(dtype)) || !aligned(w_b, esize(dtype)) || !aligned(wmax_a, 4) || !aligned(wmax_b, 4))
    return AMOE_EALIGN;
  if (input_range != nullptr) {
    if (ir_dtype != AMOE_F32 && ir_dtype != AMOE_BF16 && ir_dtype != AMOE_F16) return AMOE_EINVAL;
    if (n_up < 1 || n_dn < 1 || n_up > ir_cols || n_dn > ir_cols || ir_cols > AMOE_MAX_TILES) return AMOE_EINVAL;
    if (!ir_up || !ir_dn) return AMOE_ENULL;
    if (!aligned(input_range, esize(ir_dtype)) || !aligned(ir_up, 4) || !aligned(ir_dn, 4)) return AMOE_EALIGN;
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  const long long per_a = (long long)K_a * N_a, per_b = (long long)K_b * N_b;
  const long long per = per_a > per_b ? per_a : per_b;
  int chunks = (int)((per + 32 * kThreads - 1) / (32 * kThreads));
  chunks = chunks < 1 ? 1 : (chunks > 64 ? 64 : chunks);
  const int vec_a = aligned(w_a, 16) && (per_a % 16 == 0), vec_b = aligned(w_b, 16) && (per_b % 16 == 0);
  {
    // one small launch: the zero fill the reduction's atomic maxima start from, and the input-range tables
    const int most = input_range ? E * (n_up > n_dn ? n_up : n_dn) : E;
    const dim3 pg((most + kThreads - 1) / kThreads);
    uint32_t* za = reinterpret_cast<uint32_t*>(wmax_a);
    uint32_t* zb = reinterpret_cast<uint32_t*>(wmax_b);
    if (ir_dtype == AMOE_F32 || input_range == nullptr)
      hipLaunchKernelGGL((&layer_tables_prep_kernel<float>), pg, dim3(kThreads), 0, st, za, zb, (int)E,
                         static_cast<const float*>(input_range), (int)ir_cols, (int)n_up, ir_up, (int)n_dn, ir_dn);
    else if (ir_dtype == AMOE_BF16)
      hipLaunchKernelGGL((&layer_tables_prep_kernel<uint16_t>), pg, dim3(kThreads), 0, st, za, zb, (int)E,
                         static_cast<const uint16_t*>(input_range), (int)ir_cols, (int)n_up, ir_up, (int)n_dn, ir_dn);
    else
      hipLaunchKernelGGL((&layer_tables_prep_kernel<f16_t>), pg, dim3(kThreads), 0, st, za, zb, (int)E,
                         static_cast<const f16_t*>(input_range), (int)ir_cols, (int)n_up, ir_up, (int)n_dn, ir_dn);
  }
  if (int rc = launch_rc()) return rc;
  const dim3 grid(chunks, E, 2);
  if (dtype == AMOE_F32) {
    auto kf = &weight_abs_max_kernel<float>;
    hipLaunchKernelGGL(kf, grid, dim3(kThreads), 0, st, static_cast<const float*>(w_a), per_a, wmax_a, vec_a,
                       static_cast<const float*>(w_b), per_b, wmax_b, vec_b);
  } else if (dtype == AMOE_BF16) {
    auto kf = &weight_abs_max_kernel<uint16_t>;
    hipLaunchKernelGGL(kf, grid, dim3(kThreads), 0, st, static_cast<const uint16_t*>(w_a), per_a, wmax_a, vec_a,
                       static_cast<const uint16_t*>(w_b), per_b, wmax_b, vec_b);
  } else {
    auto kf = &weight_abs_max_kernel<f16_t>;
    hipLaunchKernelGGL(kf, grid, dim3(kThreads), 0, st, static_cast<const f16_t*>(w_a), per_a, wmax_a, vec_a,
                       static_cast<const f16_t*>(w_b), per_b, wmax_b, vec_b);
  }
  return launch_rc();
}

int amoe_weight_abs_max(int32_t dtype, const void* w, int32_t E, int32_t K, int32_t N, int32_t cols, float* wmax,
                        void* stream) {
  if (dtype != AMOE_F32 && dtype != AMOE_BF16 && dtype != AMOE_F16) return AMOE_EINVAL;
  if (E < 1 || K < 1 || N < 1 || (cols != 1 && cols != N)) return AMOE_EINVAL;
  if (!w || !wmax) return AMOE_ENULL;
  if (!aligned(w, esize(dtype)) || !aligned(wmax, 4)) return AMOE_EALIGN;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (cols == 1 || N == 1) {
    const long long per = (long long)K * N;
    int chunks = (int)((per + 32 * kThreads - 1) / (32 * kThreads));
    chunks = chunks < 1 ? 1 : (chunks > 64 ? 64 : chunks);
    const int vec = aligned(w, 16) && (per % 16 == 0);
    hipLaunchKernelGGL(fill_zero_kernel, dim3((E + kThreads - 1) / kThreads), dim3(kThreads), 0, st,
                       reinterpret_cast<uint32_t*>(wmax), (int)E);
    if (int rc = launch_rc()) return rc;
    if (dtype == AMOE_F32) {
      auto kf = &weight_abs_max_kernel<float>;
      hipLaunchKernelGGL(kf, dim3(chunks, E), dim3(kThreads), 0, st, static_cast<const float*>(w), per, wmax, vec,
                         static_cast<const float*>(nullptr), 0LL, static_cast<float*>(nullptr), 0);
    } else if (dtype == AMOE_BF16) {
      auto kf = &weight_abs_max_kernel<uint16_t>;
      hipLaunchKernelGGL(kf, dim3(chunks, E), dim3(kThreads), 0, st, static_cast<const uint16_t*>(w), per, wmax, vec,
                         static_cast<const uint16_t*>(nullptr), 0LL, static_cast<float*>(nullptr), 0);
    } else {
      auto kf = &weight_abs_max_kernel<f16_t>;
      hipLaunchKernelGGL(kf, dim3(chunks, E), dim3(kThreads), 0, st, static_cast<const f16_t*>(w), per, wmax, vec,
                         static_cast<const f16_t*>(nullptr), 0LL, static_cast<float*>(nullptr), 0);
    }
  } else if (dtype == AMOE_BF16) {
    if ((long long)E * N > 0x7fffffffLL) return AMOE_EUNSUPPORTED;
    hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)(((long long)E * N + kThreads - 1) / kThreads)), dim3(kThreads), 0,
                       st, reinterpret_cast<uint32_t*>(wmax), (int)(E * N));
    if (int rc = launch_rc()) return rc;
    const ColSplit cs = col_split(dtype, E, K, N);
    const int width = cs.width;
    const int vec = aligned(w, 16) && (N % (16 / (int)esize(dtype)) == 0);
    dim3 grid(cs.col_blocks, cs.slices, E);
    if (dtype == AMOE_F32) {
      auto kf = &weight_col_abs_max_kernel<float>;
      hipLaunchKernelGGL(kf, grid, dim3(kThreads), 0, st, static_cast<const float*>(w), (int)K, (int)N, width, wmax, vec);
    } else {
      auto kf = &weight_col_abs_max_kernel<uint16_t>;
      hipLaunchKernelGGL(kf, grid, dim3(kThreads), 0, st, static_cast<const uint16_t*>(w), (int)K, (int)N, width, wmax,
                         vec);
    }
  } else {
    if ((long long)E * N > 0x7fffffffLL) return AMOE_EUNSUPPORTED;
    hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)(((long long)E * N + kThreads - 1) / kThreads)), dim3(kThreads), 0,
                       st, reinterpret_cast<uint32_t*>(wmax), (int)(E * N));
    if (int rc = launch_rc()) return rc;
    const ColSplit cs = col_split(dtype, E, K, N);
    const int width = cs.width;
    const int vec = aligned(w, 16) && (N % (16 / (int)esize(dtype)) == 0);
    dim3 grid(cs.col_blocks, cs.slices, E);
    if (dtype == AMOE_F32) {
      auto kf = &weight_col_abs_max_kernel<float>;
      hipLaunchKernelGGL(kf, grid, dim3(kThreads), 0, st, static_cast<const float*>(w), (int)K, (int)N, width, wmax, vec);
    } else {
      auto kf = &weight_col_abs_max_kernel<f16_t>;
      hipLaunchKernelGGL(kf, grid, dim3(kThreads), 0, st, static_cast<const f16_t*>(w), (int)K, (int)N, width, wmax,
                         vec);
    }
  }
  return launch_rc();
}

int amoe_segment_sum(const float* v, const int32_t* offsets, int32_t E, int32_t n_tiles, int32_t out_dtype, void* out,
                     int64_t ldout, int32_t zero_cols, void* stream) {
  if (out_dtype != AMOE_F32 && out_dtype != AMOE_BF16 && out_dtype != AMOE_F16) return AMOE_EINVAL;
  if (E < 1 || n_tiles < 1 || n_tiles > AMOE_MAX_TILES || zero_cols < 0 || zero_cols > AMOE_MAX_TILES ||
      ldout < n_tiles + zero_cols)
    return AMOE_EINVAL;
  if (!v || !offsets || !out) return AMOE_ENULL;
  if (!aligned(v, 4) || !aligned(offsets, 4) || !aligned(out, esize(out_dtype))) return AMOE_EALIGN;
  const dim3 grid(E, n_tiles + zero_cols), block(seg_threads((long long)E * (n_tiles + zero_cols)));
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (out_dtype == AMOE_F32) {
    auto kf = &segment_sum_kernel<float>;
    hipLaunchKernelGGL(kf, grid, block, 0, st, v, offsets, (int)n_tiles, static_cast<float*>(out),
                       (long long)ldout);
  } else if (out_dtype == AMOE_BF16) {
    auto kf = &segment_sum_kernel<uint16_t>;
    hipLaunchKernelGGL(kf, grid, block, 0, st, v, offsets, (int)n_tiles, static_cast<uint16_t*>(out),
                       (long long)ldout);
  } else {
    auto kf = &segment_sum_kernel<f16_t>;
    hipLaunchKernelGGL(kf, grid, block, 0, st, v, offsets, (int)n_tiles, static_cast<f16_t*>(out),
                       (long long)ldout);
  }
  return launch_rc();
}

int amoe_expert_std(int32_t dtype, const void* x, int64_t ldx, int32_t K, const int32_t* in_index,
                    const int32_t* offsets, int32_t E, float* out, void* stream) {
  if (dtype != AMOE_F32 && dtype != AMOE_BF16 && dtype != AMOE_F16) return AMOE_EINVAL;
  if (K < 1 || E < 1 || ldx < K) return AMOE_EINVAL;
  if (!x || !in_index || !offsets || !out) return AMOE_ENULL;
  if (!aligned(x, esize(dtype)) || !aligned(in_index, 4) || !aligned(offsets, 4) || !aligned(out, 4))
    return AMOE_EALIGN;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == AMOE_F32) {
    auto kf = &expert_std_kernel<float>;
    hipLaunchKernelGGL(kf, dim3(E), dim3(kThreads), 0, st, static_cast<const float*>(x), (long long)ldx, (int)K,
                       in_index, offsets, out);
  } else if (dtype == AMOE_BF16) {
    auto kf = &expert_std_kernel<uint16_t>;
    hipLaunchKernelGGL(kf, dim3(E), dim3(kThreads), 0, st, static_cast<const uint16_t*>(x), (long long)ldx, (int)K,
                       in_index, offsets, out);
  } else {
    auto kf = &expert_std_kernel<f16_t>;
    hipLaunchKernelGGL(kf, dim3(E), dim3(kThreads), 0, st, static_cast<const f16_t*>(x), (long long)ldx, (int)K,
                       in_index, offsets, out);
  }
  return launch_rc();
}

int amoe_modify_weight(int32_t dtype, const void* w, int32_t E, int32_t K, int32_t N, const float* wmax,
                       int32_t wmax_cols, float n_states, float std_dev, const float* noise, int32_t round_noise,
                       uint64_t noise_seed, const uint64_t* noise_seed_dev, void* out, void* stream) {
  if (dtype != AMOE_F32 && dtype != AMOE_BF16 && dtype != AMOE_F16) return AMOE_EINVAL;
  if (E < 1 || K < 1 || N < 1 || (wmax_cols != 1 && wmax_cols != N)) return AMOE_EINVAL;
  if (!w || !out || !wmax) return AMOE_ENULL;
  if (!aligned(w, esize(dtype)) || !aligned(out, esize(dtype)) || !aligned(wmax, 4) || !aligned(noise, 4) ||
      !aligned(noise_seed_dev, 8))
    return AMOE_EALIGN;
  const int CH = 16 / esize(dtype);
  const long long rows = (long long)E * K;
  const long long blocks = (rows * ((N + CH - 1) / CH) + kThreads - 1) / kThreads;
  if (blocks > 0x7fffffffLL || rows > 0x7fffffffLL) return AMOE_EUNSUPPORTED;
  ModifyParams p{};
  p.w = w; p.out = out; p.wmax = wmax; p.noise = noise; p.rows = rows; p.K = K; p.N = N; p.wmax_cols = wmax_cols;
  p.inv_states = n_states > 0.f ? 1.0f / n_states : 0.f; p.std_dev = std_dev; p.round_noise = round_noise; p.seed = noise_seed;
  p.seed_dev = noise_seed_dev;
  p.vec = aligned(w, 16) && aligned(out, 16) && (N % CH == 0);
  p.cvec = aligned(wmax, 16) && (N % CH == 0);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == AMOE_F32) {
    auto kf = &modify_weight_kernel<float>;
    hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, p);
  } else if (dtype == AMOE_BF16) {
    auto kf = &modify_weight_kernel<uint16_t>;
    hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, p);
  } else {
    auto kf = &modify_weight_kernel<f16_t>;
    hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, p);
  }
  return launch_rc();
}

static int std_slices(long long per_expert) {
  const long long s = (per_expert + 32 * kThreads - 1) / (32 * kThreads);
  return s < 1 ? 1 : (s > kStdMaxSlices ? kStdMaxSlices : (int)s);
}

size_t amoe_weight_std_workspace(int32_t E, int32_t K, int32_t N, int32_t cols) {
  if (E < 1 || K < 1 || N < 1) return 0;
  if (cols == N && N != 1) return (size_t)E * col_split(AMOE_F32, E, K, N).slices * N * 2 * sizeof(double);
  return (size_t)E * std_slices((long long)K * N) * 2 * sizeof(double);
}

int amoe_weight_std(int32_t dtype, const void* w, int32_t E, int32_t K, int32_t N, int32_t cols, float* std_out,
                    void* workspace, size_t workspace_bytes, void* stream) {
  if (dtype != AMOE_F32 && dtype != AMOE_BF16 && dtype != AMOE_F16) return AMOE_EINVAL;
  if (E < 1 || K < 1 || N < 1 || (cols != 1 && cols != N)) return AMOE_EINVAL;
  if (!w || !std_out) return AMOE_ENULL;
  if (!aligned(w, esize(dtype)) || !aligned(std_out, 4) || !aligned(workspace, 8)) return AMOE_EALIGN;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (!workspace) return AMOE_ENULL;
  if (workspace_bytes < amoe_weight_std_workspace(E, K, N, cols)) return AMOE_EWORKSPACE;
  double* partial = static_cast<double*>(workspace);
  if (cols == N && N != 1) {
    if ((long long)E * N > 0x7fffffffLL) return AMOE_EUNSUPPORTED;
    ColSplit cs = col_split(dtype, E, K, N);
    const int most = col_split(AMOE_F32, E, K, N).slices;        // what the workspace was sized for
    if (cs.slices > most) cs.slices = most;
    const int vec = aligned(w, 16) && (N % (16 / (int)esize(dtype)) == 0);
    dim3 grid(cs.col_blocks, cs.slices, E);
    if (dtype == AMOE_F32) {
      auto kf = &weight_col_moments_kernel<float>;
      hipLaunchKernelGGL(kf, grid, dim3(kThreads), 0, st, static_cast<const float*>(w), (int)K, (int)N, cs.width, partial,
                         vec);
    } else if (dtype == AMOE_BF16) {
      auto kf = &weight_col_moments_kernel<uint16_t>;
      hipLaunchKernelGGL(kf, grid, dim3(kThreads), 0, st, static_cast<const uint16_t*>(w), (int)K, (int)N, cs.width,
                         partial, vec);
    } else {
      auto kf = &weight_col_moments_kernel<f16_t>;
      hipLaunchKernelGGL(kf, grid, dim3(kThreads), 0, st, static_cast<const f16_t*>(w), (int)K, (int)N, cs.width,
                         partial, vec);
    }
    if (int rc = launch_rc()) return rc;
    hipLaunchKernelGGL(weight_col_std_finalize_kernel, dim3((unsigned)(((long long)E * N + kThreads - 1) / kThreads)),
                       dim3(kThreads), 0, st, partial, cs.slices, (int)K, (int)N, (int)E, std_out);
    return launch_rc();
  }
  const long long per = (long long)K * N;
  const int slices = std_slices(per);
  const int vec = aligned(w, 16) && (per % 16 == 0);
  if (dtype == AMOE_F32) {
    auto kf = &weight_moments_kernel<float>;
    hipLaunchKernelGGL(kf, dim3(slices, E), dim3(kThreads), 0, st, static_cast<const float*>(w), per, partial, vec);
  } else if (dtype == AMOE_BF16) {
    auto kf = &weight_moments_kernel<uint16_t>;
    hipLaunchKernelGGL(kf, dim3(slices, E), dim3(kThreads), 0, st, static_cast<const uint16_t*>(w), per, partial, vec);
  } else {
    auto kf = &weight_moments_kernel<f16_t>;
    hipLaunchKernelGGL(kf, dim3(slices, E), dim3(kThreads), 0, st, static_cast<const f16_t*>(w), per, partial, vec);
  }
  if (int rc = launch_rc()) return rc;
  hipLaunchKernelGGL(weight_std_finalize_kernel, dim3((E + kThreads - 1) / kThreads), dim3(kThreads), 0, st, partial,
                     slices, per, (int)E, std_out);
  return launch_rc();
}

int amoe_clamp_weights(int32_t dtype, void* w, int32_t E, int32_t K, int32_t N, const float* bound, int32_t cols,
                       void* stream) {
  if (dtype != AMOE_F32 && dtype != AMOE_BF16 && dtype != AMOE_F16) return AMOE_EINVAL;
  if (E < 1 || K < 1 || N < 1 || (cols != 1 && cols != N)) return AMOE_EINVAL;
  if (!w || !bound) return AMOE_ENULL;
  if (!aligned(w, esize(dtype)) || !aligned(bound, 4)) return AMOE_EALIGN;
  const int CH = 16 / esize(dtype);
  const long long rows = (long long)E * K;
  const long long blocks = (rows * ((N + CH - 1) / CH) + kThreads - 1) / kThreads;
  if (blocks > 0x7fffffffLL) return AMOE_EUNSUPPORTED;
  const int vec = aligned(w, 16) && (N % CH == 0);
  const int cvec = aligned(bound, 16) && (N % CH == 0);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == AMOE_F32) {
    auto kf = &clamp_weights_kernel<float>;
    hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, static_cast<float*>(w), bound, rows, (int)K,
                       (int)N, (int)cols, vec, cvec);
  } else if (dtype == AMOE_BF16) {
    auto kf = &clamp_weights_kernel<uint16_t>;
    hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, static_cast<uint16_t*>(w), bound, rows,
                       (int)K, (int)N, (int)cols, vec, cvec);
  } else {
    auto kf = &clamp_weights_kernel<f16_t>;
    hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, static_cast<f16_t*>(w), bound, rows,
                       (int)K, (int)N, (int)cols, vec, cvec);
  }
  return launch_rc();
}

static long long select_blocks(long long T) {
  const int per_block = 4 * select_rows_per_wave(T);
  return (T + per_block - 1) / per_block;
}

size_t amoe_select_workspace(int64_t T, int32_t E) {
  if (T < 1 || E < 1) return 0;
  const long long blocks = select_blocks(T);
  return (size_t)(blocks + (blocks + kSelSumChunk - 1) / kSelSumChunk) * E * sizeof(float);
}

int amoe_select_fwd(int32_t dtype, const void* logits, int64_t T, int32_t E, int32_t k, void* sel_val, int64_t* sel_idx,
                    float* reg, float* reg_c, void* workspace, size_t workspace_bytes, void* stream) {
  if (dtype != AMOE_F32 && dtype != AMOE_BF16 && dtype != AMOE_F16) return AMOE_EINVAL;
  if (T < 0 || E < 1 || k < 1 || k > E) return AMOE_EINVAL;
  if (E > 64 * kSelPerLane) return AMOE_EUNSUPPORTED;
  if (T == 0) return AMOE_OK;
  if (!logits || !sel_val || !sel_idx) return AMOE_ENULL;
  if ((reg != nullptr) != (reg_c != nullptr)) return AMOE_EINVAL;
  if (!aligned(logits, esize(dtype)) || !aligned(sel_val, esize(dtype)) || !aligned(sel_idx, 8) || !aligned(reg, 4) ||
      !aligned(reg_c, 4) || !aligned(workspace, 4))
    return AMOE_EALIGN;
  const long long blocks = select_blocks(T);
  if (blocks > 0x7fffffffLL) return AMOE_EUNSUPPORTED;
  float* partial = nullptr;
  if (reg != nullptr) {
    if (!workspace) return AMOE_ENULL;
    if (workspace_bytes < amoe_select_workspace(T, E)) return AMOE_EWORKSPACE;
    partial = static_cast<float*>(workspace);
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int rpw = select_rows_per_wave(T);
#define AMOE_SELECT_FWD(PER)                                                                                           \
  do {                                                                                                                 \
    if (dtype == AMOE_F32) {                                                                                           \
      auto kf = &select_fwd_kernel<float, PER>;                                                                        \
      hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, static_cast<const float*>(logits),         \
                         (long long)T, (int)E, (int)k, rpw, static_cast<float*>(sel_val), sel_idx, partial);           \
    } else if (dtype == AMOE_BF16) {                                                                                   \
      auto kf = &select_fwd_kernel<uint16_t, PER>;                                                                     \
      hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, static_cast<const uint16_t*>(logits),      \
                         (long long)T, (int)E, (int)k, rpw, static_cast<uint16_t*>(sel_val), sel_idx, partial);        \
    } else {                                                                                                           \
      auto kf = &select_fwd_kernel<f16_t, PER>;                                                                        \
      hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, static_cast<const f16_t*>(logits),         \
                         (long long)T, (int)E, (int)k, rpw, static_cast<f16_t*>(sel_val), sel_idx, partial);           \
    }                                                                                                                  \
  } while (0)
  if (E <= 64) AMOE_SELECT_FWD(1);
  else if (E <= 128) AMOE_SELECT_FWD(2);
  else if (E <= 256) AMOE_SELECT_FWD(4);
  else AMOE_SELECT_FWD(8);
#undef AMOE_SELECT_FWD
  if (int rc = launch_rc()) return rc;
  if (reg != nullptr) {
    const int groups = (int)((blocks + kSelSumChunk - 1) / kSelSumChunk);
    float* level2 = partial + blocks * E;
    hipLaunchKernelGGL(select_usage_sum_kernel, dim3(groups), dim3(kThreads), 0, st, partial, (int)blocks, (int)E, level2);
    if (int rc = launch_rc()) return rc;
    hipLaunchKernelGGL(select_reg_kernel, dim3(1), dim3(kThreads), 0, st, level2, groups, (int)E, (long long)T, reg,
                       reg_c);
    return launch_rc();
  }
  return AMOE_OK;
}

int amoe_select_bwd(int32_t dtype, const void* logits, int64_t T, int32_t E, int32_t k, const int64_t* sel_idx,
                    const void* grad_val, const float* reg_c, const float* grad_reg, void* grad_logits, void* stream) {
  if (dtype != AMOE_F32 && dtype != AMOE_BF16 && dtype != AMOE_F16) return AMOE_EINVAL;
  if (T < 0 || E < 1 || k < 1 || k > E) return AMOE_EINVAL;
  if (E > 64 * kSelPerLane) return AMOE_EUNSUPPORTED;
  if (T == 0) return AMOE_OK;
  if (!logits || !grad_logits || (grad_val && !sel_idx)) return AMOE_ENULL;
  if ((reg_c != nullptr) != (grad_reg != nullptr)) return AMOE_EINVAL;
  if (!aligned(logits, esize(dtype)) || !aligned(grad_logits, esize(dtype)) || !aligned(grad_val, esize(dtype)) ||
      !aligned(sel_idx, 8) || !aligned(reg_c, 4) || !aligned(grad_reg, 4))
    return AMOE_EALIGN;
  const long long blocks = (T + 3) / 4;
  if (blocks > 0x7fffffffLL) return AMOE_EUNSUPPORTED;
  hipStream_t st = static_cast<hipStream_t>(stream);
#define AMOE_SELECT_BWD(PER)                                                                                           \
  do {                                                                                                                 \
    if (dtype == AMOE_F32) {                                                                                           \
      auto kf = &select_bwd_kernel<float, PER>;                                                                        \
      hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, static_cast<const float*>(logits),         \
                         (long long)T, (int)E, (int)k, sel_idx, static_cast<const float*>(grad_val), reg_c, grad_reg,  \
                         static_cast<float*>(grad_logits));                                                            \
    } else if (dtype == AMOE_BF16) {                                                                                   \
      auto kf = &select_bwd_kernel<uint16_t, PER>;                                                                     \
      hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, static_cast<const uint16_t*>(logits),      \
                         (long long)T, (int)E, (int)k, sel_idx, static_cast<const uint16_t*>(grad_val), reg_c,         \
                         grad_reg, static_cast<uint16_t*>(grad_logits));                                               \
    } else {                                                                                                           \
      auto kf = &select_bwd_kernel<f16_t, PER>;                                                                        \
      hipLaunchKernelGGL(kf, dim3((unsigned)blocks), dim3(kThreads), 0, st, static_cast<const f16_t*>(logits),         \
                         (long long)T, (int)E, (int)k, sel_idx, static_cast<const f16_t*>(grad_val), reg_c,            \
                         grad_reg, static_cast<f16_t*>(grad_logits));                                                  \
    }                                                                                                                  \
  } while (0)
  if (E <= 64) AMOE_SELECT_BWD(1);
  else if (E <= 128) AMOE_SELECT_BWD(2);
  else if (E <= 256) AMOE_SELECT_BWD(4);
  else AMOE_SELECT_BWD(8);
#undef AMOE_SELECT_BWD
  return launch_rc();
}

}  // extern "C"

