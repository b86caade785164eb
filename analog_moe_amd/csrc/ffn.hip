// The expert feed-forward of a layer as one call per direction: the single entry points in their order, in the backward
// direction on two streams where the launches are long enough to gain from it.
#include <amoe.h>

#include "host_util.h"
#include "ffn_kernels.h"

using namespace amoe;

namespace {

// Scratch memory of one call, handed out in 256-byte pieces; with base == nullptr it only counts.
struct Arena {
  char* base;
  size_t used = 0;
  void* take(size_t bytes) {
    void* p = base ? base + used : nullptr;
    used += (bytes + 255) / 256 * 256;
    return p;
  }
};

struct FwdScratch { int32_t* sel_sorted; void* sort; void* p1q; float* wmax_up; float* wmax_dn; };
struct BwdScratch { void* gp1; void* p1c; void* full; float* irg_dn; float* irg_up; void* ws_dn; void* ws_up; void* ws_clip; void* ws_w; };

inline int64_t rows_of(const amoe_ffn_args* a) { return a->T * a->k; }
// The up-projection also leaves the DAC image of its result for the down-projection: each row belongs to one expert,
// so the image is made once instead of once per block of output columns.
inline bool has_ranges(const amoe_ffn_args* a) { return a->ir_up != nullptr; }
inline bool chained(const amoe_ffn_args* a) { return has_ranges(a) && a->inp_res > 0 && a->n_dn == 1; }
inline bool generates_noise(const amoe_ffn_args* a) { return a->noise_std > 0 && !a->noise_up; }
inline bool needs_wmax(const amoe_ffn_args* a) { return a->out_bound > 0 || generates_noise(a); }

FwdScratch fwd_scratch(const amoe_ffn_args* a, Arena& m) {
  FwdScratch s{};
  const int64_t M = rows_of(a);
  s.sel_sorted = static_cast<int32_t*>(m.take((size_t)M * 4));
  s.sort = m.take(amoe_prepare_sel_workspace(M, (int32_t)a->E));
  if (chained(a)) s.p1q = m.take((size_t)(M * a->F) * esize((int)a->dtype));
  if (needs_wmax(a) && !a->wmax_up) {
    s.wmax_up = static_cast<float*>(m.take((size_t)(a->E * (a->noise_per_channel ? a->F : 1)) * 4));
    s.wmax_dn = static_cast<float*>(m.take((size_t)(a->E * (a->noise_per_channel ? a->V : 1)) * 4));
  }
  return s;
}

// The up-projection's clip is applied by the sum over the heads where that kernel takes the case.
inline bool clips_in_head_sum(const amoe_ffn_args* a) {
  const int ch = a->dtype == AMOE_F32 ? 4 : 8;
  return has_ranges(a) && a->k > 1 && a->k <= 8 && a->ldx % ch == 0 && aligned(a->x, 16) &&
         bounds_multiple_of((int)a->n_up, a->bounds_up, ch);
}

void fill_bwd_w(amoe_bwd_w_args& w, const amoe_ffn_args* a, bool up) {
  w.dtype = (int32_t)a->dtype;
  w.M = (int32_t)rows_of(a); w.E = (int32_t)a->E;
  w.K = (int32_t)(up ? a->D : a->F); w.N = (int32_t)(up ? a->F : a->V);
  w.n_tiles = 1; w.tile_bounds[0] = 0; w.tile_bounds[1] = w.K;
  if (up) {
    w.n_tiles = (int32_t)a->n_up;
    for (int t = 0; t <= a->n_up; t++) w.tile_bounds[t] = a->bounds_up[t];
  }
}

BwdScratch bwd_scratch(const amoe_ffn_args* a, Arena& m) {
  BwdScratch s{};
  const int64_t M = rows_of(a);
  const size_t es = esize((int)a->dtype);
  s.gp1 = m.take((size_t)(M * a->F) * es);
  s.p1c = m.take((size_t)(M * a->F) * es);
  if (a->k > 1) s.full = m.take((size_t)(M * a->D) * es);
  if (has_ranges(a)) {
    s.irg_dn = static_cast<float*>(m.take((size_t)(M * a->n_dn) * 4));
    s.irg_up = static_cast<float*>(m.take((size_t)(M * a->n_up) * 4));
    s.ws_dn = m.take(amoe_bwd_x_workspace(M, (int32_t)a->F, (int32_t)a->n_dn));
    if (clips_in_head_sum(a)) s.ws_clip = m.take(amoe_ksum_clip_workspace(a->T, (int32_t)a->k, (int32_t)a->n_up));
    else s.ws_up = m.take(amoe_bwd_x_workspace(M, (int32_t)a->D, (int32_t)a->n_up));
  }
  amoe_bwd_w_args w{};                              // (the two weight gradients follow each other on one stream)
  fill_bwd_w(w, a, false);
  size_t ws = amoe_bwd_w_workspace(&w);
  fill_bwd_w(w, a, true);
  const size_t ws_up = amoe_bwd_w_workspace(&w);
  s.ws_w = m.take(ws > ws_up ? ws : ws_up);
  return s;
}

// A fork and a join cost 10 to 20 us of the GPU's time.  The forward call has nothing long enough to hide behind the other
// branch: its tables beside the sort lost at every size (us per call, one stream and two: one token of 64 experts, 16 MB of
// weights 33 / 55, 64 MB 50 / 72; 1000 tokens 100 / 118; 16384 tokens 294 / 304; 32768 tokens, 512 MB 1054 / 1065).  In the
// backward call the companions stream the k-head tensors beside the weight gradients, whose last tiles leave CUs idle where
// the loads are uneven.  us per call, one stream and two, by the bytes of those tensors (z: load of the
// experts by Zipf(1.2), otherwise even):
//   16 experts, bf16: 8 MB 76 / 81, 16 MB 99 / 99, z 24 MB 103 / 101, 32 MB 105 / 111, 40 MB 115 / 118, z 125 / 120, 128 MB
//   238 / 228, z 256 / 233; fp32: 40 MB 179 / 178, 64 MB 228 / 222, 96 MB 252 / 243, z 292 / 279; 412 features: 19 MB 146 / 150,
//   31 MB 179 / 174, fp32 63 MB 260 / 250
//   64 experts, bf16: 16 MB 117 / 132, z 48 MB 184 / 178, 128 MB 203 / 207, z 285 / 273, 512 MB 529 / 535, z 748 / 692
// The line lies where uneven loads begin to gain; even loads lose up to 6 % beyond it, and gain 2 to 5 % where experts are few.
constexpr long long kOverlapBytes = 24LL << 20;
inline bool overlap_companions(const amoe_ffn_args* a) {
  return rows_of(a) * (a->D + a->V) * (long long)esize((int)a->dtype) >= kOverlapBytes;
}

// `to` continues after what `from` has been given so far
int order_after(hipStream_t to, hipStream_t from, hipEvent_t e) {
  hipError_t rc = hipEventRecord(e, from);
  if (rc == hipSuccess) rc = hipStreamWaitEvent(to, e, 0);
  return (int)rc;
}

// Launches on the second stream beside those on the first.  However the call ends, the first stream continues after both:
// what a launch uses belongs to the caller again once the call has returned.  Both events are there before anything is
// launched on the second stream, so that joining it needs nothing that could still be refused.
struct Fork {
  hipStream_t main, side;
  hipEvent_t start = nullptr, done = nullptr;
  bool open = false;
  Fork(hipStream_t main_, void* side_stream, bool wanted)
      : main(main_), side(wanted && side_stream ? static_cast<hipStream_t>(side_stream) : main_) {}
  int begin() {
    if (side == main) return AMOE_OK;
    hipError_t rc = hipEventCreateWithFlags(&start, hipEventDisableTiming);
    if (rc == hipSuccess) rc = hipEventCreateWithFlags(&done, hipEventDisableTiming);
    if (rc != hipSuccess) return (int)rc;
    const int ordered = order_after(side, main, start);
    open = ordered == AMOE_OK;
    return ordered;
  }
  int join() {
    if (!open) return AMOE_OK;
    open = false;
    return order_after(main, side, done);
  }
  ~Fork() {
    (void)join();
    if (start) (void)hipEventDestroy(start);         // (released once the streams have passed them)
    if (done) (void)hipEventDestroy(done);
  }
  Fork(const Fork&) = delete;
  Fork& operator=(const Fork&) = delete;
};

const char* const kFwdStages[] = {"prepare_sel", "tables", "fwd_up", "fwd_down", "gate_reduce"};
const char* const kBwdStages[] = {"xgrad_down", "xgrad_up", "gate_grad", "head_sum", "wgrad_down", "wgrad_up", "ir_sums"};

// records the stage's pair of events around what is launched while it lives
struct Stage {
  void* const* ev;
  hipStream_t st;
  Stage(const amoe_ffn_args* a, int i, hipStream_t st_) : ev(a->stage_events ? a->stage_events + 2 * i : nullptr), st(st_) {
    if (ev) (void)hipEventRecord(static_cast<hipEvent_t>(ev[0]), st);
  }
  ~Stage() {
    if (ev) (void)hipEventRecord(static_cast<hipEvent_t>(ev[1]), st);
  }
};

int check_args(const amoe_ffn_args* a) {
  if (!a) return AMOE_ENULL;
  if (a->dtype != AMOE_F32 && a->dtype != AMOE_BF16 && a->dtype != AMOE_F16) return AMOE_EINVAL;
  const int64_t lim = 0x7fffffffLL;
  if (a->T < 0 || a->D < 1 || a->E < 1 || a->F < 1 || a->V < 1 || a->k < 1) return AMOE_EINVAL;
  if (a->D > lim || a->F > lim || a->V > lim || a->k > lim || a->E > kSelMaxExperts || rows_of(a) > lim) return AMOE_EUNSUPPORTED;
  if (!a->bounds_up || !a->bounds_dn) return AMOE_ENULL;
  if (int rc = check_bounds((int)a->n_up, a->bounds_up, (int)a->D)) return rc;
  if (int rc = check_bounds((int)a->n_dn, a->bounds_dn, (int)a->F)) return rc;
  if (!a->ir_up != !a->ir_dn) return AMOE_ENULL;
  if (!a->x || !a->keys || !a->values || !a->sel || !a->gate || !a->p1 || !a->z || !a->perm || !a->in_index || !a->offsets)
    return AMOE_ENULL;
  if (a->z_is_codes && !a->z_scale) return AMOE_ENULL;
  return AMOE_OK;
}

int tables(const amoe_ffn_args* a, const FwdScratch& s, hipStream_t st) {
  const int32_t dt = (int32_t)a->dtype, E = (int32_t)a->E, D = (int32_t)a->D, F = (int32_t)a->F, V = (int32_t)a->V;
  if (s.wmax_up && !a->noise_per_channel)            // both max |W| tables and both range tables
    return amoe_layer_tables(dt, a->keys, D, F, s.wmax_up, a->values, F, V, s.wmax_dn, E, (int32_t)a->ir_dtype,
                             has_ranges(a) ? a->input_range : nullptr, (int32_t)a->ir_cols, (int32_t)a->n_up, a->ir_up, (int32_t)a->n_dn, a->ir_dn, st);
  if (has_ranges(a)) {
    if (int rc = launch_ir_tables((int)a->ir_dtype, a->input_range, (int)a->ir_cols, E, (int)a->n_up, a->ir_up, (int)a->n_dn,
                                  a->ir_dn, st))
      return rc;
  }
  if (s.wmax_up) {
    if (int rc = amoe_weight_abs_max(dt, a->keys, E, D, F, F, s.wmax_up, st)) return rc;
    if (int rc = amoe_weight_abs_max(dt, a->values, E, F, V, V, s.wmax_dn, st)) return rc;
  }
  return AMOE_OK;
}

}  // namespace

extern "C" {

size_t amoe_ffn_args_bytes(void) { return sizeof(amoe_ffn_args); }

const char* amoe_ffn_stage_name(int32_t backward, int32_t i) {
  const int n = backward ? (int)(sizeof(kBwdStages) / sizeof(char*)) : (int)(sizeof(kFwdStages) / sizeof(char*));
  return i < 0 || i >= n ? nullptr : backward ? kBwdStages[i] : kFwdStages[i];
}

size_t amoe_ffn_fwd_workspace(const amoe_ffn_args* a) {
  if (check_args(a)) return 0;
  Arena m{nullptr};
  fwd_scratch(a, m);
  return m.used;
}

size_t amoe_ffn_bwd_workspace(const amoe_ffn_args* a) {
  if (check_args(a)) return 0;
  Arena m{nullptr};
  bwd_scratch(a, m);
  return m.used;
}

int amoe_ffn_fwd(const amoe_ffn_args* a, void* workspace, size_t workspace_bytes, void* stream, void* /* side_stream */) {
  if (int rc = check_args(a)) return rc;
  if (!workspace || !a->y || (has_ranges(a) && !a->input_range)) return AMOE_ENULL;
  if (has_ranges(a) && (a->ir_cols < a->n_up || a->ir_cols < a->n_dn)) return AMOE_ESHAPE;
  if (!aligned(workspace, 16)) return AMOE_EALIGN;
  if (workspace_bytes < amoe_ffn_fwd_workspace(a)) return AMOE_EWORKSPACE;
  Arena m{static_cast<char*>(workspace)};
  const FwdScratch s = fwd_scratch(a, m);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t M = rows_of(a);
  const bool ranges = has_ranges(a), gen = generates_noise(a), chain = chained(a);
  if (s.wmax_up || ranges) {
    Stage t(a, 1, st);
    if (int rc = tables(a, s, st)) return rc;
  }
  {
    Stage t(a, 0, st);
    if (int rc = amoe_prepare_sel(a->sel, (int32_t)a->sel_is_i64, M, (int32_t)a->E, (int32_t)a->k, s.sel_sorted, a->perm,
                                  a->in_index, a->offsets, nullptr, s.sort, amoe_prepare_sel_workspace(M, (int32_t)a->E), st))
      return rc;
  }
  const float* wmax_up = a->wmax_up ? a->wmax_up : s.wmax_up;
  const float* wmax_dn = a->wmax_dn ? a->wmax_dn : s.wmax_dn;

  amoe_fwd_args f{};
  f.dtype = (int32_t)a->dtype;
  f.M = (int32_t)M; f.K = (int32_t)a->D; f.N = (int32_t)a->F; f.E = (int32_t)a->E;
  f.n_in_rows = (int32_t)a->T; f.n_out_rows = (int32_t)M;
  f.x = a->x; f.ldx = a->ldx;
  f.w = a->keys; f.w_stride_e = a->keys_se; f.w_stride_k = a->keys_sk; f.w_stride_n = a->keys_sn;
  f.out = a->p1; f.ldo = a->F;
  f.sel_sorted = s.sel_sorted; f.offsets = a->offsets; f.in_index = a->in_index; f.out_index = a->perm;
  f.ir = ranges ? a->ir_up : nullptr; f.ir_by_expert = ranges; f.inp_res = (float)a->inp_res;
  f.n_tiles = (int32_t)a->n_up;
  for (int t = 0; t <= a->n_up; t++) f.tile_bounds[t] = a->bounds_up[t];
  f.noise = a->noise_up; f.noise_tile_stride = M * a->F; f.ldnoise = a->F;
  f.noise_std = gen ? (float)a->noise_std : 0.f; f.noise_seed = (uint64_t)a->noise_seed; f.noise_seed_dev = a->noise_seed_dev;
  f.wmax = wmax_up; f.wmax_cols = a->noise_per_channel ? f.N : 1;
  f.out_bound = (float)a->out_bound; f.out_res = (float)a->out_res;
  f.relu = 1;
  if (chain) { f.xq_out = s.p1q; f.ldxq = a->F; f.xq_ir = a->ir_dn; f.xq_inp_res = (float)a->inp_res; }
  {
    Stage t(a, 2, st);
    if (int rc = amoe_cvmm_fwd(&f, st)) return rc;
  }
  if (a->down_ready)
    if (hipError_t rc = hipStreamWaitEvent(st, static_cast<hipEvent_t>(a->down_ready), 0)) return (int)rc;
  f.K = (int32_t)a->F; f.N = (int32_t)a->V; f.n_in_rows = (int32_t)M;
  f.x = chain ? s.p1q : a->p1; f.ldx = a->F; f.x_is_quantized = chain;
  f.w = a->values; f.w_stride_e = a->values_se; f.w_stride_k = a->values_sk; f.w_stride_n = a->values_sn;
  f.in_index = a->perm; f.out_index = nullptr;
  f.ir = ranges ? a->ir_dn : nullptr;
  f.n_tiles = (int32_t)a->n_dn;
  for (int t = 0; t <= a->n_dn; t++) f.tile_bounds[t] = a->bounds_dn[t];
  f.noise = a->noise_dn; f.noise_tile_stride = M * a->V; f.ldnoise = a->V;
  f.noise_seed = (uint64_t)a->noise_seed + 1;
  f.wmax = wmax_dn; f.wmax_cols = a->noise_per_channel ? f.N : 1;
  f.relu = 0; f.xq_out = nullptr; f.xq_ir = nullptr; f.xq_inp_res = 0.f; f.ldxq = 0;
  // read twice more and never as a matrix operand (gate reduction now, gate gradient in the backward pass): where the
  // kernel can, the down-projection leaves its ADC codes, one byte per value, with two factors per expert
  if (a->z_is_codes) { f.code_out = static_cast<uint8_t*>(a->z); f.ldcode = a->V; f.code_scale_out = a->z_scale; }
  else { f.out = a->z; f.ldo = a->V; }
  if (a->z_is_codes) { f.out = nullptr; f.ldo = a->V; }
  {
    Stage t(a, 3, st);
    if (int rc = amoe_cvmm_fwd(&f, st)) return rc;
  }
  // the gate reduction follows the last launch that draws noise: it moves the device seed word on
  int64_t* counter = a->seed_bump ? reinterpret_cast<int64_t*>(const_cast<uint64_t*>(a->noise_seed_dev)) : nullptr;
  Stage t(a, 4, st);
  if (a->z_is_codes)
    return amoe_gate_reduce_codes(f.dtype, static_cast<const uint8_t*>(a->z), a->z_scale, a->sel, (int32_t)a->sel_is_i64, a->gate,
                                  a->y, a->T, (int32_t)a->k, (int32_t)a->V, counter, a->seed_bump, st);
  return amoe_gate_reduce(f.dtype, a->z, a->gate, a->y, a->T, (int32_t)a->k, (int32_t)a->V, counter, a->seed_bump, st);
}

int amoe_ffn_bwd(const amoe_ffn_args* a, void* workspace, size_t workspace_bytes, void* stream, void* side_stream) {
  if (int rc = check_args(a)) return rc;
  if (!workspace || !a->dy || !a->grad_x || !a->grad_keys || !a->grad_values || !a->grad_gate) return AMOE_ENULL;
  if (!aligned(workspace, 16)) return AMOE_EALIGN;
  if (workspace_bytes < amoe_ffn_bwd_workspace(a)) return AMOE_EWORKSPACE;
  Arena m{static_cast<char*>(workspace)};
  const BwdScratch s = bwd_scratch(a, m);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t M = rows_of(a);
  const int32_t dt = (int32_t)a->dtype, E = (int32_t)a->E, k = (int32_t)a->k, D = (int32_t)a->D, F = (int32_t)a->F, V = (int32_t)a->V;
  const bool ranges = has_ranges(a), late_clip = clips_in_head_sum(a);
  void* full = a->k > 1 ? s.full : a->grad_x;

  // The input gradient reads p1 for its masks anyway; it also leaves gate * clamp(p1), which is the x operand of the
  // weight gradient (otherwise every block of its output columns clips and scales).
  amoe_bwd_x_args b{};
  b.dtype = dt; b.M = (int32_t)M; b.N = V; b.K = F; b.E = E;
  b.g = a->dy; b.ldg = V; b.n_g_rows = (int32_t)a->T;
  b.w = a->values; b.w_stride_e = a->values_se; b.w_stride_k = a->values_sk;
  b.grad_x_full = s.gp1; b.ldo = F;
  b.x = a->p1; b.ldx = F;
  b.offsets = a->offsets; b.g_index = a->in_index; b.out_index = a->perm; b.xf_index = a->perm;
  b.gate = a->gate;
  b.ir = ranges ? a->ir_dn : nullptr; b.ir_by_expert = ranges; b.ir_grad = s.irg_dn;
  b.n_tiles = (int32_t)a->n_dn;
  for (int t = 0; t <= a->n_dn; t++) b.tile_bounds[t] = a->bounds_dn[t];
  b.gradient_relative = (int32_t)a->gradient_relative; b.gradient_scale = (float)a->gradient_scale;
  b.decay = (float)a->decay; b.input_min_percentage = (float)a->input_min_percentage;
  b.relu_mask = 1;
  b.workspace = s.ws_dn; b.workspace_bytes = amoe_bwd_x_workspace(M, F, (int32_t)a->n_dn);
  b.xc_out = s.p1c; b.ldxc = F;
  {
    Stage t(a, 0, st);
    if (int rc = amoe_cvmm_bwd_x(&b, st)) return rc;
  }
  // The clip mask of the up-projection's input gradient depends on the token's input row, which its k heads share:
  // where the sum over the heads can apply it, the GEMM runs without a mask tile.
  b.N = F; b.K = D;
  b.g = s.gp1; b.ldg = F; b.n_g_rows = (int32_t)M;
  b.w = a->keys; b.w_stride_e = a->keys_se; b.w_stride_k = a->keys_sk;
  b.grad_x_full = full; b.ldo = D;
  b.g_index = a->perm; b.gate = nullptr; b.relu_mask = 0; b.xc_out = nullptr; b.ldxc = 0;
  if (late_clip || !ranges) {
    b.x = nullptr; b.xf_index = nullptr; b.ir = nullptr; b.ir_by_expert = 0; b.ir_grad = nullptr; b.workspace = nullptr;
    b.n_tiles = 1; b.tile_bounds[0] = 0; b.tile_bounds[1] = D;
  } else {
    b.x = a->x; b.ldx = a->ldx; b.xf_index = a->in_index;
    b.ir = a->ir_up; b.ir_grad = s.irg_up;
    b.n_tiles = (int32_t)a->n_up;
    for (int t = 0; t <= a->n_up; t++) b.tile_bounds[t] = a->bounds_up[t];
    b.workspace = s.ws_up; b.workspace_bytes = amoe_bwd_x_workspace(M, D, (int32_t)a->n_up);
  }
  {
    Stage t(a, 1, st);
    if (int rc = amoe_cvmm_bwd_x(&b, st)) return rc;
  }
  // The gate gradient and the sum over the k heads only stream z, dy and the per-head input gradient; they run next to
  // the two weight gradients.  With evenly loaded experts the launches take as long side by side as one after the other
  // (together they are bound by memory traffic); with uneven loads the streaming kernels fill the CUs that the weight
  // gradients' last tiles leave idle (2 - 3 % of the step).
  Fork fork(st, side_stream, overlap_companions(a));
  hipStream_t side = fork.side;
  if (int rc = fork.begin()) return rc;
  {
    Stage t(a, 2, side);
    const int rc = a->z_is_codes
        ? amoe_gate_grad_codes(dt, static_cast<const uint8_t*>(a->z), a->z_scale, a->sel, (int32_t)a->sel_is_i64, a->dy, a->grad_gate,
                               a->T, k, V, side)
        : amoe_gate_grad(dt, a->z, a->dy, a->grad_gate, a->T, k, V, side);
    if (rc) return rc;
  }
  {
    Stage t(a, 3, side);
    if (late_clip) {
      amoe_ksum_clip_args c{};
      c.dtype = dt; c.T = a->T; c.k = k; c.D = D; c.E = E;
      c.full = full; c.x = a->x; c.ldx = a->ldx; c.sel = a->sel; c.sel_is_i64 = (int32_t)a->sel_is_i64;
      c.perm = a->perm; c.offsets = a->offsets; c.ir = a->ir_up;
      c.n_tiles = (int32_t)a->n_up;
      for (int t = 0; t <= a->n_up; t++) c.tile_bounds[t] = a->bounds_up[t];
      c.grad_x = a->grad_x; c.ir_grad = s.irg_up;
      c.gradient_relative = b.gradient_relative; c.gradient_scale = b.gradient_scale;
      c.decay = b.decay; c.input_min_percentage = b.input_min_percentage;
      c.workspace = s.ws_clip; c.workspace_bytes = amoe_ksum_clip_workspace(a->T, k, (int32_t)a->n_up);
      if (int rc = amoe_ksum_clip(&c, side)) return rc;
    } else if (a->k > 1) {
      if (int rc = amoe_ksum(dt, full, a->grad_x, a->T, k, D, side)) return rc;
    }
  }
  // The per-expert sums of the input-range gradient are written in the parameter's type, each launch clearing the
  // columns its projection does not have.  The down-projection's go here, where the second stream keeps the GPU busy.
  const int nt = (int)(a->n_up > a->n_dn ? a->n_up : a->n_dn);
  char* gir = static_cast<char*>(a->grad_ir);
  const size_t ires = ranges ? esize((int)a->ir_dtype) : 0;
  if (ranges && gir)
    if (int rc = amoe_segment_sum(s.irg_dn, a->offsets, E, (int32_t)a->n_dn, (int32_t)a->ir_dtype, gir + (size_t)(a->E * nt) * ires, nt,
                                  nt - (int32_t)a->n_dn, st))
      return rc;
  amoe_bwd_w_args w{};
  fill_bwd_w(w, a, false);
  w.x = s.p1c; w.ldx = F; w.g = a->dy; w.ldg = V; w.grad_w = a->grad_values;
  w.offsets = a->offsets; w.in_index = a->perm; w.g_index = a->in_index;
  w.n_x_rows = M; w.n_g_rows = a->T;
  w.workspace_bytes = amoe_bwd_w_workspace(&w); w.workspace = w.workspace_bytes ? s.ws_w : nullptr;
  {
    Stage t(a, 4, st);
    if (int rc = amoe_cvmm_bwd_w(&w, st)) return rc;
  }
  fill_bwd_w(w, a, true);
  w.x = a->x; w.ldx = a->ldx; w.g = s.gp1; w.ldg = F; w.grad_w = a->grad_keys;
  w.in_index = a->in_index; w.g_index = a->perm;
  w.n_x_rows = a->T; w.n_g_rows = M;
  w.ir = ranges ? a->ir_up : nullptr; w.ir_by_expert = ranges;
  w.workspace_bytes = amoe_bwd_w_workspace(&w); w.workspace = w.workspace_bytes ? s.ws_w : nullptr;
  {
    Stage t(a, 5, st);
    if (int rc = amoe_cvmm_bwd_w(&w, st)) return rc;
  }
  if (int rc = fork.join()) return rc;
  if (ranges && gir) {
    Stage t(a, 6, st);
    return amoe_segment_sum(s.irg_up, a->offsets, E, (int32_t)a->n_up, (int32_t)a->ir_dtype, gir, nt, nt - (int32_t)a->n_up, st);
  }
  return AMOE_OK;
}

}  // extern "C"
