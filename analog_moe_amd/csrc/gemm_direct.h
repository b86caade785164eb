// Forward products with few rows per expert or few output columns: the contraction of one small output tile is split
// over the waves of a workgroup, and the operands go from global memory straight to the matrix fragments.
//
// What bounds these launches is latency: a 128-row tiled kernel gives a batch of 48 tokens (6 rows per expert) or a
// router (64 output columns) one workgroup per expert or per 128 rows, which walks the contraction in steps of 32 to 64
// with a barrier each -- 32 to 16 memory round trips in a row on a chip that is three quarters idle.  Here a workgroup
// owns 32 rows x 64 columns; each of its 8 waves takes every eighth step of 128 bytes of every row, so a contraction of
// 1024 16-bit elements is two steps per wave, all loads of which are in flight at once; no LDS and no barrier until the
// 8 partial tiles are added (in wave order: fixed summation order).
//
// Fragments: a lane holds 16 bytes of one token row per group (the layout of the matrix instructions' operands needs no
// transpose when both sides name the contraction indices alike); weights whose contraction is contiguous are read the
// same way; weights whose output column is contiguous are read as column PAIRS, 32 lanes side by side (128-byte rows),
// and one byte permute per two contraction indices makes the fragment of the even and of the odd column.
#pragma once
#include "host_util.h"

namespace amoe {

constexpr int kDirWaves = 8, kDirThreads = 64 * kDirWaves;
constexpr int kDirLd = kDirCols + 4;        // floats per row of a partial tile in LDS (16-byte rows, banks apart)

// A 16-byte load from a 4-byte aligned address (one instruction; the rows of odd models are no more aligned than that).
__device__ __forceinline__ Raw load16_al4(const void* p) {
  typedef u32x4 __attribute__((aligned(4))) RawU;
  return *static_cast<const RawU*>(p);
}

// The contraction elements of one step (128 bytes of a row): 4 groups, each 16 bytes per lane and operand row.
template <typename T> inline constexpr int kDirStep = 128 / (int)sizeof(T);

// What a lane holds of one step: x[i] its token row's piece of group i; w[i] the weights of group i,
//   W_KC                : words 4 * f .. 4 * f + 3 = column 32 * f + lane % 32
//   16-bit, column pairs: word r = contraction index r of the piece, columns 2 * (lane % 32) (low half) and + 1 (high)
//   32-bit, column pairs: words 2 * r, 2 * r + 1
// NF: blocks of 32 columns (2, and with W_KC also 4).
template <int NF = 2>
struct DirectStep {
  Raw x[4];
  uint32_t w[4][4 * NF];
};

template <typename T, bool W_KC, int NF = 2>
struct DirectLoader {
  static_assert(W_KC || NF == 2, "column pairs cover 64 columns");
  const T* xrow;                // this lane's token row
  const T* wcol[NF];            // W_KC: its columns
  BufRsrc w_rsrc;               // otherwise: W[e], addressed with 32-bit byte offsets
  uint32_t w_lane, w_ks;        // byte offset of (contraction index 0, this lane's column pair), bytes per index
  int lh;

  __device__ __forceinline__ void load(DirectStep<NF>& s, int k0, int khi) const {
    constexpr int CH = Elem<T>::kChunk, STEP = kDirStep<T>;
    if (k0 + STEP <= khi) {                                  // (the same for the whole wave)
#pragma unroll
      for (int i = 0; i < 4; i++) s.x[i] = load16_al4(xrow + k0 + (2 * i + lh) * CH);
      if constexpr (W_KC) {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
          for (int f = 0; f < NF; f++) {
            const Raw v = load16_al4(wcol[f] + k0 + (2 * i + lh) * CH);
#pragma unroll
            for (int d = 0; d < 4; d++) s.w[i][4 * f + d] = v[d];
          }
      } else {
        const uint32_t lane = w_lane + (uint32_t)(lh * CH) * w_ks;
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
          for (int r = 0; r < CH; r++) {
            const uint32_t off = (uint32_t)(k0 + 2 * i * CH + r) * w_ks;
            if constexpr (sizeof(T) == 2) {
              s.w[i][r] = buffer_load_b32(w_rsrc, lane, off);
            } else {
              const u32x2 v = buffer_load_b64(w_rsrc, lane, off);
              s.w[i][2 * r] = v[0];
              s.w[i][2 * r + 1] = v[1];
            }
          }
      }
      return;
    }
    // the step that the contraction ends in: both operands read as zero past its end
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int kpos = k0 + (2 * i + lh) * CH;
      int nv = khi - kpos;
      nv = nv < 0 ? 0 : (nv > CH ? CH : nv);
      s.x[i] = raw_load<T>(xrow + kpos, nv, false);
      if constexpr (W_KC) {
#pragma unroll
        for (int f = 0; f < NF; f++) {
          const Raw v = raw_load<T>(wcol[f] + kpos, nv, false);
#pragma unroll
          for (int d = 0; d < 4; d++) s.w[i][4 * f + d] = v[d];
        }
      } else {
#pragma unroll
        for (int r = 0; r < CH; r++) {
          const bool ok = r < nv;
          const uint32_t off = w_lane + (uint32_t)(ok ? kpos + r : 0) * w_ks;
          if constexpr (sizeof(T) == 2) {
            const uint32_t v = buffer_load_b32(w_rsrc, off, 0u);
            s.w[i][r] = ok ? v : 0u;
          } else {
            const u32x2 v = buffer_load_b64(w_rsrc, off, 0u);
            s.w[i][2 * r] = ok ? v[0] : 0u;
            s.w[i][2 * r + 1] = ok ? v[1] : 0u;
          }
        }
      }
    }
  }
};

// The input stage of a row: clip to its range, scale, round; 16-bit types keep the integer codes.
struct DirectDac {
  bool on;
  float r, rinv, kq, res, resinv, margin;
  __device__ __forceinline__ void set_range(float range) {
    r = range;
    rinv = 1.0f / range;
    kq = rinv * resinv;
  }
  template <typename T>
  __device__ __forceinline__ void apply(Raw& x) const {
    constexpr int CH = Elem<T>::kChunk;
    constexpr bool B16 = sizeof(T) == 2;
    float v[CH], c[CH];
    raw_unpack<T>(x, v);
    float tie = 0.f;
#pragma unroll
    for (int j = 0; j < CH; j++) {
      v[j] = clamp_sym(v[j], r);
      c[j] = dac_code<B16>(v[j], r, rinv, res, resinv, kq, tie);
      if (!B16) c[j] *= res;
    }
    if (B16 && tie > margin) {              // rare: a product next to a rounding tie
#pragma unroll
      for (int j = 0; j < CH; j++) c[j] = dac_code_exact(v[j], r, rinv, res, resinv);
    }
    if constexpr (B16) x = raw_pack_codes<T>(c);
    else x = raw_pack<T>(c);
  }
};

// acc[f] += step (f: W_KC columns 32 * f + i, otherwise columns 2 * i + f of the tile, i the instruction's row index)
template <typename T, bool W_KC, int NF = 2>
__device__ __forceinline__ void direct_multiply(f32x16 (&acc)[NF], DirectStep<NF>& s, const DirectDac& dac) {
#pragma unroll
  for (int i = 0; i < 4; i++) {
    if (dac.on) dac.apply<T>(s.x[i]);
    if constexpr (sizeof(T) == 2) {
      u32x4 wf[NF];
#pragma unroll
      for (int d = 0; d < 4; d++) {
        if constexpr (W_KC) {
#pragma unroll
          for (int f = 0; f < NF; f++) wf[f][d] = s.w[i][4 * f + d];
        } else {
          wf[0][d] = pack_low_halves(s.w[i][2 * d + 1], s.w[i][2 * d]);
          wf[1][d] = pack_high_halves(s.w[i][2 * d + 1], s.w[i][2 * d]);
        }
      }
#pragma unroll
      for (int f = 0; f < NF; f++) acc[f] = mfma_32x32x16<T>(wf[f], s.x[i], acc[f]);
    } else if constexpr (W_KC) {
      // A half wave holds four consecutive indices; with the halves' odd and even words exchanged an instruction takes
      // two consecutive ones, in order: the sums come out as the tiled kernel's, bit for bit.
      uint32_t x[4] = {s.x[i][0], s.x[i][1], s.x[i][2], s.x[i][3]};
      swap_half_waves(x[0], x[1]);
      swap_half_waves(x[2], x[3]);
#pragma unroll
      for (int f = 0; f < NF; f++) {
        swap_half_waves(s.w[i][4 * f], s.w[i][4 * f + 1]);
        swap_half_waves(s.w[i][4 * f + 2], s.w[i][4 * f + 3]);
      }
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int d = j == 0 ? 0 : j == 1 ? 2 : j == 2 ? 1 : 3;      // words of indices 2 * j and 2 * j + 1
#pragma unroll
        for (int f = 0; f < NF; f++) acc[f] = mfma_32x32x2_f32(as_f32(s.w[i][4 * f + d]), as_f32(x[d]), acc[f]);
      }
    } else {
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int f = 0; f < NF; f++)
          acc[f] = mfma_32x32x2_f32(as_f32(s.w[i][2 * j + f]), as_f32(s.x[i][j]), acc[f]);
    }
  }
}

// A wave's partial tile -> LDS, [row][column]
template <bool W_KC, int NF = 2>
__device__ __forceinline__ void direct_store_partial(float* __restrict__ tile, const f32x16 (&acc)[NF], int l32, int lh) {
  float* __restrict__ row = tile + l32 * (32 * NF + 4);
#pragma unroll
  for (int q = 0; q < 4; q++) {
    if constexpr (W_KC) {
#pragma unroll
      for (int f = 0; f < NF; f++)
        *reinterpret_cast<f32x4*>(row + 32 * f + 8 * q + 4 * lh) =
            f32x4{acc[f][4 * q], acc[f][4 * q + 1], acc[f][4 * q + 2], acc[f][4 * q + 3]};
    } else {
      *reinterpret_cast<f32x4*>(row + 16 * q + 8 * lh) = f32x4{acc[0][4 * q], acc[1][4 * q], acc[0][4 * q + 1], acc[1][4 * q + 1]};
      *reinterpret_cast<f32x4*>(row + 16 * q + 8 * lh + 4) =
          f32x4{acc[0][4 * q + 2], acc[1][4 * q + 2], acc[0][4 * q + 3], acc[1][4 * q + 3]};
    }
  }
}

// Workgroup b's tile of `rows` rows: (expert, first sorted position, end position); expert -1: there is none.
// Every thread calls it; `info` int[3] and `sums` int[8] are LDS.
__device__ __forceinline__ void direct_find_tile(const int32_t* __restrict__ offsets, int E, int tile, int* info, int* sums) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int per = (E + kDirThreads - 1) / kDirThreads;
  const int e0 = tid * per;
  int mine = 0;
  for (int j = 0; j < per; j++)
    if (e0 + j < E) mine += (offsets[e0 + j + 1] - offsets[e0 + j] + kDirRows - 1) / kDirRows;
  int incl = mine;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int up = wave_shfl_up(incl, d);
    if (lane >= d) incl += up;
  }
  if (tid == 0) info[0] = -1;
  if (lane == 63) sums[wave] = incl;
  __syncthreads();
  int t = incl - mine;
  for (int w = 0; w < wave; w++) t += sums[w];
  if (tile >= t && tile < t + mine) {
    for (int j = 0; j < per; j++) {
      if (e0 + j >= E) break;
      const int lo = offsets[e0 + j], hi = offsets[e0 + j + 1];
      const int nt = (hi - lo + kDirRows - 1) / kDirRows;
      if (tile < t + nt) {
        const int r0 = lo + (tile - t) * kDirRows;
        info[0] = e0 + j;
        info[1] = r0;
        info[2] = r0 + kDirRows < hi ? r0 + kDirRows : hi;
        break;
      }
      t += nt;
    }
  }
  __syncthreads();
}

// out[out_index[i], :] = output stage(input stage(a[a_index[i], :]) @ W[e]) for 32 sorted positions x 64 columns per
// workgroup.  The stages and their order of operations are gemm_rows_kernel's; the K-tiles follow each other.
template <typename T, bool W_KC>
__global__ __launch_bounds__(kDirThreads, 2) void direct_fwd_kernel(const RowsParams p) {
  constexpr bool B16 = sizeof(T) == 2;
  constexpr int STEP = kDirStep<T>;
  __shared__ __attribute__((aligned(16))) float sPart[kDirWaves][kDirRows * kDirLd];
  __shared__ int sInfo[3], sSums[kDirWaves];

  const int tid = threadIdx.x, lane = tid & 63, wave = wave_uniform(tid >> 6);
  const int l32 = lane & 31, lh = lane >> 5;
  const int ncb = p.n_col_blocks;
  const int lb = xcd_contiguous_id(blockIdx.x, gridDim.x);
  const int cb = lb % ncb;
  direct_find_tile(p.offsets, p.E, lb / ncb, sInfo, sSums);
  const int e = wave_uniform(sInfo[0]);
  if (e < 0) return;                                         // the same for the whole workgroup
  const int row0 = wave_uniform(sInfo[1]), row_end = wave_uniform(sInfo[2]);
  const int c0 = cb * kDirCols, N = p.ND;

  // this lane's row: rows past the end of the tile read its first row, and are not stored
  const bool valid = row0 + l32 < row_end;
  const int r = valid ? row0 + l32 : row0;
  const bool has_ir = p.ir != nullptr;
  const bool quant = p.inp_res > 0.f;
  const bool codes_mode = B16 && quant;
  const bool adc_clip = p.out_bound > 0.f, adc_quant = adc_clip && p.out_half_states > 0.f;
  const bool gen_noise = p.noise_std > 0.f;
  const uint64_t seed = p.seed + ((gen_noise && p.seed_dev != nullptr) ? *p.seed_dev : 0);
  const int64_t ir_row = (int64_t)(p.ir_by_expert ? e : r) * p.ir_cols;

  DirectLoader<T, W_KC> ld;
  ld.lh = lh;
  ld.xrow = static_cast<const T*>(p.a) + (int64_t)p.a_index[r] * p.lda;
  const T* __restrict__ W = static_cast<const T*>(p.w) + (int64_t)e * p.w_se;
  if constexpr (W_KC) {
#pragma unroll
    for (int f = 0; f < 2; f++) {
      const int col = c0 + 32 * f + l32;
      ld.wcol[f] = W + (int64_t)(col < N ? col : N - 1) * p.w_snd;
    }
  } else {
    const int col = c0 + 2 * l32;
    ld.w_rsrc = make_rsrc(W);
    ld.w_ks = (uint32_t)(p.w_skd * (int64_t)sizeof(T));
    ld.w_lane = (uint32_t)(col + 1 < N ? col : N - 2) * (uint32_t)sizeof(T);
  }
  DirectDac dac;
  dac.on = quant && p.a_prequant == 0;
  dac.res = p.inp_res;
  dac.resinv = quant ? 1.0f / p.inp_res : 0.f;
  dac.margin = dac_tie_margin(dac.resinv);

  // the part of the output this lane finishes: row l32, columns oc .. oc + 3 of the tile
  const int blk = wave >> 2, q = wave & 3;
  const int oc = 32 * blk + 8 * q + 4 * lh;
  const int orow = valid ? (p.out_index != nullptr ? p.out_index[r] : p.a_index[r]) : 0;
  const float wm = p.wmax != nullptr ? p.wmax[e] : 1.f;
  const float u_nz = p.noise_std * wm, u_bound = p.out_bound * wm;
  const float u_q = adc_quant ? p.out_half_states / u_bound : 0.f;
  const float u_qinv = adc_quant ? u_bound / p.out_half_states : 0.f;
  float total[4] = {0.f, 0.f, 0.f, 0.f};

  for (int t = 0; t < p.n_kd_tiles; t++) {
    const int klo = p.kd_bounds[t], khi = p.kd_bounds[t + 1];
    const int nsteps = (khi - klo + STEP - 1) / STEP;
    const float ir_r = has_ir ? p.ir[ir_row + t] : 1.f;
    if (dac.on) dac.set_range(ir_r);
    f32x16 acc[2];
#pragma unroll
    for (int f = 0; f < 2; f++)
#pragma unroll
      for (int i = 0; i < 16; i++) acc[f][i] = 0.f;
    if (wave < nsteps) {                    // two steps in flight: the next one is fetched before this one is multiplied
      DirectStep<> s0, s1;
      ld.load(s0, klo + wave * STEP, khi);
      for (int s = wave; s < nsteps; s += 2 * kDirWaves) {
        const int s_b = s + kDirWaves, s_c = s + 2 * kDirWaves;
        if (s_b < nsteps) ld.load(s1, klo + s_b * STEP, khi);
        direct_multiply<T, W_KC>(acc, s0, dac);
        if (s_b < nsteps) {
          if (s_c < nsteps) ld.load(s0, klo + s_c * STEP, khi);
          direct_multiply<T, W_KC>(acc, s1, dac);
        }
      }
    }
    if (t > 0) __syncthreads();             // the previous K-tile's partial sums have been read
    direct_store_partial<W_KC>(sPart[wave], acc, l32, lh);
    __syncthreads();
    float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kDirWaves; w++) {
      const f32x4 part = *reinterpret_cast<const f32x4*>(&sPart[w][l32 * kDirLd + oc]);
#pragma unroll
      for (int j = 0; j < 4; j++) v[j] += part[j];
    }
    if (codes_mode) {
#pragma unroll
      for (int j = 0; j < 4; j++) v[j] *= p.inp_res;
    }
    if (gen_noise) {
      const NoiseKey key = noise_key(seed, t);
      const int cb0 = c0 + 32 * blk;
      const i32x16 z = noise_block(noise_row_key(key, (uint32_t)orow), noise_col_key(key, (uint32_t)(cb0 + l32)),
                                   (uint32_t)cb0 >> 5, (uint32_t)row0, lh);
#pragma unroll
      for (int j = 0; j < 4; j++) {         // this wave's quarter of the block
        const int zj = q == 0 ? z[j] : q == 1 ? z[4 + j] : q == 2 ? z[8 + j] : z[12 + j];
        v[j] = fmaf((float)zj, u_nz * kNoiseScale, v[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
      if (adc_clip) v[j] = clamp_sym(v[j], u_bound);
      if (adc_quant) v[j] = rintf(v[j] * u_q) * u_qinv;
      if (has_ir) v[j] *= ir_r;
      total[j] = t == 0 ? v[j] : total[j] + v[j];
    }
  }

  const int col = c0 + oc;
  int nv = valid ? N - col : 0;
  nv = nv < 0 ? 0 : (nv > 4 ? 4 : nv);
  if (nv == 0) return;
  if (p.relu) {
#pragma unroll
    for (int j = 0; j < 4; j++) total[j] = fmaxf(total[j], 0.f);
  }
  store4<T>(static_cast<T*>(p.out) + (int64_t)orow * p.ldo + col, total, nv, p.out_vec != 0);
  if (p.xq_out != nullptr) {                // the DAC image of the value as stored, for the projection that follows
    const float qr = p.xq_ir[e], qrinv = 1.0f / qr, qresinv = 1.0f / p.xq_inp_res, kq = qrinv * qresinv;
    float tie = 0.f, xc[4], c[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const float x = B16 ? Elem<T>::to_f32(Elem<T>::cvt(total[j])) : total[j];
      xc[j] = clamp_sym(x, qr);
      c[j] = dac_code<B16>(xc[j], qr, qrinv, p.xq_inp_res, qresinv, kq, tie);
      if (!B16) c[j] *= p.xq_inp_res;
    }
    if (B16 && tie > dac_tie_margin(qresinv)) {
#pragma unroll
      for (int j = 0; j < 4; j++) c[j] = dac_code_exact(xc[j], qr, qrinv, p.xq_inp_res, qresinv);
    }
    store4<T>(static_cast<T*>(p.xq_out) + (int64_t)orow * p.ldxq + col, c, nv, p.xq_vec != 0);
  }
}

// The same tile and operand path with the whole contraction in ONE wave and nothing shared between waves: for launches
// of many rows whose contraction or width is short or ends raggedly.  There a 128-row tiled kernel has one workgroup
// per CU (a wave per SIMD, which waits for its own loads, input stage and matrix instructions in turn) and twice that
// on the CUs that get the experts' last tiles; 32-row tiles of single waves fill two waves per SIMD and even out.
// (The tile's operands pass the L1 once per wave: 12 KB per 128-byte step, a third of the 16-bit matrix rate, twice the
// fp32 one.)  Wave w of the launch takes (row tile w / column blocks, column block w % column blocks).
constexpr int kDirWaveThreads = 256;

// This wave's row tile: (expert, first sorted position, end position); expert -1: there is none.  No barriers.
__device__ __forceinline__ void direct_find_wave_tile(const int32_t* __restrict__ offsets, int E, int tile, int& e, int& row0,
                                                      int& row_end) {
  const int lane = lane_id();
  e = -1;
  row0 = row_end = 0;
  for (int e0 = 0; e0 < E; e0 += 64) {          // 64 experts at a time
    const int ee = e0 + lane;
    const int lo = ee < E ? offsets[ee] : 0, hi = ee < E ? offsets[ee + 1] : 0;
    const int nt = (hi - lo + kDirRows - 1) / kDirRows;
    int incl = nt;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int up = wave_shfl_up(incl, d);
      if (lane >= d) incl += up;
    }
    const uint64_t past = wave_ballot(incl > tile);
    if (past != 0) {                            // the first expert whose tiles reach past `tile`
      const int src = ctz64(past);
      const int before = (int)wave_read((uint32_t)(incl - nt), src);
      e = e0 + src;
      row0 = (int)wave_read((uint32_t)lo, src) + (tile - before) * kDirRows;
      const int end = (int)wave_read((uint32_t)hi, src);
      row_end = row0 + kDirRows < end ? row0 + kDirRows : end;
      return;
    }
    tile -= (int)wave_read((uint32_t)incl, 63);
  }
}

template <typename T, bool W_KC, bool SPLIT>
__global__ __launch_bounds__(kDirWaveThreads, 2) void direct_wave_kernel(const RowsParams p) {
  constexpr bool B16 = sizeof(T) == 2;
  constexpr int STEP = kDirStep<T>;
  const int lane = lane_id(), l32 = lane & 31, lh = lane >> 5;
  const int ncb = p.n_col_blocks;
  const int id = xcd_contiguous_id(blockIdx.x, gridDim.x) * (kDirWaveThreads / 64) + wave_uniform((int)threadIdx.x >> 6);
  const int cb = id % ncb;
  int e, row0, row_end;
  direct_find_wave_tile(p.offsets, p.E, id / ncb, e, row0, row_end);
  if (e < 0) return;                            // the same for the whole wave
  const int c0 = cb * kDirCols, N = p.ND;
  const bool valid = row0 + l32 < row_end;
  const int r = valid ? row0 + l32 : row0;
  const bool has_ir = p.ir != nullptr;
  const bool quant = p.inp_res > 0.f;
  const bool codes_mode = B16 && quant;
  const bool adc_clip = p.out_bound > 0.f, adc_quant = adc_clip && p.out_half_states > 0.f;
  const bool gen_noise = p.noise_std > 0.f;
  const uint64_t seed = p.seed + ((gen_noise && p.seed_dev != nullptr) ? *p.seed_dev : 0);
  const int64_t ir_row = (int64_t)(p.ir_by_expert ? e : r) * p.ir_cols;

  DirectLoader<T, W_KC> ld;
  ld.lh = lh;
  ld.xrow = static_cast<const T*>(p.a) + (int64_t)p.a_index[r] * p.lda;
  const T* __restrict__ W = static_cast<const T*>(p.w) + (int64_t)e * p.w_se;
  if constexpr (W_KC) {
#pragma unroll
    for (int f = 0; f < 2; f++) {
      const int col = c0 + 32 * f + l32;
      ld.wcol[f] = W + (int64_t)(col < N ? col : N - 1) * p.w_snd;
    }
  } else {
    const int col = c0 + 2 * l32;
    ld.w_rsrc = make_rsrc(W);
    ld.w_ks = (uint32_t)(p.w_skd * (int64_t)sizeof(T));
    ld.w_lane = (uint32_t)(col + 1 < N ? col : N - 2) * (uint32_t)sizeof(T);
  }
  DirectDac dac;
  dac.on = quant && p.a_prequant == 0;
  dac.res = p.inp_res;
  dac.resinv = quant ? 1.0f / p.inp_res : 0.f;
  dac.margin = dac_tie_margin(dac.resinv);
  const int orow = p.out_index != nullptr ? p.out_index[r] : p.a_index[r];
  const float wm = p.wmax != nullptr ? p.wmax[e] : 1.f;
  const float u_nzs = p.noise_std * wm * kNoiseScale, u_bound = p.out_bound * wm;
  const float u_q = adc_quant ? p.out_half_states / u_bound : 0.f;
  const float u_qinv = adc_quant ? u_bound / p.out_half_states : 0.f;

  f32x16 acc[2], total[2];
  for (int t = 0; t < (SPLIT ? p.n_kd_tiles : 1); t++) {
    const int klo = p.kd_bounds[t], khi = p.kd_bounds[t + 1];
    const float ir_r = has_ir ? p.ir[ir_row + t] : 1.f;
    if (dac.on) dac.set_range(ir_r);
#pragma unroll
    for (int f = 0; f < 2; f++)
#pragma unroll
      for (int i = 0; i < 16; i++) acc[f][i] = 0.f;
    DirectStep<> s0, s1;
    ld.load(s0, klo, khi);
    for (int k0 = klo; k0 < khi; k0 += 2 * STEP) {
      if (k0 + STEP < khi) ld.load(s1, k0 + STEP, khi);
      direct_multiply<T, W_KC>(acc, s0, dac);
      if (k0 + STEP < khi) {
        if (k0 + 2 * STEP < khi) ld.load(s0, k0 + 2 * STEP, khi);
        direct_multiply<T, W_KC>(acc, s1, dac);
      }
    }
    // slot (f, 4 * q + j): column 32 * f + i (W_KC) or 2 * i + f of the tile, i = 8 * q + 4 * lh + j
#pragma unroll
    for (int f = 0; f < 2; f++) {
      if (codes_mode) {
#pragma unroll
        for (int i = 0; i < 16; i++) acc[f][i] *= p.inp_res;
      }
      if (gen_noise) {
        // The noise of a 32-column block of the output is one product; the columns 2 * i + f of the tile are the even
        // or odd ones of both blocks: two products, and each slot takes the one of its column's block.
        const NoiseKey key = noise_key(seed, t);
        const uint32_t row_key = noise_row_key(key, (uint32_t)orow);
        const uint32_t col_key = noise_col_key(key, (uint32_t)(c0 + (W_KC ? 32 * f + l32 : 2 * l32 + f)));
        const uint32_t block = (uint32_t)(c0 >> 5) + (W_KC ? (uint32_t)f : 0u);
        const i32x16 z = noise_block(row_key, col_key, block, (uint32_t)row0, lh);
#pragma unroll
        for (int i = 0; i < (W_KC ? 16 : 8); i++) acc[f][i] = fmaf((float)z[i], u_nzs, acc[f][i]);
        if constexpr (!W_KC) {
          const i32x16 z1 = noise_block(row_key, col_key, block + 1u, (uint32_t)row0, lh);
#pragma unroll
          for (int i = 8; i < 16; i++) acc[f][i] = fmaf((float)z1[i], u_nzs, acc[f][i]);
        }
      }
      if (adc_clip) {
#pragma unroll
        for (int i = 0; i < 16; i++) {
          float v = clamp_sym(acc[f][i], u_bound);
          if (adc_quant) v = rintf(v * u_q) * u_qinv;
          acc[f][i] = v;
        }
      }
      if (has_ir) {
#pragma unroll
        for (int i = 0; i < 16; i++) acc[f][i] *= ir_r;
      }
      if constexpr (SPLIT) {
#pragma unroll
        for (int i = 0; i < 16; i++) total[f][i] = t == 0 ? acc[f][i] : total[f][i] + acc[f][i];
      }
    }
  }
  if constexpr (SPLIT) {
    acc[0] = total[0];
    acc[1] = total[1];
  }
  if (!valid) return;                           // nothing of a whole wave follows

  // eight runs of four consecutive columns
  const float qr = p.xq_out != nullptr ? p.xq_ir[e] : 1.f;
  const float qrinv = 1.0f / qr, qresinv = 1.0f / p.xq_inp_res, qkq = qrinv * qresinv, qmargin = dac_tie_margin(qresinv);
#pragma unroll
  for (int run = 0; run < 8; run++) {
    float v[4];
    int oc;
    if constexpr (W_KC) {
      const int f = run >> 2, q = run & 3;
      oc = 32 * f + 8 * q + 4 * lh;
#pragma unroll
      for (int j = 0; j < 4; j++) v[j] = acc[f][4 * q + j];
    } else {
      const int q = run >> 1, h = run & 1;
      oc = 16 * q + 8 * lh + 4 * h;
#pragma unroll
      for (int j = 0; j < 4; j++) v[j] = acc[j & 1][4 * q + 2 * h + (j >> 1)];
    }
    const int col = c0 + oc;
    int nv = N - col;
    nv = nv < 0 ? 0 : (nv > 4 ? 4 : nv);
    if (p.relu) {
#pragma unroll
      for (int j = 0; j < 4; j++) v[j] = fmaxf(v[j], 0.f);
    }
    if (nv > 0) store4<T>(static_cast<T*>(p.out) + (int64_t)orow * p.ldo + col, v, nv, p.out_vec != 0);
    if (p.xq_out != nullptr) {                  // the DAC image of the value as stored
      float tie = 0.f, xc[4], c[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        xc[j] = clamp_sym(B16 ? Elem<T>::to_f32(Elem<T>::cvt(v[j])) : v[j], qr);
        c[j] = dac_code<B16>(xc[j], qr, qrinv, p.xq_inp_res, qresinv, qkq, tie);
        if (!B16) c[j] *= p.xq_inp_res;
      }
      if (B16 && tie > qmargin) {
#pragma unroll
        for (int j = 0; j < 4; j++) c[j] = dac_code_exact(xc[j], qr, qrinv, p.xq_inp_res, qresinv);
      }
      if (nv > 0) store4<T>(static_cast<T*>(p.xq_out) + (int64_t)orow * p.ldxq + col, c, nv, p.xq_vec != 0);
    }
  }
}

}  // namespace amoe
