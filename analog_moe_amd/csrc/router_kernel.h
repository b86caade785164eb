// The analog router at inference in one launch: logits = output stage(input stage(x) @ W^T), sigmoid, top-k.
//
// Separately these are a max |W| reduction, a 64-column product, the top-k and the conversions between them: nine
// launches whose work is a microsecond each.  The product is the one of gemm_direct.h (the contraction split over the
// waves of a workgroup); a workgroup reads all of W for its rows, so max |W| falls out of the operand loads, and the
// logits of its rows go through LDS to one wave per row for the top-k (select_rank.h).
#pragma once
#include "gemm_direct.h"
#include "select_rank.h"

namespace amoe {

struct RouterParams {
  const void* x; int64_t ldx;
  const void* w; int64_t ldw;                       // [E, K], contraction contiguous
  int T, K, E, k;
  int rows_per_block;                               // 8, 16 or 32
  int n_tiles; int bounds[kDirWaves + 1];           // K-tiles: 1, 2, 4 or 8 (each has as many waves)
  const void* ir;                                   // input range per K-tile, in the element type
  float inp_res, out_bound, out_half_states;
  void* sel_val; int64_t* sel_idx;
};

template <typename T, int NF>
__global__ __launch_bounds__(kDirThreads, 2) void router_kernel(const RouterParams p) {
  constexpr bool B16 = sizeof(T) == 2;
  constexpr int STEP = kDirStep<T>, CH = Elem<T>::kChunk, LD = 32 * NF + 4, PER = (NF + 1) / 2;
  __shared__ __attribute__((aligned(16))) float sPart[kDirWaves][kDirRows * LD];
  __shared__ float sLogit[kDirRows][32 * NF];
  __shared__ float sMax[kDirWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_uniform(tid >> 6);
  const int l32 = lane & 31, lh = lane >> 5;
  const int row0 = (int)blockIdx.x * p.rows_per_block;
  const int rows = p.T - row0 < p.rows_per_block ? p.T - row0 : p.rows_per_block;

  DirectLoader<T, true, NF> ld;
  ld.lh = lh;
  ld.xrow = static_cast<const T*>(p.x) + (int64_t)(row0 + (l32 < rows ? l32 : 0)) * p.ldx;
#pragma unroll
  for (int f = 0; f < NF; f++) {
    const int col = 32 * f + l32;
    ld.wcol[f] = static_cast<const T*>(p.w) + (int64_t)(col < p.E ? col : p.E - 1) * p.ldw;
  }
  // wave -> K-tile t and its place among that tile's waves
  const int per_tile = kDirWaves / p.n_tiles, t = wave / per_tile, place = wave - t * per_tile;
  const int klo = p.bounds[t], khi = p.bounds[t + 1];
  const int nsteps = (khi - klo + STEP - 1) / STEP;
  const T* __restrict__ IR = static_cast<const T*>(p.ir);
  const bool quant = p.inp_res > 0.f;
  DirectDac dac;
  dac.on = quant;
  dac.res = p.inp_res;
  dac.resinv = 1.0f / p.inp_res;
  dac.margin = dac_tie_margin(dac.resinv);
  dac.set_range(Elem<T>::load(IR + t));

  float wmax = 0.f;
  auto see = [&](const DirectStep<NF>& s) {
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int f = 0; f < NF; f++) {
        float v[CH];
        raw_unpack<T>(Raw{s.w[i][4 * f], s.w[i][4 * f + 1], s.w[i][4 * f + 2], s.w[i][4 * f + 3]}, v);
#pragma unroll
        for (int j = 0; j < CH; j++) wmax = fmaxf(wmax, fabsf(v[j]));
      }
  };
  f32x16 acc[NF];
#pragma unroll
  for (int f = 0; f < NF; f++)
#pragma unroll
    for (int i = 0; i < 16; i++) acc[f][i] = 0.f;
  if (place < nsteps) {                      // as direct_fwd_kernel: the next step in flight behind the current one
    DirectStep<NF> s0, s1;
    ld.load(s0, klo + place * STEP, khi);
    for (int s = place; s < nsteps; s += 2 * per_tile) {
      const int s_b = s + per_tile, s_c = s + 2 * per_tile;
      if (s_b < nsteps) ld.load(s1, klo + s_b * STEP, khi);
      see(s0);
      direct_multiply<T, true, NF>(acc, s0, dac);
      if (s_b < nsteps) {
        if (s_c < nsteps) ld.load(s0, klo + s_c * STEP, khi);
        see(s1);
        direct_multiply<T, true, NF>(acc, s1, dac);
      }
    }
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) wmax = fmaxf(wmax, wave_shfl_xor(wmax, d));
  if (lane == 0) sMax[wave] = wmax;
  direct_store_partial<true, NF>(sPart[wave], acc, l32, lh);
  __syncthreads();
  wmax = sMax[0];
#pragma unroll
  for (int w = 1; w < kDirWaves; w++) wmax = fmaxf(wmax, sMax[w]);

  const bool adc_clip = p.out_bound > 0.f, adc_quant = adc_clip && p.out_half_states > 0.f;
  const float bound = p.out_bound * wmax;
  const float u_q = adc_quant ? p.out_half_states / bound : 0.f, u_qinv = adc_quant ? bound / p.out_half_states : 0.f;
  for (int i = tid; i < kDirRows * 8 * NF; i += kDirThreads) {
    const int r = i / (8 * NF), c = (i % (8 * NF)) * 4;
    if (r >= rows) break;
    float total[4];
    for (int tt = 0; tt < p.n_tiles; tt++) {
      float v[4] = {0.f, 0.f, 0.f, 0.f};
      for (int w = 0; w < per_tile; w++) {
        const f32x4 part = *reinterpret_cast<const f32x4*>(&sPart[tt * per_tile + w][r * LD + c]);
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] += part[j];
      }
      const float ir = Elem<T>::load(IR + tt);
#pragma unroll
      for (int j = 0; j < 4; j++) {
        if (B16 && quant) v[j] *= p.inp_res;
        if (adc_clip) v[j] = clamp_sym(v[j], bound);
        if (adc_quant) v[j] = rintf(v[j] * u_q) * u_qinv;
        v[j] *= ir;
        total[j] = tt == 0 ? v[j] : total[j] + v[j];
      }
    }
#pragma unroll
    for (int j = 0; j < 4; j++) sLogit[r][c + j] = Elem<T>::to_f32(Elem<T>::cvt(total[j]));   // as stored in T
  }
  __syncthreads();
  for (int r = wave; r < rows; r += kDirWaves) {
    float s[PER];
#pragma unroll
    for (int j = 0; j < PER; j++) {
      const int e = lane + 64 * j;
      s[j] = e < p.E ? gate_value<T>(sLogit[r][e < 32 * NF ? e : 0]) : -__builtin_inff();
    }
    const int64_t at = (int64_t)(row0 + r) * p.k;
    select_by_rank<T, PER>(s, lane, p.E, p.k, static_cast<T*>(p.sel_val) + at, p.sel_idx + at);
  }
}

}  // namespace amoe
