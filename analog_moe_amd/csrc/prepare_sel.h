// Expert sort of the CVMM path: stable counting sort of expert ids with wavefront ballots.
//   pass 1  per-wave histograms of 1024-element units (LDS atomics)
//   pass 2  a wave per expert scans its unit counts (bases in place), then one workgroup scans
//           the per-expert totals -> offsets[E+1]
//   pass 3  per wave: rank every element among equal keys of its 64-lane batch with a
//           match-any built from ballots over the key bits, add the running per-key base kept
//           in LDS, scatter (sorted id, flat index, flat index / k)
// (up to 256 experts: two launches or one, sel_group_hist_kernel / sel_group_scatter_kernel)
// Stable by construction: batches, units and lanes are all visited in ascending flat index.
#pragma once
#include "common.h"

namespace amoe {

constexpr int kSelUnitMax = 1024;   // elements per wave: 64 .. 1024, fewer for short inputs so that
                                    // the sort still spreads over the chip (see sel_unit)
__host__ __device__ inline int sel_unit(long long M) {
  int u = 64;
  while (u < kSelUnitMax && M / u > 2048) u <<= 1;   // aim at <= 2048 units
  return u < 256 ? 256 : u;
}

struct SelParams {
  const void* sel; int sel_is_i64;
  long long M; int E, k, n_units, key_bits, unit;
  int32_t* sel_sorted; int32_t* perm; int32_t* in_index; int32_t* offsets; int32_t* bad_flag;
  int32_t* unit_hist;               // workspace [n_units][E]
  int table_vec;                    // its rows are on 16-byte pieces
};

__device__ __forceinline__ int sel_key(const SelParams& p, long long i, bool& bad) {
  long long v = p.sel_is_i64 ? static_cast<const long long*>(p.sel)[i]
                             : (long long)static_cast<const int32_t*>(p.sel)[i];
  bad = v < 0 || v >= p.E;
  if (v < 0) v = 0;                      // out-of-range ids are flagged and clamped
  if (v >= p.E) v = p.E - 1;
  return (int)v;
}

__global__ __launch_bounds__(kThreads) void sel_hist_kernel(const SelParams p) {
  __shared__ int hist[4 * kSelMaxExperts];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int i = tid; i < 4 * p.E; i += kThreads) hist[i] = 0;
  __syncthreads();
  const int unit = blockIdx.x * 4 + wave;
  bool any_bad = false;
  if (unit < p.n_units) {
    for (int it = 0; it < p.unit / 64; it++) {
      const long long i = (long long)unit * p.unit + it * 64 + lane;
      if (i < p.M) {
        bool bad;
        const int key = sel_key(p, i, bad);
        any_bad |= bad;
        atomicAdd(&hist[wave * p.E + key], 1);
      }
    }
  }
  if (any_bad && p.bad_flag != nullptr) atomicOr(p.bad_flag, 1);
  __syncthreads();
  for (int w = 0; w < 4; w++) {
    const int u = blockIdx.x * 4 + w;
    if (u < p.n_units)
      for (int e = tid; e < p.E; e += kThreads) p.unit_hist[(long long)u * p.E + e] = hist[w * p.E + e];
  }
}

// pass 2a: one wave per expert turns its column of unit counts into unit bases relative to the
// expert's segment start and writes the expert's total to offsets[e + 1].
__global__ __launch_bounds__(kThreads) void sel_unit_scan_kernel(const SelParams p) {
  const int lane = threadIdx.x & 63;
  const int e = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (e >= p.E) return;
  int carry = 0;
  for (int u0 = 0; u0 < p.n_units; u0 += 64) {
    const int u = u0 + lane;
    const int c = u < p.n_units ? p.unit_hist[(long long)u * p.E + e] : 0;
    int incl = c;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int up = wave_shfl_up(incl, d);
      if (lane >= d) incl += up;
    }
    if (u < p.n_units) p.unit_hist[(long long)u * p.E + e] = carry + incl - c;
    carry += wave_shfl(incl, 63);
  }
  if (lane == 0) p.offsets[e + 1] = carry;
}

// pass 2b: one workgroup turns the per-expert totals (in offsets[1..E]) into offsets[0..E].
__global__ __launch_bounds__(kThreads) void sel_offsets_kernel(const SelParams p) {
  constexpr int kPer = kSelMaxExperts / kThreads;
  __shared__ int wave_sums[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int e0 = tid * kPer;
  int c[kPer];
  int mine = 0;
#pragma unroll
  for (int j = 0; j < kPer; j++) {
    c[j] = e0 + j < p.E ? p.offsets[e0 + j + 1] : 0;
    mine += c[j];
  }
  int incl = mine;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int up = wave_shfl_up(incl, d);
    if (lane >= d) incl += up;
  }
  if (lane == 63) wave_sums[wave] = incl;
  __syncthreads();                     // also orders every read of the totals before the writes below
  int run = incl - mine;
  for (int w = 0; w < wave; w++) run += wave_sums[w];
#pragma unroll
  for (int j = 0; j < kPer; j++) {
    if (e0 + j < p.E) p.offsets[e0 + j] = run;
    run += c[j];
  }
  if (tid == 0) p.offsets[p.E] = (int)p.M;
}

__global__ __launch_bounds__(kThreads) void sel_scatter_kernel(const SelParams p) {
  __shared__ int base[4 * kSelMaxExperts];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int w = 0; w < 4; w++) {
    const int u = blockIdx.x * 4 + w;
    if (u < p.n_units)
      for (int e = tid; e < p.E; e += kThreads) base[w * p.E + e] = p.offsets[e] + p.unit_hist[(long long)u * p.E + e];
  }
  __syncthreads();
  const int unit = blockIdx.x * 4 + wave;
  int* my_base = &base[wave * p.E];
  const uint64_t lt_mask = ((uint64_t)1 << lane) - 1;
  for (int it = 0; it < p.unit / 64; it++) {
    const long long i = (long long)unit * p.unit + it * 64 + lane;
    const bool valid = unit < p.n_units && i < p.M;
    bool bad;
    const int key = valid ? sel_key(p, i, bad) : 0;
    uint64_t same = wave_ballot(valid);
    for (int b = 0; b < p.key_bits; b++) {
      const bool bit = (key >> b) & 1;
      const uint64_t bal = wave_ballot(valid && bit);
      same &= bit ? bal : ~bal;
    }
    const int rank = popc64(same & lt_mask);
    const int count = popc64(same);
    int pos = 0;
    if (valid) pos = my_base[key] + rank;
    wave_sync();
    if (valid && rank == 0) my_base[key] += count;
    wave_sync();
    if (valid) {
      p.sel_sorted[pos] = key;
      p.perm[pos] = (int)i;
      p.in_index[pos] = (int)(i / p.k);
    }
  }
}

// ---- the same sort with at most kThreads experts --------------------------------------------------------------
// A group is `span` consecutive elements, one workgroup, a quarter per wave.  Two launches: the groups' histograms as a
// table [n_groups][E], then every workgroup sums the whole table for itself (per expert: the total, and the part of the
// groups before its own), scans the totals into the experts' segment starts, counts its own waves' keys again in LDS
// and scatters.  Up to kSelSmall elements the second launch counts the keys themselves instead of a table and is the
// only one.  The sort is on the path to the first GEMM of every step, so what matters is the number of launches and
// the length of the dependent chain inside them, not the bytes.
//   Span: the smallest that leaves at most kSelGroups groups, or as many as make a table of kSelTable counts, so that the
//   table every workgroup reads stays at or below 128 KB and few experts still get many short groups.  One table row per
//   wave, as the general path has it, is a table four times as large: 131 072 elements of 128 experts 19.9 us, 13.0 by
//   groups, of 64 experts 18.5 and 11.5.  128 groups of up to 16384 elements whatever E is were too few and too long for few
//   experts (8 experts, 262 144 elements 14.9 us, 1 000 000 40.1; as it is now 10.5 and 16.7), and a row of no multiple of
//   four counts was read in one chain (250 experts, 131 072 elements 41.7 us; with eight loads in flight 18.1).
//   kSelSpanMax: beyond it the general path is as fast (1 000 000 elements of 128 experts 56.2 us in spans of 8192, 55.4).
//   kSelSmall: one launch that counts all keys takes 3.3 us at 8 elements, 4.0 at 512 (two launches: 5.9, 8.1) and grows
//   by 0.8 us per 1024 elements; two launches take 7 us from there on.
constexpr int kSelSmall = 4096;
constexpr int kSelGroups = 128, kSelTable = 8192;
constexpr int kSelSpanMax = 4096;
__host__ __device__ inline int sel_groups_max(int E) { return kSelTable / E > kSelGroups ? kSelTable / E : kSelGroups; }
__host__ __device__ inline int sel_span(long long M, int E) {
  int s = kThreads;
  if (M > kSelSmall)
    while (s < kSelSpanMax && (M + s - 1) / s > sel_groups_max(E)) s <<= 1;
  return s;
}
__host__ __device__ inline bool sel_by_groups(long long M, int E) {
  return E <= kThreads && (M + sel_span(M, E) - 1) / sel_span(M, E) <= sel_groups_max(E);
}

// counts of n keys from `first` into hist (LDS, zeroed), eight loads in flight per thread; true: an id out of range
__device__ __forceinline__ bool sel_count(const SelParams& p, long long first, long long n, int* hist) {
  bool any_bad = false;
  for (long long i0 = threadIdx.x; i0 < n; i0 += 8 * kThreads) {
    int key[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const long long i = i0 + j * kThreads;
      bool bad = false;
      key[j] = i < n ? sel_key(p, first + i, bad) : -1;
      any_bad |= bad;
    }
#pragma unroll
    for (int j = 0; j < 8; j++)
      if (key[j] >= 0) atomicAdd(&hist[key[j]], 1);
  }
  return any_bad;
}

__global__ __launch_bounds__(kThreads) void sel_group_hist_kernel(const SelParams p) {
  __shared__ int hist[kThreads];
  const int tid = threadIdx.x;
  hist[tid] = 0;
  __syncthreads();
  const long long first = (long long)blockIdx.x * p.unit;
  const long long n = p.M - first < p.unit ? p.M - first : p.unit;
  const bool any_bad = sel_count(p, first, n, hist);
  if (any_bad && p.bad_flag != nullptr) atomicOr(p.bad_flag, 1);
  __syncthreads();
  if (tid < p.E) p.unit_hist[(long long)blockIdx.x * p.E + tid] = hist[tid];
}

template <bool SMALL>
__global__ __launch_bounds__(kThreads) void sel_group_scatter_kernel(const SelParams p) {
  __shared__ int base[4 * kThreads];          // [wave][expert]: where the next element of that expert goes
  __shared__ __attribute__((aligned(16))) int part_total[4 * kThreads], part_before[4 * kThreads];
  __shared__ int wave_sums[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int E = p.E, group = blockIdx.x;
  const long long first = (long long)group * p.unit;      // this workgroup's elements
  const int per_wave = p.unit / 4;
#pragma unroll
  for (int w = 0; w < 4; w++) base[w * kThreads + tid] = 0;
  int my_total = 0, my_before = 0;                  // thread e < E: the expert's two sums
  if constexpr (SMALL) {
    part_before[tid] = part_total[tid] = 0;
    __syncthreads();
    bool bad = sel_count(p, 0, first < p.M ? first : p.M, part_before);
    bad |= sel_count(p, first, p.M - first, part_total);
    if (bad && group == 0 && p.bad_flag != nullptr) atomicOr(p.bad_flag, 1);
    __syncthreads();
    if (tid < E) {
      my_before = part_before[tid];
      my_total = my_before + part_total[tid];
    }
  } else if (p.table_vec) {
    // the table in rows (one group's counts), several rows per pass of the workgroup, four experts per thread
    typedef __attribute__((ext_vector_type(4))) int i32x4v;
    const int tpr = E >> 2;                         // threads per row (<= 64)
    const int rpp = kThreads / tpr;                 // rows per pass
    const int c4 = tid % tpr, row = tid / tpr;
    i32x4v tot = {0, 0, 0, 0}, bef = {0, 0, 0, 0};
    if (row < rpp) {
#pragma unroll 4
      for (int u = row; u < p.n_units; u += rpp) {
        const i32x4v c = *reinterpret_cast<const i32x4v*>(p.unit_hist + (long long)u * E + 4 * c4);
        tot += c;
        if (u < group) bef += c;
      }
      *reinterpret_cast<i32x4v*>(&part_total[row * E + 4 * c4]) = tot;
      *reinterpret_cast<i32x4v*>(&part_before[row * E + 4 * c4]) = bef;
    }
    __syncthreads();
    if (tid < E)
      for (int r = 0; r < rpp; r++) {
        my_total += part_total[r * E + tid];
        my_before += part_before[r * E + tid];
      }
  } else {
    int epad = 1;
    while (epad < E) epad <<= 1;
    const int groups = kThreads / epad;
    const int e = tid & (epad - 1), grp = tid / epad;
    int total = 0, before = 0;
    if (e < E) {
#pragma unroll 8
      for (int u = grp; u < p.n_units; u += groups) {
        const int c = p.unit_hist[(long long)u * E + e];
        total += c;
        before += u < group ? c : 0;
      }
    }
    part_total[tid] = total;
    part_before[tid] = before;
    __syncthreads();
    if (tid < E)
      for (int g = 0; g < groups; g++) {
        my_total += part_total[g * epad + tid];
        my_before += part_before[g * epad + tid];
      }
  }
  // the waves' own counts (base was cleared before the barriers above)
  for (int it = 0; it < per_wave; it += 64) {
    const long long i = first + (long long)wave * per_wave + it + lane;
    bool bad;
    if (i < p.M) atomicAdd(&base[wave * kThreads + sel_key(p, i, bad)], 1);
  }
  // exclusive scan of the totals over the experts (thread = expert)
  int incl = my_total;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int up = wave_shfl_up(incl, d);
    if (lane >= d) incl += up;
  }
  if (lane == 63) wave_sums[wave] = incl;
  __syncthreads();
  int start = incl - my_total;
  for (int w = 0; w < wave; w++) start += wave_sums[w];
  if (tid < E) {
    if (group == 0) {
      p.offsets[tid] = start;
      if (tid == E - 1) p.offsets[E] = (int)p.M;
    }
    int run = start + my_before;
#pragma unroll
    for (int w = 0; w < 4; w++) {
      const int c = base[w * kThreads + tid];
      base[w * kThreads + tid] = run;
      run += c;
    }
  }
  __syncthreads();
  int* my_base = &base[wave * kThreads];
  const uint64_t lt_mask = ((uint64_t)1 << lane) - 1;
  for (int it = 0; it < per_wave; it += 64) {
    const long long i = first + (long long)wave * per_wave + it + lane;
    const bool valid = i < p.M;
    bool bad;
    const int key = valid ? sel_key(p, i, bad) : 0;
    uint64_t same = wave_ballot(valid);
    for (int b = 0; b < p.key_bits; b++) {
      const bool bit = (key >> b) & 1;
      const uint64_t bal = wave_ballot(valid && bit);
      same &= bit ? bal : ~bal;
    }
    const int rank = popc64(same & lt_mask);
    const int count = popc64(same);
    int pos = 0;
    if (valid) pos = my_base[key] + rank;
    wave_sync();
    if (valid && rank == 0) my_base[key] += count;
    wave_sync();
    if (valid) {
      p.sel_sorted[pos] = key;
      p.perm[pos] = (int)i;
      p.in_index[pos] = (int)((uint32_t)i / (uint32_t)p.k);
    }
  }
}

// offsets[E+1] from sorted ids: position i owns every expert in (sel[i-1], sel[i]].
__global__ __launch_bounds__(kThreads) void offsets_from_sorted_kernel(const int32_t* __restrict__ sel,
                                                                        long long M, int E,
                                                                        int32_t* __restrict__ offsets) {
  const long long i = (long long)blockIdx.x * kThreads + threadIdx.x;
  if (i > M) return;
  const int prev = (i == 0) ? -1 : sel[i - 1];
  int cur = (i == M) ? E : sel[i];
  if (cur > E) cur = E;
  for (int e = prev + 1; e <= cur; e++)
    if (e >= 0) offsets[e] = (int)i;
}

}  // namespace amoe
