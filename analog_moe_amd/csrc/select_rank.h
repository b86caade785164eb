// Gate values of the router and the choice of the k largest of a row.
#pragma once
#include "common.h"

namespace amoe {

// The gate value as the tensor expression sigmoid(logits) holds it: computed in fp32, stored in T.
template <typename T>
__device__ __forceinline__ float gate_value(float x) {
  return Elem<T>::to_f32(Elem<T>::cvt(1.0f / (1.0f + expf(-x))));
}

// The k largest of a row's gate values s (lane owns the experts lane, lane + 64, ...; NaN: never chosen): an expert's
// place is the number of experts with a larger value, or with the same value and a lower id.  Gate values are not
// negative, so their bit patterns order as they do; 0 marks what cannot be chosen.
template <typename T, int PER>
__device__ __forceinline__ void select_by_rank(const float (&s)[PER], int lane, int E, int k, T* __restrict__ val,
                                               int64_t* __restrict__ idx) {
  uint32_t key[PER];
  int place[PER], n = 0;
#pragma unroll
  for (int j = 0; j < PER; j++) {
    key[j] = s[j] >= 0.f ? as_u32(s[j]) + 1u : 0u;
    place[j] = 0;
    n += popc64(wave_ballot(key[j] != 0u));
  }
#pragma unroll
  for (int jj = 0; jj < PER; jj++) {
    const int here = E - 64 * jj < 64 ? E - 64 * jj : 64;
#pragma unroll 8
    for (int l = 0; l < here; l++) {
      const uint32_t other = wave_read(key[jj], l);
#pragma unroll
      for (int j = 0; j < PER; j++) {
        const bool lower_id = jj < j || (jj == j && l < lane);
        place[j] += other > key[j] - (lower_id ? 1u : 0u) ? 1 : 0;
      }
    }
  }
#pragma unroll
  for (int j = 0; j < PER; j++)
    if (key[j] != 0u && place[j] < k) {
      val[place[j]] = Elem<T>::cvt(s[j]);
      idx[place[j]] = lane + 64 * j;
    }
  if (lane >= n && lane < k) {                    // fewer than k experts can be chosen
    val[lane] = Elem<T>::cvt(-__builtin_inff());
    idx[lane] = 0x7fffffff;
  }
  for (int t = 64 + lane; t < k; t += 64)
    if (t >= n) {
      val[t] = Elem<T>::cvt(-__builtin_inff());
      idx[t] = 0x7fffffff;
    }
}

}  // namespace amoe
