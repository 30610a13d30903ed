// One query row of attention by one thread: f32 dot products, online softmax in registers. A serial
// chain over the keys, so its time grows with them.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels.h"
#include "numeric.h"

namespace ku::hipbk {

namespace {

// query qi (< a.s) of `head`; keys after it are not read when a.causal
template <int D, int DT, class T>
__device__ __forceinline__ void attn_row(const AttnArgs& a, int64_t head, int64_t qi) {
  const T* Q = static_cast<const T*>(a.q) + head * a.s * D;
  const T* K = static_cast<const T*>(a.k) + head * a.s * D;
  const T* Vv = static_cast<const T*>(a.v) + head * a.s * D;
  float q[D], acc[D];
#pragma unroll
  for (int t = 0; t < D; ++t) {
    q[t] = load_elem<DT, T, float>(Q[qi * D + t]);
    acc[t] = 0.f;
  }
  float m = -INFINITY, l = 0.f;
  const int64_t kend = a.causal ? qi + 1 : a.s;
  for (int64_t j = 0; j < kend; ++j) {
    float sc = 0.f;
#pragma unroll
    for (int t = 0; t < D; ++t) sc = fmaf(q[t], load_elem<DT, T, float>(K[j * D + t]), sc);
    sc *= a.scale;
    float mn = fmaxf(m, sc);
    float corr = expf(m - mn);
    float p = expf(sc - mn);
    l = l * corr + p;
#pragma unroll
    for (int t = 0; t < D; ++t) acc[t] = acc[t] * corr + p * load_elem<DT, T, float>(Vv[j * D + t]);
    m = mn;
  }
  T* O = static_cast<T*>(a.o) + head * a.s * D;
  const float inv = 1.f / l;
#pragma unroll
  for (int t = 0; t < D; ++t) O[qi * D + t] = store_elem<DT, T, float>(acc[t] * inv);
}

}  // namespace

}  // namespace ku::hipbk
