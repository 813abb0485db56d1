// LayerNorm of one row by one wavefront, shared by the prompt kernels.
#pragma once

#include "mie_common.h"

namespace mie {

// out = LayerNorm(x) over dim elements (a multiple of 4): float32, biased
// variance, the result rounded to T; b may be NULL.  P > 0: the row and the
// parameters are read in one memory round and stay in registers (dim <= 256 P;
// lane l holds elements 256 p + 4 l ..), and the rounded row is returned in
// `y` (when given; zero past dim).  P = 0: any dim, in three passes.
template <typename T, int P>
__device__ __forceinline__ void norm_row(const T* x, const T* w, const T* b, T* out, int dim, float eps, int lane,
                                         mem_f32x4* y = nullptr) {
  if constexpr (P > 0) {
    typename Mem<T>::raw4 rx[P], rw[P], rb[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int i = p * 256 + lane * 4 < dim ? p * 256 + lane * 4 : 0;  // in bounds; dropped below
      rx[p] = Mem<T>::load_raw(x + i);
      rw[p] = Mem<T>::load_raw(w + i);
      rb[p] = Mem<T>::load_raw((b ? b : w) + i);
    }
    mem_f32x4 v[P];
    float s = 0.f;
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const bool live = p * 256 + lane * 4 < dim;
      v[p] = live ? Mem<T>::widen(rx[p]) : mem_f32x4{0.f, 0.f, 0.f, 0.f};
      s += (v[p].x + v[p].y) + (v[p].z + v[p].w);
    }
    const float mean = wave_sum(s) / dim;
    float q = 0.f;
#pragma unroll
    for (int p = 0; p < P; ++p) {
      if (p * 256 + lane * 4 >= dim) continue;
      const mem_f32x4 d = v[p] - mean;
      q += (d.x * d.x + d.y * d.y) + (d.z * d.z + d.w * d.w);
    }
    const float rstd = rsqrtf(wave_sum(q) / dim + eps);
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int i = p * 256 + lane * 4;
      mem_f32x4 r = {0.f, 0.f, 0.f, 0.f};
      if (i < dim) {
        r = (v[p] - mean) * rstd * Mem<T>::widen(rw[p]);
        if (b) r += Mem<T>::widen(rb[p]);
        r = Mem<T>::R4(r);
        Mem<T>::put4(out + i, r);
      }
      if (y) y[p] = r;
    }
  } else {
    float s = 0.f;
    for (int i = lane * 4; i < dim; i += 256) {
      const mem_f32x4 v = Mem<T>::load4(x + i);
      s += (v.x + v.y) + (v.z + v.w);
    }
    const float mean = wave_sum(s) / dim;
    float q = 0.f;
    for (int i = lane * 4; i < dim; i += 256) {
      const mem_f32x4 d = Mem<T>::load4(x + i) - mean;
      q += (d.x * d.x + d.y * d.y) + (d.z * d.z + d.w * d.w);
    }
    const float rstd = rsqrtf(wave_sum(q) / dim + eps);
    for (int i = lane * 4; i < dim; i += 256) {
      mem_f32x4 r = (Mem<T>::load4(x + i) - mean) * rstd * Mem<T>::load4(w + i);
      if (b) r += Mem<T>::load4(b + i);
      Mem<T>::put4(out + i, r);
    }
  }
}

}  // namespace mie
