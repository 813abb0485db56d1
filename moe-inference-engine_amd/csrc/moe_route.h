// Top-k routing over a wavefront, shared by the one-token MoE kernels and the
// prompt MoE's routing kernel.
#pragma once

#include <math.h>

#include "mie_common.h"

namespace mie {
namespace route {

constexpr int kMaxExperts = 64;
constexpr int kMaxTopK = 8;

typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float dot4(f32x4_t a, f32x4_t b, float s) {
  s = fmaf(a.x, b.x, s);
  s = fmaf(a.y, b.y, s);
  s = fmaf(a.z, b.z, s);
  return fmaf(a.w, b.w, s);
}

// Dot product of a row with a vector over one wavefront (four elements per
// lane per step), in float32.
template <typename T>
__device__ __forceinline__ float wave_dot(const T* __restrict__ row, const T* __restrict__ v, int n, int lane) {
  float s = 0.f;
  for (int i = lane * 4; i < n; i += 256) s = dot4(Mem<T>::load4(row + i), Mem<T>::load4(v + i), s);
  return wave_sum(s);
}

// (v, i) against (ov, oi): the larger logit wins, the lower expert id on
// ties, and NaN counts as larger than every number (torch.topk's order) - a
// total order, so any reduction tree gives the same pick, and a NaN logit is
// picked like any other, so the pick is always an expert that is not yet
// taken (a taken expert holds -inf and an id past 63).  Compares and selects,
// no branches.
__device__ __forceinline__ void topk_take(float& v, int& i, float ov, int oi) {
  const bool v_nan = v != v, o_nan = ov != ov;
  const bool lower = oi < i;
  // ov > v and ov == v are false when either is NaN.
  const bool b = (o_nan & (!v_nan | lower)) | (ov > v) | ((ov == v) & lower);
  v = b ? ov : v;
  i = b ? oi : i;
}

template <int CTRL>
__device__ __forceinline__ void topk_dpp(float& v, int& i) {
  topk_take(v, i, dpp<CTRL>(v), __builtin_amdgcn_update_dpp(0, i, CTRL, 0xF, 0xF, false));
}

// Top-k over a wave: lane e holds expert e's logit (-inf for lanes >= E).
// Round kk takes the largest logit not yet taken, the lower expert id on ties;
// ids and weights (the softmax of the selected logits) come out uniform across
// the wave.  Fixed-size loops keep both arrays in registers; top_k <= K.
template <int K = kMaxTopK>
__device__ __forceinline__ void wave_topk(float logit, int top_k, int num_experts, int lane, int* ids,
                                          float* weights) {
  bool taken = false;
  float vals[K];
#pragma unroll
  for (int kk = 0; kk < K; ++kk) {
    ids[kk] = 0;
    vals[kk] = 0.f;
    if (kk < top_k) {
      // A taken expert also loses every tie, so a repeated -inf cannot pick it twice.
      float v = taken ? -INFINITY : logit;
      int idx = taken ? lane + 64 : lane;
      // Only the lanes holding experts take part: DPP stages over 2, 4, 8 and
      // 16 lanes (quad xor-1 and xor-2, then half-row and row mirrors), then
      // cross-row exchanges for more than 16 experts.
      topk_dpp<0xB1>(v, idx);
      topk_dpp<0x4E>(v, idx);
      if (num_experts > 4) topk_dpp<0x141>(v, idx);
      if (num_experts > 8) topk_dpp<0x140>(v, idx);
      if (num_experts > 16) topk_take(v, idx, __shfl_xor(v, 16), __shfl_xor(idx, 16));
      if (num_experts > 32) topk_take(v, idx, __shfl_xor(v, 32), __shfl_xor(idx, 32));
      // Lane 0 holds the pick; every lane takes it from a scalar register.
      idx = __builtin_amdgcn_readfirstlane(idx);
      v = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
      ids[kk] = idx;
      vals[kk] = v;
      taken = taken || lane == idx;
    }
  }
  // softmax over the selected logits; vals[0] is their maximum
  float sum = 0.f;
#pragma unroll
  for (int kk = 0; kk < K; ++kk) {
    weights[kk] = kk < top_k ? expf(vals[kk] - vals[0]) : 0.f;
    sum += weights[kk];
  }
#pragma unroll
  for (int kk = 0; kk < K; ++kk) weights[kk] /= sum;
}

}  // namespace route
}  // namespace mie
