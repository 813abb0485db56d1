// A workgroup's tile of C = A . W^T on the matrix cores: A rows and W rows are
// both K-contiguous ("NT"), float32 or bfloat16, accumulated in float32.
//
// 256 threads, four waves as WM x WN over a BM x BN tile, each wave MT x NT
// blocks of 16 x 16.  One 16-byte LDS read per lane is one fragment: four
// v_mfma_f32_16x16x4_f32 steps of float32, or one v_mfma_f32_16x16x32_bf16.
// A lane's fragment holds consecutive K of one row, so a float32 step j
// multiplies K = 4 g + j of lane group g: a permutation of the contraction,
// the same for both operands.  W is the instruction's first operand, so a
// lane's four results are four consecutive columns of one row and the
// epilogue stores 16-byte vectors.
//
// K goes in steps of KB bytes per row through two LDS buffers: step s + 1 is
// written while step s is multiplied, step s + 2 is in flight in registers.
// The barrier orders LDS only (a workgroup fence on the local address space),
// so the loads in flight stay in flight across it.  Rows are padded by 16
// bytes: the 16 rows of a fragment read then start in 16 different groups of
// four banks.
#pragma once

#include "mie_common.h"

namespace mie {
namespace gemm {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Orders this workgroup's LDS accesses; global loads may stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <typename T>
__device__ __forceinline__ f32x4 mfma_fragment(u32x4 a, u32x4 b, f32x4 c);
template <>
__device__ __forceinline__ f32x4 mfma_fragment<float>(u32x4 a, u32x4 b, f32x4 c) {
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.x), __uint_as_float(b.x), c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.y), __uint_as_float(b.y), c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.z), __uint_as_float(b.z), c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.w), __uint_as_float(b.w), c, 0, 0, 0);
}
template <>
__device__ __forceinline__ f32x4 mfma_fragment<uint16_t>(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                 0, 0);
}

template <typename T, int BM_, int BN_, int KB_, int WM_, int WN_>
struct Tile {
  static constexpr int BM = BM_, BN = BN_, KB = KB_, WM = WM_, WN = WN_;
  static constexpr int MT = BM / WM / 16, NT = BN / WN / 16;
  static constexpr int kStride = KB + 16;         // LDS bytes per row
  static constexpr int kVec = KB / 16;            // 16-byte vectors per row and step
  static constexpr int kRows = 256 / kVec;        // rows one pass of the workgroup loads
  static constexpr int kA = BM / kRows, kW = BN / kRows;  // passes over the A and W rows
  static constexpr int kBuffer = (BM + BN) * kStride;
  static constexpr int kLds = 2 * kBuffer;  // bytes of LDS
  static_assert(WM * WN == 4 && MT >= 1 && NT >= 1 && kA >= 1 && kW >= 1, "tile does not fit four waves");
  static_assert(BM % kRows == 0 && BN % kRows == 0 && KB % 64 == 0, "tile does not divide into passes");

  // acc[n][m] += the tile's product over row bytes [k0, k1): a_row(r) and
  // w_row(r) give the byte address of tile row r's first element (any valid
  // row past the edge: its results are dropped by the caller).  k0 and k1 are
  // multiples of 16; lds holds kLds bytes, free to overwrite (the caller has
  // a barrier behind its last use).  On return no wave still reads it.
  template <typename ARow, typename WRow>
  static __device__ __forceinline__ void run(char* lds, ARow a_row, WRow w_row, int k0, int k1,
                                             f32x4 (&acc)[NT][MT]) {
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WM, wn = wave / WM;
    const int vr = tid / kVec, vc = (tid % kVec) * 16;
    const char* ap[kA];
    const char* wp[kW];
#pragma unroll
    for (int i = 0; i < kA; ++i) ap[i] = a_row(vr + i * kRows) + vc;
#pragma unroll
    for (int i = 0; i < kW; ++i) wp[i] = w_row(vr + i * kRows) + vc;
    u32x4 av[kA], wv[kW];
    // Loads are unconditional (a vector past k1 reads the row's first one and
    // is zeroed when stored), so a step's loads all go out together.
    auto load = [&](int k) {
      const int off = k + vc < k1 ? k : -vc;
#pragma unroll
      for (int i = 0; i < kW; ++i) wv[i] = *reinterpret_cast<const u32x4*>(wp[i] + off);
#pragma unroll
      for (int i = 0; i < kA; ++i) av[i] = *reinterpret_cast<const u32x4*>(ap[i] + off);
    };
    auto store = [&](int k, char* buf) {
      const bool live = k + vc < k1;
      const u32x4 zero = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int i = 0; i < kA; ++i)
        *reinterpret_cast<u32x4*>(buf + (vr + i * kRows) * kStride + vc) = live ? av[i] : zero;
#pragma unroll
      for (int i = 0; i < kW; ++i)
        *reinterpret_cast<u32x4*>(buf + (BM + vr + i * kRows) * kStride + vc) = live ? wv[i] : zero;
    };
    const int frag = (lane & 15) * kStride + (lane >> 4) * 16;
    const int a_frag = wm * MT * 16 * kStride + frag;
    const int w_frag = (BM + wn * NT * 16) * kStride + frag;
    auto multiply = [&](const char* buf) {
#pragma unroll
      for (int c = 0; c < KB; c += 64) {
        u32x4 a[MT], w[NT];
#pragma unroll
        for (int m = 0; m < MT; ++m) a[m] = *reinterpret_cast<const u32x4*>(buf + a_frag + m * 16 * kStride + c);
#pragma unroll
        for (int n = 0; n < NT; ++n) w[n] = *reinterpret_cast<const u32x4*>(buf + w_frag + n * 16 * kStride + c);
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
          for (int m = 0; m < MT; ++m) acc[n][m] = mfma_fragment<T>(w[n], a[m], acc[n][m]);
      }
    };
    if (k0 >= k1) return;
    load(k0);
    store(k0, lds);
    if (k0 + KB < k1) load(k0 + KB);
    lds_barrier();
    int cur = 0;
    for (int k = k0; k < k1; k += KB) {
      multiply(lds + cur);
      cur = kBuffer - cur;
      if (k + KB < k1) {
        store(k + KB, lds + cur);
        if (k + 2 * KB < k1) load(k + 2 * KB);
      }
      lds_barrier();
    }
  }

  // Tile row and first column of the four results a lane holds in acc[n][m].
  static __device__ __forceinline__ int row(int m) {
    return ((__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) % WM) * MT + m) * 16 + (threadIdx.x & 15);
  }
  static __device__ __forceinline__ int col(int n) {
    return ((__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) / WM) * NT + n) * 16 + ((threadIdx.x & 63) >> 4) * 4;
  }
};

}  // namespace gemm
}  // namespace mie
