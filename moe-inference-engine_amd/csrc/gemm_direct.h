// A small tile of C = A . W^T without LDS staging: 16 MT rows x 16 NT columns per
// workgroup of four waves, the waves splitting K.  For few rows, where a
// launch is bound by how many bytes of W it has in flight and by its memory
// rounds: each wave's fragments go from memory to the matrix cores' operands
// (16 rows x 64 bytes per load), two windows of KF of them in flight, no
// barrier until the waves' sums meet in LDS at the end.  Operand layout as in
// gemm_tile.h (W first, so a lane ends with four consecutive columns).
#pragma once

#include "gemm_tile.h"

namespace mie {
namespace gemm {

template <typename T, int NT_, int KF_>
struct Direct {
  static constexpr int NT = NT_, KF = KF_;
  static constexpr int BN = 16 * NT;
  static constexpr int kWindow = 4 * KF * 64;  // bytes of K per window, all four waves
  template <int MT> static constexpr int kLds = 4 * MT * NT * 64 * 16;  // every wave's sums

  template <int N> struct Set {
    u32x4 v[N][KF];
  };

  // Byte offset of this lane's piece of fragment u of the window at `k`.
  static __device__ __forceinline__ int piece(int k, int u) {
    return k + (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * KF + u) * 64 + ((threadIdx.x & 63) >> 4) * 16;
  }

  // One window of N operand blocks' fragments; row[n] is the address of this
  // lane's row (16 n + lane % 16).  Loads are unconditional: pieces past k1
  // read the row's piece at k0 and are zeroed in multiply().
  template <int N>
  static __device__ __forceinline__ void load(Set<N>& s, const char* const (&row)[N], int k, int k0, int k1) {
#pragma unroll
    for (int u = 0; u < KF; ++u) {
      const int off = piece(k, u);
#pragma unroll
      for (int n = 0; n < N; ++n) s.v[n][u] = *reinterpret_cast<const u32x4*>(row[n] + (off < k1 ? off : k0));
    }
  }
  template <int MT>
  static __device__ __forceinline__ void multiply(const Set<NT>& ws, const Set<MT>& as, int k, int k1,
                                                  f32x4 (&acc)[NT][MT]) {
    const bool whole = k + kWindow <= k1;
#pragma unroll
    for (int u = 0; u < KF; ++u) {
      u32x4 w[NT], a[MT];
#pragma unroll
      for (int n = 0; n < NT; ++n) w[n] = ws.v[n][u];
#pragma unroll
      for (int m = 0; m < MT; ++m) a[m] = as.v[m][u];
      if (!whole) {
        const bool live = piece(k, u) < k1;
        const u32x4 zero = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int n = 0; n < NT; ++n) w[n] = live ? w[n] : zero;
#pragma unroll
        for (int m = 0; m < MT; ++m) a[m] = live ? a[m] : zero;
      }
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[n][m] = mfma_fragment<T>(w[n], a[m], acc[n][m]);
    }
  }

  // The first two windows' W fragments.
  static __device__ __forceinline__ void prefetch(Set<NT> (&ws)[2], const char* const (&w)[NT], int k0, int k1) {
    load<NT>(ws[0], w, k0, k0, k1);
    if (k0 + kWindow < k1) load<NT>(ws[1], w, k0 + kWindow, k0, k1);
  }

  // The product of MT blocks of rows over row bytes [k0, k1): `ws` holds the
  // first two windows' W fragments (prefetch), already in flight.  The
  // waves' sums meet in lds (kLds<MT> bytes, free to overwrite) and the blocks
  // are dealt out: store(n, m, sum) runs for each block on one wave, with four
  // consecutive columns 16 n + 4 (lane / 16) .. of row 16 m + lane % 16 per lane.
  template <int MT, typename Store>
  static __device__ __forceinline__ void run(char* lds, Set<NT> (&ws)[2], const char* const (&a)[MT],
                                             const char* const (&w)[NT], int k0, int k1, Store store) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    f32x4 acc[NT][MT];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    Set<MT> a0, a1;
    load<MT>(a0, a, k0, k0, k1);
    if (k0 + kWindow < k1) load<MT>(a1, a, k0 + kWindow, k0, k1);
    for (int k = k0; k < k1; k += 2 * kWindow) {
      multiply<MT>(ws[0], a0, k, k1, acc);
      if (k + 2 * kWindow < k1) {
        load<NT>(ws[0], w, k + 2 * kWindow, k0, k1);
        load<MT>(a0, a, k + 2 * kWindow, k0, k1);
      }
      if (k + kWindow < k1) {
        multiply<MT>(ws[1], a1, k + kWindow, k1, acc);
        if (k + 3 * kWindow < k1) {
          load<NT>(ws[1], w, k + 3 * kWindow, k0, k1);
          load<MT>(a1, a, k + 3 * kWindow, k0, k1);
        }
      }
    }
    f32x4* sums = reinterpret_cast<f32x4*>(lds) + lane;
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int m = 0; m < MT; ++m) sums[(wave * NT * MT + n * MT + m) * 64] = acc[n][m];
    lds_barrier();
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        if ((n * MT + m) % 4 != wave) continue;
        f32x4 sum = sums[(n * MT + m) * 64];
#pragma unroll
        for (int v = 1; v < 4; ++v) sum += sums[(v * NT * MT + n * MT + m) * 64];
        store(n, m, sum);
      }
  }
};

}  // namespace gemm
}  // namespace mie
