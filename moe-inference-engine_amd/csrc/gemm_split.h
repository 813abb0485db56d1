// A workgroup's tile of C = A . W^T for float32 operands on the bfloat16 matrix
// cores, at float32's precision.
//
// A float32 is the exact sum of three bfloat16 values: its upper half, the
// upper half of what is left, and the rest (8 + 8 + 8 bits).  Products of
// bfloat16 values are exact in float32.  Six of the nine partial products are
// kept.  The other three are left out, always toward zero: together below 2^-21
// of the product (largest seen 4.0e-7, root mean square 5.5e-8, mean 3.8e-8),
// where the float32 instruction keeps a product whole.  The product of the
// upper halves has an accumulator of its own, so the small ones are not rounded
// to its size at every step, which more than makes up for it in sums of 16
// products and more; callers give shorter ones to float32 instructions.  Error
// against float64, N(0, 1) rows times U(-1, 1) rows, relative 2-norm: K 768
// 1.7e-7 (float32 instruction 5.0e-7), K 3072 3.4e-7 (9.8e-7).  Sums of bfloat16
// parts for float32 products: G. Henry, P. T. P. Tang, A. Heinecke, "Leveraging
// the bfloat16 Artificial Intelligence Datatype For Higher-Precision
// Computations", 2019.
//
// Low parts of very small values would underflow, and an infinity has no
// parts: results of an A or W row whose largest value is outside [2^-50, 2^50]
// are computed again by the float32 instruction, so a result depends on its
// own two rows only.  NaNs reach the results either way.
//
// 256 threads, four waves side by side over the columns: 16 MT rows x 64 NT
// columns.  A wave's W rows are its own, so their fragments go from memory to
// registers and are split there; A is split once on its way into LDS (two
// buffers, the three parts of a row side by side) and read by all.  K goes in
// steps of 32, the loads two steps ahead.  The three parts of a step need six
// v_mfma_f32_16x16x32_bf16 where float32 takes eight instructions of twice the
// time, and about 6.5 vector instructions per value for the split, which share
// the issue with them: measured, a step takes about 410 + 120 MT NT + 30 (2 MT
// + 8 NT) cycles, so larger tiles pay.  MI355X, 2048 x 3072 x 768, 64 x 128
// tile: 60 us (160 TFLOP/s; 95 us with float32's instruction).
#pragma once

#include <type_traits>

#include "gemm_tile.h"

namespace mie {
namespace gemm {

template <int MT_, int NT_>
struct SplitTile {
  static constexpr int MT = MT_, NT = NT_, BM = 16 * MT, BN = 64 * NT, KB = 128;
  static constexpr int kStride = 3 * KB / 2 + 16;  // 208 bytes: 16 rows start in different groups of four banks
  static constexpr int kA = (BM + 31) / 32;        // passes over the A rows, 32 rows of 8 vectors each
  static constexpr int kBuffer = BM * kStride;
  static constexpr int kLds = 2 * kBuffer;  // bytes of LDS, the rows' largest values among them
  static_assert(kLds >= (BM + BN) * 4, "LDS");
  // Workgroups per CU by registers (waves per SIMD, for __launch_bounds__).
  static constexpr int kWaves = MT * NT <= 4 ? 3 : 2;

  typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
  struct Parts {
    u32x2 p[3];  // four values' upper, middle and lower parts
  };
  struct Raw {
    u32x4 a[kA], w[NT][2];
  };

  static __device__ __forceinline__ Parts split(u32x4 v, float& largest) {
    float x[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = __uint_as_float(v[i]);
    largest = fmaxf(fmaxf(largest, fabsf(x[0])), fabsf(x[1]));
    largest = fmaxf(fmaxf(largest, fabsf(x[2])), fabsf(x[3]));
    Parts r;
#pragma unroll
    for (int part = 0; part < 3; ++part) {
      uint32_t b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) b[i] = __float_as_uint(x[i]);
      r.p[part] = u32x2{__builtin_amdgcn_perm(b[1], b[0], 0x07060302u), __builtin_amdgcn_perm(b[3], b[2], 0x07060302u)};
      if (part < 2) {
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] -= __uint_as_float(b[i] & 0xffff0000u);
      }
    }
    return r;
  }

  // As Tile::run (a_row, w_row, k0, k1 and lds too), over the tile's first 16 ML
  // rows; acc holds zeros.  row() and col() say which results a lane holds.
  template <int ML = MT, typename ARow, typename WRow>
  static __device__ __forceinline__ void run(char* lds, ARow a_row, WRow w_row, int k0, int k1, f32x4 (&acc)[NT][MT]) {
    if (k0 >= k1) return;
    constexpr int kPasses = (16 * ML + 31) / 32;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = lane & 15, g = lane >> 4;
    const int vr = threadIdx.x / 8, vc = threadIdx.x % 8 * 16;
    const char* ap[kPasses];
    const char* wp[NT];
#pragma unroll
    for (int j = 0; j < kPasses; ++j) ap[j] = a_row(min(vr + j * 32, 16 * ML - 1)) + vc;
#pragma unroll
    for (int n = 0; n < NT; ++n) wp[n] = w_row((wave * NT + n) * 16 + i) + g * 16;
    // WHOLE: K is whole steps; loads past the end read the last step again and
    // are not used.  Otherwise a vector past the end reads the row's first one
    // and is zeroed when split.
    auto load = [&](auto whole, Raw& r, int k) {
      const int last = decltype(whole)::value ? min(k, k1 - KB) : k;
      const int ao = decltype(whole)::value || k + vc < k1 ? last : -vc;
#pragma unroll
      for (int j = 0; j < kPasses; ++j) r.a[j] = *reinterpret_cast<const u32x4*>(ap[j] + ao);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int wo = decltype(whole)::value || k + u * 64 + g * 16 < k1 ? last + u * 64 : -g * 16;
#pragma unroll
        for (int n = 0; n < NT; ++n) r.w[n][u] = *reinterpret_cast<const u32x4*>(wp[n] + wo);
      }
    };
    // A lane's W fragment is its row's vectors g and 4 + g of a step; A's are
    // put in the same order.
    const int a_put = vr * kStride + (vc & 63) + vc / 64 * 8;
    float a_max[kPasses], w_max[NT];  // of this lane's vectors of each row
#pragma unroll
    for (int j = 0; j < kPasses; ++j) a_max[j] = 0.f;
#pragma unroll
    for (int n = 0; n < NT; ++n) w_max[n] = 0.f;
    auto stage = [&](auto whole, Raw& r, int k, char* buf, u32x4 (&w)[NT][3]) {
      if constexpr (!decltype(whole)::value) {
        const u32x4 zero = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int j = 0; j < kPasses; ++j) r.a[j] = k + vc < k1 ? r.a[j] : zero;
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
          for (int u = 0; u < 2; ++u) r.w[n][u] = k + u * 64 + g * 16 < k1 ? r.w[n][u] : zero;
      }
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const Parts x = split(r.w[n][0], w_max[n]), y = split(r.w[n][1], w_max[n]);
#pragma unroll
        for (int p = 0; p < 3; ++p) w[n][p] = u32x4{x.p[p].x, x.p[p].y, y.p[p].x, y.p[p].y};
      }
#pragma unroll
      for (int j = 0; j < kPasses; ++j) {
        if (j * 32 + 32 > 16 * ML && wave >= 2) break;  // the last pass has 16 rows: waves 0 and 1
        const Parts x = split(r.a[j], a_max[j]);
#pragma unroll
        for (int p = 0; p < 3; ++p) *reinterpret_cast<u32x2*>(buf + a_put + j * 32 * kStride + p * 64) = x.p[p];
      }
    };
    const int frag = i * kStride + g * 16;
    f32x4 rest[NT][ML];  // every product but upper x upper
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int m = 0; m < ML; ++m) rest[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const char* buf, const u32x4 (&w)[NT][3]) {
      u32x4 a[3][ML];
#pragma unroll
      for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int m = 0; m < ML; ++m) a[p][m] = *reinterpret_cast<const u32x4*>(buf + frag + m * 16 * kStride + p * 64);
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < ML; ++m) acc[n][m] = mfma_fragment<uint16_t>(w[n][0], a[0][m], acc[n][m]);
      constexpr int kWPart[5] = {1, 2, 0, 1, 0}, kAPart[5] = {0, 0, 1, 1, 2};
#pragma unroll
      for (int q = 0; q < 5; ++q)
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
          for (int m = 0; m < ML; ++m) rest[n][m] = mfma_fragment<uint16_t>(w[n][kWPart[q]], a[kAPart[q]][m], rest[n][m]);
    };
    Raw raw[2];
    u32x4 wf[2][NT][3];
    auto loop = [&](auto whole) {
      load(whole, raw[0], k0);
      load(whole, raw[1], k0 + KB);
      stage(whole, raw[0], k0, lds, wf[0]);
      load(whole, raw[0], k0 + 2 * KB);
      lds_barrier();
      // No branch in a step: the last ones stage what nothing reads.
      auto step = [&](int k, Raw& next, const char* buf, char* other, u32x4 (&w)[NT][3], u32x4 (&wn)[NT][3]) {
        multiply(buf, w);
        stage(whole, next, k + KB, other, wn);
        load(whole, next, k + 3 * KB);
        lds_barrier();
      };
      for (int k = k0;;) {
        step(k, raw[1], lds, lds + kBuffer, wf[0], wf[1]);
        if ((k += KB) >= k1) break;
        step(k, raw[0], lds + kBuffer, lds, wf[1], wf[0]);
        if ((k += KB) >= k1) break;
      }
    };
    if ((k1 - k0) % KB == 0) {
      loop(std::true_type{});
    } else {
      loop(std::false_type{});
    }
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int m = 0; m < ML; ++m) acc[n][m] += rest[n][m];
    // Rows the split does not hold: each row's largest value, through LDS (the
    // last step's buffers are read).
    float* a_row_max = reinterpret_cast<float*>(lds);
    float* w_row_max = a_row_max + BM;
#pragma unroll
    for (int j = 0; j < kPasses; ++j) {
#pragma unroll
      for (int off = 4; off >= 1; off >>= 1) a_max[j] = fmaxf(a_max[j], __shfl_xor(a_max[j], off));
      if ((lane & 7) == 0 && vr + j * 32 < 16 * ML) a_row_max[vr + j * 32] = a_max[j];
    }
#pragma unroll
    for (int n = 0; n < NT; ++n) {
#pragma unroll
      for (int off = 32; off >= 16; off >>= 1) w_max[n] = fmaxf(w_max[n], __shfl_xor(w_max[n], off));
      if (g == 0) w_row_max[(wave * NT + n) * 16 + i] = w_max[n];
    }
    lds_barrier();
    auto outside = [](float x) { return x > 0x1p50f || (x > 0.f && x < 0x1p-50f); };
    bool bad_a[ML], bad_w[NT][4], any = false;
#pragma unroll
    for (int m = 0; m < ML; ++m) any |= bad_a[m] = outside(a_row_max[row(m)]);
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) any |= bad_w[n][r] = outside(w_row_max[col(n) + r]);
    lds_barrier();
    if (__any(any)) {
      f32x4 again[NT][ML];
      plain<ML>(a_row, w_row, k0, k1, again);
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < ML; ++m)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[n][m][r] = bad_a[m] || bad_w[n][r] ? again[n][m][r] : acc[n][m][r];
    }
  }

  // The product by the float32 instruction, straight from memory (rare).
  template <int ML, typename ARow, typename WRow>
  static __device__ __forceinline__ void plain(ARow a_row, WRow w_row, int k0, int k1, f32x4 (&acc)[NT][ML]) {
    const int i = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
    const u32x4 zero = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int m = 0; m < ML; ++m) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int k = k0; k < k1; k += 64) {
      const bool live = k + g * 16 < k1;
      const int off = live ? k + g * 16 : 0;
      u32x4 w[NT];
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        w[n] = *reinterpret_cast<const u32x4*>(w_row(col(n) - g * 4 + i) + off);
        w[n] = live ? w[n] : zero;
      }
#pragma unroll
      for (int m = 0; m < ML; ++m) {
        u32x4 a = *reinterpret_cast<const u32x4*>(a_row(row(m)) + off);
        a = live ? a : zero;
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[n][m] = mfma_fragment<float>(w[n], a, acc[n][m]);
      }
    }
  }

  // Tile row and first column of the four results a lane holds in acc[n][m].
  static __device__ __forceinline__ int row(int m) { return m * 16 + (threadIdx.x & 15); }
  static __device__ __forceinline__ int col(int n) {
    return (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * NT + n) * 16 + ((threadIdx.x & 63) >> 4) * 4;
  }
};

}  // namespace gemm
}  // namespace mie
