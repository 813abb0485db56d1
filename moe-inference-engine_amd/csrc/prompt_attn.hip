// The attention half of a decoder block over a prompt at position 0 (float32
// or bfloat16): LayerNorm, QKV projection with K and V stored into the paged
// pools, causal attention over the fresh K and V, output projection and
// residual.
//
// Replaces CachedAttention.forward at position 0 (reference model.py:226-269,
// with cache.write :167-184) and, with the norm and the residual, the block's
// x + attention(attn_norm(x)) (:495).  Rounding points are the PyTorch path's:
// every product, softmax and sum in float32; in bfloat16 the norm's output,
// each projection's output (sum plus bias, once), the attention's output and
// the residual sum are rounded.  The probabilities stay float32 up to the
// product with V (float32 MFMA; for bfloat16 V they go in as the sum of two
// bfloat16 values, 16 bits of significand).
//
// Launches: norm (block form), QKV, attention, output projection.  Few tokens
// are bound by the launches and the weights, many by the matrix cores.  A
// layer on MI355X, 12 heads x 64, against library products, PyTorch's
// attention and the append launch: 1000 tokens float32 126 -> 77 us, 333
// tokens bfloat16 85 -> 25 us; with the MoE half, 62 tokens float32 through 12
// blocks and the head 4.1 -> 0.95 ms.
//
// Attention.  One workgroup per (head, 16 queries); its four waves take
// every fourth block of 32 keys and merge their softmax states in LDS once.
// Nothing else is shared, so there is no barrier in the loop.  Scores are
// computed transposed, S^T = K Q^T, so a lane holds four consecutive keys of
// one query - exactly the second operand of O^T = V^T P^T: the probabilities
// never leave their registers.  V is read in rows: lane i's vector holds dims
// 4 i .. 4 i + 3, operand rows i of four 16-row blocks (block j: dims 4 i + j),
// so a query's results end as 16 consecutive dims per lane.
#include <math.h>

#include <algorithm>

#include "gemm_direct.h"
#include "gemm_split.h"
#include "gemm_tile.h"
#include "mie_common.h"
#include "row_norm.h"

namespace {

using mie::Mem;
using mie::gemm::Direct;
using mie::gemm::f32x4;
using mie::gemm::Tile;
using mie::gemm::u32x4;

constexpr float kLog2e = 1.4426950408889634f;
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

struct NormArgs {
  const char* x;  // T [rows, dim]
  const char* w;  // T [dim]
  const char* b;  // T [dim] or NULL
  char* out;      // T [rows, dim]
  int32_t rows, dim;
  float eps;
};

// grid = ceil(rows / 4): one wave per row (float32, biased variance), the row
// and the parameters in registers (one memory round), P pieces of 256 elements.
template <typename T, int P>
__global__ __launch_bounds__(256) void prompt_norm_kernel(NormArgs a) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= a.rows) return;
  const T* x = reinterpret_cast<const T*>(a.x) + static_cast<int64_t>(row) * a.dim;
  mie::norm_row<T, P>(x, reinterpret_cast<const T*>(a.w), reinterpret_cast<const T*>(a.b),
                      reinterpret_cast<T*>(a.out) + static_cast<int64_t>(row) * a.dim, a.dim, a.eps, lane);
}

struct LinearArgs {
  const char* x;         // T [rows, k]
  const char* w;         // T [n, k]
  const char* bias;      // T [n] or NULL
  const char* residual;  // T [rows, n] or NULL
  char* out;             // T [rows, n]
  int32_t rows, n, k;
  // QKV form (pool K and V; NULL for a plain product): columns [dim, 3 dim)
  // also go to the pools through the block table, row r as token r.
  char* k_pool;
  char* v_pool;
  int64_t sblk, shead;  // elements
  int32_t num_blocks, dim, head_dim;
  const int32_t* table;
  mie::FastDiv block, head;  // block size, head_dim
};

// The pool block of row r (token r) in the QKV form; -1 when it is not stored.
__device__ __forceinline__ int32_t block_of(const LinearArgs& a, int r) {
  if (!a.k_pool) return -1;
  const int32_t id = a.table[a.block.div(min(r, a.rows - 1))];
  return id < a.num_blocks ? id : -1;
}

// Stores four consecutive results of row r, columns c .. c + 3 (before bias);
// blk is block_of(r).
template <typename T>
__device__ __forceinline__ void store_linear(const LinearArgs& a, int r, int c, f32x4 sum, f32x4 bias, int32_t blk) {
  f32x4 v = Mem<T>::R4(sum + bias);
  const int64_t at = static_cast<int64_t>(r) * a.n + c;
  if (a.residual) v = Mem<T>::load4(reinterpret_cast<const T*>(a.residual) + at) + v;
  Mem<T>::put4(reinterpret_cast<T*>(a.out) + at, v);
  if (blk >= 0 && c >= a.dim) {
    const int d = c < 2 * a.dim ? c - a.dim : c - 2 * a.dim;
    char* pool = c < 2 * a.dim ? a.k_pool : a.v_pool;
    const uint32_t h = a.head.div(d), slot = r - a.block.div(r) * a.block.d;
    Mem<T>::put4(reinterpret_cast<T*>(pool) + blk * a.sblk + h * a.shead + static_cast<int64_t>(slot) * a.head_dim +
                     (d - h * a.head_dim),
                 v);
  }
}

// Bias of columns c .. c + 3 (zeros without a bias or past the edge).
template <typename T>
__device__ __forceinline__ f32x4 bias_of(const LinearArgs& a, int c) {
  if (!a.bias || c >= a.n) return f32x4{0.f, 0.f, 0.f, 0.f};
  return Mem<T>::load4(reinterpret_cast<const T*>(a.bias) + c);
}

template <typename T, typename Tile>
__device__ __forceinline__ void linear_tile(const LinearArgs& a, char* lds) {
  const int n0 = blockIdx.x * Tile::BN, m0 = blockIdx.y * Tile::BM;
  const int64_t row_bytes = static_cast<int64_t>(a.k) * sizeof(T);
  f32x4 acc[Tile::NT][Tile::MT];
#pragma unroll
  for (int n = 0; n < Tile::NT; ++n)
#pragma unroll
    for (int m = 0; m < Tile::MT; ++m) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  Tile::run(
      lds, [&](int i) { return a.x + min(m0 + i, a.rows - 1) * row_bytes; },
      [&](int i) { return a.w + min(n0 + i, a.n - 1) * row_bytes; }, 0, static_cast<int>(row_bytes), acc);
  int32_t blk[Tile::MT];
#pragma unroll
  for (int m = 0; m < Tile::MT; ++m) blk[m] = block_of(a, m0 + Tile::row(m));
#pragma unroll
  for (int n = 0; n < Tile::NT; ++n) {
    const int c = n0 + Tile::col(n);
    if (c >= a.n) continue;  // n is a multiple of 4
    const f32x4 b = bias_of<T>(a, c);
#pragma unroll
    for (int m = 0; m < Tile::MT; ++m) {
      const int r = m0 + Tile::row(m);
      if (r < a.rows) store_linear<T>(a, r, c, acc[n][m], b, blk[m]);
    }
  }
}

// grid = (ceil(n / BN), ceil(rows / BM)).
template <typename T, typename Tile>
__global__ __launch_bounds__(256) void prompt_linear_kernel(LinearArgs a) {
  __shared__ __align__(16) char lds[Tile::kLds];
  linear_tile<T, Tile>(a, lds);
}

// The same on gemm_split.h's tiles.
template <typename Tile>
__global__ __launch_bounds__(256, Tile::kWaves) void prompt_linear_split_kernel(LinearArgs a) {
  __shared__ __align__(16) char lds[Tile::kLds];
  linear_tile<float, Tile>(a, lds);
}

// grid = (ceil(n / BN), ceil(rows / (16 MT))): few rows.
template <typename T, typename Tile, int MT>
__global__ __launch_bounds__(256, 2) void prompt_linear_direct_kernel(LinearArgs a) {
  __shared__ __align__(16) char lds[Tile::template kLds<MT>];
  const int n0 = blockIdx.x * Tile::BN, m0 = blockIdx.y * MT * 16;
  const int row_bytes = a.k * static_cast<int>(sizeof(T));
  const int i = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
  const char *ap[MT], *wp[Tile::NT];
#pragma unroll
  for (int n = 0; n < Tile::NT; ++n) wp[n] = a.w + static_cast<int64_t>(min(n0 + n * 16 + i, a.n - 1)) * row_bytes;
#pragma unroll
  for (int m = 0; m < MT; ++m) ap[m] = a.x + static_cast<int64_t>(min(m0 + m * 16 + i, a.rows - 1)) * row_bytes;
  typename Tile::template Set<Tile::NT> ws[2];
  Tile::prefetch(ws, wp, 0, row_bytes);
  // What the epilogue needs goes out with the operands.
  f32x4 bias[Tile::NT];
  int32_t blk[MT];
#pragma unroll
  for (int n = 0; n < Tile::NT; ++n) bias[n] = bias_of<T>(a, n0 + n * 16 + g * 4);
#pragma unroll
  for (int m = 0; m < MT; ++m) blk[m] = block_of(a, m0 + m * 16 + i);
  Tile::template run<MT>(lds, ws, ap, wp, 0, row_bytes, [&](int n, int m, f32x4 sum) {
    const int c = n0 + n * 16 + g * 4, r = m0 + m * 16 + i;
    if (c < a.n && r < a.rows) store_linear<T>(a, r, c, sum, bias[n], blk[m]);  // n is a multiple of 4
  });
}

struct AttnArgs {
  const char* qkv;  // T [rows, 3 dim]
  char* out;        // T [rows, dim]
  int32_t rows, dim;
  float scale;  // 1 / sqrt(head_dim) * log2(e)
};

// x combined over the four 16-lane groups (lanes i, i + 16, i + 32, i + 48).
template <bool MAX>
__device__ __forceinline__ float across_groups(float x) {
  auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  const float u = __uint_as_float(a[0]), v = __uint_as_float(a[1]);
  x = MAX ? fmaxf(u, v) : u + v;
  a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  const float s = __uint_as_float(a[0]), t = __uint_as_float(a[1]);
  return MAX ? fmaxf(s, t) : s + t;
}

// V's operands of one 64- or 32-dim group for 32 keys, and their products.
// Lane (i, g): keys 16 t + 4 g + r (t < 2, r < 4), dims VEC i .. VEC i + VEC - 1.
template <typename T, int VEC> struct ValueGroup;
template <int VEC> struct ValueGroup<float, VEC> {
  typedef float vec __attribute__((ext_vector_type(VEC)));
  vec v[2][4];
  __device__ __forceinline__ void load(int t, int r, const float* p) { v[t][r] = *reinterpret_cast<const vec*>(p); }
  __device__ __forceinline__ void multiply(const float (&p)[2][4], f32x4* o) const {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int j = 0; j < VEC; ++j)
          o[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[t][r][j], p[t][r], o[j], 0, 0, 0);
  }
};
template <int VEC> struct ValueGroup<uint16_t, VEC> {
  uint32_t v[2][4][VEC / 2];
  __device__ __forceinline__ void load(int t, int r, const uint16_t* p) {
    if constexpr (VEC == 4) {
      const u32x2 x = *reinterpret_cast<const u32x2*>(p);
      v[t][r][0] = x.x;
      v[t][r][1] = x.y;
    } else {
      v[t][r][0] = *reinterpret_cast<const uint32_t*>(p);
    }
  }
  // Contraction slot 4 t + r of lane group g is key 16 t + 4 g + r in both operands.
  __device__ __forceinline__ void multiply(const float (&p)[2][4], f32x4* o) const {
    u32x4 hi, lo;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float x = p[w / 2][2 * (w % 2)], y = p[w / 2][2 * (w % 2) + 1];
      hi[w] = mie::pack_bf16x2(x, y);
      lo[w] = mie::pack_bf16x2(x - mie::bf16_lo(hi[w]), y - mie::bf16_hi(hi[w]));
    }
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      u32x4 a;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const uint32_t x = v[w / 2][2 * (w % 2)][j / 2], y = v[w / 2][2 * (w % 2) + 1][j / 2];
        a[w] = __builtin_amdgcn_perm(y, x, j % 2 ? 0x07060302u : 0x05040100u);  // the two keys' dim j
      }
      o[j] = mie::gemm::mfma_fragment<uint16_t>(a, hi, o[j]);
      o[j] = mie::gemm::mfma_fragment<uint16_t>(a, lo, o[j]);
    }
  }
};

// grid = (heads, ceil(rows / 16)).  Sixteen queries per workgroup rather than
// 32: 1000 tokens x 12 heads make 756 workgroups instead of 384 (28.8 against
// 33.6 us, float32).  Tiles with more keys take longer, and that many
// workgroups are resident at once, dealt to the CUs in order: the first third
// of the grid takes the longest tiles, longest first, the second third the
// shortest, shortest first, so a CU's workgroups add up to about the same
// (27.4 against 30.0 us longest first throughout).
template <typename T, int D>
__global__ __launch_bounds__(256, D <= 64 ? 3 : 2) void prompt_attention_kernel(AttnArgs a) {
  constexpr int NCH = D * static_cast<int>(sizeof(T)) / 64;  // 64-byte pieces of a row
  constexpr int G4 = D / 64, G2 = D % 64 / 32;               // 64- and 32-dim groups
  constexpr int NO = G4 * 4 + G2 * 2;                        // 16-dim blocks
  constexpr int Q = 16;
  __shared__ float s_max[4][Q], s_sum[4][Q];
  __shared__ __align__(16) float s_out[4][Q][D + 4];
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = blockIdx.x;
  const int tiles = gridDim.y, third = (tiles + 2) / 3, y = blockIdx.y;
  const int q0 = (y < third ? tiles - 1 - y : y - third) * Q;
  const uint32_t stride = 3u * a.dim * sizeof(T);  // bytes
  const char* base = a.qkv + static_cast<int64_t>(h) * D * sizeof(T);
  const int last = a.rows - 1;
  const int keys = min(q0 + Q, a.rows);  // this tile's last query sees [0, keys)

  u32x4 q[NCH];
#pragma unroll
  for (int c = 0; c < NCH; ++c)
    q[c] = *reinterpret_cast<const u32x4*>(base + static_cast<int64_t>(min(q0 + i, last)) * stride + c * 64 + g * 16);
  f32x4 o[NO];
  float m = -INFINITY, l = 0.f;
#pragma unroll
  for (int n = 0; n < NO; ++n) o[n] = f32x4{0.f, 0.f, 0.f, 0.f};

  // A block's rows as offsets from its first one (a wave-uniform address): the
  // offsets change only where rows past the last token repeat it (masked).
  uint32_t k_off[2], v_off[2][4];
  auto offsets = [&](int top) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      k_off[t] = min(t * 16 + i, top) * stride + a.dim * sizeof(T) + g * 16;
#pragma unroll
      for (int r = 0; r < 4; ++r) v_off[t][r] = min(t * 16 + g * 4 + r, top) * stride + 2u * a.dim * sizeof(T);
    }
  };
  offsets(31);
  u32x4 kf[2][NCH];
  auto load_keys = [&](int k0) {
    const char* rows = base + static_cast<int64_t>(k0) * stride;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int c = 0; c < NCH; ++c) kf[t][c] = *reinterpret_cast<const u32x4*>(rows + k_off[t] + c * 64);
  };
  int k0 = wave * 32;
  if (k0 < keys) {
    if (k0 + 31 > last) offsets(last - k0);
    load_keys(k0);
  }
  for (; k0 < keys; k0 += 128) {
    ValueGroup<T, 4> v4[G4 > 0 ? G4 : 1];
    ValueGroup<T, 2> v2[G2 > 0 ? G2 : 1];
    const char* rows = base + static_cast<int64_t>(k0) * stride;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const T* v = reinterpret_cast<const T*>(rows + v_off[t][r]);
#pragma unroll
        for (int n = 0; n < G4; ++n) v4[n].load(t, r, v + n * 64 + i * 4);
#pragma unroll
        for (int n = 0; n < G2; ++n) v2[n].load(t, r, v + G4 * 64 + n * 32 + i * 2);
      }
    f32x4 s[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      s[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < NCH; ++c) s[u] = mie::gemm::mfma_fragment<T>(kf[u][c], q[c], s[u]);
    }
    if (k0 + 128 < keys) {
      if (k0 + 128 + 31 > last) offsets(last - k0 - 128);
      load_keys(k0 + 128);
    }
    float p[2][4];
    float top = m;
    const bool diagonal = k0 + 31 > q0;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        p[u][r] = s[u][r] * a.scale;
        if (diagonal) p[u][r] = k0 + u * 16 + g * 4 + r <= q0 + i ? p[u][r] : -INFINITY;
        top = fmaxf(top, p[u][r]);
      }
    top = across_groups<true>(top);
    const float ref = top == -INFINITY ? 0.f : top;
    if (__any(top > m)) {  // a later maximum: the sums so far shrink
      const float alpha = mie::fast_exp2(m - ref);
      l *= alpha;
#pragma unroll
      for (int n = 0; n < NO; ++n) o[n] *= alpha;
    }
    m = top;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        p[u][r] = mie::fast_exp2(p[u][r] - ref);
        l += p[u][r];
      }
#pragma unroll
    for (int n = 0; n < G4; ++n) v4[n].multiply(p, &o[n * 4]);
#pragma unroll
    for (int n = 0; n < G2; ++n) v2[n].multiply(p, &o[G4 * 4 + n * 2]);
  }

  // Merge the waves: the largest maximum, then the rescaled sums and outputs.
  l = across_groups<false>(l);
  if (g == 0) {
    s_max[wave][i] = m;
    s_sum[wave][i] = l;
  }
  __syncthreads();
  const float top = fmaxf(fmaxf(s_max[0][i], s_max[1][i]), fmaxf(s_max[2][i], s_max[3][i]));
  const float f = m == -INFINITY ? 0.f : mie::fast_exp2(m - top);
  // Lane (i, g) holds, of a 64-dim group, dims 16 g + 4 r + j in o[j][r]; of a
  // 32-dim group, dims 8 g + 2 r + j.
#pragma unroll
  for (int n = 0; n < G4; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const f32x4* u = &o[n * 4];
      *reinterpret_cast<f32x4*>(&s_out[wave][i][n * 64 + g * 16 + r * 4]) = f32x4{u[0][r], u[1][r], u[2][r], u[3][r]} * f;
    }
#pragma unroll
  for (int n = 0; n < G2; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const f32x4* u = &o[G4 * 4 + n * 2];
      float* dst = &s_out[wave][i][G4 * 64 + n * 32 + g * 8 + r * 2];
      dst[0] = u[0][r] * f;
      dst[1] = u[1][r] * f;
    }
  __syncthreads();
  for (int e = threadIdx.x; e < Q * (D / 4); e += 256) {
    const int row = e / (D / 4), c = e % (D / 4) * 4;
    if (q0 + row >= a.rows) break;
    float top = s_max[0][row];
#pragma unroll
    for (int w = 1; w < 4; ++w) top = fmaxf(top, s_max[w][row]);
    float sum = 0.f;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float mw = s_max[w][row];
      sum += mw == -INFINITY ? s_sum[w][row] : s_sum[w][row] * mie::fast_exp2(mw - top);
      v += *reinterpret_cast<const f32x4*>(&s_out[w][row][c]);
    }
    Mem<T>::put4(reinterpret_cast<T*>(a.out) + static_cast<int64_t>(q0 + row) * a.dim + h * D + c, v / sum);
  }
}

// ---- host ------------------------------------------------------------------

template <typename T, typename Tile>
void launch_tile(const LinearArgs& a, hipStream_t st) {
  prompt_linear_kernel<T, Tile>
      <<<dim3((a.n + Tile::BN - 1) / Tile::BN, (a.rows + Tile::BM - 1) / Tile::BM), 256, 0, st>>>(a);
}

template <int MT, int NT>
void launch_split(const LinearArgs& a, hipStream_t st) {
  using Tile = mie::gemm::SplitTile<MT, NT>;
  prompt_linear_split_kernel<Tile>
      <<<dim3((a.n + Tile::BN - 1) / Tile::BN, (a.rows + Tile::BM - 1) / Tile::BM), 256, 0, st>>>(a);
}

template <typename T, typename Tile, int MT>
void launch_direct(const LinearArgs& a, hipStream_t st) {
  prompt_linear_direct_kernel<T, Tile, MT>
      <<<dim3((a.n + Tile::BN - 1) / Tile::BN, (a.rows + 16 * MT - 1) / (16 * MT)), 256, 0, st>>>(a);
}

// Fewer than 128 tiles of 32 x 32 (few rows): direct tiles, the larger that
// still makes 128 workgroups.
//
// float32 beyond: the tile of the least estimated time.  A first round of
// workgroups over the 256 CUs takes `first`, each further one, overlapping,
// `more` (us at K 768 with the epilogue; every tile scales with K alike).  Split tiles
// win from about 320 x 2304 on; below, the small tile's rounds are few and the
// shortest (300 tokens: a layer in 35 us with it, 37 with 48x64 split).
//
// Measured on MI355X, us, products alone at K 768 (graph replays); float32:
//   rows x n (32x32 tiles)  direct 16x16  32x16  32x32 | split 32x64  48x64  64x64  64x128
//     32 x 2304    (72)         7.8   6.7    8.1        13.3   17.4   18.2   25.4
//    128 x 768     (96)         7.9   6.7    7.9        13.3   17.6   18.6   26.1
//     48 x 2304   (144)         8.0  10.0    8.1        13.3   17.5   18.4   25.9
//     62 x 2304   (144)        10.4  10.7    8.1        13.3   17.7   18.5   26.2
//     96 x 2304   (216)        13.5  11.0    8.2        13.4   17.7   18.7   26.3
//    300 x 768    (240)        13.2  10.9    8.2        13.4   17.7   18.7   26.2
//    333 x 2304   (792)        35.1  29.7   20.0        16.9   18.0   19.0   28.9
//   1000 x 768    (768)        34.0  26.9   16.5        17.1   18.5   19.5   26.7
//   1000 x 2304  (2304)        97.1  74.3   42.5        41.5   31.0   33.5   39.5
//   2048 x 3072  (6144)           -     -    103          86     77     63     60
// bfloat16, the last three columns 32x32, 32x64, 64x48 staged:
//     32 x 2304    (72)         4.7   4.2   |  4.5   6.0   7.2
//    128 x 768     (96)         4.7   4.2   |  4.5   6.0   7.2
//     62 x 2304   (144)         6.1   5.9   |  4.6   6.1   7.3
//    300 x 768    (240)         7.5   6.1   |  4.6   6.1   7.3
//    333 x 2304   (792)        19.0  16.7   |  8.2   7.9   9.2
//   1000 x 2304  (2304)        50.8  41.2   | 15.8  13.8  15.3
//
// bfloat16: the staged tile whose last round wastes least - rounds x tile area;
// on a tie the smallest tile while it makes at most 512 workgroups (more of
// them hide each other's waits), the largest beyond (less operand traffic).
template <typename T>
int32_t launch_linear(const LinearArgs& a, hipStream_t st) {
  auto tiles = [&](int bm, int bn) { return static_cast<int64_t>((a.rows + bm - 1) / bm) * ((a.n + bn - 1) / bn); };
  auto rounds = [&](int bm, int bn) { return (tiles(bm, bn) + 255) / 256; };
  if (tiles(32, 32) < 128) {
    if (tiles(32, 16) >= 128) {
      launch_direct<T, Direct<T, 1, 6>, 2>(a, st);
    } else {
      launch_direct<T, Direct<T, 1, 6>, 1>(a, st);
    }
  } else if constexpr (sizeof(T) == 4) {
    struct Form {
      int bm, bn;
      float first, more;
      void (*launch)(const LinearArgs&, hipStream_t);
    };
    static constexpr Form kForms[] = {
        {32, 32, 8.0f, 4.6f, launch_tile<T, Tile<T, 32, 32, 256, 2, 2>>},
        {32, 64, 13.9f, 6.6f, launch_split<2, 1>},
        {48, 64, 17.7f, 7.3f, launch_split<3, 1>},
        {64, 64, 18.5f, 8.6f, launch_split<4, 1>},
        {64, 128, 26.0f, 16.5f, launch_split<4, 2>},
    };
    const Form* best = nullptr;
    float least = 0.f;
    for (const Form& f : kForms) {
      const float cost = f.first + f.more * static_cast<float>(rounds(f.bm, f.bn) - 1);
      if (!best || cost < least) {
        best = &f;
        least = cost;
      }
    }
    best->launch(a, st);
  } else {
    auto cost = [&](int bm, int bn) { return rounds(bm, bn) * bm * bn; };
    const int64_t big = cost(64, 48), mid = cost(32, 64), small = cost(32, 32);
    if (tiles(32, 32) <= 512 ? small <= mid && small <= big : small < mid && small < big) {
      launch_tile<T, Tile<T, 32, 32, 256, 2, 2>>(a, st);
    } else if (mid < big) {
      launch_tile<T, Tile<T, 32, 64, 128, 2, 2>>(a, st);
    } else {
      launch_tile<T, Tile<T, 64, 48, 256, 4, 1>>(a, st);
    }
  }
  return mie::check_launch("prompt_linear_kernel");
}

template <typename T, int D>
void launch_heads(const AttnArgs& a, int32_t heads, hipStream_t st) {
  prompt_attention_kernel<T, D><<<dim3(heads, (a.rows + 15) / 16), 256, 0, st>>>(a);
}

template <typename T>
int32_t launch_attention(const AttnArgs& a, int32_t heads, int32_t head_dim, hipStream_t st) {
  switch (head_dim) {
    case 32: launch_heads<T, 32>(a, heads, st); break;
    case 64: launch_heads<T, 64>(a, heads, st); break;
    case 96: launch_heads<T, 96>(a, heads, st); break;
    default: launch_heads<T, 128>(a, heads, st); break;
  }
  return mie::check_launch("prompt_attention_kernel");
}

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

int64_t align256(int64_t n) { return (n + 255) / 256 * 256; }

bool built(int32_t heads, int32_t head_dim, int32_t dtype) {
  return (dtype == MIE_DTYPE_F32 || dtype == MIE_DTYPE_BF16) && heads > 0 && heads <= 65535 &&
         (head_dim == 32 || head_dim == 64 || head_dim == 96 || head_dim == 128) &&
         static_cast<int64_t>(heads) * head_dim <= 65536;
}

constexpr int32_t kMaxRows = 1 << 19;  // tiles of 16 rows stay below the grid's y limit

}  // namespace

extern "C" int32_t mie_attn_prefill_supported(int32_t num_heads, int32_t head_dim, int32_t dtype) {
  return built(num_heads, head_dim, dtype) ? 1 : 0;
}

extern "C" int64_t mie_attn_prefill_workspace(int32_t tokens, int32_t num_heads, int32_t head_dim, int32_t dtype) {
  if (tokens <= 0 || tokens > kMaxRows || !built(num_heads, head_dim, dtype)) return -MIE_ERR_INVALID;
  const int64_t row = static_cast<int64_t>(num_heads) * head_dim * mie::elt_size(dtype);
  return align256(3 * row * tokens) + 2 * align256(row * tokens);  // qkv; attention's output; the norm's
}

extern "C" int32_t mie_attn_prefill(const void* x, int32_t tokens, const void* ln_weight, const void* ln_bias,
                                    float ln_eps, const void* w_in, const void* b_in, const void* w_out,
                                    const void* b_out, const void* residual, void* out, void* k_pool, void* v_pool,
                                    int64_t pool_stride_block, int64_t pool_stride_head, int32_t num_blocks,
                                    const int32_t* block_table, int32_t block_table_len, int32_t num_heads,
                                    int32_t head_dim, int32_t block_size, float scale, void* workspace,
                                    int64_t workspace_bytes, int32_t dtype, void* stream) {
  mie::clear_error();
  if (!built(num_heads, head_dim, dtype))
    return mie::fail(MIE_ERR_UNSUPPORTED, "mie_attn_prefill: not built for %d heads x %d, dtype %d", num_heads,
                     head_dim, dtype);
  if (tokens <= 0 || tokens > kMaxRows || block_size <= 0 || num_blocks <= 0)
    return mie::fail(MIE_ERR_INVALID, "mie_attn_prefill: tokens=%d block_size=%d num_blocks=%d", tokens, block_size,
                     num_blocks);
  if (!x || !w_in || !w_out || !out || !k_pool || !v_pool || !block_table || !workspace)
    return mie::fail(MIE_ERR_INVALID, "mie_attn_prefill: null pointer");
  if (!ln_weight && ln_bias) return mie::fail(MIE_ERR_INVALID, "mie_attn_prefill: a norm bias needs a weight");
  if ((static_cast<int64_t>(tokens) + block_size - 1) / block_size > block_table_len)
    return mie::fail(MIE_ERR_INVALID, "mie_attn_prefill: %d tokens in blocks of %d pass the table's %d entries",
                     tokens, block_size, block_table_len);
  for (const void* p : {x, ln_weight, ln_bias, w_in, b_in, w_out, b_out, residual, static_cast<const void*>(out),
                        static_cast<const void*>(k_pool), static_cast<const void*>(v_pool),
                        static_cast<const void*>(workspace)})
    if (!aligned16(p)) return mie::fail(MIE_ERR_INVALID, "mie_attn_prefill: every pointer must be 16-byte aligned");
  if (pool_stride_block % 8 || pool_stride_head % 8)
    return mie::fail(MIE_ERR_INVALID, "mie_attn_prefill: pool strides must be multiples of 8 elements");
  const int64_t need = mie_attn_prefill_workspace(tokens, num_heads, head_dim, dtype);
  if (workspace_bytes < need)
    return mie::fail(MIE_ERR_WORKSPACE, "mie_attn_prefill: workspace of %lld bytes, needs %lld",
                     static_cast<long long>(workspace_bytes), static_cast<long long>(need));
  const hipStream_t st = static_cast<hipStream_t>(stream);
  const int32_t dim = num_heads * head_dim;
  const int64_t row = static_cast<int64_t>(dim) * mie::elt_size(dtype);
  char* qkv = static_cast<char*>(workspace);
  char* attn = qkv + align256(3 * row * tokens);
  char* normed = attn + align256(row * tokens);
  const bool f32 = dtype == MIE_DTYPE_F32;
  int32_t rc;
  const char* in = static_cast<const char*>(x);
  if (ln_weight) {
    const NormArgs n{in, static_cast<const char*>(ln_weight), static_cast<const char*>(ln_bias), normed, tokens, dim,
                     ln_eps};
    const int groups = (tokens + 3) / 4;
    if (dim <= 1024) {
      f32 ? prompt_norm_kernel<float, 4><<<groups, 256, 0, st>>>(n)
          : prompt_norm_kernel<uint16_t, 4><<<groups, 256, 0, st>>>(n);
    } else {
      f32 ? prompt_norm_kernel<float, 0><<<groups, 256, 0, st>>>(n)
          : prompt_norm_kernel<uint16_t, 0><<<groups, 256, 0, st>>>(n);
    }
    rc = mie::check_launch("prompt_norm_kernel");
    if (rc != MIE_OK) return rc;
    in = normed;
  }
  LinearArgs p{};
  p.x = in;
  p.w = static_cast<const char*>(w_in);
  p.bias = static_cast<const char*>(b_in);
  p.out = qkv;
  p.rows = tokens;
  p.n = 3 * dim;
  p.k = dim;
  p.k_pool = static_cast<char*>(k_pool);
  p.v_pool = static_cast<char*>(v_pool);
  p.sblk = pool_stride_block;
  p.shead = pool_stride_head;
  p.num_blocks = num_blocks;
  p.dim = dim;
  p.head_dim = head_dim;
  p.table = block_table;
  p.block = mie::FastDiv::make(block_size);
  p.head = mie::FastDiv::make(head_dim);
  rc = f32 ? launch_linear<float>(p, st) : launch_linear<uint16_t>(p, st);
  if (rc != MIE_OK) return rc;
  const AttnArgs t{qkv, attn, tokens, dim, scale * kLog2e};
  rc = f32 ? launch_attention<float>(t, num_heads, head_dim, st) : launch_attention<uint16_t>(t, num_heads, head_dim, st);
  if (rc != MIE_OK) return rc;
  LinearArgs y{};
  y.x = attn;
  y.w = static_cast<const char*>(w_out);
  y.bias = static_cast<const char*>(b_out);
  y.residual = static_cast<const char*>(residual);
  y.out = static_cast<char*>(out);
  y.rows = tokens;
  y.n = dim;
  y.k = dim;
  return f32 ? launch_linear<float>(y, st) : launch_linear<uint16_t>(y, st);
}
