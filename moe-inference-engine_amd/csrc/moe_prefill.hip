// Top-k mixture-of-experts over a prompt (float32 or bfloat16): routing, the
// selected experts' products and the weighted sum, with no host sync.
//
// Replaces, for several tokens, the reference's PyTorch MoE path
// (src/moe_engine/model.py:443-461), whose per-expert torch.where makes the
// host wait for the device once per expert:
//
//   logits = W_r x_t                     (float32)
//   ids    = the top_k experts by logit  (lower id on ties), w = their softmax
//   y_te   = W2_e GELU(W1_e x_t + b1_e) + b2_e         for the selected experts
//   out_t  = sum over them in increasing expert id, from 0, of round(w y)
//
// The block form adds what stands around it in a decoder block (model.py:496):
// x_t goes through a LayerNorm first and a residual is added to out_t.
//
// Rounding points are the one-token kernels' (moe_decode.hip): every sum is
// float32; in bfloat16 the norm's output, each Linear's output, GELU's, the route weight, the
// product and each partial sum are rounded, as the PyTorch path stores them.
//
// Four launches.
//   1. moe_prompt_route: two tokens per wave; the selected experts and weights
//      per token, and per expert a bit mask over the tokens (one byte per
//      workgroup of 8 tokens), so no workgroup needs another's counts.
//   2. moe_prompt_w1: h[slot] = GELU(W1_e x_t + b1_e).  Slots are the (expert,
//      token) pairs, expert by expert; each workgroup finds its expert and its
//      rows in the masks by popcounts.
//   3. moe_prompt_w2: partial sums of W2_e h over one K split.
//   4. moe_prompt_combine: the splits' sum, bias, weight and expert-order sum.
// The work follows the routing: top_k / E of what running every expert on
// every token takes, at any skew.  Row tiles (many rows per expert) do not read
// an expert without tokens; the few-rows form has the first two windows (2048
// bytes) of every expert's rows of W1, and of its share of W2's, in flight
// before the routing is known.
//
// Bounds: at few tokens the experts' bytes (768 x 2048 x 8 float32: 101 MB),
// at many the matrix cores (float32 instructions: 153 TFLOP/s; the split form
// also by the vector instructions that make the parts).  A whole layer on MI355X,
// 8 experts, top-2, before (dense-masked library products up to 512 float32
// tokens, the per-expert PyTorch path otherwise) and with these launches:
// 32 tokens, FFN 2048, float32: 228 -> 40 us; 1000 tokens, FFN 3072, float32:
// 1131 -> 186 us; 512 tokens, FFN 2048, bfloat16: 1140 -> 43 us.
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "gemm_direct.h"
#include "gemm_split.h"
#include "gemm_tile.h"
#include "mie_common.h"
#include "moe_route.h"
#include "row_norm.h"

namespace {

using namespace mie::route;
using mie::Mem;
using mie::gemm::f32x4;

constexpr int kChunk = 4096;      // tokens per set of launches: 64 mask words per expert, one per lane
constexpr int kRouteTokens = 8;   // tokens per routing workgroup: one mask byte per expert
constexpr int kMaxSplits = 8;

struct PromptArgs {
  const char* x;       // T [tokens, dim]
  const char* router;  // T [E, dim]
  const char* w1;      // T [E, hidden, dim]
  const char* b1;      // T [E, hidden]
  const char* w2;      // T [E, dim, hidden]
  const char* b2;      // T [E, dim]
  const char* ln_w;    // T [dim]; block form: the norm's weight (NULL: no norm)
  const char* ln_b;    // T [dim] or NULL
  const char* residual;  // T [tokens, dim]; block form: added to the output (or NULL)
  float ln_eps;
  char* normed;        // T [tokens, dim]: the norm's output
  int32_t tokens, E, top_k, dim, hidden;
  int32_t words;              // mask words per expert: ceil(tokens / 64)
  int32_t per_expert;         // 1: the few-rows form (a workgroup per expert); 0: row tiles of all experts
  int32_t splits, split_len;  // W2: K splits and bytes of a row per split
  unsigned long long* masks;  // [E, words]
  int32_t* counts;            // [E] tokens per expert
  int32_t* ids;               // [tokens, top_k], increasing
  float* weights;             // [tokens, top_k], the same order
  int32_t* slots;             // [tokens, top_k], the same order
  char* h;                    // T [tokens * top_k, hidden]
  float* part;                // [splits, tokens * top_k, dim]
  char* out;                  // T [tokens, dim]
};

// grid = words * 8; four waves, two tokens each.  Bound by its memory rounds.
// P > 0 (dim <= 256 P): the tokens' rows stay in registers, and up to
// kRouteRows / P experts' router rows go out with them in one round.  P = 0:
// any dim.
constexpr int kRouteRows = 24;
template <typename T, int P, int K>
__global__ __launch_bounds__(256) void moe_prompt_route(PromptArgs a) {
  __shared__ unsigned int s_mask[kMaxExperts];
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  if (threadIdx.x < kMaxExperts) s_mask[threadIdx.x] = 0u;
  __syncthreads();
  const int t0 = blockIdx.x * kRouteTokens + wave * 2;
  if (t0 < a.tokens) {
    const bool two = t0 + 1 < a.tokens;
    const T* x0 = reinterpret_cast<const T*>(a.x) + static_cast<int64_t>(t0) * a.dim;
    const T* x1 = two ? x0 + a.dim : x0;
    const T* ln_w = reinterpret_cast<const T*>(a.ln_w);
    const T* ln_b = reinterpret_cast<const T*>(a.ln_b);
    // Without a second token its norm goes where the first's goes (the same row).
    T* y0 = reinterpret_cast<T*>(a.normed) + static_cast<int64_t>(t0) * a.dim;
    T* y1 = two ? y0 + a.dim : y0;
    const T* router = reinterpret_cast<const T*>(a.router);
    float l0 = -INFINITY, l1 = -INFINITY;  // lane e: expert e's logit
    if constexpr (P > 0) {
      constexpr int G = kRouteRows / P;
      typename Mem<T>::raw4 r[G][P];
      auto load_rows = [&](int e) {
#pragma unroll
        for (int u = 0; u < G; ++u)
#pragma unroll
          for (int p = 0; p < P; ++p) {
            const int i = p * 256 + lane * 4 < a.dim ? p * 256 + lane * 4 : 0;  // in bounds; met by zeros
            r[u][p] = Mem<T>::load_raw(router + static_cast<int64_t>(min(e + u, a.E - 1)) * a.dim + i);
          }
      };
      f32x4_t v0[P], v1[P];
      if (a.ln_w) {
        load_rows(0);
        mie::norm_row<T, P>(x0, ln_w, ln_b, y0, a.dim, a.ln_eps, lane, v0);
        mie::norm_row<T, P>(x1, ln_w, ln_b, y1, a.dim, a.ln_eps, lane, v1);
      } else {
        typename Mem<T>::raw4 w0[P], w1[P];
#pragma unroll
        for (int p = 0; p < P; ++p) {
          const int i = p * 256 + lane * 4 < a.dim ? p * 256 + lane * 4 : 0;
          w0[p] = Mem<T>::load_raw(x0 + i);
          w1[p] = Mem<T>::load_raw(x1 + i);
        }
        load_rows(0);
#pragma unroll
        for (int p = 0; p < P; ++p) {
          const bool live = p * 256 + lane * 4 < a.dim;
          v0[p] = live ? Mem<T>::widen(w0[p]) : f32x4_t{0.f, 0.f, 0.f, 0.f};
          v1[p] = live ? Mem<T>::widen(w1[p]) : f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
      }
      for (int e = 0; e < a.E; e += G) {
        if (e > 0) load_rows(e);
#pragma unroll
        for (int u = 0; u < G; ++u) {
          float s0 = 0.f, s1 = 0.f;
#pragma unroll
          for (int p = 0; p < P; ++p) {
            if (p * 256 + lane * 4 >= a.dim) continue;
            s0 = dot4(Mem<T>::widen(r[u][p]), v0[p], s0);
            s1 = dot4(Mem<T>::widen(r[u][p]), v1[p], s1);
          }
          s0 = mie::wave_sum(s0);
          s1 = mie::wave_sum(s1);
          if (lane == e + u && e + u < a.E) {
            l0 = s0;
            l1 = s1;
          }
        }
      }
    } else {
      if (a.ln_w) {  // each lane reads back what it wrote itself
        mie::norm_row<T, 0>(x0, ln_w, ln_b, y0, a.dim, a.ln_eps, lane);
        mie::norm_row<T, 0>(x1, ln_w, ln_b, y1, a.dim, a.ln_eps, lane);
        x0 = y0;
        x1 = y1;
      }
      for (int e = 0; e < a.E; ++e) {
        float s0 = 0.f, s1 = 0.f;
        for (int i = lane * 4; i < a.dim; i += 256) {
          const f32x4_t r = Mem<T>::load4(router + static_cast<int64_t>(e) * a.dim + i);
          s0 = dot4(r, Mem<T>::load4(x0 + i), s0);
          s1 = dot4(r, Mem<T>::load4(x1 + i), s1);
        }
        s0 = mie::wave_sum(s0);
        s1 = mie::wave_sum(s1);
        if (lane == e) {
          l0 = s0;
          l1 = s1;
        }
      }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if (j == 1 && !two) break;
      int ids[K];
      float p[K];
      wave_topk<K>(j ? l1 : l0, a.top_k, a.E, lane, ids, p);
#pragma unroll
      for (int kk = 0; kk < K; ++kk) {
        int rank = 0;  // place in increasing expert id (ids are distinct)
#pragma unroll
        for (int o = 0; o < K; ++o) rank += o < a.top_k && ids[o] < ids[kk];
        if (kk < a.top_k && lane == kk) {
          const int64_t at = static_cast<int64_t>(t0 + j) * a.top_k + rank;
          a.ids[at] = ids[kk];
          a.weights[at] = p[kk];
          atomicOr(&s_mask[ids[kk]], 1u << (wave * 2 + j));
        }
      }
    }
  }
  __syncthreads();
  // Every byte of every word is written, also past the last token.
  if (threadIdx.x < a.E)
    reinterpret_cast<uint8_t*>(a.masks + static_cast<int64_t>(threadIdx.x) * a.words)[blockIdx.x] =
        static_cast<uint8_t>(s_mask[threadIdx.x]);
}

__device__ __forceinline__ int wave_inclusive(int v, int lane) {
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int o = __shfl_up(v, off);
    v += lane >= off ? o : 0;
  }
  return v;
}

// The rows a workgroup works on: expert e's rows from m0 (of `count`: up to
// one tile of them, or all in the few-rows form), the expert's first slot.
struct Rows {
  int e, m0, count, base;
};

// Rows of expert y or of row tile y from the experts' token counts (lane e:
// expert e's).
// Uniform over the workgroup; e < 0 when there are none.
__device__ __forceinline__ Rows find_rows(const PromptArgs& a, int cnt, int bm, int lane, int y) {
  const int tiles = (cnt + bm - 1) / bm;
  const int incl = wave_inclusive(cnt, lane);
  Rows r;
  r.m0 = 0;
  if (a.per_expert) {
    r.e = y;
  } else {
    const int incl_tiles = wave_inclusive(tiles, lane);
    const unsigned long long past = __ballot(incl_tiles > y);
    if (past == 0ull) return Rows{-1, 0, 0, 0};
    r.e = __ffsll(past) - 1;
    r.m0 = (y - __shfl(incl_tiles - tiles, r.e)) * bm;
  }
  r.e = __builtin_amdgcn_readfirstlane(r.e);
  r.m0 = __builtin_amdgcn_readfirstlane(r.m0);
  r.count = __builtin_amdgcn_readlane(cnt, r.e);
  r.base = __builtin_amdgcn_readlane(incl, r.e) - r.count;
  if (r.m0 >= r.count) r.e = -1;
  return r;
}

// Token counts of the eight experts from e0 (their mask words `word`, one per
// lane) into lanes e0 .. e0 + 7 of cnt.
__device__ __forceinline__ int count_tokens(const PromptArgs& a, const unsigned long long (&word)[8], int e0, int lane,
                                            int cnt) {
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    int c = lane < a.words ? __popcll(word[u]) : 0;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) c += __shfl_xor(c, off);
    cnt = lane == e0 + u && e0 + u < a.E ? c : cnt;
  }
  return cnt;
}

// The workgroup lists an expert's tokens of ranks m0 .. m0 + BM - 1: lane w
// holds word w of its mask and the rank of that word's first token; wave v
// takes words v, v + 4, ..., a token per lane.  Entries past the expert's last
// token name token 0 (their results are dropped).
template <int BM>
__device__ __forceinline__ void list_rows(unsigned long long mask, int first, int m0, int count, int words, int lane,
                                          int wave, int* rows) {
  const int lo = static_cast<int>(mask), hi = static_cast<int>(mask >> 32);
  for (int w = wave; w < words; w += 4) {
    const unsigned int wl = __builtin_amdgcn_readlane(lo, w), wh = __builtin_amdgcn_readlane(hi, w);
    const int rank = __builtin_amdgcn_readlane(first, w) +
                     static_cast<int>(__builtin_amdgcn_mbcnt_hi(wh, __builtin_amdgcn_mbcnt_lo(wl, 0u))) - m0;
    const bool in = (((static_cast<unsigned long long>(wh) << 32) | wl) >> lane) & 1ull;
    if (in && rank >= 0 && rank < BM) rows[rank] = w * 64 + lane;
  }
  const int i = wave * 64 + lane;
  if (i < BM && i >= count - m0) rows[i] = 0;
}

// Records where token's output of expert e is, for the combining launch.
__device__ __forceinline__ void keep_slot(const PromptArgs& a, int token, int e, int slot) {
  for (int j = 0; j < a.top_k; ++j) {
    const int64_t at = static_cast<int64_t>(token) * a.top_k + j;
    if (a.ids[at] == e) a.slots[at] = slot;
  }
}

__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.f + erff(x * 0.70710678118654752440f)); }

template <typename Tile> struct Waves {
  static constexpr int value = 1;
};
template <int MT, int NT> struct Waves<mie::gemm::SplitTile<MT, NT>> {
  static constexpr int value = mie::gemm::SplitTile<MT, NT>::kWaves;
};

// Tile's product over its first `rows` rows.
template <typename Tile, typename ARow, typename WRow>
__device__ __forceinline__ void run_tile(char* lds, ARow a_row, WRow w_row, int k0, int k1, int rows,
                                         f32x4 (&acc)[Tile::NT][Tile::MT]) {
  if constexpr (std::is_same_v<Tile, mie::gemm::SplitTile<4, 1>>) {
    if (rows > 48) {
      Tile::template run<4>(lds, a_row, w_row, k0, k1, acc);
    } else if (rows > 32) {
      Tile::template run<3>(lds, a_row, w_row, k0, k1, acc);
    } else if (rows > 16) {
      Tile::template run<2>(lds, a_row, w_row, k0, k1, acc);
    } else {
      Tile::template run<1>(lds, a_row, w_row, k0, k1, acc);
    }
  } else {
    Tile::run(lds, a_row, w_row, k0, k1, acc);
  }
}

// grid = (ceil(hidden / BN), row tiles).
template <typename T, typename Tile>
__global__ __launch_bounds__(256, Waves<Tile>::value) void moe_prompt_w1(PromptArgs a) {
  __shared__ __align__(16) char lds[Tile::kLds];
  __shared__ int s_rows[Tile::BM];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Every wave counts every expert's tokens: eight masks in one memory round.
  int cnt = 0;  // lane e: expert e's
  for (int e0 = 0; e0 < a.E; e0 += 8) {
    unsigned long long word[8];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      word[u] = a.masks[static_cast<int64_t>(min(e0 + u, a.E - 1)) * a.words + min(lane, a.words - 1)];
    cnt = count_tokens(a, word, e0, lane, cnt);
  }
  if (blockIdx.x == 0 && blockIdx.y == 0 && wave == 0 && lane < a.E) a.counts[lane] = cnt;
  const Rows r = find_rows(a, cnt, Tile::BM, lane, static_cast<int>(blockIdx.y));
  if (r.e < 0) return;
  const unsigned long long mask = lane < a.words ? a.masks[static_cast<int64_t>(r.e) * a.words + lane] : 0ull;
  const int bits = __popcll(mask);
  const int first = wave_inclusive(bits, lane) - bits;  // rank of this word's first token
  const int64_t row_bytes = static_cast<int64_t>(a.dim) * sizeof(T);
  const int n0 = blockIdx.x * Tile::BN;
  const char* x = a.ln_w ? a.normed : a.x;
  const char* w = a.w1 + static_cast<int64_t>(r.e) * a.hidden * row_bytes;
  const T* bias = reinterpret_cast<const T*>(a.b1) + static_cast<int64_t>(r.e) * a.hidden;
  list_rows<Tile::BM>(mask, first, r.m0, r.count, a.words, lane, wave, s_rows);
  __syncthreads();
  f32x4 acc[Tile::NT][Tile::MT];
#pragma unroll
  for (int n = 0; n < Tile::NT; ++n)
#pragma unroll
    for (int m = 0; m < Tile::MT; ++m) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  run_tile<Tile>(
      lds, [&](int i) { return x + s_rows[i] * row_bytes; },
      [&](int i) { return w + min(n0 + i, a.hidden - 1) * row_bytes; }, 0, static_cast<int>(row_bytes),
      r.count - r.m0, acc);
#pragma unroll
  for (int n = 0; n < Tile::NT; ++n) {
    const int c = n0 + Tile::col(n);
    if (c >= a.hidden) continue;  // hidden is a multiple of 4: all four columns or none
    const f32x4_t b = Mem<T>::load4(bias + c);
#pragma unroll
    for (int m = 0; m < Tile::MT; ++m) {
      const int rank = r.m0 + Tile::row(m);
      if (rank >= r.count) continue;
      f32x4_t v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = gelu(Mem<T>::R(acc[n][m][i] + b[i]));  // of the Linear's output
      Mem<T>::put4(reinterpret_cast<T*>(a.h) + static_cast<int64_t>(r.base + rank) * a.hidden + c, v);
    }
  }
  if (blockIdx.x == 0 && static_cast<int>(threadIdx.x) < min(Tile::BM, r.count - r.m0))
    keep_slot(a, s_rows[threadIdx.x], r.e, r.base + r.m0 + threadIdx.x);
}

// grid = (ceil(dim / BN) * splits, row tiles); blockIdx.x is column tile *
// splits + split.
template <typename T, typename Tile>
__global__ __launch_bounds__(256, Waves<Tile>::value) void moe_prompt_w2(PromptArgs a) {
  __shared__ __align__(16) char lds[Tile::kLds];
  const int lane = threadIdx.x & 63;
  const Rows r = find_rows(a, lane < a.E ? a.counts[lane] : 0, Tile::BM, lane, static_cast<int>(blockIdx.y));
  if (r.e < 0) return;
  const int tile = blockIdx.x / a.splits, split = blockIdx.x % a.splits;
  const int64_t row_bytes = static_cast<int64_t>(a.hidden) * sizeof(T);
  const int k0 = split * a.split_len;
  const int k1 = min(static_cast<int>(row_bytes), k0 + a.split_len);
  const int n0 = tile * Tile::BN;
  const char* w = a.w2 + static_cast<int64_t>(r.e) * a.dim * row_bytes;
  const char* h = a.h + r.base * row_bytes;
  float* part = a.part + (static_cast<int64_t>(split) * a.tokens * a.top_k + r.base) * a.dim;
  f32x4 acc[Tile::NT][Tile::MT];
#pragma unroll
  for (int n = 0; n < Tile::NT; ++n)
#pragma unroll
    for (int m = 0; m < Tile::MT; ++m) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  run_tile<Tile>(
      lds, [&](int i) { return h + min(r.m0 + i, r.count - 1) * row_bytes; },
      [&](int i) { return w + min(n0 + i, a.dim - 1) * row_bytes; }, k0, k1, r.count - r.m0, acc);
#pragma unroll
  for (int n = 0; n < Tile::NT; ++n) {
    const int c = n0 + Tile::col(n);
    if (c >= a.dim) continue;
#pragma unroll
    for (int m = 0; m < Tile::MT; ++m) {
      const int rank = r.m0 + Tile::row(m);
      if (rank < r.count) *reinterpret_cast<f32x4*>(part + static_cast<int64_t>(rank) * a.dim + c) = acc[n][m];
    }
  }
}

// grid = ceil(tokens * dim / 4 / 256): four outputs of a token per thread.
// Two memory rounds: the token's slots, then every partial sum of KK experts.
template <typename T, int KK>
__global__ __launch_bounds__(256) void moe_prompt_combine(PromptArgs a, mie::FastDiv row) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  const uint32_t t = row.div(i);
  if (t >= static_cast<uint32_t>(a.tokens)) return;
  const int c = (i - t * row.d) * 4;
  const int64_t all = static_cast<int64_t>(a.tokens) * a.top_k * a.dim;
  const int64_t here = static_cast<int64_t>(t) * a.dim + c;
  f32x4_t res = {0.f, 0.f, 0.f, 0.f};
  if (a.residual) res = Mem<T>::load4(reinterpret_cast<const T*>(a.residual) + here);
  f32x4_t out = {0.f, 0.f, 0.f, 0.f};
  for (int j0 = 0; j0 < a.top_k; j0 += KK) {  // increasing expert id
    int slot[KK], id[KK];
    float w[KK];
#pragma unroll
    for (int j = 0; j < KK; ++j) {
      const int64_t at = static_cast<int64_t>(t) * a.top_k + min(j0 + j, a.top_k - 1);
      slot[j] = a.slots[at];
      id[j] = a.ids[at];
      w[j] = Mem<T>::R(a.weights[at]);
    }
    f32x4_t y[KK], b[KK];
#pragma unroll
    for (int j = 0; j < KK; ++j) {
      b[j] = Mem<T>::load4(reinterpret_cast<const T*>(a.b2) + static_cast<int64_t>(id[j]) * a.dim + c);
      y[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    for (int s0 = 0; s0 < a.splits; s0 += 4) {
      f32x4_t p[KK][4];
#pragma unroll
      for (int j = 0; j < KK; ++j)
#pragma unroll
        for (int s = 0; s < 4; ++s)
          p[j][s] = *reinterpret_cast<const f32x4_t*>(a.part + min(s0 + s, a.splits - 1) * all +
                                                      static_cast<int64_t>(slot[j]) * a.dim + c);
#pragma unroll
      for (int j = 0; j < KK; ++j)
#pragma unroll
        for (int s = 0; s < 4; ++s)
          if (s0 + s < a.splits) y[j] += p[j][s];
    }
#pragma unroll
    for (int j = 0; j < KK; ++j) {
      if (j0 + j >= a.top_k) break;
#pragma unroll
      for (int u = 0; u < 4; ++u)
        out[u] = Mem<T>::R(__fadd_rn(out[u], Mem<T>::R(__fmul_rn(w[j], Mem<T>::R(y[j][u] + b[j][u])))));
    }
  }
  if (a.residual) out += res;
  Mem<T>::put4(reinterpret_cast<T*>(a.out) + here, out);
}

// ---- few rows per expert -----------------------------------------------------
// The two products where the launch streams the experts' weights: one
// workgroup per (expert, 32 columns), direct tiles (gemm_direct.h), 32 or 16
// rows at a time.  The expert is known from blockIdx, so two windows of its
// weights (2048 bytes of each row) are in flight before the routing is read.
template <typename T> using Few = mie::gemm::Direct<T, 2, 4>;

// grid = (ceil(hidden / 32), E).
template <typename T>
__global__ __launch_bounds__(256, 2) void moe_prompt_w1_few(PromptArgs a) {
  using Tile = Few<T>;
  __shared__ __align__(16) char lds[Tile::template kLds<2>];
  __shared__ int s_rows[32];
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int e = blockIdx.y, n0 = blockIdx.x * Tile::BN;
  const int row_bytes = a.dim * static_cast<int>(sizeof(T));
  const unsigned long long mask = lane < a.words ? a.masks[static_cast<int64_t>(e) * a.words + lane] : 0ull;
  unsigned long long word[8];
#pragma unroll
  for (int u = 0; u < 8; ++u)
    word[u] = a.masks[static_cast<int64_t>(min(u, a.E - 1)) * a.words + min(lane, a.words - 1)];
  const char* wp[Tile::NT];
#pragma unroll
  for (int n = 0; n < Tile::NT; ++n)
    wp[n] = a.w1 + (static_cast<int64_t>(e) * a.hidden + min(n0 + n * 16 + i, a.hidden - 1)) * row_bytes;
  typename Tile::template Set<Tile::NT> ws[2];
  Tile::prefetch(ws, wp, 0, row_bytes);
  __builtin_amdgcn_sched_barrier(0);
  int cnt = count_tokens(a, word, 0, lane, 0);
  for (int e0 = 8; e0 < a.E; e0 += 8) {
#pragma unroll
    for (int u = 0; u < 8; ++u)
      word[u] = a.masks[static_cast<int64_t>(min(e0 + u, a.E - 1)) * a.words + min(lane, a.words - 1)];
    cnt = count_tokens(a, word, e0, lane, cnt);
  }
  if (blockIdx.x == 0 && e == 0 && wave == 0 && lane < a.E) a.counts[lane] = cnt;
  const Rows r = find_rows(a, cnt, 32, lane, e);
  if (r.e < 0) return;
  const int bits = __popcll(mask);
  const int rank0 = wave_inclusive(bits, lane) - bits;
  const char* x = a.ln_w ? a.normed : a.x;
  f32x4_t bias[Tile::NT];
#pragma unroll
  for (int n = 0; n < Tile::NT; ++n)
    bias[n] = Mem<T>::load4(reinterpret_cast<const T*>(a.b1) + static_cast<int64_t>(e) * a.hidden +
                            min(n0 + n * 16 + g * 4, a.hidden - 4));
  for (int m0 = 0; m0 < r.count; m0 += 32) {
    if (m0 > 0) {
      __syncthreads();  // the last tile's rows and sums are read
      Tile::prefetch(ws, wp, 0, row_bytes);
    }
    list_rows<32>(mask, rank0, m0, r.count, a.words, lane, wave, s_rows);
    mie::gemm::lds_barrier();
    auto store = [&](int n, int m, f32x4 sum) {
      const int c = n0 + n * 16 + g * 4, rank = m0 + m * 16 + i;
      if (c >= a.hidden || rank >= r.count) return;
      f32x4_t v;
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = gelu(Mem<T>::R(sum[u] + bias[n][u]));
      Mem<T>::put4(reinterpret_cast<T*>(a.h) + static_cast<int64_t>(r.base + rank) * a.hidden + c, v);
    };
    if (r.count - m0 > 16) {
      const char* ap[2] = {x + static_cast<int64_t>(s_rows[i]) * row_bytes,
                           x + static_cast<int64_t>(s_rows[16 + i]) * row_bytes};
      Tile::template run<2>(lds, ws, ap, wp, 0, row_bytes, store);
    } else {
      const char* ap[1] = {x + static_cast<int64_t>(s_rows[i]) * row_bytes};
      Tile::template run<1>(lds, ws, ap, wp, 0, row_bytes, store);
    }
    if (blockIdx.x == 0 && static_cast<int>(threadIdx.x) < min(32, r.count - m0))
      keep_slot(a, s_rows[threadIdx.x], e, r.base + m0 + threadIdx.x);
  }
}

// grid = (ceil(dim / 32) * splits, E); blockIdx.x is column tile * splits + split.
template <typename T>
__global__ __launch_bounds__(256, 2) void moe_prompt_w2_few(PromptArgs a) {
  using Tile = Few<T>;
  __shared__ __align__(16) char lds[Tile::template kLds<2>];
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
  const int e = blockIdx.y, n0 = blockIdx.x / a.splits * Tile::BN, split = blockIdx.x % a.splits;
  const int row_bytes = a.hidden * static_cast<int>(sizeof(T));
  const int k0 = split * a.split_len, k1 = min(row_bytes, k0 + a.split_len);
  const int cnt = a.counts[min(lane, a.E - 1)];
  const char* wp[Tile::NT];
#pragma unroll
  for (int n = 0; n < Tile::NT; ++n)
    wp[n] = a.w2 + (static_cast<int64_t>(e) * a.dim + min(n0 + n * 16 + i, a.dim - 1)) * row_bytes;
  typename Tile::template Set<Tile::NT> ws[2];
  Tile::prefetch(ws, wp, k0, k1);
  __builtin_amdgcn_sched_barrier(0);
  const Rows r = find_rows(a, lane < a.E ? cnt : 0, 32, lane, e);
  if (r.e < 0) return;
  const char* h = a.h + static_cast<int64_t>(r.base) * row_bytes;
  float* part = a.part + (static_cast<int64_t>(split) * a.tokens * a.top_k + r.base) * a.dim;
  for (int m0 = 0; m0 < r.count; m0 += 32) {
    if (m0 > 0) {
      __syncthreads();
      Tile::prefetch(ws, wp, k0, k1);
    }
    auto store = [&](int n, int m, f32x4 sum) {
      const int c = n0 + n * 16 + g * 4, rank = m0 + m * 16 + i;
      if (c < a.dim && rank < r.count) *reinterpret_cast<f32x4*>(part + static_cast<int64_t>(rank) * a.dim + c) = sum;
    };
    const char* ap[2] = {h + static_cast<int64_t>(min(m0 + i, r.count - 1)) * row_bytes,
                         h + static_cast<int64_t>(min(m0 + 16 + i, r.count - 1)) * row_bytes};
    if (r.count - m0 > 16) {
      Tile::template run<2>(lds, ws, ap, wp, k0, k1, store);
    } else {
      const char* one[1] = {ap[0]};
      Tile::template run<1>(lds, ws, one, wp, k0, k1, store);
    }
  }
}

// More rows: LDS-staged tiles of 64 x 64, for float32 on the bfloat16 matrix
// cores (gemm_split.h) and over the rows a tile has, 16 to 64 (1000 tokens,
// top-2 of 8, FFN 3072: W1 127 -> 98 us, W2 116 -> 89).
// bfloat16 waits on memory and barriers, hidden by four workgroups per CU: steps
// of 256 bytes (two per CU) take 53 us a layer for 512 tokens, FFN 2048, these 43.
template <typename T> struct WideTile {
  using type = mie::gemm::Tile<T, 64, 64, 128, 2, 2>;
};
template <> struct WideTile<float> {
  using type = mie::gemm::SplitTile<4, 1>;
};
template <typename T> using Wide = typename WideTile<T>::type;

struct Plan {
  bool few;
  int32_t rows;               // blockIdx.y extent
  int32_t splits, split_len;  // W2
};

// Few rows: up to 20 per expert on average.  At 16 (62 tokens, 8 experts,
// top-2, float32) both forms take 36-38 us for the two products, at 8 the
// direct tiles 29 against 35 us, at 32 the staged ones 50 against 62 us (in float32 instructions).
Plan make_plan(int32_t tokens, int32_t E, int32_t top_k, int32_t dim, int32_t hidden, int elt) {
  Plan p;
  const int64_t slots = static_cast<int64_t>(tokens) * top_k;
  // float32 sums of fewer than 16 products stay in float32 instructions too:
  // what the split leaves out of a product (gemm_split.h) is only made up for by
  // the longer sums' own rounding.
  p.few = slots <= 20 * static_cast<int64_t>(E) || (elt == 4 && std::min(dim, hidden) < 16);
  const int bn = p.few ? 32 : 64, kb = p.few ? 1024 : 128;
  p.rows = p.few ? E : static_cast<int32_t>(slots / 64 + std::min<int64_t>(E, slots));
  // W2 has few column tiles, so its K is split.  bfloat16 and few rows wait on
  // memory: until the launch holds two workgroups per CU, and, where that can
  // be had, with a multiple of 8 column tiles x splits - workgroups are dealt
  // to the 8 XCDs in turn, so each column tile is then read through one XCD's
  // L2.  float32 tiles fill the matrix cores: the split with the least rounds
  // over the 256 CUs per split (a round more costs a tile, a third of one is
  // lost once) and partial sums (8 bytes each way per value and split, against
  // a tile's time).  Measured, us for 1, 2, 3, 4, 5, 6, 8 splits: float32 1000
  // tokens, FFN 3072, whole layer: 188, 197, 183, 181, 187, 183, 189; bfloat16
  // 512 tokens 20, 15, 18, 15, 20, 16, 17.
  const int64_t used = p.few ? std::min<int64_t>(E, slots) : slots / 64 + E / 2;
  const int64_t columns = (dim + bn - 1) / bn;
  const int64_t groups = columns * std::max<int64_t>(1, used);
  const int32_t steps = (hidden * elt + kb - 1) / kb;
  const int32_t most = std::max<int32_t>(1, std::min<int32_t>(kMaxSplits, steps / 2));
  int32_t splits = 1;
  if (p.few || elt == 2) {
    splits = static_cast<int32_t>(std::min<int64_t>(most, (511 + groups) / groups));
    if (!p.few)
      for (int32_t s = splits; s <= most; ++s)
        if (columns * s % 8 == 0) {
          splits = s;
          break;
        }
  } else {
    const double partials = 1.25 * static_cast<double>(slots) * dim / hidden;
    auto cost = [&](int32_t s) { return (static_cast<double>((groups * s + 255) / 256) * 100 + 53) / s + partials / 100 * s; };
    for (int32_t s = 2; s <= most; ++s)
      if (cost(s) < cost(splits)) splits = s;
  }
  p.split_len = (steps + splits - 1) / splits * kb;
  p.splits = (hidden * elt + p.split_len - 1) / p.split_len;
  return p;
}

int64_t align256(int64_t n) { return (n + 255) / 256 * 256; }

// Lays the workspace out for `tokens` (at most kChunk) and returns its bytes.
int64_t layout(PromptArgs& a, const Plan& p, int elt, char* base) {
  const int64_t slots = static_cast<int64_t>(a.tokens) * a.top_k;
  int64_t at = 0;
  auto take = [&](int64_t bytes) {
    char* here = base + at;
    at += align256(bytes);
    return here;
  };
  a.masks = reinterpret_cast<unsigned long long*>(take(static_cast<int64_t>(a.E) * a.words * 8));
  a.counts = reinterpret_cast<int32_t*>(take(a.E * 4));
  a.ids = reinterpret_cast<int32_t*>(take(slots * 4));
  a.weights = reinterpret_cast<float*>(take(slots * 4));
  a.slots = reinterpret_cast<int32_t*>(take(slots * 4));
  a.normed = take(static_cast<int64_t>(a.tokens) * a.dim * elt);
  a.h = take(slots * a.hidden * elt);
  a.part = reinterpret_cast<float*>(take(slots * a.dim * 4 * p.splits));
  return at;
}

template <typename T, int K>
void launch_route(const PromptArgs& a, hipStream_t st) {
  const int groups = a.words * 8;
  if (a.dim <= 768) {
    moe_prompt_route<T, 3, K><<<groups, 256, 0, st>>>(a);
  } else if (a.dim <= 1024) {
    moe_prompt_route<T, 4, K><<<groups, 256, 0, st>>>(a);
  } else {
    moe_prompt_route<T, 0, K><<<groups, 256, 0, st>>>(a);
  }
}

template <typename T>
int32_t launch(const PromptArgs& a, const Plan& p, hipStream_t st) {
  a.top_k <= 2 ? launch_route<T, 2>(a, st) : launch_route<T, kMaxTopK>(a, st);
  int32_t rc = mie::check_launch("moe_prompt_route");
  if (rc != MIE_OK) return rc;
  const int bn = p.few ? 32 : 64;
  const dim3 g1((a.hidden + bn - 1) / bn, p.rows), g2((a.dim + bn - 1) / bn * p.splits, p.rows);
  if (p.few) {
    moe_prompt_w1_few<T><<<g1, 256, 0, st>>>(a);
  } else {
    moe_prompt_w1<T, Wide<T>><<<g1, 256, 0, st>>>(a);
  }
  rc = mie::check_launch("moe_prompt_w1");
  if (rc != MIE_OK) return rc;
  if (p.few) {
    moe_prompt_w2_few<T><<<g2, 256, 0, st>>>(a);
  } else {
    moe_prompt_w2<T, Wide<T>><<<g2, 256, 0, st>>>(a);
  }
  rc = mie::check_launch("moe_prompt_w2");
  if (rc != MIE_OK) return rc;
  const int64_t threads = static_cast<int64_t>(a.tokens) * (a.dim / 4);
  const uint32_t groups = static_cast<uint32_t>((threads + 255) / 256);
  const mie::FastDiv row = mie::FastDiv::make(static_cast<uint32_t>(a.dim / 4));
  if (a.top_k == 1) {
    moe_prompt_combine<T, 1><<<groups, 256, 0, st>>>(a, row);
  } else {
    moe_prompt_combine<T, 2><<<groups, 256, 0, st>>>(a, row);
  }
  return mie::check_launch("moe_prompt_combine");
}

int32_t check(int64_t tokens, int32_t E, int32_t top_k, int32_t dim, int32_t hidden, int32_t dtype) {
  if (dtype != MIE_DTYPE_F32 && dtype != MIE_DTYPE_BF16)
    return mie::fail(MIE_ERR_UNSUPPORTED, "mie_moe_prefill: float32 or bfloat16 only (dtype %d)", dtype);
  if (tokens <= 0 || E <= 0 || E > kMaxExperts || top_k <= 0 || top_k > kMaxTopK || top_k > E)
    return mie::fail(MIE_ERR_INVALID, "mie_moe_prefill: tokens=%lld experts=%d top_k=%d (at most %d and %d)",
                     static_cast<long long>(tokens), E, top_k, kMaxExperts, kMaxTopK);
  const int vec = 16 / mie::elt_size(dtype);
  if (dim <= 0 || hidden <= 0 || dim % vec != 0 || hidden % vec != 0 || dim > (1 << 20) || hidden > (1 << 20))
    return mie::fail(MIE_ERR_INVALID, "mie_moe_prefill: dim=%d hidden=%d must be multiples of %d up to 2^20", dim,
                     hidden, vec);
  return MIE_OK;
}

PromptArgs shape_args(int32_t tokens, int32_t E, int32_t top_k, int32_t dim, int32_t hidden) {
  PromptArgs a{};
  a.tokens = tokens;
  a.E = E;
  a.top_k = top_k;
  a.dim = dim;
  a.hidden = hidden;
  a.words = (tokens + 63) / 64;
  return a;
}

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

}  // namespace

extern "C" int64_t mie_moe_prefill_workspace(int64_t tokens, int32_t num_experts, int32_t top_k, int32_t dim,
                                             int32_t hidden, int32_t dtype) {
  const int32_t rc = check(tokens, num_experts, top_k, dim, hidden, dtype);
  if (rc != MIE_OK) return -rc;
  const int elt = mie::elt_size(dtype);
  int64_t need = 0;
  // The last chunk is shorter and may split K more ways.
  for (int64_t n : {std::min<int64_t>(tokens, kChunk), tokens % kChunk}) {
    if (n == 0) continue;
    PromptArgs a = shape_args(static_cast<int32_t>(n), num_experts, top_k, dim, hidden);
    need = std::max(need, layout(a, make_plan(a.tokens, num_experts, top_k, dim, hidden, elt), elt, nullptr));
  }
  return need;
}

extern "C" int32_t mie_moe_prefill(const void* x, int64_t tokens, const void* ln_weight, const void* ln_bias,
                                   float ln_eps, const void* residual, const void* router_weight, const void* w1,
                                   const void* b1, const void* w2, const void* b2, int32_t num_experts, int32_t top_k, int32_t dim,
                                   int32_t hidden, void* out, void* workspace, int64_t workspace_bytes, int32_t dtype,
                                   void* stream) {
  mie::clear_error();
  int32_t rc = check(tokens, num_experts, top_k, dim, hidden, dtype);
  if (rc != MIE_OK) return rc;
  if (!x || !router_weight || !w1 || !b1 || !w2 || !b2 || !out || !workspace)
    return mie::fail(MIE_ERR_INVALID, "mie_moe_prefill: null pointer");
  if (!ln_weight && ln_bias) return mie::fail(MIE_ERR_INVALID, "mie_moe_prefill: a norm bias needs a weight");
  for (const void* p : {x, ln_weight, ln_bias, residual, router_weight, w1, b1, w2, b2, static_cast<const void*>(out),
                        static_cast<const void*>(workspace)})
    if (!aligned16(p)) return mie::fail(MIE_ERR_INVALID, "mie_moe_prefill: every pointer must be 16-byte aligned");
  const int64_t need = mie_moe_prefill_workspace(tokens, num_experts, top_k, dim, hidden, dtype);
  if (workspace_bytes < need)
    return mie::fail(MIE_ERR_WORKSPACE, "mie_moe_prefill: workspace of %lld bytes, needs %lld",
                     static_cast<long long>(workspace_bytes), static_cast<long long>(need));
  const int elt = mie::elt_size(dtype);
  for (int64_t t0 = 0; t0 < tokens; t0 += kChunk) {
    PromptArgs a = shape_args(static_cast<int32_t>(std::min<int64_t>(kChunk, tokens - t0)), num_experts, top_k, dim,
                              hidden);
    const Plan p = make_plan(a.tokens, num_experts, top_k, dim, hidden, elt);
    layout(a, p, elt, static_cast<char*>(workspace));
    a.x = static_cast<const char*>(x) + t0 * dim * elt;
    a.ln_w = static_cast<const char*>(ln_weight);
    a.ln_b = static_cast<const char*>(ln_bias);
    a.ln_eps = ln_eps;
    a.residual = residual ? static_cast<const char*>(residual) + t0 * dim * elt : nullptr;
    a.router = static_cast<const char*>(router_weight);
    a.w1 = static_cast<const char*>(w1);
    a.b1 = static_cast<const char*>(b1);
    a.w2 = static_cast<const char*>(w2);
    a.b2 = static_cast<const char*>(b2);
    a.out = static_cast<char*>(out) + t0 * dim * elt;
    a.per_expert = p.few;
    a.splits = p.splits;
    a.split_len = p.split_len;
    const hipStream_t st = static_cast<hipStream_t>(stream);
    rc = dtype == MIE_DTYPE_F32 ? launch<float>(a, p, st) : launch<uint16_t>(a, p, st);
    if (rc != MIE_OK) return rc;
  }
  return MIE_OK;
}
