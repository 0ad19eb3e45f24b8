// Device core of the decode kernels for f32 activations or f32 caches (the
// bf16 / bf16 kernels have theirs in decode_mfma.hpp): one workgroup scans a
// token range of one KV head for one or all four query heads of its GQA group and
// one slice of the output dims, keeping an online-softmax state per head.
//
// Lane layout (wave64 = 4 row-groups of 16 lanes): row-group g takes one token
// per step, and a row is read in 16-byte pieces, 16 lanes on one contiguous
// 256-byte stretch (whole 128-byte lines; a bf16 V slice of 64 dims in 8-byte
// pieces, one line).  q.k partial dots reduce inside the
// 16-lane row with four DPP steps; the softmax runs in the exp2 domain with
// log2(e)/sqrt(D) folded into q.
#pragma once

#include "common.hpp"

namespace raftinfer::amd {

constexpr int kHeadDim = 256;
constexpr int kQueryHeads = 16;
constexpr int kKvHeads = 4;
constexpr int kGroup = kQueryHeads / kKvHeads;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

// Element index of (token, kv_head, dim 0) in one cache plane
// (cpp/kernels/qwen35_online_attention.cu:240-252).
__device__ __forceinline__ std::size_t cache_row(bool head_major, std::size_t token,
                                                 std::size_t kv_head, std::size_t max_ctx) {
  return head_major ? (kv_head * max_ctx + token) * kHeadDim
                    : (token * kKvHeads + kv_head) * kHeadDim;
}

// W contiguous cache elements as loaded (kStream: nontemporal).
template <typename T, int W, bool kStream> struct Piece {
  static_assert(W * sizeof(T) <= 16);
  typedef T vec __attribute__((ext_vector_type(W == 1 ? 2 : W)));
  using Raw = std::conditional_t<W == 1, T, vec>;
  Raw raw;
  __device__ __forceinline__ void load(const T *p) {
    const auto *v = reinterpret_cast<const Raw *>(p);
    if constexpr (kStream) raw = __builtin_nontemporal_load(v); else raw = *v;
  }
  __device__ __forceinline__ void set(int i, T x) {
    if constexpr (W == 1) raw = x; else raw[i] = x;
  }
  __device__ __forceinline__ float get(int i) const {
    T x;
    if constexpr (W == 1) x = raw; else x = raw[i];
    return Elem<T>::load(&x, 0);
  }
};

// What the scan reads: query [16][256], the new token's key / value rows
// [4][256] (its cache rows are not read) and the cache planes.
template <typename ActT, typename CacheT> struct ScanArgs {
  const ActT *query, *key_new, *value_new;
  CacheT *cache;
  std::size_t max_ctx;
  bool head_major;
};

// Per-head combined state after a workgroup scan, staged in LDS.
template <int NH, int DS, int WAVES> struct ScanShared {
  float m[WAVES][NH];
  float l[WAVES][NH];
  float acc[WAVES][NH][kHeadDim / DS];
};

// Scans tokens [begin, end) for the query heads head .. head + NH - 1 of one KV
// head, dims slice dq of 256 / DS for the output, and leaves the per-wave states in `sh`.  The row of position `pos` (if
// in range) comes from key_new / value_new, as the cache stores it.  U tokens per
// row-group and step.  Every wave returns after writing its slot; the caller
// synchronizes.
template <typename ActT, typename CacheT, int NH, int DS, int WAVES, int U>
__device__ __forceinline__ void scan_slice(const ScanArgs<ActT, CacheT> &a, std::size_t head, int dq,
                                           std::size_t begin, std::size_t end, std::size_t pos,
                                           ScanShared<NH, DS, WAVES> &sh) {
  static_assert(kGroup % NH == 0, "the heads of one KV head");
  const std::size_t kv_head = head / kGroup;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int g = lane >> 4;
  const int r = lane & 15;
  const float qscale = kLog2e / 16.0f; // log2(e) / sqrt(256)
  constexpr int kDims = kHeadDim / DS, kPerLane = kDims / 16; // output dims of the slice, of a lane
  constexpr int KW = 16 / sizeof(CacheT), KP = 16 / KW;       // K piece width, pieces per lane
  constexpr int VW = kPerLane < KW ? kPerLane : KW, VP = kPerLane / VW;
  // Which rows are streamed past the caches: in a split step K where one workgroup
  // reads it, and V, each slice its own.  From memory (1 GB of caches in turn, us, both
  // / K alone / neither): f32, 16384 tokens 31.3 / 32.5 / 34.6, 8000 in two slices 22.3
  // / 23.3, 4096 in four 16.4 / 17.0; bf16, 16384: 23.0 / 23.4 / 24.2.  (One layer over
  // and over, 268 MB that the memory-side cache half holds, 32768 tokens: 61 / 54 / 55.)
  // The short rows of a single-block step are better left alone (700 tokens 18.8 with
  // V streamed, 15.3 without).
  constexpr bool kSplit = NH == kGroup, kStreamK = kSplit && DS == 1, kStreamV = kSplit;
  // Element of piece p of a lane: 16 KW p + KW r (K), 16 VW p + VW r of the slice (V).
  const CacheT *k_plane = a.cache + cache_row(a.head_major, 0, kv_head, a.max_ctx);
  const CacheT *v_plane = k_plane + a.max_ctx * kKvHeads * kHeadDim + dq * kDims;
  const std::size_t token_stride = a.head_major ? kHeadDim : kKvHeads * kHeadDim;

  float q[NH][16];
#pragma unroll
  for (int h = 0; h < NH; ++h) {
    const ActT *qh = a.query + (head + h) * kHeadDim;
#pragma unroll
    for (int i = 0; i < 16; ++i) q[h][i] = Elem<ActT>::load(qh, 16 * KW * (i / KW) + KW * r + i % KW) * qscale;
  }

  float m[NH], l[NH], acc[NH][kPerLane];
#pragma unroll
  for (int h = 0; h < NH; ++h) {
    m[h] = -INFINITY;
    l[h] = 0.f;
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) acc[h][i] = 0.f;
  }

  constexpr int kTile = 4 * U; // tokens per wave step
  for (std::size_t tile = begin + static_cast<std::size_t>(wave) * kTile; tile < end;
       tile += static_cast<std::size_t>(WAVES) * kTile) {
    Piece<CacheT, KW, kStreamK> k[U][KP];
    Piece<CacheT, VW, kStreamV> v[U][VP];
    const bool whole = tile + kTile <= end; // (uniform)
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // tokens past the range re-read its last row (masked below)
      const std::size_t tok = tile + 4 * u + g;
      const std::size_t row = (tok < end ? tok : end - 1) * token_stride;
#pragma unroll
      for (int p = 0; p < KP; ++p) k[u][p].load(k_plane + row + 16 * KW * p + KW * r);
#pragma unroll
      for (int p = 0; p < VP; ++p) v[u][p].load(v_plane + row + 16 * VW * p + VW * r);
    }
    if (pos >= tile && pos < tile + kTile) { // (uniform) this step holds the new token
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (tile + 4 * u + g != pos) continue;
        const ActT *kn = a.key_new + kv_head * kHeadDim, *vn = a.value_new + kv_head * kHeadDim + dq * kDims;
        CacheT x;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          Elem<CacheT>::store(&x, 0, Elem<ActT>::load(kn, 16 * KW * (i / KW) + KW * r + i % KW));
          k[u][i / KW].set(i % KW, x);
        }
#pragma unroll
        for (int i = 0; i < kPerLane; ++i) {
          Elem<CacheT>::store(&x, 0, Elem<ActT>::load(vn, 16 * VW * (i / VW) + VW * r + i % VW));
          v[u][i / VW].set(i % VW, x);
        }
      }
    }
    float s[NH][U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int h = 0; h < NH; ++h) {
        float d0 = 0.f, d1 = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          d0 = fmaf(q[h][i], k[u][i / KW].get(i % KW), d0);
          d1 = fmaf(q[h][8 + i], k[u][(8 + i) / KW].get((8 + i) % KW), d1);
        }
        s[h][u] = row16_sum(d0 + d1);
      }
    }
    if (!whole) {
      // no weight, and no value either: the row read in its place may be the
      // new token's, which the cache does not hold yet
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (tile + 4 * u + g < end) continue;
#pragma unroll
        for (int h = 0; h < NH; ++h) s[h][u] = -INFINITY;
#pragma unroll
        for (int i = 0; i < kPerLane; ++i) v[u][i / VW].set(i % VW, CacheT{});
      }
    }
#pragma unroll
    for (int h = 0; h < NH; ++h) {
      float mt = m[h];
#pragma unroll
      for (int u = 0; u < U; ++u) mt = fmaxf(mt, s[h][u]);
      const float ref = mt == -INFINITY ? 0.f : mt; // a row-group may have seen no token yet
      const float so = __builtin_amdgcn_exp2f(m[h] - ref);
      float p[U];
      float psum = 0.f;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        p[u] = __builtin_amdgcn_exp2f(s[h][u] - ref);
        psum += p[u];
      }
      l[h] = l[h] * so + psum;
#pragma unroll
      for (int i = 0; i < kPerLane; ++i) {
        float x = acc[h][i] * so;
#pragma unroll
        for (int u = 0; u < U; ++u) x = fmaf(p[u], v[u][i / VW].get(i % VW), x);
        acc[h][i] = x;
      }
      m[h] = mt;
    }
  }

  // Combine the four row-groups of the wave (lanes r, r^16, r^32, r^48 own
  // the same dims).
#pragma unroll
  for (int h = 0; h < NH; ++h) {
    float mm = fmaxf(m[h], xor16(m[h]));
    mm = fmaxf(mm, xor32(mm));
    const float w = m[h] == -INFINITY ? 0.f : exp2f(m[h] - mm);
    float lw = l[h] * w;
    lw += xor16(lw);
    lw += xor32(lw);
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) {
      float x = acc[h][i] * w;
      x += xor16(x);
      x += xor32(x);
      acc[h][i] = x;
    }
    if (lane == 0) {
      sh.m[wave][h] = mm;
      sh.l[wave][h] = lw;
    }
    if (lane < 16) {
#pragma unroll
      for (int i = 0; i < kPerLane; ++i) sh.acc[wave][h][16 * VW * (i / VW) + VW * r + i % VW] = acc[h][i];
    }
  }
}

// Merges the per-wave states of `sh` for output element (h, d of the slice):
// returns the exp2-domain max, the sum and the unnormalised accumulator.
template <int NH, int DS, int WAVES>
__device__ __forceinline__ void combine_waves(const ScanShared<NH, DS, WAVES> &sh, int h, int d,
                                              float &m_out, float &l_out, float &a_out) {
  float mm = -INFINITY;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) mm = fmaxf(mm, sh.m[w][h]);
  float l = 0.f, a = 0.f;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    const float mw = sh.m[w][h];
    const float sc = mw == -INFINITY ? 0.f : exp2f(mw - mm);
    l = fmaf(sh.l[w][h], sc, l);
    a = fmaf(sh.acc[w][h][d], sc, a);
  }
  m_out = mm;
  l_out = l;
  a_out = a;
}

// Stores the new token's K and V rows of kv_head at `pos`, cast to the cache
// dtype (round to nearest even).
template <typename ActT, typename CacheT>
__device__ __forceinline__ void append_rows(const ScanArgs<ActT, CacheT> &a, std::size_t kv_head, std::size_t pos) {
  if (threadIdx.x >= kHeadDim) return;
  const std::size_t row = cache_row(a.head_major, pos, kv_head, a.max_ctx) + threadIdx.x;
  const std::size_t src = kv_head * kHeadDim + threadIdx.x;
  Elem<CacheT>::store(a.cache, row, Elem<ActT>::load(a.key_new, src));
  Elem<CacheT>::store(a.cache, a.max_ctx * kKvHeads * kHeadDim + row, Elem<ActT>::load(a.value_new, src));
}

// sigmoid(x) = 1 / (1 + 2^(-x log2 e)) with the hardware exp2 and reciprocal
// (about 1 ulp each; outputs are rounded to bf16 or compared at 1e-2).
__device__ __forceinline__ float sigmoid_gate(float x) {
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-x * kLog2e));
}

} // namespace raftinfer::amd
