// Device pieces shared by the bf16 MFMA prefill kernels: swizzled LDS reads,
// AGPR-resident accumulators and the q producer applied to staged rows.
#pragma once

#include "decode_scan.hpp"
#include "norm_rope.hpp"

namespace raftinfer::amd {
namespace prefill {

constexpr int kKTile = 32;           // keys per tile
constexpr int kWaves = 4;            // waves per workgroup
constexpr int kThreads = kWaves * kWave;
constexpr float kLazyRescale = 8.0f; // log2 units
constexpr int kHalfElems = kKTile * kHeadDim / 2; // one half of a K / V tile (128 dims)

typedef short short4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) short4v lds_short4v;

// The q producer fused into the prefill kernel (NormQ).
struct PrefillNormRope {
  const void *weight; // q norm weight [256], bf16 or f32
  bool weight_f32;
  int pairs;    // rotary_dim / 2 (rotary_dim a multiple of 8)
  double ratio; // rope_base^(-2 / rotary_dim)
  float epsilon;
};
// Physical 16-byte chunk of logical chunk c in tile row r: c ^ (r & 7).  The
// LDS bank-conflict counter, calibrated on these access patterns alone, shows
// this leaves 2-way conflicts on the K/Q ds_read_b128 (16 rows per pass) and
// 4-way on the V ds_read_b64_tr_b16; c ^ (4 (r % 4) + (r / 4) % 4) is free of
// both, but measured PP512 13.2 -> 13.1 us, PP2048 80 -> 78, PP128 7.13 ->
// 7.3 (more lane bases held across the loop), so the loop is not bound by
// these reads and the simpler swizzle stays.
__device__ __forceinline__ int swz(int r) { return r & 7; }

__device__ __forceinline__ int chunk_offset(int r, int c) { // in bf16 elements
  return r * kHeadDim + ((c ^ swz(r)) << 3);
}

__device__ __forceinline__ bf16x8 lds_b128(const bf16_bits *p) {
  return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(p));
}

__device__ __forceinline__ u32x2 lds_tr16(const bf16_bits *p) {
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4v *)(p)));
}

__host__ __device__ constexpr std::size_t ceil_div_u(std::size_t n, std::size_t d) {
  return (n + d - 1) / d;
}

// o += a * b (v_mfma_f32_32x32x16_bf16) with the accumulator pinned to AGPRs.
// The compiler would otherwise move all 128 accumulator registers between
// AGPRs and VGPRs around every tile because of the (rare) rescale code.  The
// s_nop covers the VALU-write -> MFMA-read hazard of the operands, which the
// hazard recognizer does not see through asm.  For the same reason the
// compiler does not know the MFMA's result latency: a register copy of `o`
// placed right after this statement would read it before it is written.  The
// build (raftinfer_amd/asm_check.py) scans this file's assembly and fails on
// any such read; the drain below covers the reads the kernel itself makes.
__device__ __forceinline__ void mfma_acc_agpr(floatx16 &o, bf16x8 a, bf16x8 b) {
  asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(o) : "v"(a), "v"(b));
}
// o *= s for an AGPR-resident accumulator.  The empty asm statements pin the
// copy to VGPRs inside this (rare) rescale path; without them the compiler
// hoists the AGPR -> VGPR copies of all accumulators onto every tile.
__device__ __forceinline__ void scale_agpr(floatx16 &o, float s) {
  floatx16 x = o;
  asm volatile("" : "+v"(x));
#pragma unroll
  for (int i = 0; i < 16; ++i) x[i] *= s;
  asm volatile("" : "+v"(x));
  o = x;
}
// Wait states after the last such MFMA before VALU code reads its result.
__device__ __forceinline__ void mfma_drain() { asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3" ::: "memory"); }

__device__ __forceinline__ float fexp2(float x) { return __builtin_amdgcn_exp2f(x); }

// The q producer's RMSNorm + RoPE applied in place to the staged Q rows, bit
// for bit.  Sliced form (rotary pairs a multiple of 32; norm_rope_256_slice):
// eight lanes per row, so a wave finishes its 8 rows at once with one LDS
// round trip.
__device__ __forceinline__ void norm_rope_rows_sliced(bf16_bits *q, int r, int g, const float *weight,
                                                      bool weight_f32, int pairs, const float *rot,
                                                      float epsilon) {
  bf16_bits *row = q + r * kHeadDim;
  u32x4 raw[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) raw[j] = *reinterpret_cast<const u32x4 *>(row + (((4 * g + j) ^ swz(r)) << 3));
  float x[32], w[32], v[32];
  unpack_bf16x32(raw, x);
  load_slice_weights(weight, weight_f32, g, w);
  norm_rope_256_slice(x, w, g, pairs, rot, epsilon, v);
  u32x4 out[4];
  pack_bf16x32(v, out);
#pragma unroll
  for (int j = 0; j < 4; ++j) *reinterpret_cast<u32x4 *>(row + (((4 * g + j) ^ swz(r)) << 3)) = out[j];
}

// Lane-wise form (any rotary width): rows row0 .. row0+7 (one per token slot,
// rot[0..7]) one at a time, lane l owning dims 4l .. 4l+3 (8 bytes of logical
// chunk l / 2).
__device__ __forceinline__ void norm_rope_rows_lanewise(bf16_bits *q, int row0, int lane, const float *weight,
                                                        bool weight_f32, int pairs, const float (*rot)[kHeadDim],
                                                        float epsilon) {
  float w[4];
  if (weight_f32) {
    const float4 x = reinterpret_cast<const float4 *>(weight)[lane];
    w[0] = x.x; w[1] = x.y; w[2] = x.z; w[3] = x.w;
  } else {
    const u32x2 x = reinterpret_cast<const u32x2 *>(weight)[lane];
    w[0] = bf16_lo(x[0]); w[1] = bf16_hi(x[0]); w[2] = bf16_lo(x[1]); w[3] = bf16_hi(x[1]);
  }
#pragma unroll
  for (int rr = 0; rr < 8; ++rr) {
    const int r = row0 + rr;
    u32x2 *slot = reinterpret_cast<u32x2 *>(q + chunk_offset(r, lane >> 1) + 4 * (lane & 1));
    const u32x2 raw = *slot;
    const float x[4] = {bf16_lo(raw[0]), bf16_hi(raw[0]), bf16_lo(raw[1]), bf16_hi(raw[1])};
    float v[4];
    norm_rope_256_lane(x, w, lane, pairs, rot[rr], epsilon, v);
    *slot = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
  }
}

} // namespace prefill
} // namespace raftinfer::amd
