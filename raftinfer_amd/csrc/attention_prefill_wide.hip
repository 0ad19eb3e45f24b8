// Causal gated GQA prefill attention for long key ranges (gfx950 bf16 MFMA, the
// Qwen3.5 signature): the same arithmetic as prefill_mfma_kernel on a schedule
// that keeps the matrix units busy.
//
// prefill_mfma_kernel runs each wave's tile as a chain (wait, QK^T, softmax, PV)
// at one wave per SIMD, so the matrix units idle through the softmax and through
// most of the loads: 1.75 us per round of four 32-key tiles, where the MFMAs of
// its 32 columns take 0.5.  Here
//   - a wave holds NB = 1 or 2 blocks of 32 columns (4 heads x 8 tokens), so a K
//     or V operand read from LDS feeds NB MFMAs, with the Q operands in registers
//     and the O^T accumulators in the accumulation registers by number;
//   - S(n + 1) = K Q^T runs on the matrix unit while the vector unit turns S(n)
//     into probabilities, and the rest of them and the max of S(n + 1) are formed
//     behind the MFMAs of PV(n).  One wave issues at most an instruction every
//     four clocks, so the instructions around the MFMAs are counted: loads set
//     their LDS address once each and take their row from the instruction's
//     offset, operand addresses of a pair of steps share an exclusive-or;
//   - K and V tiles stream through a ring of five LDS slots per key group, loaded
//     by LDS-direct loads three or four ring items ahead, one load behind each
//     MFMA group;
//   - KS = 4 key groups: each wave streams its own 32-key tiles (no barriers in
//     the loop); KS = 2: two waves with 64 columns each share a group's tiles,
//     which halves the bytes and LDS writes per column for one barrier per item.
//     Counters (share of the wave cycles that the matrix units are busy / that vector
//     instructions issue / that a wave waits): NB = 1, 512
//     tokens behind 3584: 32 / 30 / 27%, one chain per SIMD; NB = 2, 2000 tokens: 26 /
//     35 / 33%, the start, the end and the last workgroups; 6001 tokens: 49 / 34 / 19%
//     at 2.07 GHz; 2048 behind 30000: 60 / 36 / 16% at 1.70 GHz, where the other kernels
//     run at 2.3 to 2.4: the card's power bounds the last two (1.0 to 1.2 PFLOP/s, the
//     rate that a bf16 matrix product of 8192^3 reaches here).
//   - a masked key has probability 0, and 0 times an infinite or NaN value is not 0:
//     with NB = 2, a workgroup whose own tokens have such values throws its sums away
//     and forms them again, the tiles that mask key by key (careful_tile).  With 8
//     tokens per workgroup (here and in prefill_mfma_kernel) such a value reaches the
//     up to seven tokens before it in its workgroup; the look for them would take
//     0.8 of 54 us there (512 tokens behind 3584).
// prefill_plan (attention_prefill_mfma.hip) says which form takes a call.
#include "prefill_mfma.hpp"
#include "prefill_tile.hpp"

#include <type_traits>
#include <utility>

namespace raftinfer::amd {
namespace {

using namespace prefill;

__device__ __forceinline__ bf16x8 lds_read_b128(unsigned addr) {
  return __builtin_bit_cast(bf16x8, *(const __attribute__((address_space(3))) u32x4 *)(std::uintptr_t)(addr));
}
__device__ __forceinline__ u32x2 lds_read_tr16(unsigned addr) {
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4v *)(std::uintptr_t)(addr)));
}
template <typename T> __device__ __forceinline__ T *lds_ptr(unsigned addr) {
  return (T *)(__attribute__((address_space(3))) T *)(std::uintptr_t)(addr);
}
// off ^ x and off + a, as asm so that the results are formed where they are used:
// hoisted out of the tile loop, the offsets of all loads took registers from the
// Q operands.
template <unsigned kXor, unsigned kAdd> __device__ __forceinline__ std::uint32_t load_offset(std::uint32_t off) {
  std::uint32_t x = off;
  if constexpr (kXor != 0) asm volatile("v_xor_b32 %0, %2, %1" : "=v"(x) : "v"(off), "n"(kXor));
  if constexpr (kAdd != 0) asm volatile("v_add_u32 %0, %2, %1" : "=v"(x) : "v"(x), "n"(kAdd));
  return x;
}
// load_lds_b128 with an instruction offset, which the hardware adds to both the
// memory and the LDS address.
template <int kOffset>
__device__ __forceinline__ void load_lds_b128_at(const void *base, std::uint32_t voff, unsigned lds) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2 offset:%3"
               :
               : "s"(lds), "v"(voff), "s"(base), "n"(kOffset)
               : "memory");
}

// The O^T accumulators (2 column blocks x 8 dim blocks x 16 registers) fill the
// 256 accumulation registers, and are addressed by number from asm: block
// `kAcc` (8 b + nb) is a[16 kAcc : 16 kAcc + 15].  Left to the register
// allocator, values of this size were copied and spilled around every tile.  What is
// left of the vector registers does not hold everything with NB = 2: 23 to 28 (KS
// = 4) or 33 and 34 (KS = 2) are spilled, none of them inside the loop over whole
// tiles; two steps of the loop over the last tiles have 16 to 19 scratch accesses, and
// the wait for a reload also waits for the LDS-direct loads in front of it.
// acc_fence clobbers the whole file around every tile, so the compiler keeps
// nothing of its own there (the statements in between carry no clobber list,
// which took minutes to compile); the build checks that no instruction outside
// asm uses an accumulation register (raftinfer_amd/asm_check.py).
#define RAFT_AGPR10(n) \
  "a" #n "0", "a" #n "1", "a" #n "2", "a" #n "3", "a" #n "4", "a" #n "5", "a" #n "6", "a" #n "7", "a" #n "8", "a" #n "9"
#define RAFT_ALL_AGPRS \
  "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", \
      RAFT_AGPR10(1), RAFT_AGPR10(2), RAFT_AGPR10(3), RAFT_AGPR10(4), \
      RAFT_AGPR10(5), RAFT_AGPR10(6), RAFT_AGPR10(7), RAFT_AGPR10(8), \
      RAFT_AGPR10(9), RAFT_AGPR10(10), RAFT_AGPR10(11), RAFT_AGPR10(12), \
      RAFT_AGPR10(13), RAFT_AGPR10(14), RAFT_AGPR10(15), RAFT_AGPR10(16), \
      RAFT_AGPR10(17), RAFT_AGPR10(18), RAFT_AGPR10(19), RAFT_AGPR10(20), \
      RAFT_AGPR10(21), RAFT_AGPR10(22), RAFT_AGPR10(23), RAFT_AGPR10(24), \
      "a250", "a251", "a252", "a253", "a254", "a255"

__device__ __forceinline__ void acc_fence() { asm volatile("" : : : RAFT_ALL_AGPRS); }
template <int kAcc> __device__ __forceinline__ void acc_mfma(bf16x8 a, bf16x8 b) {
  asm volatile("v_mfma_f32_32x32x16_bf16 a[%0:%1], %2, %3, a[%0:%1]"
               :
               : "n"(16 * kAcc), "n"(16 * kAcc + 15), "v"(a), "v"(b));
}
// s = a b and s += a b with s in vector registers.  A statement writes no
// result for another 19 wait states: new_max reads S(t + 4) only after PV(t),
// and after the first tile's chain the kernel drains.
__device__ __forceinline__ void s_mfma_zero(floatx16 &s, bf16x8 a, bf16x8 b) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(s) : "v"(a), "v"(b));
}
__device__ __forceinline__ void s_mfma(floatx16 &s, bf16x8 a, bf16x8 b) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(s) : "v"(a), "v"(b));
}
template <int kReg> __device__ __forceinline__ void acc_set(float x) {
  asm volatile("v_accvgpr_write_b32 a[%0], %1" : : "n"(kReg), "v"(x));
}
template <int kReg> __device__ __forceinline__ float acc_get() {
  float x;
  asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(x) : "n"(kReg));
  return x;
}
// max(a, b, c).  As asm: on results of the asm MFMAs fmaxf adds a canonicalising
// instruction per operand.
__device__ __forceinline__ float max3(float a, float b, float c) {
  float x;
  asm volatile("v_max3_f32 %0, %1, %2, %3" : "=v"(x) : "v"(a), "v"(b), "v"(c));
  return x;
}
// The wait states between the last s_mfma of a chain and the first use of s.
template <int NB> __device__ __forceinline__ void s_drain(floatx16 (&s)[NB]) {
  if constexpr (NB == 2)
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3" : "+v"(s[0]), "+v"(s[1]));
  else
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3" : "+v"(s[0]));
}
// f(integral_constant<int, 0>) .. f(integral_constant<int, N - 1>)
template <int N, typename F> __device__ __forceinline__ void static_for(F &&f) {
  [&]<int... I>(std::integer_sequence<int, I...>) __attribute__((always_inline)) { (f(std::integral_constant<int, I>{}), ...); }
  (std::make_integer_sequence<int, N>{});
}

// NB column blocks of 32 per wave, KS key groups (see the head of the file).
template <int NB, int KS> struct Plan {
  static constexpr int kShare = kWaves / KS;            // waves that share a key group's tiles
  static constexpr int kTok = 8 * NB * kShare;          // query tokens per workgroup
  static constexpr int kRows = 4 * kTok;                // columns, one staged row each
  static constexpr unsigned kSlot = 8192u * kShare;     // ring slot: 16 / 32 rows of 512 bytes
  static constexpr unsigned kArea = 5 * kSlot;          // a key group's part of LDS
  static constexpr int kGroupRows = kRows / KS;         // staged rows in each group's area
  static constexpr unsigned kRowsAt = kShare == 1 ? 4 * kSlot : 3 * kSlot;
  static constexpr int kParts = 8 / KS;                 // dims blocks that a wave finishes
};

// ---- f32 cache (F32).  K, V, the probabilities and all sums stay f32: f32 MFMAs
// have a sixteenth of the bf16 rate, so a value is split into three bf16 parts of
// 8 bits (x = h + m + l exactly, by truncation), and the products of parts that
// matter at f32 precision are summed in f32.  Cache rows appended from bf16
// activations have m = l = 0; each half tile is checked, and takes the products
// with m and l only if some value has more bits.  A tile is 16 keys, so its halves
// are the same 8 KiB ring items; S and PV are not overlapped.  It is a chain at one
// wave per SIMD: 35 to 39% of the wave cycles issue vector instructions (the checks and
// packing of 8192 values per wave and tile), 32 to 35% wait, the matrix units are busy
// for 12 to 16%; with general f32 values 51, 31 and 14%.  512 tokens on a token-major
// f32 cache: 866 us with one wave per row and fp32 FMAs, now 31 to 33; behind 4000
// tokens 17,900 us, now 197 where the past is exact in bf16 (rows that bf16 activations
// appended) and 507 where it is not.
__device__ __forceinline__ std::uint32_t high_pair(float a, float b) { // truncated bf16 of (a, b)
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
// What x - h is; 0 for an infinity.
__device__ __forceinline__ float rest_part(float x) {
  const float h = __uint_as_float(__float_as_uint(x) & 0xFFFF0000u);
  return __builtin_isinf(x) ? 0.f : x - h;
}
__device__ __forceinline__ bf16x8 high_operand(const float (&x)[8]) {
  return __builtin_bit_cast(bf16x8, u32x4{high_pair(x[0], x[1]), high_pair(x[2], x[3]), high_pair(x[4], x[5]),
                                          high_pair(x[6], x[7])});
}
__device__ __forceinline__ floatx4 lds_read_f4(unsigned addr) {
  return *(const __attribute__((address_space(3))) floatx4 *)(std::uintptr_t)(addr);
}
__device__ __forceinline__ float lds_read_f1(unsigned addr) {
  return *(const __attribute__((address_space(3))) float *)(std::uintptr_t)(addr);
}
template <bool F32> using CacheElem = std::conditional_t<F32, float, bf16_bits>;

// The output of a workgroup's tile (kTok query tokens of one KV head, as
// prefill_wide_kernel deals them) where its own tokens have infinite or NaN values:
// one column block (4 heads x 8 tokens) per wave over all keys, a 32-key tile at a
// time in the wave's own part of LDS (K and V rows of 512 bytes, 16-byte chunk c of
// row r at c ^ swz(r)), the tiles that mask key by key.  A chain of latencies, about
// 3.4 us a tile (6001 tokens, every value NaN: 1.27 ms in place of 0.34).  It derives
// everything anew and is not the streaming loop run again: values kept for either
// took registers in the streaming loop and its ends (6001 tokens of finite values:
// 308 us, 313 to 318 with a second run of the loop, 449 with the Q operands kept).
// Its arguments are the kernel's, loaded again for the same reason: kept in scalar
// registers they were spilled (fused, 1500 tokens behind 2000: 115.5 us in place of
// 107.2).
struct WideArguments { // as the kernel argument segment holds those of prefill_wide_kernel
  const bf16_bits *query, *key_in, *value_in, *gate;
  bf16_bits *output;
  const bf16_bits *cache;
  std::size_t tokens, max_ctx, past;
  PrefillNormRope nq;
};
static_assert(sizeof(WideArguments) == 104, "the arguments lie without padding in between");
template <int kTok, bool HeadMajor, bool FromInput, bool NormQ>
__device__ __forceinline__ void careful_tile(unsigned lds0) {
  auto arguments = reinterpret_cast<std::uintptr_t>(__builtin_amdgcn_kernarg_segment_ptr());
  asm volatile("" : "+s"(arguments));
  const auto &args = *(const __attribute__((address_space(4))) WideArguments *)arguments;
  const bf16_bits *query = args.query, *key_in = args.key_in, *value_in = args.value_in, *gate = args.gate;
  const bf16_bits *cache = args.cache;
  bf16_bits *output = args.output;
  const std::size_t tokens = args.tokens, max_ctx = args.max_ctx, past = args.past;
  const PrefillNormRope nq{args.nq.weight, args.nq.weight_f32, args.nq.pairs, args.nq.ratio, args.nq.epsilon};
  int tid = threadIdx.x;
  unsigned block = blockIdx.x;
  asm volatile("" : "+v"(tid), "+s"(block)); // (nothing of this is formed before the streaming loop)
  const int lane = tid & 63, col = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (wave >= kTok / 8) return;
  const std::size_t qtile = ceil_div_u(tokens, kTok) - 1 - (2 * (block >> 3) + (block & 1u));
  const std::size_t kv_head = (block & 7u) >> 1, t0 = qtile * kTok;
  const std::size_t q_rows = tokens - t0 < kTok ? tokens - t0 : kTok, key_end = past + t0 + q_rows;
  // Token slot and head of row r (0..31) of the wave's block.
  auto slot = [&](int r) __attribute__((always_inline)) {
    const std::size_t tt = 8 * wave + (r & 7);
    return tt < q_rows ? tt : q_rows - 1;
  };
  auto io_row = [&](int r) __attribute__((always_inline)) {
    return ((t0 + slot(r)) * kQueryHeads + kv_head * kGroup + (r >> 3)) * kHeadDim;
  };
  const unsigned k_at = lds0 + 40960u * wave, v_at = k_at + 16384u;
  constexpr std::size_t q_row_elems = NormQ ? 2 * kHeadDim : kHeadDim;
  // ---- Q rows in the place of K, normalised there, then in registers
#pragma unroll 1
  for (int i = 0; i < 16; ++i) {
    const int r = 2 * i + half;
    load_lds_b128(query + (t0 * kQueryHeads + kv_head * kGroup) * q_row_elems,
                  static_cast<std::uint32_t>(slot(r) * kQueryHeads + (r >> 3)) * (q_row_elems * 2) + 16u * (col ^ swz(r)),
                  k_at + 1024u * i);
  }
  if constexpr (NormQ) { // weight and rotation tables in the place of V
    const std::uint32_t bytes = nq.weight_f32 ? 1024u : 512u;
    load_lds_b128(nq.weight, 16u * lane < bytes ? 16u * lane : bytes - 16u, v_at);
    auto rot = reinterpret_cast<float(*)[kHeadDim]>(lds_ptr<float>(v_at + 1024u));
    for (int i = lane; i < 8 * nq.pairs; i += kWave) {
      const int s = i / nq.pairs, pp = i - s * nq.pairs;
      float cs, sn;
      rope_cos_sin(pp, past + t0 + slot(s), nq.ratio, cs, sn);
      rot[s][pp] = cs;
      rot[s][nq.pairs + pp] = sn;
    }
    wait_vm<0>();
    wave_lds_order();
    const float *weight = lds_ptr<float>(v_at);
#pragma unroll 1
    for (int h = 0; h < 4; ++h) { // the 8 token slots of a head
      bf16_bits *staged = lds_ptr<bf16_bits>(k_at + 4096u * h);
      if (nq.pairs % 32 == 0)
        norm_rope_rows_sliced(staged, lane >> 3, lane & 7, weight, nq.weight_f32, nq.pairs, rot[lane >> 3], nq.epsilon);
      else
        norm_rope_rows_lanewise(staged, 0, lane, weight, nq.weight_f32, nq.pairs, rot, nq.epsilon);
    }
    wave_lds_order();
  }
  wait_vm<0>();
  const unsigned k_lane = k_at + col * 512u + 16u * (half ^ swz(col)); // chunk 2 kk + half: exclusive-or 32 kk
  bf16x8 q[16];
#pragma unroll
  for (int kk = 0; kk < 16; ++kk) q[kk] = lds_read_b128(k_lane ^ (32u * kk));
  // V^T operand of dims block nb, key step kb: as in prefill_wide_kernel
  const int vg = (lane >> 4) & 1, vr = lane & 15, vrow = 4 * half + (vr >> 2);
  const unsigned v_lane = v_at + vrow * 512u + 16u * ((2 * vg + ((vr & 3) >> 1)) ^ swz(vrow)) + 8u * (vr & 1);
  constexpr std::uint32_t row_bytes = (HeadMajor && !FromInput ? kHeadDim : kKvHeads * kHeadDim) * 2;
  const bf16_bits *k_src = FromInput ? key_in + kv_head * kHeadDim : cache + cache_row(HeadMajor, 0, kv_head, max_ctx);
  const bf16_bits *v_src = FromInput ? value_in + kv_head * kHeadDim : k_src + max_ctx * kKvHeads * kHeadDim;
  const float scale = kLog2e / 16.0f;
  const std::ptrdiff_t pos = static_cast<std::ptrdiff_t>(past + t0 + slot(col));
  acc_fence();
  static_for<128>([&](auto i) __attribute__((always_inline)) { acc_set<i>(0.f); });
  float m_run = -INFINITY, l_run = 0.f;
#pragma unroll 1
  for (std::size_t k0 = 0; k0 < key_end; k0 += kKTile) {
    const std::uint32_t last = static_cast<std::uint32_t>(key_end - 1 - k0 < 31 ? key_end - 1 - k0 : 31);
    wait_lgkm0(); // the last tile has been read
#pragma unroll 1
    for (int i = 0; i < 16; ++i) {
      const std::uint32_t r = 2 * i + half, voff = (r < last ? r : last) * row_bytes + 16u * (col ^ swz(r));
      load_lds_b128(k_src + k0 * (row_bytes / 2), voff, k_at + 1024u * i);
      load_lds_b128(v_src + k0 * (row_bytes / 2), voff, v_at + 1024u * i);
    }
    wait_vm<0>();
    floatx16 s;
    static_for<16>([&](auto kk) __attribute__((always_inline)) {
      bf16x8 a = lds_read_b128(k_lane ^ (32u * kk));
      asm volatile("s_nop 1" : "+v"(a)); // (wait states before the MFMA)
      if constexpr (kk == 0) s_mfma_zero(s, a, q[kk]); else s_mfma(s, a, q[kk]);
    });
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3" : "+v"(s));
    const std::ptrdiff_t lim = pos - static_cast<std::ptrdiff_t>(k0); // last visible key
    float x[16], top = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      x[i] = (i >> 2) * 8 + 4 * half + (i & 3) > lim ? -INFINITY : s[i] * scale;
      top = fmaxf(top, x[i]);
    }
    top = max_xor32(top);
    const bool grow = top > m_run + kLazyRescale;
    if (__builtin_amdgcn_ballot_w64(grow) != 0) {
      const float sc = grow ? fexp2(m_run - top) : 1.0f;
      l_run *= sc;
      m_run = grow ? top : m_run;
      static_for<128>([&](auto i) __attribute__((always_inline)) { acc_set<i>(acc_get<i>() * sc); });
    }
    const float m_ref = m_run == -INFINITY ? 0.f : m_run;
    std::uint32_t p[8]; // P^T, bf16 pairs in accumulator order
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      p[i] = pack_bf16x2(fexp2(x[2 * i] - m_ref), fexp2(x[2 * i + 1] - m_ref));
      l_run = dot2_bf16(p[i], 0x3F803F80u, l_run);
    }
    acc_fence();
    if (k0 + kKTile - 1 <= past + t0) {
      static_for<16>([&](auto st) __attribute__((always_inline)) {
        constexpr int kb = st & 1, nb = st >> 1;
        const unsigned a = (v_lane ^ (64u * nb)) + 8192u * kb;
        const u32x2 lo = lds_read_tr16(a), hi = lds_read_tr16(a + 4096u);
        bf16x8 v = __builtin_bit_cast(bf16x8, u32x4{lo[0], lo[1], hi[0], hi[1]});
        bf16x8 w = __builtin_bit_cast(bf16x8, u32x4{p[4 * kb], p[4 * kb + 1], p[4 * kb + 2], p[4 * kb + 3]});
        asm volatile("s_nop 1" : "+v"(v), "+v"(w));
        acc_mfma<nb>(v, w);
      });
    } else {
#pragma unroll 1
      for (int key = 0; key < kKTile; ++key) {
        std::uint32_t pair = p[0]; // the key's probability, in the lanes of its half, then in the whole column
#pragma unroll
        for (int i = 1; i < 8; ++i) {
          pair = i == 2 * (key >> 3) + ((key & 3) >> 1) ? p[i] : pair;
          asm volatile("" : "+v"(pair)); // a chain of selects, not an array in scratch
        }
        float w = (key & 1) != 0 ? bf16_hi(pair) : bf16_lo(pair);
        const float other = xor32(w);
        w = ((key >> 2) & 1) != half ? other : w;
        const unsigned row = v_at + key * 512u;
        static_for<32>([&](auto quad) __attribute__((always_inline)) { // dims 8 quad + 4 half .. +3
          const u32x2 y = *lds_ptr<u32x2>(row + 16u * (quad ^ swz(key)) + 8u * half);
          static_for<4>([&](auto e) __attribute__((always_inline)) {
            const float v = (e & 1) != 0 ? bf16_hi(y[e >> 1]) : bf16_lo(y[e >> 1]);
            const float was = acc_get<4 * quad + e>();
            acc_set<4 * quad + e>(key <= lim ? fmaf(w, v, was) : was);
          });
        });
        acc_fence();
      }
    }
    mfma_drain();
  }
  const float inv = 1.0f / (l_run + xor32(l_run));
  const bf16_bits *gate_row = NormQ ? query + 2 * io_row(col) + kHeadDim : gate + io_row(col);
  if (static_cast<std::size_t>(8 * wave + (col & 7)) >= q_rows) return;
  static_for<32>([&](auto quad) __attribute__((always_inline)) {
    constexpr int d = 8 * quad;
    const u32x2 g = *reinterpret_cast<const u32x2 *>(gate_row + d + 4 * half);
    *reinterpret_cast<u32x2 *>(output + io_row(col) + d + 4 * half) =
        u32x2{pack_bf16x2(acc_get<4 * quad>() * inv * sigmoid_gate(bf16_lo(g[0])),
                          acc_get<4 * quad + 1>() * inv * sigmoid_gate(bf16_hi(g[0]))),
              pack_bf16x2(acc_get<4 * quad + 2>() * inv * sigmoid_gate(bf16_lo(g[1])),
                          acc_get<4 * quad + 3>() * inv * sigmoid_gate(bf16_hi(g[1])))};
  });
}

template <int NB, int KS, bool HeadMajor, bool FromInput, bool NormQ, bool F32 = false>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1))) void prefill_wide_kernel(
    const bf16_bits *__restrict__ query, const bf16_bits *key_in, const bf16_bits *value_in,
    const bf16_bits *gate, bf16_bits *__restrict__ output, CacheElem<F32> *__restrict__ cache,
    std::size_t tokens, std::size_t max_ctx, std::size_t past, PrefillNormRope nq) {
  static_assert(!(NormQ && FromInput), "the fused producer path reads K/V from the cache");
  static_assert(!F32 || (NB == 1 && KS == 4 && !FromInput && !NormQ), "the form of the f32 cache");
  constexpr int kTileKeys = F32 ? 16 : kKTile;
  using P = Plan<NB, KS>;
  constexpr int kTok = P::kTok, kShare = P::kShare;
  constexpr unsigned kSlot = P::kSlot;
  __shared__ __attribute__((aligned(16384))) unsigned char sh[KS * P::kArea];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int col = lane & 31;  // MFMA column of a block: head_in_group * 8 + token
  const int half = lane >> 5; // k-half of the MFMA operands
  const std::size_t n_qtiles = ceil_div_u(tokens, kTok);
  const unsigned xcd = blockIdx.x & 7u;
  const std::size_t slot_index = 2 * (blockIdx.x >> 3) + (xcd & 1u);
  if (slot_index >= n_qtiles) return; // padding of an odd tile count
  const std::size_t qtile = n_qtiles - 1 - slot_index;
  const std::size_t kv_head = xcd >> 1;
  const std::size_t t0 = qtile * kTok;
  const std::size_t q_rows = tokens - t0 < kTok ? tokens - t0 : kTok;
  const std::size_t key_end = past + t0 + q_rows;
  const std::size_t n_tiles = (key_end + kTileKeys - 1) / kTileKeys;
  const std::size_t plane = max_ctx * kKvHeads * kHeadDim;
  const float scale = kLog2e / 16.0f;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave % KS, cg = wave / KS; // key group, column group
  // Token slot of staged row r = 32 blk + c, clamped to the tile's tokens, and
  // the element offset of its row in the query / gate / output layout [T][16][256].
  auto slot_row = [&](int r) __attribute__((always_inline)) {
    const std::size_t tt = 8 * (r >> 5) + (r & 7);
    return tt < q_rows ? tt : q_rows - 1;
  };
  auto io_row = [&](int r) __attribute__((always_inline)) {
    return ((t0 + slot_row(r)) * kQueryHeads + kv_head * kGroup + ((r & 31) >> 3)) * kHeadDim;
  };
  constexpr std::size_t q_row_elems = NormQ ? 2 * kHeadDim : kHeadDim;
  const bf16_bits *gate_src = NormQ ? query + kHeadDim : gate;
  const unsigned lds0 = lds_address(sh);
  const unsigned ring = lds0 + kg * P::kArea;
  // LDS address of a staged row (Q, gate, output): 16-byte chunk k at k ^ swz(r).
  auto row_at = [&](int r) __attribute__((always_inline)) {
    return lds0 + (r / P::kGroupRows) * P::kArea + P::kRowsAt + (r % P::kGroupRows) * 512u;
  };

  // The lane index again: what is derived from it is not computed before the tile
  // loop and kept (or spilled) over it.  With NB = 2 the index is counted anew as well:
  // kept in a register, it had the tail of the loop spill 55 in place of 34 (KS = 2,
  // NormQ: 2500 tokens 100 us in place of 92; without NormQ, 600 behind 800: 36.5 in
  // place of 35.6).  With KS = 4 and NormQ it is better kept (1500: 56.8 against 59.3).
  auto late_lane = [&]() __attribute__((always_inline)) {
    int l;
    if constexpr (NB == 2 && (kShare > 1 || !NormQ)) {
      asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    } else {
      l = threadIdx.x & 63;
      asm volatile("" : "+v"(l));
    }
    return l;
  };
  // ---- staging: ring items of 8 loads (1 KiB) per wave.
  //   K, own tiles: one dims half of the 32-key tile, 4 half-rows a load (rows
  //     4i + lane / 16), 16-byte chunk c (0..15) at c ^ f, f = 4 (row % 4) + row / 4 % 4;
  //   K, shared tiles: 16 rows, two whole rows a load (2i + lane / 32), chunk c
  //     (0..31) at c ^ f, f = row / 2 % 8 + 8 (row % 2);
  //   V: 16 rows likewise, f = 4 (row / 2 % 2) + 8 (row % 2).
  // The 16 rows of a ds_read_b128 pass over K then share no bank, nor do the 4
  // rows x 64 bytes of a ds_read_b64_tr_b16 pass over V, whose rows 8 apart have
  // the same f.  A load's offset is the lane's, an exclusive-or and an addition.
  constexpr std::uint32_t row_bytes =
      (HeadMajor && !FromInput ? kHeadDim : kKvHeads * kHeadDim) * sizeof(CacheElem<F32>);
  const CacheElem<F32> *k_src, *v_src;
  if constexpr (FromInput) {
    k_src = key_in + kv_head * kHeadDim;
    v_src = value_in + kv_head * kHeadDim;
  } else {
    k_src = cache + cache_row(HeadMajor, 0, kv_head, max_ctx);
    v_src = k_src + plane;
  }
  constexpr int k_rows = kShare == 1 ? 4 : 2; // rows per K load
  const int hrow = kShare == 1 ? lane >> 4 : half;
  const std::uint32_t v_off = half * row_bytes + 16u * (col ^ (8 * half));
  const std::uint32_t k_off = kShare == 1 ? hrow * row_bytes + 16u * ((lane & 15) ^ (4 * hrow)) : v_off;
  auto load_k = [&](const unsigned char *base, unsigned to, auto ic) __attribute__((always_inline)) {
    constexpr int i = ic, x = kShare == 1 ? i & 3 : i;
    load_lds_b128_at<1024 * (i & 3)>(base + 4096 * (i >> 2), load_offset<16u * x, i *(k_rows * row_bytes - 1024)>(k_off),
                                     to + 4096u * (i >> 2));
  };
  auto load_v = [&](const unsigned char *base, unsigned to, auto ic) __attribute__((always_inline)) {
    constexpr int i = ic;
    load_lds_b128_at<1024 * (i & 3)>(base + 4096 * (i >> 2), load_offset<64u * (i & 1), i *(2 * row_bytes - 1024)>(v_off),
                                     to + 4096u * (i >> 2));
  };
  auto base_of = [&](const CacheElem<F32> *src, std::size_t row) __attribute__((always_inline)) {
    return reinterpret_cast<const unsigned char *>(src) + row * row_bytes;
  };
  // The same for items that may reach past key_end: those rows re-read the last
  // one (their scores are masked).  k0: first row; for K of own tiles `half_tile`
  // is the dims half.
  auto load_clamped = [&](const CacheElem<F32> *src, auto is_v, std::size_t k0, int half_tile, unsigned to, auto ic)
      __attribute__((always_inline)) {
    constexpr int i = ic;
    constexpr bool dims_half = kShare == 1 && !is_v;
    const std::size_t first = k0 < key_end ? k0 : key_end - 1;
    const std::uint32_t last = static_cast<std::uint32_t>(key_end - 1 - first < 31 ? key_end - 1 - first : 31);
    const int l = late_lane();
    const std::uint32_t r = dims_half ? 4 * i + (l >> 4) : 2 * i + (l >> 5);
    const std::uint32_t chunk = dims_half ? (l & 15) ^ (4 * (l >> 4)) ^ (i & 3)
                                          : (l & 31) ^ (8 * (l >> 5)) ^ (is_v ? 4 * (i & 1) : i);
    // (no instruction offset here: less 1024 i, the offset of a clamped row could
    // be negative, and it is unsigned)
    load_lds_b128_at<0>(base_of(src, first) + (dims_half ? 256 * half_tile : 0), (r < last ? r : last) * row_bytes + 16u * chunk,
                        to + 1024u * i);
  };
  // Tile of this wave's key group, counted from its first, and the first row of
  // its share `sub` of it.
  auto tile_row = [&](std::size_t n, int sub) __attribute__((always_inline)) {
    return (n * KS + kg) * kTileKeys + 16 * sub;
  };
  constexpr std::false_type kIsK{};
  constexpr std::true_type kIsV{};
  // An f32 half tile (16 rows of 128 dims, two rows a load): chunk c (0..31) at
  // c ^ row for K (a ds_read_b128 pass takes one chunk of 16 rows), at c ^ 8
  // (row / 4 % 2) for V (a ds_read_b32 takes 32 dims of two rows 4 apart).
  auto load_f32 = [&](bool is_v, std::size_t tile, int hh, unsigned to) __attribute__((always_inline)) {
    const std::size_t k0 = (tile * KS + kg) * kTileKeys;
    const int l = late_lane();
    const std::uint32_t last = static_cast<std::uint32_t>(key_end - 1 - k0 < 15 ? key_end - 1 - k0 : 15);
    const unsigned char *base = base_of(is_v ? v_src : k_src, k0) + 512 * hh;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const std::uint32_t r = 2 * i + (l >> 5), f = is_v ? 8 * ((i >> 1) & 1) : r;
      load_lds_b128_at<0>(base, (r < last ? r : last) * row_bytes + 16u * ((l & 31) ^ f), to + 1024u * i);
    }
  };
  auto load_item = [&](const CacheElem<F32> *src, auto is_v, std::size_t k0, int half_tile, unsigned to)
      __attribute__((always_inline)) {
    static_for<8>([&](auto i) __attribute__((always_inline)) { load_clamped(src, is_v, k0, half_tile, to, i); });
  };
  // This wave's kRows / 4 staged rows from a [T][16][row elems] source, two per load.
  auto issue_rows = [&](const bf16_bits *src, int lane) __attribute__((always_inline)) {
    constexpr int n = P::kRows / kWaves;
    const unsigned to = row_at(n * wave);
#pragma unroll
    for (int i = 0; i < n / 2; ++i) {
      const int r = n * wave + 2 * i + (lane >> 5);
      const std::uint32_t voff =
          static_cast<std::uint32_t>(slot_row(r) * kQueryHeads + ((r & 31) >> 3)) * (q_row_elems * 2) +
          16u * ((lane & 31) ^ swz(r));
      load_lds_b128(src + (t0 * kQueryHeads + kv_head * kGroup) * q_row_elems, voff, to + 1024u * i);
    }
  };
  // Tiles of this key group; with shared tiles every wave runs the same number
  // (the barriers), the tiles past n_tiles fully masked.
  const std::size_t m = kShare > 1 ? ceil_div_u(n_tiles, KS)
                                   : (n_tiles > static_cast<std::size_t>(kg) ? ceil_div_u(n_tiles - kg, KS) : 0);
  // Ring items of 8 loads per wave each (i = tile):
  //   own tiles (half tiles h):     K0 K1(0) K0 K1(1) V0 V1(0) K0 K1(2) V0 V1(1) ...
  //   shared tiles (whole tiles):   K(0) K(1) V(0) K(2) V(1) K(3) V(2) ...
  // Item n uses slot n % 5.  While item n is read, item n + 4 is loaded into the
  // slot of n - 1 (own tiles), or item n + 3 into the slot of n - 2, which every
  // wave has left when it passes the barrier in front of item n (shared tiles).
  issue_rows(query, lane);
  const int my = kShare > 1 ? cg : 0; // this wave's share of an item
  const unsigned part = 8192u * my;
  auto issue_start = [&](int from, int to) __attribute__((always_inline)) {
    if constexpr (F32) { // K0 K1 V0 V1 of tile 0
      for (int n = from; n < to; ++n)
        if (m != 0) load_f32(n >= 2, 0, n & 1, ring + n * kSlot);
    } else if constexpr (kShare == 1) {
      for (int n = from; n < to; ++n)
        if (static_cast<std::size_t>(n >> 1) < m) load_item(k_src, kIsK, tile_row(n >> 1, 0), n & 1, ring + n * kSlot);
    } else {
      for (int n = from; n < to; ++n)
        if (n == 0) load_item(k_src, kIsK, tile_row(0, my), 0, ring + part);
        else if (n == 1 && m > 1) load_item(k_src, kIsK, tile_row(1, my), 0, ring + kSlot + part);
        else if (n == 2) load_item(v_src, kIsV, tile_row(0, my), 0, ring + 2 * kSlot + part);
    }
  };
  constexpr int kFirstItems = kShare == 1 ? 2 : 1; // before the norm, 2 / 1 items (K(0))
  constexpr int kStartItems = kShare == 1 ? 4 : 3;
  if constexpr (NormQ) {
    // The norm weight (512 B bf16 or 1 KiB f32) into the second-last group's
    // slot 2, the rotation tables of the tile's (up to kTok) positions into the
    // last group's slots 2, 3 (own tiles) or 1, 2; the items of those slots go
    // out once they have been used.
    const unsigned w_at = lds0 + (KS - 2) * P::kArea + 2 * kSlot;
    const unsigned rot_at = lds0 + (KS - 1) * P::kArea + (kShare == 1 ? 2 : 1) * kSlot;
    if (wave == 0) {
      const std::uint32_t bytes = nq.weight_f32 ? 1024u : 512u;
      const std::uint32_t off = 16u * lane < bytes ? 16u * lane : bytes - 16u;
      load_lds_b128(nq.weight, off, w_at);
    }
    issue_start(0, kFirstItems);
    auto rot = reinterpret_cast<float(*)[kHeadDim]>(lds_ptr<float>(rot_at));
    for (int i = tid; i < kTok * nq.pairs; i += kThreads) {
      const int s = i / nq.pairs, pp = i - s * nq.pairs;
      const std::size_t tt = static_cast<std::size_t>(s) < q_rows ? s : q_rows - 1;
      float cs, sn;
      rope_cos_sin(pp, past + t0 + tt, nq.ratio, cs, sn);
      rot[s][pp] = cs;
      rot[s][nq.pairs + pp] = sn;
    }
    if (m != 0) wait_vm<8 * kFirstItems>(); else wait_vm<0>();
    __syncthreads();
    const float *weight = lds_ptr<float>(w_at);
    constexpr int n = P::kRows / kWaves;
#pragma unroll
    for (int g8 = 0; g8 < n / 8; ++g8) { // eight rows (one head, the 8 token slots of a block) at a time
      const int row0 = n * wave + 8 * g8;
      const float(*rows)[kHeadDim] = rot + 8 * (row0 >> 5);
      bf16_bits *staged = lds_ptr<bf16_bits>(row_at(row0));
      if (nq.pairs % 32 == 0)
        norm_rope_rows_sliced(staged, lane >> 3, lane & 7, weight, nq.weight_f32, nq.pairs, rows[lane >> 3],
                              nq.epsilon);
      else
        norm_rope_rows_lanewise(staged, 0, lane, weight, nq.weight_f32, nq.pairs, rows, nq.epsilon);
    }
    __syncthreads(); // every row is normalised, the tables have been read
    issue_start(kFirstItems, kStartItems);
  } else {
    issue_start(0, kStartItems);
  }
  acc_fence();
  static_for<128 * NB>([](auto r) __attribute__((always_inline)) { acc_set<r>(0.f); });
  acc_fence();
  float m_run[NB], l_run[NB]; // reference max (exp2 domain) and this lane's sum, of column `col`
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    m_run[b] = -INFINITY;
    l_run[b] = 0.f;
  }
  if constexpr (!NormQ) {
    // this wave's Q rows have landed, then every other wave's
    if constexpr (F32) {
      if (m != 0) wait_vm<32>(); else wait_vm<0>();
    } else if constexpr (kShare == 1) {
      if (m > 1) wait_vm<32>(); else if (m != 0) wait_vm<16>(); else wait_vm<0>();
    } else {
      if (m > 1) wait_vm<24>(); else wait_vm<16>();
    }
    __syncthreads();
  }
  // Q^T operands stay in registers: block b, k-step kk holds chunk 2 kk + half
  // of the staged row of its column.
  bf16x8 qa[NB][16];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const unsigned row = row_at(32 * (NB * cg + b) + col);
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) qa[b][kk] = lds_read_b128(row + 16u * ((2 * kk + half) ^ swz(col)));
  }
  wait_lgkm0();
  __syncthreads(); // the staged rows' slots are free

  // Slot addresses of ring items n - 1, n, n + 1, n + 2, n + 3 (n = the next to
  // be read); the slot of n - 2 is that of n + 3.
  unsigned p0 = ring + 4 * kSlot, p1 = ring, p2 = ring + kSlot, p3 = ring + 2 * kSlot, p4 = ring + 3 * kSlot;
  auto advance = [&](int items) __attribute__((always_inline)) {
    for (int i = 0; i < items; ++i) {
      const unsigned x = p0;
      p0 = p1; p1 = p2; p2 = p3; p3 = p4; p4 = x;
    }
  };
  // K operand of k-step kk: chunk 2 kk + half of row col.  V^T operand
  // (transposed read) of dims block nb and key step kb: rows 16 kb + 4 half +
  // r / 4 and 8 below, dims 32 nb + 16 (g & 1) + 4 (r & 3).
  const unsigned k_lane = kShare == 1 ? col * 256u + 16u * (half ^ (4 * (col & 3) + ((col >> 2) & 3)))
                                      : col * 512u + 16u * (half ^ (((col >> 1) & 7) + 8 * (col & 1)));
  const int vg = (lane >> 4) & 1, vr = lane & 15, vrow = 4 * half + (vr >> 2);
  const unsigned v_lane = vrow * 512u + 16u * ((2 * vg + ((vr & 3) >> 1)) ^ (4 * ((vrow >> 1) & 1) + 8 * (vrow & 1))) +
                          8u * (vr & 1);
  bf16x8 op[4];       // operands of the next four MFMA groups, across phases
  unsigned at = 0;    // lane address of the tile part being read
  unsigned at_x = 0;  // ... of the exclusive-or group being read
  // Order within a phase, s = 0..15: with own tiles k-step s (the dims halves
  // one after the other), with shared tiles k-steps s / 2 and s / 2 + 8 in turn;
  // for V, key step s / 8 and dims blocks s / 2 % 4 and s / 2 % 4 + 4 in turn.
  // Such pairs share their exclusive-or.
  auto k_operand = [&](auto sc) __attribute__((always_inline)) {
    constexpr int s = sc;
    if constexpr (kShare == 1) return lds_read_b128(at ^ (32u * (s & 7)));
    if constexpr (s % 2 == 0) at_x = at ^ (32u * (s >> 1));
    return lds_read_b128(at_x + 256u * (s & 1));
  };
  auto v_operand = [&](auto sc) __attribute__((always_inline)) {
    constexpr int s = sc;
    constexpr unsigned off = 256u * (s & 1) + (kShare > 1 ? 8192u * (s >> 3) : 0u);
    if constexpr (s % 2 == 0) at_x = at ^ (64u * ((s >> 1) & 3));
    const u32x2 lo = lds_read_tr16(at_x + off), hi = lds_read_tr16(at_x + off + 4096u);
    return __builtin_bit_cast(bf16x8, u32x4{lo[0], lo[1], hi[0], hi[1]});
  };

  floatx16 s0[NB], s1[NB];
  std::uint32_t pk[NB][8]; // P^T, bf16 pairs in accumulator order
  float m_ref[NB], mx[NB]; // mx: max of the next S over this lane's keys

  // Pair u of the probabilities (blocks in turn): registers 2i, 2i+1 of an S.
  // The sum takes the same bf16 probabilities as the PV product.  The empty asm
  // keeps the pair where it is written, among the MFMAs.
  auto soft_pair = [&](const floatx16(&s)[NB], auto uc) __attribute__((always_inline)) {
    constexpr int b = uc % NB, i = uc / NB;
    const float x0 = fexp2(fmaf(s[b][2 * i], scale, -m_ref[b]));
    const float x1 = fexp2(fmaf(s[b][2 * i + 1], scale, -m_ref[b]));
    pk[b][i] = pack_bf16x2(x0, x1);
    l_run[b] = dot2_bf16(pk[b][i], 0x3F803F80u, l_run[b]);
    asm volatile("" : "+v"(pk[b][i]), "+v"(l_run[b]));
  };
  // Pairs [A, B) spread over the steps of a part of `steps` steps.
  auto soft_step = [&](const floatx16(&s)[NB], auto sc, auto from, auto count, auto steps) __attribute__((always_inline)) {
    constexpr int u0 = sc * count / steps, u1 = (sc + 1) * count / steps;
    static_for<u1 - u0>([&](auto k) __attribute__((always_inline)) {
      soft_pair(s, std::integral_constant<int, from + u0 + k>{});
    });
  };
  constexpr std::integral_constant<int, 0> c0{};
  constexpr std::integral_constant<int, 6 * NB> kQkPairs{}; // of 8 NB; all of key step 0 among them
  constexpr std::integral_constant<int, 2 * NB> kPvPairs{};
  constexpr std::integral_constant<int, 16> c16{};
  constexpr std::integral_constant<int, 8> c8{};
  auto lane_max = [&](const floatx16(&s)[NB]) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      mx[b] = max3(s[b][0], s[b][1], s[b][2]);
#pragma unroll
      for (int i = 3; i < 15; i += 2) mx[b] = max3(mx[b], s[b][i], s[b][i + 1]);
      mx[b] = max3(mx[b], s[b][15], s[b][15]);
    }
  };
  // The new reference max from mx, and the (rare) rescale of the accumulators:
  // it moves only when a column max grows by more than 2^8.
  auto new_max = [&](bool first) __attribute__((always_inline)) {
    float mm[NB];
    bool grow[NB], any_grow = false;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      mm[b] = max_xor32(mx[b]) * scale;
      grow[b] = mm[b] > m_run[b] + kLazyRescale;
      any_grow |= grow[b];
    }
    if (first) { // nothing is accumulated yet
#pragma unroll
      for (int b = 0; b < NB; ++b) m_run[b] = grow[b] ? mm[b] : m_run[b];
    } else if (__builtin_amdgcn_ballot_w64(any_grow) != 0) {
      mfma_drain();
      static_for<NB>([&](auto b) __attribute__((always_inline)) {
        const float sc = grow[b] ? fexp2(m_run[b] - mm[b]) : 1.0f;
        l_run[b] *= sc;
        m_run[b] = grow[b] ? mm[b] : m_run[b];
        static_for<128>([&](auto r) __attribute__((always_inline)) { acc_set<128 * b + r>(acc_get<128 * b + r>() * sc); });
      });
    }
    // a column whose keys so far are all masked keeps m = -inf
#pragma unroll
    for (int b = 0; b < NB; ++b) m_ref[b] = m_run[b] == -INFINITY ? 0.f : m_run[b];
  };
  // Keys past each column's position score -inf (register i: key 8 (i / 4) +
  // 4 half + i % 4 of the tile at row k0).
  auto mask = [&](floatx16(&s)[NB], std::size_t k0) __attribute__((always_inline)) {
    const int le = late_lane();
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const std::ptrdiff_t rel = static_cast<std::ptrdiff_t>(past + t0 + slot_row(32 * (NB * cg + b) + (le & 31))) -
                                 static_cast<std::ptrdiff_t>(k0) - 4 * (le >> 5);
      const int lim = rel < -1 ? -1 : (rel > kKTile ? kKTile : static_cast<int>(rel));
#pragma unroll
      for (int i = 0; i < 16; ++i) s[b][i] = (i >> 2) * 8 + (i & 3) > lim ? -INFINITY : s[b][i];
    }
    lane_max(s);
  };
  auto none = [](auto) __attribute__((always_inline)) {};
  // Waits until the wave's share of the next ring item has landed, with n of its
  // later loads outstanding, and with shared tiles until every wave's has.
  auto ready = [&](auto n) __attribute__((always_inline)) {
    wait_vm<n>();
    if constexpr (kShare > 1) __builtin_amdgcn_s_barrier();
  };
  // out = K Q^T of the tile at `at`, on the matrix unit, while (soft) the vector
  // unit turns s into probabilities.  load(step) issues the wave's loads of this
  // phase, second_ready / next_ready wait for the second half tile and for V.
  auto qk = [&](auto soft, const floatx16(&s)[NB], floatx16(&out)[NB], auto load, auto second_ready, auto next_ready,
                unsigned k_second, unsigned v_slot)
      __attribute__((always_inline)) {
    static_for<16>([&](auto st) __attribute__((always_inline)) {
      constexpr int q = st & 3, kk = kShare == 1 ? +st : (st >> 1) + 8 * (st & 1);
      if constexpr (st == 0) s_mfma_zero(out[0], op[q], qa[0][kk]); else s_mfma(out[0], op[q], qa[0][kk]);
      if constexpr (soft) soft_step(s, st, c0, kQkPairs, c16);
      if constexpr (NB == 2) {
        if constexpr (st == 0) s_mfma_zero(out[1], op[q], qa[1][kk]); else s_mfma(out[1], op[q], qa[1][kk]);
      }
      if constexpr (kShare == 1 && st == 4) {
        second_ready();
        at = k_second + k_lane;
      }
      if constexpr (soft && st == 12) {
        next_ready();
        at = v_slot + v_lane;
      }
      if constexpr (st < 12) op[q] = k_operand(std::integral_constant<int, st + 4>{});
      else if constexpr (soft) op[q] = v_operand(std::integral_constant<int, st - 12>{});
      load(st);
      if constexpr (st % 2 == 1) acc_fence();
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  // O += V^T P^T, the remaining probabilities of s formed on the way; with kMax
  // the max of `next` over this lane's keys is taken and the next K tile begun.
  auto pv = [&](auto kMax, const floatx16(&s)[NB], const floatx16(&next)[NB], auto load, auto second_ready,
                auto next_ready, unsigned v_second, unsigned k_a) __attribute__((always_inline)) {
    acc_fence();
    auto p_operand = [&](int b, int kb) __attribute__((always_inline)) {
      return __builtin_bit_cast(bf16x8, u32x4{pk[b][4 * kb], pk[b][4 * kb + 1], pk[b][4 * kb + 2], pk[b][4 * kb + 3]});
    };
    static_for<16>([&](auto st) __attribute__((always_inline)) {
      constexpr int q = st & 3, kb = st >> 3, nb = ((st >> 1) & 3) + 4 * (st & 1);
      acc_mfma<nb>(op[q], p_operand(0, kb));
      if constexpr (st < 8) soft_step(s, st, kQkPairs, kPvPairs, c8);
      if constexpr (NB == 2) acc_mfma<8 + nb>(op[q], p_operand(1, kb));
      if constexpr (st == 4 && kShare == 1) {
        second_ready();
        at = v_second + v_lane;
      }
      if constexpr (kMax && st == 12) {
        next_ready();
        at = k_a + k_lane;
      }
      if constexpr (st < 12) op[q] = v_operand(std::integral_constant<int, st + 4>{});
      else if constexpr (kMax) op[q] = k_operand(std::integral_constant<int, st - 12>{});
      if constexpr (kMax && st >= 8) { // two values of each block per step
        constexpr int i = 2 * (st - 8);
#pragma unroll
        for (int b = 0; b < NB; ++b) mx[b] = max3(st == 8 ? next[b][0] : mx[b], next[b][i], next[b][i + 1]);
      }
      load(st);
      if constexpr (st % 4 == 3) acc_fence();
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  // Step n: tile n (its S in s, mx its max) -> O, with S(n + 1) formed on the
  // way.  kSteady: every item loaded in the step exists and is whole.  The two S
  // buffers alternate by name: a copy placed right behind the MFMA that writes
  // it would read it too early.
  std::size_t n = 0;
  const std::size_t full = key_end / kKTile; // whole tiles, then those of the group
  const std::size_t whole = full > static_cast<std::size_t>(kg) ? ceil_div_u(full - kg, KS) : 0;
  auto step = [&](auto kSteady, floatx16(&s)[NB], floatx16(&next)[NB]) __attribute__((always_inline)) {
    if constexpr (!kSteady)
      if (tile_row(n, 0) + kKTile - 1 > past + t0) mask(s, tile_row(n, 0));
    new_max(n == 0);
    if constexpr (kShare == 1) {
      // QK reads K(n+1) (items n', n'+1) and loads K(n+2), PV reads V(n) and loads V(n+1).
      const bool more = kSteady || n + 2 < m;
      auto wait = [&]() __attribute__((always_inline)) { if (more) wait_vm<20>(); else wait_vm<4>(); };
      const unsigned char *kb0 = base_of(k_src, tile_row(n + 2, 0)), *vb0 = base_of(v_src, tile_row(n + 1, 0));
      qk(std::true_type{}, s, next,
         [&](auto st) __attribute__((always_inline)) {
           constexpr std::integral_constant<int, st & 7> i{};
           const unsigned to = st < 8 ? p0 : p1;
           if constexpr (kSteady) load_k(st < 8 ? kb0 : kb0 + 256, to, i);
           else if (more) load_clamped(k_src, kIsK, tile_row(n + 2, 0), st >> 3, to, i);
         },
         wait, wait, p2, p3);
      pv(std::true_type{}, s, next,
         [&](auto st) __attribute__((always_inline)) {
           constexpr std::integral_constant<int, st & 7> i{};
           const unsigned to = st < 8 ? p2 : p3; // V0(n) has been read after half the phase
           if constexpr (kSteady) load_v(st < 8 ? vb0 : vb0 + 16 * row_bytes, to, i);
           else load_clamped(v_src, kIsV, tile_row(n + 1, st >> 3), 0, to, i);
         },
         wait, wait, p4, p0);
      advance(4);
    } else {
      // QK reads K(n+1) and loads V(n+1), PV reads V(n) and loads K(n+3).
      const bool more2 = kSteady || n + 2 < m, more3 = kSteady || n + 3 < m;
      const unsigned char *vb0 = base_of(v_src, tile_row(n + 1, my)), *kb0 = base_of(k_src, tile_row(n + 3, my));
      qk(std::true_type{}, s, next,
         [&](auto st) __attribute__((always_inline)) {
           if constexpr (st % 2 == 0) {
             constexpr std::integral_constant<int, st / 2> i{};
             const unsigned to = p4 + part; // item n' + 3
             if constexpr (kSteady) load_v(vb0, to, i);
             else load_clamped(v_src, kIsV, tile_row(n + 1, my), 0, to, i);
           }
         },
         [] {}, [&]() __attribute__((always_inline)) { if (more2) ready(std::integral_constant<int, 14>{}); else ready(std::integral_constant<int, 6>{}); },
         0, p2);
      pv(std::true_type{}, s, next,
         [&](auto st) __attribute__((always_inline)) {
           if constexpr (st % 2 == 0) {
             constexpr std::integral_constant<int, st / 2> i{};
             const unsigned to = p0 + part; // item n' + 4, the slot of n' - 1
             if constexpr (kSteady) load_k(kb0, to, i);
             else if (more3) load_clamped(k_src, kIsK, tile_row(n + 3, my), 0, to, i);
           }
         },
         [] {},
         [&]() __attribute__((always_inline)) { if (more3) ready(std::integral_constant<int, 14>{}); else ready(std::integral_constant<int, 0>{}); },
         0, p3);
      advance(2);
    }
    ++n;
  };
  if constexpr (F32) {
    // Ring items K0 K1 V0 V1 of one tile after the other; while item n is read,
    // n + 4 (the same part of the next tile) is loaded into the slot of n - 1.
    const int row = lane & 15;
    const bool low = (lane & 16) != 0;
    const unsigned kf_lane = row * 512u + 16u * ((2 * half) ^ row);
    const unsigned vf_lane = half * 2048u + 128u * half + 4u * col;
    for (; n < m; ++n) {
      const bool more = n + 1 < m;
      auto next_item = [&](bool is_v, int hh, int left) __attribute__((always_inline)) {
        if (more || left == 3) wait_vm<24>(); else if (left == 2) wait_vm<16>(); else if (left == 1) wait_vm<8>(); else wait_vm<0>();
        if (more) load_f32(is_v, n + 1, hh, p0);
      };
      // S^T: A rows r and r + 16 both hold key r.  High parts first (rows 16..
      // repeat them and are not used); if some value has more bits, rows 0..15
      // the middle and rows 16.. the low parts into a second accumulator.
      floatx16 sm = floatx16{};
      bool rest = false;
      static_for<2>([&](auto hh) __attribute__((always_inline)) {
        next_item(false, hh, 3 - hh);
        const unsigned a0 = p1 + kf_lane;
        auto values = [&](unsigned base, int kk, float(&y)[8]) __attribute__((always_inline)) { // kk in the half
          const unsigned a = (base ^ (64u * (kk & 3))) + 256u * (kk >> 2);
          const floatx4 u = lds_read_f4(a), w = lds_read_f4(a ^ 16u);
          y[0] = u[0]; y[1] = u[1]; y[2] = u[2]; y[3] = u[3];
          y[4] = w[0]; y[5] = w[1]; y[6] = w[2]; y[7] = w[3];
        };
        std::uint32_t bits = 0;
        float y[4][8];
        static_for<4>([&](auto j) __attribute__((always_inline)) { values(a0, j, y[j]); });
        static_for<8>([&](auto kk) __attribute__((always_inline)) {
          float(&v)[8] = y[kk & 3];
#pragma unroll
          for (int j = 0; j < 8; ++j) bits |= __float_as_uint(v[j]);
          bf16x8 a = high_operand(v);
          asm volatile("s_nop 1" : "+v"(a)); // (wait states before the MFMA)
          if constexpr (hh == 0 && kk == 0) s_mfma_zero(s0[0], a, qa[0][0]); else s_mfma(s0[0], a, qa[0][8 * hh + kk]);
          if constexpr (kk < 4) values(a0, kk + 4, y[kk & 3]);
          __builtin_amdgcn_sched_barrier(0);
        });
        if (__builtin_amdgcn_ballot_w64((bits & 0xFFFFu) != 0) != 0) {
          rest = true;
          static_for<8>([&](auto kk) __attribute__((always_inline)) {
            float v[8];
            values(a0, kk, v);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
              v[j] = rest_part(v[j]);
              v[j] = low ? rest_part(v[j]) : v[j];
            }
            bf16x8 a = high_operand(v);
            asm volatile("s_nop 1" : "+v"(a), "+v"(sm));
            s_mfma(sm, a, qa[0][8 * hh + kk]);
            __builtin_amdgcn_sched_barrier(0);
          });
        }
        advance(1);
      });
      asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3" : "+v"(s0[0]), "+v"(sm));
      float x[8]; // scores, then probabilities, of keys 4 half + 0..3 and 8 + 4 half + 0..3
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = s0[0][i];
      if (rest)
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] += sm[i] + sm[8 + i];
      const std::ptrdiff_t rel = static_cast<std::ptrdiff_t>(past + t0 + slot_row(col)) -
                                 static_cast<std::ptrdiff_t>(tile_row(n, 0));
      const int lim = rel < -1 ? -1 : (rel > kTileKeys ? kTileKeys : static_cast<int>(rel)); // last visible key
      float mxs = -INFINITY;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        x[i] = (i >> 2) * 8 + 4 * half + (i & 3) > lim ? -INFINITY : x[i] * scale;
        mxs = fmaxf(mxs, x[i]);
      }
      mxs = max_xor32(mxs);
      const bool grow = mxs > m_run[0] + kLazyRescale;
      if (n == 0) {
        m_run[0] = grow ? mxs : m_run[0];
      } else if (__builtin_amdgcn_ballot_w64(grow) != 0) {
        mfma_drain();
        const float sc = grow ? fexp2(m_run[0] - mxs) : 1.0f;
        l_run[0] *= sc;
        m_run[0] = grow ? mxs : m_run[0];
        static_for<128>([&](auto r) __attribute__((always_inline)) { acc_set<r>(acc_get<r>() * sc); });
      }
      const float mref = m_run[0] == -INFINITY ? 0.f : m_run[0];
      float pr[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        x[i] = fexp2(x[i] - mref);
        l_run[0] += x[i];
        pr[i] = rest_part(x[i]);
      }
      const bf16x8 ph = high_operand(x), pm = high_operand(pr);
#pragma unroll
      for (int i = 0; i < 8; ++i) pr[i] = rest_part(pr[i]);
      const bf16x8 pl = high_operand(pr);
      // O^T += V^T P^T, 4 dims blocks per half tile.
      static_for<2>([&](auto hh) __attribute__((always_inline)) {
        next_item(true, hh, 1 - hh);
        acc_fence();
        const unsigned a0 = p1 + vf_lane;
        auto values = [&](int nb, float(&y)[8]) __attribute__((always_inline)) { // dim 32 nb + col of the half
#pragma unroll
          for (int i = 0; i < 8; ++i) y[i] = lds_read_f1((a0 ^ (128u * nb)) + 512u * (8 * (i >> 2) + (i & 3)));
        };
        std::uint32_t bits = 0;
        float finite = 0.f; // NaN if some value is an infinity or a NaN
        bf16x8 vh[4];
        static_for<4>([&](auto nb) __attribute__((always_inline)) {
          float y[8];
          values(nb, y);
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            bits |= __float_as_uint(y[i]);
            finite = fmaf(y[i], 0.f, finite);
          }
          vh[nb] = high_operand(y);
        });
        if (__builtin_amdgcn_ballot_w64(finite != finite) != 0) {
          // key by key: a zero part of a probability times an infinity is not 0,
          // and a masked key must not count
          mfma_drain();
#pragma unroll 1
          for (int key = 0; key < kTileKeys; ++key) {
            float w = x[0]; // the key's probability, in the lanes of its half, then in the whole column
#pragma unroll
            for (int i = 1; i < 8; ++i) {
              w = i == 4 * (key >> 3) + (key & 3) ? x[i] : w;
              asm volatile("" : "+v"(w)); // a chain of selects, not an array in scratch
            }
            const float other = xor32(w);
            w = ((key >> 2) & 1) != half ? other : w;
            const unsigned a = p1 + key * 512u;
            static_for<64>([&](auto r) __attribute__((always_inline)) {
              constexpr int i = r & 15, d = 32 * (r >> 4) + 8 * (i >> 2) + (i & 3); // + 4 half
              const float y = lds_read_f1(a + 16u * ((((d + 4 * half) >> 2)) ^ (8 * ((key >> 2) & 1))) + 4u * (d & 3));
              const float was = acc_get<64 * hh + r>();
              acc_set<64 * hh + r>(key <= lim ? fmaf(w, y, was) : was);
            });
            acc_fence();
          }
        } else {
          // the smallest products first
          asm volatile("s_nop 1" : "+v"(vh[0]), "+v"(vh[1]), "+v"(vh[2]), "+v"(vh[3]));
          static_for<4>([&](auto nb) __attribute__((always_inline)) { acc_mfma<4 * hh + nb>(vh[nb], pl); });
          static_for<4>([&](auto nb) __attribute__((always_inline)) { acc_mfma<4 * hh + nb>(vh[nb], pm); });
          static_for<4>([&](auto nb) __attribute__((always_inline)) { acc_mfma<4 * hh + nb>(vh[nb], ph); });
          if (__builtin_amdgcn_ballot_w64((bits & 0xFFFFu) != 0) != 0) {
            static_for<4>([&](auto nb) __attribute__((always_inline)) {
              float y[8];
              values(nb, y);
#pragma unroll
              for (int i = 0; i < 8; ++i) y[i] = rest_part(y[i]);
              bf16x8 vm = high_operand(y);
#pragma unroll
              for (int i = 0; i < 8; ++i) y[i] = rest_part(y[i]);
              bf16x8 vl = high_operand(y);
              asm volatile("s_nop 1" : "+v"(vm), "+v"(vl));
              acc_mfma<4 * hh + nb>(vl, ph);
              acc_mfma<4 * hh + nb>(vm, pm);
              acc_mfma<4 * hh + nb>(vm, ph);
            });
          }
        }
        acc_fence();
        advance(1);
      });
    }
    mfma_drain();
    wait_lgkm0();
  } else if (m != 0) {
    // S of the first tile: items 0, 1 (own) or 0 (shared) are read, V(0) or K(2) loaded.
    if constexpr (kShare == 1) {
      if (m > 1) wait_vm<24>(); else wait_vm<8>(); // K(0), first half
      at = p1 + k_lane;
      static_for<4>([&](auto i) __attribute__((always_inline)) { op[i] = k_operand(i); });
      qk(std::false_type{}, s0, s0,
         [&](auto st) __attribute__((always_inline)) {
           load_clamped(v_src, kIsV, tile_row(0, st >> 3), 0, st < 8 ? p0 : p1,
                        std::integral_constant<int, st & 7>{});
         },
         [&]() __attribute__((always_inline)) { if (m > 1) wait_vm<20>(); else wait_vm<4>(); }, [] {}, p2, 0);
      advance(2);
    } else {
      if (m > 1) wait_vm<16>(); else wait_vm<8>();
      __builtin_amdgcn_s_barrier();
      at = p1 + k_lane;
      static_for<4>([&](auto i) __attribute__((always_inline)) { op[i] = k_operand(i); });
      qk(std::false_type{}, s0, s0,
         [&](auto st) __attribute__((always_inline)) {
           if constexpr (st % 2 == 0)
             if (m > 2) load_clamped(k_src, kIsK, tile_row(2, my), 0, p4 + part, std::integral_constant<int, st / 2>{});
         },
         [] {}, [] {}, 0, 0);
      advance(1);
    }
    s_drain(s0);
    lane_max(s0);
    if (m > 1) { // K(1)
      if constexpr (kShare == 1)
        wait_vm<24>(); // first half
      else if (m > 2)
        ready(std::integral_constant<int, 16>{});
      else
        ready(std::integral_constant<int, 8>{});
      at = p1 + k_lane;
      static_for<4>([&](auto i) __attribute__((always_inline)) { op[i] = k_operand(i); });
    }
    constexpr std::size_t kReach = kShare == 1 ? 2 : 3; // the furthest tile that a step loads
    while (n + kReach + 1 < whole) {
      step(std::true_type{}, s0, s1);
      step(std::true_type{}, s1, s0);
    }
    while (n + 1 < m) {
      step(std::false_type{}, s0, s1);
      if (n + 1 >= m) {
        s_drain(s1);
#pragma unroll
        for (int b = 0; b < NB; ++b) s0[b] = s1[b];
        break;
      }
      step(std::false_type{}, s1, s0);
    }
    if (tile_row(n, 0) + kKTile - 1 > past + t0) mask(s0, tile_row(n, 0));
    new_max(n == 0);
    static_for<kQkPairs>([&](auto u) __attribute__((always_inline)) { soft_pair(s0, u); });
    if constexpr (kShare == 1) {
      wait_vm<8>(); // V(last), first half
      at = p3 + v_lane;
    } else {
      ready(std::integral_constant<int, 0>{});
      at = p2 + v_lane;
    }
    static_for<4>([&](auto i) __attribute__((always_inline)) { op[i] = v_operand(i); });
    pv(std::false_type{}, s0, s0, none, [] { wait_vm<0>(); }, [] {}, p4, 0);
    mfma_drain();
    wait_lgkm0();
  }
  // ---- epilogue.  The gate rows take the staged rows' place, and the partials
  // are merged one column block at a time: wave (kg, cg) finishes dims 256 / KS
  // kg .. of the columns that it shares with the other waves of column group cg.
  if constexpr (kShare > 1) __syncthreads(); // every wave has left the ring
  const int lane_e = late_lane(), col_e = lane_e & 31, half_e = lane_e >> 5;
  issue_rows(gate_src, lane_e);
  constexpr int kApp = FromInput ? kTok / 4 : 1; // this workgroup's cache rows: 2 planes x kTok tokens x 32 pieces
  [[maybe_unused]] u32x4 app[kApp];
  auto app_at = [&](int j, int &pl, int &tok, int &piece) __attribute__((always_inline)) {
    const int idx = kWave * wave + lane_e + kThreads * j;
    pl = idx / (kTok * 32);
    tok = (idx >> 5) % kTok;
    piece = idx & 31;
  };
  if constexpr (FromInput) {
#pragma unroll
    for (int j = 0; j < kApp; ++j) {
      int pl, tok, piece;
      app_at(j, pl, tok, piece);
      const std::size_t tt = static_cast<std::size_t>(tok) < q_rows ? tok : q_rows - 1;
      app[j] = *reinterpret_cast<const u32x4 *>((pl ? value_in : key_in) +
                                                ((t0 + tt) * kKvHeads + kv_head) * kHeadDim + 8 * piece);
    }
  }
  auto store_app = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < kApp; ++j) {
      int pl, tok, piece;
      app_at(j, pl, tok, piece);
      if (static_cast<std::size_t>(tok) < q_rows)
        *reinterpret_cast<u32x4 *>(cache + pl * plane + cache_row(HeadMajor, t0 + tok, kv_head, max_ctx) + 8 * piece) =
            app[j];
    }
  };
  // Pieces of the V rows that some of the tile's columns must not see, or that are
  // read again in the place of rows past the last (with FromInput the V half of app).
  constexpr bool kWatch = NB == 2;
  constexpr int kOwn = kWatch && !FromInput ? kTok / 8 : 1;
  [[maybe_unused]] u32x4 own[kOwn];
  if constexpr (kWatch && !FromInput) {
#pragma unroll
    for (int j = 0; j < kOwn; ++j) {
      const std::size_t idx = kWave * wave + lane_e + kThreads * j, tt = idx >> 5 == 0 ? 1 : idx >> 5;
      own[j] = *reinterpret_cast<const u32x4 *>(base_of(v_src, past + t0 + (tt < q_rows ? tt : q_rows - 1)) +
                                                16 * (idx & 31));
    }
  }
  bool again = false; // one of them is an infinity or a NaN
  // Partials of wave (g, cg) for the finisher of part q (q != g): [dims block of
  // the part][register quad][lane] float4; its (max, sum) of each block, [2 NB][lane].
  constexpr unsigned kPartBytes = P::kParts * 4 * kWave * sizeof(float4);
  auto part_at = [&](int g, int q) __attribute__((always_inline)) {
    return lds_ptr<float4>(lds0 + g * P::kArea + (kShare == 1 ? q : cg) * kPartBytes);
  };
  auto ml_at = [&](int g) __attribute__((always_inline)) {
    return lds_ptr<float>(lds0 + g * P::kArea + (kShare == 1 ? g * kPartBytes : 2 * kPartBytes + cg * 1024u));
  };
  auto flag_at = [&](int w) __attribute__((always_inline)) { // what wave w found in its pieces
    return lds_ptr<unsigned>(lds0 + (w % KS) * P::kArea + (kShare == 1 ? w % KS : 2) * kPartBytes + 4096u + 4u * (w / KS));
  };
  static_for<NB>([&](auto bc) __attribute__((always_inline)) {
    constexpr int b = bc;
    if (b != 0) __syncthreads(); // block b - 1 has been merged
    floatx16 f[P::kParts]; // this wave's share of its own part
#pragma unroll
    for (int j = 0; j < P::kParts; ++j) f[j] = floatx16{};
    acc_fence();
    static_for<KS>([&](auto q) __attribute__((always_inline)) {
      constexpr int r0 = 16 * (8 * b + P::kParts * q);
      if (q != kg) {
        float4 *to = part_at(kg, q);
        static_for<4 * P::kParts>([&](auto ji) __attribute__((always_inline)) {
          constexpr int r = r0 + 4 * ji;
          to[kWave * ji + lane_e] = make_float4(acc_get<r>(), acc_get<r + 1>(), acc_get<r + 2>(), acc_get<r + 3>());
        });
      } else {
        static_for<16 * P::kParts>([&](auto i) __attribute__((always_inline)) { f[i / 16][i % 16] = acc_get<r0 + i>(); });
      }
    });
    acc_fence();
    if (b == 0) {
#pragma unroll
      for (int bb = 0; bb < NB; ++bb) {
        ml_at(kg)[(2 * bb) * kWave + lane_e] = m_run[bb];
        ml_at(kg)[(2 * bb + 1) * kWave + lane_e] = l_run[bb];
      }
      if constexpr (kWatch) {
        std::uint32_t bad = 0; // an exponent of all ones, plus one, carries into the sign's place
        auto look = [&](const u32x4 &x) __attribute__((always_inline)) {
#pragma unroll
          for (int e = 0; e < 4; ++e) bad |= ((x[e] & 0x7F807F80u) + 0x00800080u) & 0x80008000u;
        };
#pragma unroll
        for (int j = 0; j < (FromInput ? kApp / 2 : kOwn); ++j)
          if constexpr (FromInput) look(app[kApp / 2 + j]); else look(own[j]);
        const unsigned any = __builtin_amdgcn_ballot_w64(bad != 0) != 0;
        if (lane_e == 0) *flag_at(wave) = any;
      }
      wait_vm<0>(); // this wave's gate rows
    }
    __syncthreads();
    // The gate pieces of this lane (its column's row, dims 8 k + 4 half .. +3 of
    // the part), read before the partials so that no round trip waits for another.
    constexpr int kChunks = 4 * P::kParts; // 16-byte chunks of a row's part
    const int r0 = 32 * (NB * cg + b);
    const unsigned row = row_at(r0 + col_e);
    auto gate_at = [&](int k) __attribute__((always_inline)) {
      return row + 16u * ((kChunks * kg + k) ^ swz(col_e)) + 8u * half_e;
    };
    u32x2 gp[kChunks];
#pragma unroll
    for (int k = 0; k < kChunks; ++k) gp[k] = *lds_ptr<u32x2>(gate_at(k));
    float mw[KS], lw[KS], mm = -INFINITY, lsum = 0.f;
#pragma unroll
    for (int g = 0; g < KS; ++g) {
      mw[g] = ml_at(g)[(2 * b) * kWave + lane_e];
      lw[g] = ml_at(g)[(2 * b + 1) * kWave + lane_e];
    }
    if constexpr (b == 0 && kWatch) {
      unsigned any = 0;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) any |= *flag_at(w);
      again = __builtin_amdgcn_readfirstlane(any) != 0;
    }
#pragma unroll
    for (int g = 0; g < KS; ++g) mm = fmaxf(mm, mw[g]);
#pragma unroll
    for (int g = 0; g < KS; ++g) {
      mw[g] = fexp2(mw[g] - mm); // a wave that saw no key has m = -inf and weight 0
      lsum += mw[g] * lw[g];
    }
    const float a_own = fexp2(m_run[b] - mm);
#pragma unroll
    for (int j = 0; j < P::kParts; ++j)
#pragma unroll
      for (int i = 0; i < 16; ++i) f[j][i] *= a_own;
#pragma unroll
    for (int g = 0; g < KS; ++g) {
      if (g == kg) continue;
      const float4 *from = part_at(g, kg);
#pragma unroll
      for (int j = 0; j < P::kParts; ++j)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
          const float4 x = from[kWave * (4 * j + i4) + lane_e];
          f[j][4 * i4] += mw[g] * x.x;
          f[j][4 * i4 + 1] += mw[g] * x.y;
          f[j][4 * i4 + 2] += mw[g] * x.z;
          f[j][4 * i4 + 3] += mw[g] * x.w;
        }
    }
    const float inv = 1.0f / (lsum + xor32(lsum));
    // The gate pieces become the gated outputs, which leave as whole lines.
#pragma unroll
    for (int j = 0; j < P::kParts; ++j)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        const u32x2 g = gp[4 * j + i4];
        const floatx16 &x = f[j];
        gp[4 * j + i4] = u32x2{pack_bf16x2(x[4 * i4] * inv * sigmoid_gate(bf16_lo(g[0])),
                                           x[4 * i4 + 1] * inv * sigmoid_gate(bf16_hi(g[0]))),
                               pack_bf16x2(x[4 * i4 + 2] * inv * sigmoid_gate(bf16_lo(g[1])),
                                           x[4 * i4 + 3] * inv * sigmoid_gate(bf16_hi(g[1])))};
      }
#pragma unroll
    for (int k = 0; k < kChunks; ++k) *lds_ptr<u32x2>(gate_at(k)) = gp[k];
    wave_lds_order(); // the rows' pieces are read back by other lanes of this wave
    constexpr int kPerStore = kWave / kChunks; // rows
#pragma unroll
    for (int i = 0; i < 32 / kPerStore; ++i) {
      const int c = kPerStore * i + lane_e / kChunks, k = kChunks * kg + lane_e % kChunks, r = r0 + c;
      if (!again && static_cast<std::size_t>(8 * (r >> 5) + (r & 7)) < q_rows)
        *reinterpret_cast<u32x4 *>(output + io_row(r) + 8 * k) = *lds_ptr<u32x4>(row_at(r) + 16u * (k ^ swz(c)));
    }
  });
  if constexpr (FromInput) store_app();
  if constexpr (kWatch) {
    if (!again) return;
    __syncthreads(); // the flags have been read
    careful_tile<kTok, HeadMajor, FromInput, NormQ>(lds0);
  }
}

void launch_f32(const bf16_bits *q, const bf16_bits *gate, bf16_bits *out, float *cache, std::size_t tokens,
                std::size_t max_ctx, std::size_t past, bool head_major, hipStream_t stream) {
  const unsigned grid = static_cast<unsigned>(8 * ceil_div_unchecked(ceil_div_unchecked(tokens, Plan<1, 4>::kTok), 2));
  auto go = [&](auto kernel) {
    kernel<<<grid, kThreads, 0, stream>>>(q, nullptr, nullptr, gate, out, cache, tokens, max_ctx, past,
                                          PrefillNormRope{});
  };
  go(head_major ? prefill_wide_kernel<1, 4, true, false, false, true>
                : prefill_wide_kernel<1, 4, false, false, false, true>);
}

template <int NB, int KS>
void launch(const bf16_bits *q, const bf16_bits *key, const bf16_bits *value, const bf16_bits *gate, bf16_bits *out,
            bf16_bits *cache, std::size_t tokens, std::size_t max_ctx, std::size_t past, bool head_major,
            bool fused_append, const PrefillNormRope *nq, hipStream_t stream) {
  // 8 workgroups (one per XCD) per pair of query tiles
  const unsigned grid =
      static_cast<unsigned>(8 * ceil_div_unchecked(ceil_div_unchecked(tokens, Plan<NB, KS>::kTok), 2));
  const PrefillNormRope arg = nq != nullptr ? *nq : PrefillNormRope{};
  auto go = [&](auto kernel) {
    kernel<<<grid, kThreads, 0, stream>>>(q, key, value, gate, out, cache, tokens, max_ctx, past, arg);
  };
  if (nq != nullptr)
    go(head_major ? prefill_wide_kernel<NB, KS, true, false, true> : prefill_wide_kernel<NB, KS, false, false, true>);
  else if (fused_append)
    go(head_major ? prefill_wide_kernel<NB, KS, true, true, false> : prefill_wide_kernel<NB, KS, false, true, false>);
  else
    go(head_major ? prefill_wide_kernel<NB, KS, true, false, false> : prefill_wide_kernel<NB, KS, false, false, false>);
}
} // namespace

void launch_prefill_f32_cache(const bf16_bits *q, const bf16_bits *gate, bf16_bits *out, float *cache,
                              std::size_t tokens, std::size_t max_ctx, std::size_t past, bool head_major,
                              hipStream_t stream) {
  launch_f32(q, gate, out, cache, tokens, max_ctx, past, head_major, stream);
}

void launch_prefill_wide(PrefillForm form, const bf16_bits *q, const bf16_bits *key, const bf16_bits *value,
                         const bf16_bits *gate, bf16_bits *out, bf16_bits *cache, std::size_t tokens,
                         std::size_t max_ctx, std::size_t past, bool head_major, bool fused_append,
                         const prefill::PrefillNormRope *nq, hipStream_t stream) {
  switch (form) {
  case PrefillForm::stream8:
    return launch<1, 4>(q, key, value, gate, out, cache, tokens, max_ctx, past, head_major, fused_append, nq, stream);
  case PrefillForm::stream16:
    return launch<2, 4>(q, key, value, gate, out, cache, tokens, max_ctx, past, head_major, fused_append, nq, stream);
  default:
    return launch<2, 2>(q, key, value, gate, out, cache, tokens, max_ctx, past, head_major, fused_append, nq, stream);
  }
}

} // namespace raftinfer::amd
