// gemm_units.hpp: what the grouped dequant GEMM's kernels (gemm.hip,
// gemm_tall.hip) share: code unpacking to f16, the f16 operand form of a stored
// value, and counted waits.
#pragma once
#include "moe_common.hpp"
#include "moe_internal.hpp"

namespace moe {

typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 h2_t __attribute__((ext_vector_type(2)));

// vector-memory instructions of one bload_unit
template <int BITS>
constexpr int kUnitLoads = (BITS == 5 || BITS == 6 || BITS == 8) ? 2 : 1;

// s_waitcnt for at most N outstanding vector-memory operations (gfx9
// encoding: vmcnt in bits 3:0 and 15:14; expcnt 6:4 and lgkmcnt 11:8 left
// at their maxima)
template <int N>
__device__ __forceinline__ void vmcnt_wait() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// Block barrier for LDS written by this block's LDS stores and by its
// memory-to-LDS copies of earlier chunks: waits for the wave's own LDS
// operations (lgkmcnt 0) only. A release fence on LDS would also wait for
// every memory-to-LDS copy in flight, including the ones issued for chunks
// two ahead; the callers wait for the copies that must have landed
// (vmcnt_wait) themselves. The signal fences keep the compiler from moving
// memory operations across the barrier.
__device__ __forceinline__ void lds_barrier_copies_in_flight() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0); vmcnt and expcnt at their maxima
  __builtin_amdgcn_s_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// Values 8 s + 2 p and 8 s + 2 p + 1 (p < 4) of a 32-value unit as 16-bit
// pairs 0x6400 | q, i.e. 1024 + q in f16 (exact for q < 1024). Not for 4 bits
// (quarter_codes).
template <int BITS>
__device__ __forceinline__ void quarter_pairs(const uint32_t (&w)[BITS], int s, uint32_t (&pr)[4]) {
  const uint32_t M = opaque_vgpr(0x64006400u);
  if constexpr (BITS == 8) {
#pragma unroll
    for (int p = 0; p < 4; p++) {  // bytes [b(2p), 0, b(2p+1), 0] of word 2 s + p / 2
      const int bb = 2 * (p & 1);
      pr[p] = __builtin_amdgcn_perm(0u, w[2 * s + (p >> 1)],
                                    (uint32_t)bb | 0x0C00u | ((uint32_t)(bb + 1) << 16) | 0x0C000000u) | M;
    }
  } else if constexpr (BITS <= 3) {
    // Two pairs per 4 * BITS-bit field y (values a, b, c, d from bit 0):
    // m = y | y << (16 - BITS) has a at bit 0, b at bit 16, c at bit 2 * BITS
    // and d at bit 16 + 2 * BITS, and the two copies of y do not overlap
    // (4 * BITS <= 16 - BITS), so one mask per pair picks them out.
    constexpr uint32_t kField = (1u << (4 * BITS)) - 1u, kPair = ((1u << BITS) - 1u) * 0x10001u;
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int bit = (2 * s + h) * 4 * BITS, lo = bit >> 5, sh = bit & 31;
      uint32_t y;
      if (sh + 4 * BITS <= 32)
        y = (w[lo] >> sh) & kField;
      else
        y = __builtin_amdgcn_alignbit(w[lo + 1], w[lo], (uint32_t)sh) & kField;
      const uint32_t m = y | (y << (16 - BITS));
      pr[2 * h] = (m & kPair) | M;
      pr[2 * h + 1] = ((m >> (2 * BITS)) & kPair) | M;
    }
  } else {  // 5 and 6 bits
    // A pair's 2 * BITS bits lie inside the 16 bits from the byte holding its
    // first bit: one byte permute puts those 16 bits in both halves, and one
    // packed 16-bit shift right by (o, o + BITS) brings each value to the
    // bottom of its half.
    typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));
    constexpr uint32_t kPair = ((1u << BITS) - 1u) * 0x10001u;
#pragma unroll
    for (int p = 0; p < 4; p++) {
      const int bit = (8 * s + 2 * p) * BITS, byte = bit >> 3, o = bit & 7;
      const int wi = byte >> 2, bw = byte & 3, wj = wi + 1 < BITS ? wi + 1 : BITS - 1;
      const uint32_t sel = (uint32_t)bw | ((uint32_t)(bw + 1) << 8) | ((uint32_t)bw << 16) |
                           ((uint32_t)(bw + 1) << 24);
      const u16x2_t z = __builtin_bit_cast(u16x2_t, __builtin_amdgcn_perm(w[wj], w[wi], sel));
      const u16x2_t t = z >> u16x2_t{(unsigned short)o, (unsigned short)(o + BITS)};
      pr[p] = (__builtin_bit_cast(uint32_t, t) & kPair) | M;
    }
  }
}

// Codes of values 8 s + 2 p and 8 s + 2 p + 1 (p < 4) of a 32-value unit as
// f16 pairs. 4-bit: the nibbles are spread one per byte, and a byte q < 16 is
// the OCP e4m3 number q * 2^-9 (subnormal below 8), so the scaled fp8
// conversion at 2^9 gives q exactly, two values per instruction. Other widths:
// 1024 + q pairs less 1024.
template <int BITS>
__device__ __forceinline__ void quarter_codes(const uint32_t (&w)[BITS], int s, h2_t (&q)[4]) {
  if constexpr (BITS == 4) {
    const uint32_t t = w[s] & 0x0F0F0F0Fu, u = (w[s] >> 4) & 0x0F0F0F0Fu;
    const uint32_t z0 = __builtin_amdgcn_perm(u, t, 0x05010400u);  // bytes [t0, u0, t1, u1]
    const uint32_t z1 = __builtin_amdgcn_perm(u, t, 0x07030602u);  // bytes [t2, u2, t3, u3]
    q[0] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(z0, 512.0f, false);
    q[1] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(z0, 512.0f, true);
    q[2] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(z1, 512.0f, false);
    q[3] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(z1, 512.0f, true);
  } else {
    uint32_t pr[4];
    quarter_pairs<BITS>(w, s, pr);
#pragma unroll
    for (int p = 0; p < 4; p++)
      q[p] = __builtin_bit_cast(h2_t, pr[p]) - h2_t{(_Float16)1024.0f, (_Float16)1024.0f};
  }
}

// One stored output value (fp32, already in the output's units) as the f16 A
// operand of the next GEMM: round to the layer dtype first (the reference
// stores the activation in it), then scale into f16 range, saturating.
template <typename XT>
__device__ __forceinline__ _Float16 to_a16(float v) {
  v = round_to<XT>(v);
  if constexpr (__is_same(XT, bf16_t)) {
    v = __builtin_ldexpf(v, -kA16Shift);
    v = fminf(fmaxf(v, -65504.0f), 65504.0f);
  }
  return (_Float16)v;
}

}  // namespace moe
