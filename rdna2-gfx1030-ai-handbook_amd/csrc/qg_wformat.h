// Weight formats of the streaming kernels (skinny_gemm.hip, mid_gemm.hip):
// expansion to MFMA fragments and the LDS layout of their operands.
#pragma once
#include "qg_common.h"

namespace qg {

namespace {

enum SkinnyFormat { SK_I8 = 0, SK_E4M3 = 1, SK_E5M2 = 2, SK_W4 = 3, SK_UINT4 = 4 };

// 8 nibbles (K order; high: nibble 7 first) -> 8 fp16 256 + 4 u or bf16 128 + u.
template <bool F16A>
struct NibbleExpand {
  uint32_t sel[4], mask, magic;
  __device__ __forceinline__ explicit NibbleExpand(bool high) {
    static_for<0, 4>([&](auto ic) {
      constexpr uint32_t i = decltype(ic)::value;
      // halves of register i: elements 2 i and 2 i + 1, from the word (bytes
      // 0-3) and the word shifted right by 4 (bytes 4-7), 0x0c = zero byte
      sel[i] = high ? (0x0C000C00u | ((3u - i) << 16) | (7u - i)) : (0x0C000C00u | ((4u + i) << 16) | i);
    });
    mask = F16A ? 0x00F000F0u : 0x000F000Fu;
    magic = F16A ? 0x5C005C00u : 0x43004300u;
    asm volatile("" : "+v"(mask), "+v"(magic));
  }
  __device__ __forceinline__ i32x4 operator()(uint32_t w) const {
    const uint32_t lo = F16A ? w << 4 : w, hi = F16A ? w : w >> 4;
    i32x4 r;
    static_for<0, 4>([&](auto i) {
      r[int(i)] = static_cast<int>((__builtin_amdgcn_perm(hi, lo, sel[int(i)]) & mask) | magic);
    });
    return r;
  }
};

template <bool F16A>
__device__ __forceinline__ f32x4 mfma_half(const i32x4& a, const i32x4& b, const f32x4& c) {
  if constexpr (F16A)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
}

// XOR of the 16-byte chunk index of an LDS row: 256-byte rows of 2-byte
// activations, 128-byte rows (int8, fp8), 64-byte rows (INT4). The 16 rows of
// a fragment, read at chunk c + q by lane quarter q, then hit different banks
// within a ds_read_b128 phase (lanes 0-3, 12-15, 20-23, 24-27, and so on).
template <int ROW>
__device__ __forceinline__ int lds_row_xor(int row) {
  if constexpr (ROW == 256) return row & 15;
  else if constexpr (ROW == 128) return 2 * ((row >> 1) & 3);
  else return (-(row >> 2)) & 3;
}

// Lane quarter q holds 16 fp8 bytes 16 q .. 16 q + 15 of 64: words 2 h, 2 h + 1
// become bytes 32 h + 8 q .. + 7 (the K order of two 32-element steps).
__device__ __forceinline__ i32x4 k_order_bytes(const i32x4& w) {
  int w0 = w[0], w1 = w[1], w2 = w[2], w3 = w[3];
  swap16(w0, w2);
  swap32(w0, w2);
  swap16(w1, w3);
  swap32(w1, w3);
  return i32x4{w0, w1, w2, w3};
}
// Lane quarter q holds INT4 words 4 q .. 4 q + 3 of 16: word j becomes 4 j + q.
__device__ __forceinline__ i32x4 k_order_words(const i32x4& w) {
  int w0 = w[0], w1 = w[1], w2 = w[2], w3 = w[3];
  swap16(w0, w1);
  swap16(w2, w3);
  swap32(w0, w2);
  swap32(w1, w3);
  return i32x4{w0, w1, w2, w3};
}

}  // namespace

}  // namespace qg
