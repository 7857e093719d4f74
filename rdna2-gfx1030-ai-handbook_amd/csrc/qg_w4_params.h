// Where the few-row INT4 kernel (skinny_gemm.hip) finds the group parameters of
// a column: LDS pitches and the reads behind them. Plain C++, so that the reads
// can be checked on the host against the arrays' ends.
#pragma once
#include <cstdint>

namespace qg {

// LDS words per column of the scales and zero points: odd, so that a group's 16
// columns lie in different banks. bf16 scales of a column may start in the
// upper half of a word.
constexpr int w4_scale_pitch(int ng, bool f32) { return (f32 ? ng : ng / 2 + 1) | 1; }
constexpr int w4_zero_pitch(int ng, int zw, bool packed) { return (packed ? zw : ng) | 1; }

// The read that fills word w (from 0; those past the column's own repeat its
// last one) of column n < N: byte offset from the array's base and bytes. Scales
// [N, ng] are read as words from the one holding group 0; of an odd number of
// bf16 scales the last is half a word, read alone.
struct W4Read {
  uint32_t offset, bytes;
};
constexpr W4Read w4_scale_read(uint32_t n, uint32_t N, uint32_t ng, bool f32, uint32_t w) {
  const uint32_t used = f32 ? ng : (ng + 1) / 2;
  const uint32_t word = (f32 ? n * ng : (n * ng) >> 1) + (w < used ? w : used - 1);
  return W4Read{4 * word, !f32 && 2 * word + 1 == N * ng ? 2u : 4u};
}
// Zero points [N, per] (one word per group, or zw words of packed nibbles).
constexpr W4Read w4_zero_read(uint32_t n, uint32_t per, uint32_t w) {
  return W4Read{4 * (n * per + (w < per ? w : per - 1)), 4u};
}

}  // namespace qg
