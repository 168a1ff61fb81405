// Row addresses of the sub-chunk DGDA prefill's loads: a uniform base at a sub-chunk's first row
// and 32-bit byte offsets from it.  Plain C++, so that the arithmetic is tested on the host too.
#pragma once
#include <cstdint>

namespace maba {

constexpr int SC = 16;   // tokens per sub-chunk

// Offset of the last row a sub-chunk's loads may touch: row `most` of the window, or the last
// of the sequence, `left` rows after the base.  The rows are clamped before they are multiplied:
// the sequence's whole remainder times the row step leaves 32 bits on long sequences.
constexpr uint32_t row_end(int left, int most, int step, int first) {
  return (uint32_t)(left < most ? left : most) * (uint32_t)step + (uint32_t)first;
}
// Offset of row `row` after the lane's first one, at most `end`; a row before the base (the fused
// layer's conv taps ahead of token 0) wraps and is `end` too.
constexpr uint32_t row_offset(uint32_t lane0, int row, int step, uint32_t end) {
  return lane0 + (uint32_t)(row * step) < end ? lane0 + (uint32_t)(row * step) : end;
}

}  // namespace maba
