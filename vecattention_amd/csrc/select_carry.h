// The record that the maxima pass of a two-pass selection leaves per (row, key
// segment) for the carry pass.
#pragma once
#include <stdint.h>

namespace va {

constexpr int kCarryTiles = 4;  // near-max tiles a segment passes on

// The segment's MFMA maximum, the exact maximum of what was resolved exactly
// (-inf: nothing), and the tiles that can hold the segment's exact maximum
// besides, whose exact scores are left to the carry pass's rare path.
struct SegCarry {
  float m, ex;
  int32_t n, pad;
  int32_t tile[kCarryTiles];
};
static_assert(sizeof(SegCarry) == 32, "the host sizes carry buffers at 32 bytes per record");

}  // namespace va
