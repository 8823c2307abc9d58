// The buffer window that the MFMA epilogues store a wave tile of D through: plain arithmetic, one definition for the kernels
// and for the host program that checks it over shapes (tests/host_c/store_window_check.cpp).
//
// The window starts at the wave tile's corner.  A store's place in it is the lane's byte offset plus a uniform one, the sum is
// compared with the window's size without a sign, and what is not inside is dropped by the hardware:
//   * columns past the last one of D lie behind the window's end,
//   * lanes past the end of P (D's unit-stride index) take kStoreNowhere as their offset.
// So no window may reach beyond that offset, however much of D lies behind the corner.  Nothing wanted lies there: a pitch
// is below kNarrowPitch elements (the dispatchers check it) and a wave tile has at most kWaveTile columns.
#pragma once
#include <cstdint>

namespace zluda_amd {

constexpr uint32_t kWindowEnd = 0x80000000u;
constexpr int kStoreNowhere = (int)kWindowEnd;
constexpr int64_t kNarrowPitch = 1 << 22;
constexpr int kWaveTile = 128;
// (4-byte elements; the last column starts below 2 GiB with room for its rows)
static_assert((kWaveTile - 1) * (kNarrowPitch - 1) * 4 + kWaveTile * 4 <= (int64_t)kWindowEnd, "a wave tile reaches past its window");

// `base_elems`: the corner, in elements from this batch's D; NQ columns of pitch d_sq, the last one NP long
constexpr uint32_t tile_window_bytes(int64_t d_sq, int NP, int NQ, int64_t base_elems, int esz) {
  const int64_t left = ((int64_t)(NQ - 1) * d_sq + NP - base_elems) * esz;
  return left <= 0 ? 0u : left > (int64_t)kWindowEnd ? kWindowEnd : (uint32_t)left;
}

} // namespace zluda_amd
