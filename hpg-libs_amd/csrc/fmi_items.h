// fmi_items.h -- how the items of a wavefront's 64 lanes are shared out among
// wavefronts (wave_items): the arithmetic alone, for host and device code.
#pragma once

#include <algorithm>
#include <cstdint>

namespace fmi {

// The most items per lane whose sum over a wavefront fits in 32 bits.
constexpr uint64_t kItems32 = (1ull << 26) - 1;

// Wavefronts per 64 lanes: one where there are enough to fill the device twice
// (256 CUs of 32), else as many as do, at most one per 64 items the 64 lanes
// can bring.
inline uint32_t item_parts(uint64_t lanes, uint64_t items_per_lane) {
  const uint64_t waves = (lanes + 63) / 64;
  const uint64_t fill = std::max<uint64_t>(16384 / std::max<uint64_t>(waves, 1), 1);
  return (uint32_t)std::min<uint64_t>(fill, items_per_lane);
}

// From the wavefront's 64 items at base (below total) to its next 64, parts of
// 64 further on; false when there are none.  What is left is compared before
// the step: base + 64 parts need not fit in T.
template <class T>
constexpr bool items_next(T &base, T total, uint32_t parts) {
  const T step = (T)64u * (T)parts;
  if (total - base <= step) return false;
  base += step;
  return true;
}

}  // namespace fmi
