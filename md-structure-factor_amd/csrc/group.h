// How many frames a plan's slots hold: host rules without device calls.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace mdsf {

// Frames per group.  A small grid's frame leaves most of the chip idle (64
// tiles of a 64^3 grid for 256 CUs) and its dozen and a half launches each take
// their few microseconds of latency, so the frame loops hand every kernel the
// frames of a group at once, as blockIdx.y: as many as make kGroupTiles tiles,
// at most kMaxGroup, within kGroupBytes of state for the slots together.  Grids
// of kGroupTiles tiles and more fill the chip with one frame.  Before and after:
// ten frames of 2,700 atoms at 64^3 1,091 -> 292 us, sixteen forward and backward
// frames at 128^3 4,865 -> 3,242 us, eight systems of 64^3 to 192^3 in one graph
// 11,778 -> 9,012 us; one frame per group at 256^3, 4,930 and 4,915 us.
constexpr int kGroupTiles = 2048;
constexpr int kMaxGroup = 16;
constexpr size_t kGroupBytes = (size_t)2 << 30;
// What groups take beyond one frame comes out of the first half of the device's
// memory, a plan's at most this share of what is free of it, so that any number of
// plans that fits half the device with one frame each still fits (150 plans of
// 140 MB took 21 GB with one frame each and would take 300 GB with whole groups).
constexpr size_t kGroupShare = 16;

// Frames whose state of `bytes` each fits kGroupBytes and the device's memory (free
// and total: 0 if unknown), at least 1.
inline int group_fit(size_t bytes, size_t free, size_t total) {
  if (bytes == 0) return kMaxGroup;
  size_t extra = kGroupBytes;
  if (total > 0) {
    const size_t used = total / 2 + bytes;
    extra = free > used ? (free - used) / kGroupShare : 0;
  }
  const size_t fit = std::min(kGroupBytes / bytes, 1 + extra / bytes);
  return (int)std::min<size_t>(std::max<size_t>(fit, 1), kMaxGroup);
}

// The group of a grid of `tiles` tiles for calls of at most `frames` frames (0: any).
inline int group_frames(long long tiles, int64_t frames, size_t bytes, size_t free, size_t total) {
  const long long want = (kGroupTiles + tiles - 1) / std::max(tiles, 1LL);
  long long g = std::min<long long>(want, group_fit(bytes, free, total));
  if (frames > 0) g = std::min<long long>(g, frames);
  return (int)std::max(1LL, g);
}

// Allocates with attempt(group), halving the group while memory is out; returns what
// the last attempt returned, `out_of_memory` if one frame does not fit either.
template <typename E, typename Attempt>
E take_group(int* group, E out_of_memory, Attempt attempt) {
  for (;;) {
    const E e = attempt(*group);
    if (e != out_of_memory || *group == 1) return e;
    *group /= 2;
  }
}

}  // namespace mdsf
