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
// What groups take beyond one frame is at most 1 / kGroupTotal of the device's memory
// over all plans of the process, and a plan's at most 1 / kGroupShare of what is free,
// so that plans which fit three quarters of the device with one frame each fit it still
// (150 plans of 140 MB took 21 GB with one frame each and would take 300 GB with whole
// groups).
constexpr size_t kGroupShare = 16;
constexpr size_t kGroupTotal = 4;

// The device's memory (total 0: unknown) and what groups hold of it beyond one frame.
struct GroupMemory {
  size_t free = 0, total = 0, taken = 0;
};

// Frames whose state of `bytes` each fits kGroupBytes and the memory, at least 1.
inline int group_fit(size_t bytes, const GroupMemory& mem) {
  if (bytes == 0) return kMaxGroup;
  size_t extra = kGroupBytes;
  if (mem.total > 0) {
    const size_t most = mem.total / kGroupTotal;
    extra = std::min(mem.free > bytes ? (mem.free - bytes) / kGroupShare : 0,
                     most > mem.taken ? most - mem.taken : 0);
  }
  const size_t fit = std::min(kGroupBytes / bytes, 1 + extra / bytes);
  return (int)std::min<size_t>(std::max<size_t>(fit, 1), kMaxGroup);
}

// The group of a grid of `tiles` tiles for calls of at most `frames` frames (0: any).
inline int group_frames(long long tiles, int64_t frames, size_t bytes, const GroupMemory& mem) {
  const long long want = (kGroupTiles + tiles - 1) / std::max(tiles, 1LL);
  long long g = std::min<long long>(want, group_fit(bytes, mem));
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
