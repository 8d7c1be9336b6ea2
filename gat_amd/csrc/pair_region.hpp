// Which pairs a digest reads of one query's region of a pair buffer.  Plain
// constexpr arithmetic, so the same functions run in the kernels and in a host
// program that walks every case around a buffer's end.
#pragma once

#include <cstdint>

namespace gat {

// Pairs [begin, end) of the buffer, read from the even pair `first` at or below
// begin on.  All zero when the region holds nothing inside the buffer: a region
// of a batch that outgrew the buffer may start anywhere past it.
struct PairRegion {
  uint64_t first, begin, end;
};

constexpr PairRegion pair_region(uint64_t base, uint64_t count, uint64_t capacity) {
  const uint64_t room = base < capacity ? capacity - base : 0;
  const uint64_t n = count < room ? count : room;
  return n == 0 ? PairRegion{0, 0, 0} : PairRegion{base & ~uint64_t(1), base, base + n};
}

// Whether both pairs of the last even group below `end` lie inside the buffer.
constexpr bool whole_groups(uint64_t end, uint64_t capacity) { return end <= (capacity & ~uint64_t(1)); }

// The even pair at `at`, or the last group's below end >= 1.
constexpr uint64_t clamped_group(uint64_t at, uint64_t end) {
  const uint64_t last = (end - 1) & ~uint64_t(1);
  return at < last ? at : last;
}

}  // namespace gat
