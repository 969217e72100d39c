// Positions in the lists of a binning, as 32-bit integers: a batch's capacity
// reaches 2^31 - 256, so the sum of two positions need not fit an int.
#pragma once
#include <cstdint>

namespace jsa {

// a + b, at most cap (a and b are at most cap themselves, both not negative).
constexpr int clamped_sum(int a, uint32_t b, int cap) {
    const uint32_t sum = (uint32_t)a + b;
    return sum < (uint32_t)cap ? (int)sum : cap;
}

// Partitions of up to `size` entries that [begin, end) makes, and the end of the
// one from `at` (in [begin, end)).
constexpr int part_count(int begin, int end, int size) {
    return (int)(((uint32_t)(end - begin) + (uint32_t)size - 1u) / (uint32_t)size);
}
constexpr int part_end(int at, int end, int size) {
    return end - at < size ? end : at + size;
}

}  // namespace jsa
