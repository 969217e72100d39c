// Index arithmetic that also compiles for the host.
#pragma once
#include <cstdint>

namespace jsa {

// Positions in the lists of a binning, as 32-bit integers: a batch's capacity
// reaches 2^31 - 256, so the sum of two positions need not fit an int.
//
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

// Tile of workgroup b in a grid of xcd_grid(num_tiles, chunk) workgroups:
// workgroups are dealt to the 8 XCDs round robin, so XCD b & 7 gets chunks of
// `chunk` consecutive tiles, which share Gaussians in its L2, and the chunks
// are dealt to the XCDs in turn (indexes past num_tiles are the caller's to
// skip).  num_tiles up to 2^30, chunk up to num_tiles / 8 rounded up, or 64.
constexpr int xcd_grid(int num_tiles, int chunk) {
    const long long round = 8ll * chunk;
    return (int)((num_tiles + round - 1) / round * round);
}
constexpr int xcd_tile(int b, int chunk) {
    const int j = b >> 3, q = (int)((uint32_t)j / (uint32_t)chunk);
    return (q * 8 + (b & 7)) * chunk + (j - q * chunk);
}

}  // namespace jsa
