// How many films share a launch whose grid covers the widest and the tallest of
// them for each.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace lucida {

// Grid pixels outside every film that a launch may cover whatever its films'
// size: 4,096 blocks that return at once, 0.8 us.
constexpr uint64_t EMPTY_PIXELS = 1u << 20;

// The films of `in` (count of them, at least one; anything with width and
// height), from the first on, that go into one launch of at most `most`: as long
// as the grid stays within twice the films' own pixels and EMPTY_PIXELS. An empty
// block costs a thirtieth of a full one, but wide and tall films together make
// any number: of the blocks for 131,072 x 16 and 128 x 16,384 one in 1,024 had
// pixels, and a pass over crops of the two took 14.7 ms in shared launches,
// 0.9 in launches of their own.
template <class Film>
inline size_t films_together(const Film* const* in, size_t count, size_t most) {
    uint64_t w = 0, h = 0, pixels = 0;  // sides fit 32 bits; the grid's product may not fit 64
    size_t n = 0;
    for (; n < count && n < most; ++n) {
        w = std::max<uint64_t>(w, in[n]->width);
        h = std::max<uint64_t>(h, in[n]->height);
        pixels += (uint64_t)in[n]->width * in[n]->height;
        if (n > 0 && (double)(n + 1) * (double)(w * h) > 2.0 * (double)pixels + (double)EMPTY_PIXELS) break;
    }
    return n;
}

}  // namespace lucida
