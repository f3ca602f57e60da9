// Integer formulas of the kernels whose range matters more than their speed:
// plain constexpr functions, so that the device code and a host program that
// checks them over their whole range compile the same text.
#pragma once

#include <stddef.h>

namespace ak {

// Elements from the first row of a page to token t's row, for pages of bs
// tokens, a power of two.  In 64 bits: a page may hold every token of a context
// (one page per sequence), and 2^24 rows of 128 elements no longer fit an int.
constexpr size_t page_row_offset(int t, int bs, int d) { return (size_t)(t & (bs - 1)) * d; }

// ceil(c / size) for 0 <= c < 2^24 and size >= 32, from the hardware's
// reciprocal of size.  With that and the product each off by a unit in the last
// place the quotient is off by less than 1, so its whole part is the true one
// or a neighbour: the remainder tells which, and one past it either way.
constexpr int split_count(int c, int size, float reciprocal) {
    const int n = (int)((float)c * reciprocal), r = c - n * size;
    return n + (r > 0) + (r > size) - (r <= -size);
}

}  // namespace ak
