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

}  // namespace ak
