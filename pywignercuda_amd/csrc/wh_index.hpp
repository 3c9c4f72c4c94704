// Element indices of arrays that may hold more than 2^32 bytes.
#pragma once
#include <cstddef>

namespace wh {

// Element (row, col) of an array of rows of X elements.  X is a caller's batch: 64 rows of five
// million complex128 columns already span 2^32 bytes, so that the product needs 64 bits (a 32-bit byte
// offset read and wrote other columns).
constexpr size_t col_element(int row, int X, int col) { return size_t(row) * size_t(X) + size_t(col); }

}  // namespace wh
