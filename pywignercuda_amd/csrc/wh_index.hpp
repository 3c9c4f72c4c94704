// Element indices of arrays that may hold more than 2^32 bytes.
#pragma once
#include <cstddef>

namespace wh {

// Element (row, col) of an array of rows of X elements.  X is a caller's batch: 64 rows of five
// million complex128 columns already span 2^32 bytes, so that the product needs 64 bits (a 32-bit byte
// offset read and wrote other columns).
constexpr size_t col_element(int row, int X, int col) { return size_t(row) * size_t(X) + size_t(col); }

// Whether the byte offset of every element of the first `rows` rows fits 32 bits.  Kernels then address
// a uniform base and one offset register per lane (with 64-bit lane addresses 512 transforms of 1024
// take 7.4 us instead of 7.1); the others are instantiations of their own, as a branch around the loads
// costs up to 13%.
constexpr bool offsets_fit_32(int rows, int X, size_t element) { return size_t(rows) * size_t(X) * element <= size_t(1) << 32; }

}  // namespace wh
