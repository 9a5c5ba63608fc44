// Which operand rows a tile of the matrix products can address by one scalar address and 32-bit offsets. Host code only.
#pragma once

namespace sd3 {

// Offsets of a tile's bytes from its first one: `rows` rows of `row_bytes`, of each of which a K tile asks for 128 bytes (which the scalar address moves
// along with K)
constexpr bool offsets_fit(int rows, long long row_bytes) { return (rows - 1) * row_bytes + 128 <= 1LL << 32; }

}  // namespace sd3
