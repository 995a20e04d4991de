// Byte offsets of a wavefront's tile of Q8_0 rows within its (sequence, kv head) slice
// (attn_decode_q8.hip), plain arithmetic that a host program can check.  A slice has size = S x row
// bytes, at most 2^32 - 1, and last16 = size - 16 is where its last 16 bytes start.  A tile's end can lie
// past 2^32, so sums that may pass the slice's end are only compared as differences.
#pragma once

#include <cstdint>

namespace gtq8 {

// Whether the tile of tb bytes at t0 (a multiple of 16) holds a 16-byte piece that the slice ends in.
constexpr bool ends_inside_piece(uint32_t t0, uint32_t tb, uint32_t last16) {
    return (last16 & 15) != 0 && t0 <= last16 && last16 + 16 - t0 < tb;
}

// Where the piece at `off` is read: in place, or the slice's last 16 bytes (`off` may have wrapped past
// 2^32: some piece inside the slice, of rows that do not exist).
constexpr uint32_t read_at(uint32_t off, uint32_t last16) { return off < last16 ? off : last16; }

// Dwords by which a piece read at last16 precedes `off` when the slice ends inside it (1 to 3), else 0.
constexpr uint32_t dwords_early(uint32_t off, uint32_t last16) {
    return off > last16 && off - last16 < 16 ? (off - last16) / 4 : 0;
}

}  // namespace gtq8
