// Byte offsets of direct loads whose rows or keys may lie past an operand's end.
//
// A raw buffer load is out of range, and returns zeros, where its per-lane offset is not below
// num_records - soffset (the ISA documents state the check in this form).  The subtraction is only
// meaningful while soffset itself is in range, so the scalar offsets below never leave the resource:
// a load whose rows all lie past the end reads rows that exist instead.
#pragma once

namespace laya {

// Ring GEMM, A rows: load q of a half-slab is 64 rows further on, but no further than the last 64-row group
// with a row.  rows_left: the operand's rows from the tile's first one on; row_bytes: bytes per row.
constexpr unsigned ring_row_limit(int rows_left, unsigned row_bytes) {
  return static_cast<unsigned>((rows_left - 1) / 64 * 64) * row_bytes;
}
constexpr unsigned ring_row_offset(int q, unsigned row_bytes, unsigned limit) {
  return 64u * static_cast<unsigned>(q) * row_bytes < limit ? 64u * static_cast<unsigned>(q) * row_bytes : limit;
}

// Attention, K rows of 128 bytes: the first row of half `half` (32 keys) of the 64-key block at kb.
constexpr unsigned key_half_offset(int kb, int half, int m) {
  return static_cast<unsigned>(kb + 32 * half < m ? kb + 32 * half : kb) * 128u;
}

// Attention, V^T rows of m keys: the first of the eight keys of 16-byte chunk c of the block at kb; chunks
// past the end take the row's last eight keys, values of the same head dim.
constexpr int value_chunk_key(int kb, int c, int m) { return kb + 8 * c < m - 8 ? kb + 8 * c : m - 8; }

}  // namespace laya
