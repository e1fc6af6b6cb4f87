// Index rules of the tiled products that can be checked without a GPU (no HIP headers).
#pragma once

#if defined(__HIPCC__)
#define BDH_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define BDH_HOST_DEVICE inline
#endif

// A thread of a k-major tile owns `ch` adjacent rows that start at row r0 + lead of the operand (lead a multiple of ch, r0 of
// the tile) and reads them with one access per k where `rows` is a multiple of ch, and one by one elsewhere.  The row that
// its c-th value comes from: its own, or, past the end, one of the last whole group -- every access of ch values then starts
// at a multiple of ch and ends inside the operand.  What a repeated row adds up to is not stored.
BDH_HOST_DEVICE int bdh_kmajor_row(int r0, int lead, int c, int ch, int rows) {
  if (rows % ch == 0) {
    const int first = r0 + lead < rows - ch ? r0 + lead : rows - ch;
    return first + c;
  }
  return r0 + lead + c < rows - 1 ? r0 + lead + c : rows - 1;
}

// A thread owns the `piece` columns from c on (a multiple of piece) of rows of `cols` values that lie one behind the other: how
// many of them exist.  Where cols % piece == 0 that is all or none, and a row's pieces are aligned as the first one is: one
// access each.  Elsewhere a row starts anywhere and its last piece ends inside the next row, or behind the last one: one by one.
BDH_HOST_DEVICE int bdh_columns_of_piece(int c, int piece, int cols) {
  return c >= cols ? 0 : cols - c < piece ? cols - c : piece;
}

// Byte offset of the value at (row, col) of a tile from the tile's first value, in 32 bits: what a copy adds to a base that is
// the same for a whole wavefront.  It holds while the last row of the tile lies less than 4 GiB behind the first one.
BDH_HOST_DEVICE unsigned int bdh_tile_offset(int row, int ld, int col) { return ((unsigned int)row * (unsigned int)ld + (unsigned int)col) * 2u; }
// ... which it does for bf16 rows of ld values in tiles of up to `tile` rows of `tile` columns.
BDH_HOST_DEVICE bool bdh_tile_offsets_fit(int tile, int ld) { return ((long long)(tile - 1) * ld + tile) * 2 <= 0xffffffffLL; }
