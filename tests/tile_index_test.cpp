// The rows that the threads of a k-major tile read (bdh_kmajor_row), for every width up to 640 and every tile: inside the
// operand, aligned where a group is read at once, and the thread's own row wherever it has one.  And the columns that the
// pieces of a 64 wide tile read (bdh_columns_of_piece): each column of a row once, none behind it, all of an aligned piece or
// none of it where it is read at once.  And the 32-bit offsets inside a bf16 tile (bdh_tile_offset): those of 64 bits wherever
// bdh_tile_offsets_fit says so, which is up to the widest rows for which all of them are.
#include <cstdio>
#include <initializer_list>

#include "../burn_dragon_amd/csrc/tile_index.h"

int main() {
  const int tiles[3] = {128, 64, 32}, threads = 256;
  long checked = 0;
  for (int rows = 1; rows <= 640; ++rows)
    for (int R : tiles) {
      const int ch = R * 4 / threads > 0 ? R * 4 / threads : 1;
      for (int r0 = 0; r0 < rows; r0 += R)
        for (int lead = 0; lead < R; lead += ch) {
          for (int c = 0; c < ch; ++c) {
            const int at = bdh_kmajor_row(r0, lead, c, ch, rows);
            if (at < 0 || at >= rows) return std::printf("rows %d tile %d: row %d\n", rows, R, at), 1;
            if (r0 + lead + c < rows && at != r0 + lead + c) return std::printf("rows %d tile %d: %d for %d\n", rows, R, at, r0 + lead + c), 1;
            ++checked;
          }
          if (rows % ch == 0) {  // read at once, from the first of the group
            const int first = bdh_kmajor_row(r0, lead, 0, ch, rows);
            if (first % ch != 0 || first + ch > rows) return std::printf("rows %d tile %d: group at %d\n", rows, R, first), 1;
          }
        }
    }
  for (int cols = 1; cols <= 640; ++cols)
    for (int piece : {4, 8}) {
      int read = 0;
      for (int c0 = 0; c0 < cols; c0 += 64)
        for (int cc = 0; cc < 64; cc += piece) {
          const int n = bdh_columns_of_piece(c0 + cc, piece, cols);
          if (n < 0 || n > piece || (n > 0 && c0 + cc + n > cols)) return std::printf("cols %d piece of %d at %d: %d\n", cols, piece, c0 + cc, n), 1;
          if (cols % piece == 0 && n != 0 && n != piece) return std::printf("cols %d: a part of an aligned piece of %d\n", cols, piece), 1;
          read += n;
        }
      if (read != cols) return std::printf("cols %d: %d read in pieces of %d\n", cols, read, piece), 1;
      checked += cols;
    }
  for (int tile : {64, 128})
    for (long long ld = 8; ld <= 0x7fffffff; ld += ld < 16000000 || (ld > 17000000 && ld < 33000000) || ld > 35000000 ? 999992 : 8) {
      bool same = true;
      for (int row : {0, 1, tile / 2 - 1, tile - 2, tile - 1})
        for (int col : {0, 56, tile - 8})
          same = same && bdh_tile_offset(row, (int)ld, col) == (unsigned long long)(row * ld + col) * 2;
      if (bdh_tile_offsets_fit(tile, (int)ld) != same) return std::printf("tile %d rows of %lld: %d\n", tile, ld, same), 1;
      ++checked;
    }
  std::printf("ok %ld\n", checked);
  return 0;
}
