// Where the pieces of a row tile lie that a block copies to LDS (stage_rows_v in ssd_f32.hip). Plain constexpr
// functions, so that the host can check them over every width and row stride.
//
// Piece id is the four floats at columns 4 (id % cpr) of row id / cpr, cpr pieces to a row. A thread takes id0,
// id0 + nthr, id0 + 2 nthr, ...; cpr divides the 64 lanes of a wave and nthr, so its columns stay and its row grows by
// nthr / cpr each time. The row stride is the whole tensor's (heads times head width, up to 65535 * 128 floats), also
// where the tile is a part of a head: 64 rows of it are 2 GiB. So the buffer resource of each piece starts at the row
// of the wave's first lane, and a lane's offset from it spans the rows of one wave only, 64 / cpr of them.
#pragma once

#include <cstdint>

constexpr int stage_row(int id, int cpr) { return id / cpr; }
constexpr int stage_col(int id, int cpr) { return id % cpr * 4; }
// first row of the resource for the piece q of the threads whose wave starts at id w0
constexpr int stage_base(int w0, int q, int nthr, int cpr) { return w0 / cpr + q * (nthr / cpr); }
// floats from there to the thread's piece, the same for every q
constexpr int stage_off(int id0, int w0, int cpr, int64_t ld) {
  return (id0 / cpr - w0 / cpr) * (int)ld + stage_col(id0, cpr);
}
