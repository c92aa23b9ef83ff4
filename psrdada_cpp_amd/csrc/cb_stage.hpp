// Coherent beamformer: the byte offsets of the FTPA staging loads (cb_tr_k,
// cb_ws_k) and of the operands read back, as plain constexpr functions, so
// that the kernels and a check on the host run the same arithmetic.
#pragma once

namespace fbf {

// One 16-byte load of a staged FTPA tile (32 columns, `kpad` bytes each in
// LDS, `vstride` bytes apart in memory): the load that fills tile byte `off`
// (a multiple of 16).  The bank swizzle is on the memory side: physical piece
// pp of column col holds K piece (pp + col * kpad / 256) % (kpad / 16); pieces
// past the column's K bytes re-read piece 0, whose weights there are zero.
// Where K % 16 == 8 the last piece runs 8 bytes into the next column (zero
// weights again), and past the block's end in its very last column: in the
// block's last tile that load starts `early` bytes before `offset`.  With 4
// antennas (K = 8) piece 0 is the last one, so the loads that re-read it are
// early as well.
struct StagedLoad {
    int offset;   // from the tile's first column
    int early;
};

constexpr StagedLoad staged_load(int off, int kpad, int K, int vstride)
{
    const int col = off / kpad;
    const int pp = (off - col * kpad) >> 4;
    const int j = (pp + ((col * kpad) >> 8)) % (kpad / 16);
    const int kpieces = (K + 15) / 16;
    const int piece = j < kpieces ? j : 0;
    return StagedLoad{col * vstride + 16 * piece, (K & 15) && col == 31 && piece == kpieces - 1 ? 8 : 0};
}

// Tile byte of K piece `piece` of column `col`.
constexpr int staged_piece(int col, int piece, int kpad)
{
    const int pr = kpad / 16;
    return col * kpad + 16 * ((piece - ((col * kpad) >> 8) + 32 * pr) % pr);
}

// The K piece of column 31 whose operand, loaded early in the block's last
// tile, is moved down 8 bytes where K % 16 == 8.
constexpr int staged_tail_piece(int K) { return K / 16; }

}  // namespace fbf
