// The staging loads of FTPA tiles (cb_stage.hpp) on the host: every load of
// the block's last tile lies within the block, and each column's operands come
// out of the tile as the column holds them.  4 to 128 antennas in fours, as
// the whole block, and as a subset at the start, the end and inside a wider one.
// Exit status 0 = passed.
#include <cstdio>
#include <vector>

#include "../../psrdada_cpp_amd/csrc/cb_stage.hpp"

using namespace fbf;

namespace {

int check(int A, int vstride, int voff)
{
    const int K = 2 * A;
    const int ksteps = (K + 31) / 32, kpad = 32 * ksteps, kpieces = (K + 15) / 16;
    // The block's last tile, after one more column so that early loads show.
    const int start = vstride, bytes = 33 * vstride;
    std::vector<int> mem(bytes), tile(32 * kpad);
    for (int i = 0; i < bytes; ++i) mem[i] = i;
    for (int off = 0; off < 32 * kpad; off += 16) {
        const StagedLoad ld = staged_load(off, kpad, K, vstride);
        const int src = start + voff + ld.offset - ld.early;
        if (src < start || src + 16 > bytes) {
            std::printf("%d antennas, stride %d, offset %d: load of tile byte %d reads bytes %d .. %d of the last tile's %d\n",
                        A, vstride, voff, off, src - start, src - start + 15, 32 * vstride);
            return 1;
        }
        for (int i = 0; i < 16; ++i) tile[off + i] = mem[src + i];
    }
    for (int col = 0; col < 32; ++col)
        for (int piece = 0; piece < kpieces; ++piece) {
            const int at = staged_piece(col, piece, kpad);
            const bool moved = (K & 15) && col == 31 && piece == staged_tail_piece(K);
            for (int i = 0; i < 16 && 16 * piece + i < K; ++i) {
                const int got = tile[at + (moved ? i + 8 : i)];
                const int want = start + voff + col * vstride + 16 * piece + i;
                if (got != want) {
                    std::printf("%d antennas, stride %d, offset %d: byte %d of column %d is %d, not %d\n", A, vstride,
                                voff, 16 * piece + i, col, got, want);
                    return 1;
                }
            }
        }
    return 0;
}

}  // namespace

int main()
{
    int bad = 0;
    for (int A = 4; A <= 128; A += 4)
        for (int more = 0; more <= 64; more += 4)         // antennas of the block beside the subset's
            for (int a0 = 0; a0 <= more; a0 += 4) bad += check(A, 2 * (A + more), 2 * a0);
    std::printf("%d geometries out of range or out of place\n", bad);
    return bad != 0;
}
