// qmag_wimage.h -- which bytes of a weight matrix a wave's LDS image requests
// (WImage in qmag_mfma.h): integer arithmetic only, without device code, so
// that a host program can walk through every request of every lane.
//
// A matrix is n_out rows of nb super-blocks.  The image of one super-block of
// ROWS rows is PIECES 16-byte pieces a row plus its last two bytes (the tail),
// piece p = lane + 64 k (row p / PIECES, its piece p % PIECES) belonging to
// lane and request k.  The requests are whole waves: the lanes past the last
// piece repeat it and drop it, and so take its step as well (with a step of
// their own number they ran past the end of repacked matrices).
#pragma once

#include <stdint.h>

#include "../../include/qma_gpu.h"

namespace qmag {

template <int WT, int ROWS>
struct WImageMap {
    static constexpr bool Q4 = WT == QMAG_TYPE_Q4_K, REP = WT == QMAG_TYPE_Q6_K_R;
    static constexpr int BLOCK = Q4 ? 144 : 210, PIECES = Q4 ? 9 : 13;
    static constexpr int STRIDE = Q4 ? 144 : 240;      // 36 or 60 words: 16 rows' reads on distinct banks
    static constexpr int BYTES = ROWS * STRIDE, NP = ROWS * PIECES, WP = (NP + 63) / 64;

    static constexpr int piece(int lane, int k) { return lane + 64 * k < NP ? lane + 64 * k : NP - 1; }
    // row r of a wave that starts at row0 (past the last row: the last), and
    // its offset from the wave's first
    static constexpr int row(int r, int row0, int n_out) { return row0 + r < n_out - 1 ? row0 + r : n_out - 1; }
    static constexpr int row_off(int r, int row0, int n_out, int rb)
    {
        return (row(r, row0, n_out) - row(0, row0, n_out)) * rb;
    }
    // where piece j of a row starts in the row's super-block 0, how far on it
    // is per super-block, and where the image holds row r's
    static constexpr int src(int j, int nb)
    {
        if (!REP) return 16 * j;
        if (j < 8) return 64 * nb * ((j >> 1) & 1) + 16 * (2 * (j >> 2) + (j & 1));
        return j < 12 ? 128 * nb + 16 * (j - 8) : 192 * nb;
    }
    static constexpr uint32_t step(int j) { return REP ? (j < 12 ? 64u : 16u) : (uint32_t)BLOCK; }
    static constexpr int dst(int r, int j) { return r * STRIDE + 16 * j; }
    // A Q6_K block is read from the dword it starts in, `lead` bytes ahead of it.
    // Offsets count from the dword that the wave's first row starts in, `skew`
    // bytes ahead of that row (a row that starts inside a dword is not the
    // matrix's first), so that no difference below is negative: counted from the
    // row itself, a first row 2 bytes into a dword gave 2^32 - 2.
    static constexpr uint32_t lead(uint32_t off) { return WT == QMAG_TYPE_Q6_K ? off & 2 : 0; }
    static constexpr uint32_t skew(int row, int rb) { return lead((uint32_t)row * (uint32_t)rb); }
    // where super-block ib's piece j is read from, start its block 0's offset
    static constexpr uint32_t from(uint32_t start, int ib, int j)
    {
        const uint32_t o = start + (uint32_t)ib * step(j);
        return o - lead(o);
    }
    // the tail of super-block ib in its row (Q6_K formats)
    static constexpr int tail0(int nb) { return REP ? 208 * nb : 208; }
    static constexpr int tail_step() { return REP ? 2 : BLOCK; }
};

}  // namespace qmag
