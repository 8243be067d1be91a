"""CPU check of the weight image of the matrix-core matmul kernels: every byte
that any lane of any wave requests lies within the matrix.  The requests'
arithmetic (qmag_wimage.h) is compiled for the host and walked through; a read
past the end that is dropped afterwards shows in no result."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

WALK = r"""
#include <stdio.h>
#include <stdlib.h>
#include "qmag_wimage.h"
using namespace qmag;

template <int WT, int ROWS>
static long walk(int nb, int n_out)
{
    using M = WImageMap<WT, ROWS>;
    const int rb = nb * M::BLOCK;
    const long end = (long)n_out * rb;
    long bad = 0;
    auto in = [&](long from, long bytes, const char *what, int row0, int lane, int k, int ib) {
        if (from >= 0 && from + bytes <= end) return;
        if (!bad++) printf("%d rows %d nb %d n_out %d: %s of row0 %d lane %d request %d block %d is [%ld, %ld) of %ld\n",
                           WT, ROWS, nb, n_out, what, row0, lane, k, ib, from, from + bytes, end);
    };
    // row0 also past the last row: the surplus waves of a workgroup
    for (int row0 = 0; row0 < n_out + 4 * ROWS; row0 += ROWS) {
        const int fr = M::row(0, row0, n_out);
        const uint32_t skew = M::skew(fr, rb);
        const long base = (long)fr * rb - skew;                 // may not lie ahead of the matrix either
        in(base, 1, "base", row0, 0, 0, 0);
        for (int ib = 0; ib < nb; ib++)
            for (int lane = 0; lane < 64; lane++) {
                for (int k = 0; k < M::WP; k++) {
                    const int p = M::piece(lane, k), r = p / M::PIECES, j = p % M::PIECES;
                    const long block = M::row(r, row0, n_out) * (long)rb + ib * (long)M::BLOCK;
                    const uint32_t o = M::from(skew + (uint32_t)(M::row_off(r, row0, n_out, rb) + M::src(j, nb)), ib, j);
                    in(base + (long)o, 16, "piece", row0, lane, k, ib);
                    if (!M::REP && base + (long)o != block + 16 * j - (long)M::lead((uint32_t)block) && !bad++)
                        printf("%d rows %d nb %d n_out %d: piece %d of row0 %d block %d from %ld\n", WT, ROWS, nb, n_out, p,
                               row0, ib, base + (long)o);
                }
                if (M::Q4) continue;
                const uint32_t t = skew + (uint32_t)M::row_off(lane % ROWS, row0, n_out, rb) +
                                   (uint32_t)(M::tail0(nb) + ib * M::tail_step());
                in(base + (long)(uint32_t)(t - M::lead(t)), 2, "tail", row0, lane, 0, ib);
                in(base + (long)t, 2, "tail", row0, lane, 0, ib);
            }
    }
    return bad;
}

int main(int argc, char **argv)
{
    long bad = 0;
    for (int a = 1; a + 1 < argc; a += 2) {
        const int nb = atoi(argv[a]), n_out = atoi(argv[a + 1]);
        bad += walk<QMAG_TYPE_Q4_K, 16>(nb, n_out) + walk<QMAG_TYPE_Q4_K, 32>(nb, n_out);
        bad += walk<QMAG_TYPE_Q6_K, 16>(nb, n_out) + walk<QMAG_TYPE_Q6_K, 32>(nb, n_out);
        if (nb % 8 == 0) bad += walk<QMAG_TYPE_Q6_K_R, 16>(nb, n_out) + walk<QMAG_TYPE_Q6_K_R, 32>(nb, n_out);
    }
    printf("%ld requests out of range\n", bad);
    return bad != 0;
}
"""


def test_every_request_lies_in_the_matrix(tmp_path):
    """All three layouts, images of 16 and 32 rows, one row, rows off a tile
    and whole tiles, one to 128 super-blocks, in the kernels' own 32-bit
    arithmetic; and a block's pieces are the block's."""
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no host compiler")
    src, exe = tmp_path / "walk.cpp", tmp_path / "walk"
    src.write_text(WALK)
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-I",
                    os.path.join(ROOT, "qwen-mobile-agent_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    shapes = [(nb, n) for nb in (1, 3, 8, 16, 24, 32, 128) for n in (1, 15, 16, 33, 64, 100)]
    r = subprocess.run([str(exe), *[str(v) for s in shapes for v in s]], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
