"""The weight loads of the batched fp32 kernels stay inside the weights: every piece of every unit of every tile,
evaluated on the host with the kernels' own offsets (memvanta_amd/csrc/mvh_stage.h)."""
import os
import subprocess

from conftest import ROOT

# the two staging forms of a 16-row tile (a larger one has the same rows more often): 2-byte pieces at any K,
# 16-byte pieces at whole units
PROG = r"""
#include <stdio.h>
#include "mvh_stage.h"
int main(void) {
    long bad = 0, n = 0;
    const int kinds[2] = {18, 34};
    for (int t = 0; t < 2; ++t)
        for (int nb = 1; nb <= 33; ++nb)
            for (int rows = 1; rows <= 17; ++rows)
                for (int bytes = 2; bytes <= 16; bytes += 14) {
                    if (bytes == 16 && nb % 8) continue;
                    const int kb = kinds[t], per_row = 8 * kb / bytes, pieces = 16 * per_row, row_bytes = nb * kb;
                    for (int row0 = 0; row0 < rows; row0 += 16)
                        for (int p = 0; p < pieces + 256; ++p) {
                            const MvhStagePiece q = mvh_stage_piece(p, pieces, per_row, bytes, rows - row0, row_bytes);
                            for (int c = 0; c < (nb + 7) / 8; ++c) {
                                const int at = 8 * kb * c;
                                const long o = (long)row0 * row_bytes + mvh_stage_at(q, at, row_bytes);
                                ++n;
                                bad += o < 0 || o + bytes > (long)rows * row_bytes;
                                /* a piece inside its row is the one it should be */
                                const int row = row0 + (p < pieces ? p : pieces - 1) / per_row;
                                if (row < rows && at + q.off < row_bytes)
                                    bad += o != (long)row * row_bytes + at + q.off;
                            }
                        }
                }
    printf("%ld %ld\n", bad, n);
    return 0;
}
"""


def test_every_piece_inside_the_weights(tmp_path):
    src = tmp_path / "stage.cpp"
    src.write_text(PROG)
    exe = tmp_path / "stage"
    subprocess.run(["g++", "-O2", "-I", os.path.join(ROOT, "memvanta_amd", "csrc"), "-o", str(exe), str(src)], check=True)
    bad, n = (int(v) for v in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split())
    assert n > 1000000
    assert bad == 0
