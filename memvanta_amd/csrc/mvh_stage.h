/*
 * mvh_stage.h -- where the batched fp32 kernels (mvh_gemm_f32.hip) read the
 * pieces of a tile of quantized weight rows.
 *
 * A row is taken in units of 8 blocks, a unit in `per_row` pieces of `bytes`
 * bytes; piece p of a unit belongs to the tile's row p / per_row.  The last
 * unit of a row may be shorter than 8 blocks (the only one, of a row with
 * fewer): its pieces past the row's end are fetched from the row's start and
 * never used, so that every load stays inside the weights.
 *
 * Plain C++ (host or HIP device: define MVH_STAGE_QUAL before including).
 */
#ifndef MVH_STAGE_H
#define MVH_STAGE_H
#include <stdint.h>

#ifndef MVH_STAGE_QUAL
#define MVH_STAGE_QUAL static inline
#endif

struct MvhStagePiece {
    uint32_t src; /* byte offset in unit 0, from the tile's first row */
    int off;      /* the same, from the piece's own row */
};

/* Piece p of a tile with `rows` rows left in the matrix; pieces and rows past
 * the last one read that one (their results are not stored). */
MVH_STAGE_QUAL MvhStagePiece mvh_stage_piece(int p, int pieces, int per_row, int bytes, int rows, int row_bytes) {
    const int pc = p < pieces ? p : pieces - 1, row = pc / per_row < rows ? pc / per_row : rows - 1;
    MvhStagePiece r;
    r.off = bytes * (pc % per_row);
    r.src = (uint32_t)row * (uint32_t)row_bytes + (uint32_t)r.off;
    return r;
}

/* Byte offset, from the tile's first row, of a piece of the unit that starts
 * `at` bytes into each row. */
MVH_STAGE_QUAL uint32_t mvh_stage_at(MvhStagePiece q, int at, int row_bytes) {
    return q.src + (uint32_t)(at + q.off < row_bytes ? at : -q.off);
}
#endif
