// f32 products on the f16 matrix cores (hgemm.hip), for the training step.
#pragma once

#include "common.h"

namespace ava {

// An operand in split form: per row (of A; column of B) hgemm_ldk(k) k values as blocks of 32 hi and 32
// lo f16 terms, and the row's exponent.
struct HgemmOp {
    const void *planes;
    const int *exps;
};
inline int hgemm_ldk(int k) { return (k + 63) / 64 * 64; }
inline size_t hgemm_plane_bytes(size_t rows, int k) { return rows * (size_t)hgemm_ldk(k) * 4; }
// x [rows][cols]: an operand of `rows` rows over k = cols
int hgemm_split_rows(const float *x, int rows, int cols, int ld, void *planes, int *exps, hipStream_t st);
// x [rows][cols]: an operand of `cols` rows over k = rows; part: hgemm_part_floats(rows, cols)
size_t hgemm_part_floats(int rows, int cols);
int hgemm_split_cols(const float *x, int rows, int cols, int ld, void *planes, int *exps, float *part, hipStream_t st);
// the parts K is cut into; with more than one, hgemm needs splits * m * n floats of scratch
int hgemm_splits(int m, int n, int k);
size_t hgemm_part_max();  // the most floats of scratch that any product needs
// C [m][n] (row-major, ldc) = A B, or C += A B
int hgemm(const HgemmOp &a, const HgemmOp &b, int m, int n, int k, float *c, int ldc, bool add, float *part,
          size_t part_floats, hipStream_t st);

}  // namespace ava
