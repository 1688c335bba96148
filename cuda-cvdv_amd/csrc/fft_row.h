// fft_row.h - the row kernel's interface (fft_row.hip) to the planner (fft.hip).
#pragma once

#include "fft_pass.h"

// Row lengths with an instance.  Shorter rows would gain too ([14,12] complex64 a displacement
// 0.51 -> 0.32 ms, [14,11] complex128 0.30 -> 0.28), but a lone transform's error against 80 bits
// grows there (1.307e-7 -> 1.319e-7 and 2.285e-16 -> 2.311e-16); at these lengths it falls.
constexpr bool row_instance(bool c128, int lgm) { return c128 ? lgm == 12 : lgm == 13 || lgm == 14; }

// Twiddles of a row of 2^lgm points, E = 2^lge elements a thread (row_values in fft.hip): the
// middle stage's, the last's.
constexpr int row_lge_of(bool c128) { return c128 ? 4 : 5; }
constexpr int row_tw_mid(int lge) { return ((1 << lge) - 1) << lge; }
constexpr int row_tw_last(int lgm, int lge) { return ((1 << (lgm - 2 * lge)) - 1) * ((1 << (lgm - 2 * lge)) + (1 << lge)); }
constexpr int row_tw_total(int lgm, int lge) { return row_tw_mid(lge) + row_tw_last(lgm, lge); }

// One transform of every row: phases (tables read by row, generic terms affine in the row
// coordinate), direction, and the index bit + 1 that turns it round (0: none).
struct RowStep {
    FastDiag pre;
    int inv, ctl;
};

struct RowArgs {
    RowStep s[FT_CHAIN_MAX];
    int m, useScale;
    double scale;   // what the tables do not hold of the steps' normalisation
    uint64_t rows;
};

// One pass over a.rows contiguous rows of 2^lgm points.
void fft_row_launch(hipStream_t stream, void* data, bool c128, int lgm, const RowArgs& a, const void* tw);
