// fft_row.h - the row kernel's interface (fft_row.hip) to the planner (fft.hip).
#pragma once

#include "fft_pass.h"

#define FFT_ROW_LGM_MIN 13
#define FFT_ROW_LGM_MAX 14

// Twiddles of a row of 2^lgm points (row_values in fft.hip): the middle stage's, the last's.
constexpr int row_tw_mid() { return 31 * 32; }
constexpr int row_tw_last(int lgm) { return ((1 << (lgm - 10)) - 1) * ((1 << (lgm - 10)) + 32); }
constexpr int row_tw_total(int lgm) { return row_tw_mid() + row_tw_last(lgm); }

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

// One pass over a.rows contiguous complex64 rows of 2^lgm points.
void fft_row_launch(hipStream_t stream, float2* data, int lgm, const RowArgs& a, const float2* tw);
