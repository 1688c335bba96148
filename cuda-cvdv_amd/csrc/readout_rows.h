// readout_rows.h - tiles of the row kernels of the phase-space readouts
// (phase_space.hip, phase_grid.hip): rows of 2^3 .. 2^13 complex128 points
// transformed in LDS, eight points a thread.
#pragma once

#include <type_traits>

#include "fft_stages.h"

// A tile is Hb rows of N points: whole rows from 2^9 points on, 512 points of several
// rows below.
#define ROWS_LGM_MIN 3
#define ROWS_LGM_MAX 13
template <int LGM> constexpr int rows_lg_hb() { return LGM >= 9 ? 0 : 9 - LGM; }
template <int LGM> constexpr int rows_threads() { return 1 << (LGM + rows_lg_hb<LGM>() - 3); }
template <int LGM> constexpr size_t rows_lds() {
    constexpr int tile = 1 << (LGM + rows_lg_hb<LGM>());
    return (size_t)(tile + tile / 8) * sizeof(double2);  // EX_ROWS layout
}

// Calls f with the register's size as a compile-time constant (ROWS_LGM_MIN ..
// ROWS_LGM_MAX points).
template <typename F>
static void rows_dispatch(int n, F f) {
    switch (n) {
#define CVDV_ROWS_CASE(L) \
    case L: f(std::integral_constant<int, L>{}); break;
        CVDV_ROWS_CASE(3) CVDV_ROWS_CASE(4) CVDV_ROWS_CASE(5) CVDV_ROWS_CASE(6) CVDV_ROWS_CASE(7) CVDV_ROWS_CASE(8)
        CVDV_ROWS_CASE(9) CVDV_ROWS_CASE(10) CVDV_ROWS_CASE(11) CVDV_ROWS_CASE(12) CVDV_ROWS_CASE(13)
#undef CVDV_ROWS_CASE
        default: throw CvdvError{CVDV_ERR_UNSUPPORTED, "readout row length without a kernel instance"};
    }
}

template <typename K>
static void rows_launch_attr(K kfn, size_t lds) {
    if (lds > 64 * 1024)
        HIPCHK(hipFuncSetAttribute((const void*)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
}
