// fft_fused.h - the two-stage fused kernel's interface (fft_fused.hip) to the planner (fft.hip).
#pragma once

#include "fft_pass.h"

#define FUSE2_LGM 7
#define FUSE2_LGC 5        // columns: 256 bytes of a row
#define FUSE2_THREADS 512

// A fused pass over digits of 2^FUSE2_LGM complex64 points in tiles of 2^FUSE2_LGC columns.
struct FusedArgs {
    FftPass d, dD;   // the tile in the state, and in the natural index of the completed transform
    int conjMid, swapSh, swapLo, swapHi;
};

// `tw`: W_128^{j q}, W_128^{j (q + 8)} at (j - 1) 8 + q, 1 <= j < 8, q < 8.  False: no instance for this shape.
bool fft_fused2_launch(hipStream_t stream, float2* data, const FusedArgs& a, const FastDiag& pre, const float4* tw,
                       const float2* tw4, unsigned blocks);
