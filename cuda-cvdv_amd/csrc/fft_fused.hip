// fft_fused.hip - the fused four-step pass (the pending half of one transform, the phases, the
// first half of the next) for digits of 2^7 complex64 points.
//
// The tile kernel (k_fft_fused in fft.hip) takes such a digit in three stages of 8 elements a
// thread (8 x 8 x 2): six stages and four exchanges a pass, 102 VALU instructions an
// element, which is what bounds it.  With 16 elements a thread a digit is two stages, 16 x 8,
// and one exchange: [14,14] complex64 (a copy of this shape takes 0.82 ms), ms a gate of the strided
// register: displacement 2.01 -> 1.81, squeezing 4.04 -> 3.61, beam splitter 4.03 -> 3.50.
// complex64 in runs of 256 bytes only: in complex128 the 16 elements take 242 VGPRs, two
// waves a SIMD, and [13,12] displacements went from 0.22 to 0.26 ms.

#include "cvdv_internal.h"
#include "fft_fused.h"
#include "fft_radix16.h"

// Element k + 2 i of the natural order (rows q + e M/16) lies at x[8 k + i]: the order in
// which stage0_load, stage0_pre and last_store deal out a thread's two radix-8 butterflies.
__device__ constexpr int fuse2_at(int e) { return 8 * (e & 1) + (e >> 1); }

// The digit's transform over a tile, the thread's rows q + e M/16 before and after.
__device__ __forceinline__ void digit_fft(float2* x, float2* lds, const float4* __restrict__ tw, int tid) {
    using C = float2;
    constexpr int LGM = FUSE2_LGM, LGC = FUSE2_LGC, M = 1 << LGM, QN = M / 16, NB = 2;
    const int c = tid & ((1 << LGC) - 1), q = (tid >> LGC) & (QN - 1), hb = tid >> (LGC + LGM - 4);
    C y[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) y[e] = x[fuse2_at(e)];
    dft16<1>(y);
    C* tile = lds + (hb << (LGM + LGC)) + c;
    {
        C* wr = tile + (q << (4 + LGC));
#pragma unroll
        for (int m = 0; m < 16; ++m) wr[m << LGC] = y[m];
    }
    lds_barrier();
    {
        const C* rd = tile + (q << LGC);
#pragma unroll
        for (int e = 0; e < 16; ++e) y[e] = rd[(e * QN) << LGC];
    }
    lds_barrier();
    // butterfly k sits at q + k QN: W_M^{j (q + k QN)}, one rounded product each, both butterflies'
    // in one load (as W_M^{j q} W_16^{j k} the second takes two products, and eight transforms of
    // [14,5] are 5.07e-7 off instead of 4.40e-7; 4.77e-7 by 8 x 8 x 2)
#pragma unroll
    for (int j = 1; j < 8; ++j) {
        const float4 w = tw[(j - 1) * QN + q];
        y[NB * j] = cmul(y[NB * j], make_float2(w.x, w.y));
        y[NB * j + 1] = cmul(y[NB * j + 1], make_float2(w.z, w.w));
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        C z[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) z[j] = y[k + 2 * j];
        dft8<false>(z);
#pragma unroll
        for (int j = 0; j < 8; ++j) y[k + 2 * j] = z[j];
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) x[fuse2_at(e)] = y[e];
}

// As k_fft_fused (fft.hip) where every table is read by row and the generic terms are affine in
// the rows.
__global__ void __launch_bounds__(FUSE2_THREADS, 5)
k_fft_fused2(float2* data, FusedArgs a, FastDiag pre, const float4* __restrict__ tw, const float2* __restrict__ tw4) {
    using C = float2;
    constexpr int LGM = FUSE2_LGM, LGC = FUSE2_LGC;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ PreLds P;
    C* lds = reinterpret_cast<C*>(smem_raw);
    const int tid = threadIdx.x, nt = blockDim.x;
    const FftPass& d = a.d;
    const FftPass& dD = a.dD;
    if (dD.usePre) {
        // constant indices: the argument is read in place
#pragma unroll
        for (int i = 0; i < CVDV_FAST_TABS; ++i)
            if (tid == i && i < pre.ntab) P.tab[i] = pre.tab[i];
#pragma unroll
        for (int i = 0; i < CVDV_FAST_GEN; ++i)
            if (tid == CVDV_FAST_TABS + i && i < pre.ngen) P.gen[i] = pre.gen[i];
        __syncthreads();
    }
    const float scale = (float)d.outScale;
    const float scaleLo = (float)(d.outScale - (double)scale);

    const uint64_t t = blockIdx.x;
    const uint64_t loBlk = t & ((1ull << d.lgNLoBlk) - 1);
    const uint64_t rr = t >> d.lgNLoBlk;
    const uint64_t h2Blk = rr & ((1ull << d.lgNH2Blk) - 1);
    const uint64_t h1 = rr >> d.lgNH2Blk;
    const uint64_t base = (h1 << d.lgInH1) + ((h2Blk << d.lgHb) << d.lgInH2) + (loBlk << LGC);
    uint64_t natBase = base;
    if (a.swapLo > 0) {
        const uint64_t ml = (1ull << a.swapLo) - 1ull, mh = (1ull << a.swapHi) - 1ull;
        const uint64_t lo = (base >> a.swapSh) & ml, hi = (base >> (a.swapSh + a.swapLo)) & mh;
        natBase = (base & ~(((mh << a.swapLo) | ml) << a.swapSh)) | (((lo << a.swapHi) | hi) << a.swapSh);
    }

    C x[16];
    stage0_load<8, 16, LGM, LGC>(data, x, d, base, tid, nt);
    if (a.conjMid) {
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i].y = -x[i].y;
    }
    stage0_pre<8, 16, LGM, LGC, true, TM_NONE>(x, d, base, P, pre, tw4, tid, nt, lds);
    digit_fft(x, lds, tw, tid);
    if (a.conjMid) {
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i].y = -x[i].y;
    }
    // opaque: the first half's last steps would be sunk into the second half and held beside its factors
#pragma unroll
    for (int e = 0; e < 16; ++e) asm volatile("" : "+v"(x[e].x), "+v"(x[e].y));
    // an opaque copy of the thread id: index math for the second half and the store would
    // otherwise be held across the first
    int t2 = tid;
    asm volatile("" : "+v"(t2));
    stage0_pre<8, 16, LGM, LGC, false, TM_STAGED>(x, dD, natBase, P, pre, tw4, t2, nt, lds);
    digit_fft(x, lds, tw, t2);
    out_finish<16>(x, d, d.conjOut, scale, scaleLo);
    last_store<8, 16, LGM, LGC>(data, x, d, base, scale, scaleLo, t2, nt);
}

bool fft_fused2_launch(hipStream_t stream, float2* data, const FusedArgs& a, const FastDiag& pre, const float4* tw,
                       const float2* tw4, unsigned blocks) {
    const int tile = 1 << (FUSE2_LGM + FUSE2_LGC + a.d.lgHb);
    const size_t lds = (size_t)tile * sizeof(float2);
    if (a.d.lgM != FUSE2_LGM || a.d.lgC != FUSE2_LGC || tile / 16 > FUSE2_THREADS || lds > 64 * 1024) return false;
    hipLaunchKernelGGL(k_fft_fused2, dim3(blocks), dim3(tile / 16), lds, stream, data, a, pre, tw, tw4);
    return true;
}
