// fft_stages.h - Stockham stages over a tile held in registers and exchanged
// through LDS, shared by the register FFT (fft.hip) and the native phase-space
// readouts (phase_space.hip).
#pragma once

#include "fft_bfly.h"

// LDS layouts of the Stockham exchanges (padding breaks power-of-two strides).
// LAY 0, every exchange of every tile unless below: one pad entry per 32.
// One-row complex64 tiles of 2^13-2^14 points write exchange 0 at a stride of 8
// entries and exchange 1 in runs of 8 lanes 64 entries apart, which puts two
// lanes of every 16 on one LDS bank under LAY 0: there exchange 0 takes one pad
// entry per 16 (LAY 1) and exchange 1 eight per 64 (LAY 2).
// LAY 3, the complex128 rows of the phase-space readouts: one pad entry per 8, so
// that exchange 0's stride of 8 16-byte entries falls on different banks.
template <int LAY>
__device__ __forceinline__ int lay_ix(int i) {
    return LAY == 0 ? i + (i >> 5) : (LAY == 1 ? i + (i >> 4) : (LAY == 2 ? i + ((i >> 6) << 3) : i + (i >> 3)));
}
template <int LAY> constexpr int lay_period() { return LAY == 0 ? 32 : (LAY == 1 ? 16 : (LAY == 2 ? 64 : 8)); }
template <int LAY> constexpr int lay_padded(int stride) {
    return stride + (LAY == 0 ? stride / 32 : (LAY == 1 ? stride / 16 : stride / 8));
}
// The exchanges of a tile: EX_TILE LAY 0, EX_ONE the one-row complex64 layouts,
// EX_ROWS LAY 3.  The layout of exchange XS (stage XS's outputs, read by stage XS + 1):
enum { EX_TILE = 0, EX_ONE = 1, EX_ROWS = 2 };
template <int EX, int XS> constexpr int ex_lay() {
    return EX == EX_TILE ? 0 : (EX == EX_ROWS ? 3 : (XS == 0 ? 1 : (XS == 1 ? 2 : 0)));
}

__device__ __forceinline__ int lds_ix(int i) { return lay_ix<0>(i); }

// Padded index of i0 + m * STRIDE.  When STRIDE is a multiple of the layout's
// period the padding is linear (adding it leaves the bits below the period
// alone), so every element is the padded base plus a compile-time offset (an
// immediate in the LDS access).
template <int STRIDE, int LAY = 0>
__device__ __forceinline__ int lds_at(int i0, int pbase, int m) {
    if constexpr (STRIDE % lay_period<LAY>() == 0) return pbase + m * lay_padded<LAY>(STRIDE);
    else return lay_ix<LAY>(i0 + m * STRIDE);
}

// Stage plan of a length-2^LGM transform: radix-8 stages, then one radix-4 or
// radix-2 stage.  Stage s has sub-length L = 8^s and its twiddles start at
// entry off(s) of the stage table (W_{RL}^{ij} at off + j (R-1) + i - 1), the
// layout stage_values() writes.
template <int LGM> struct Plan {
    static constexpr int NST = LGM / 3 + (LGM % 3 ? 1 : 0);
    static constexpr int lgr(int s) { return s < LGM / 3 ? 3 : LGM % 3; }
    static constexpr int off(int s) {
        int o = 0, L = 1;
        for (int i = 0; i < s; ++i) {
            o += L * ((1 << lgr(i)) - 1);
            L <<= lgr(i);
        }
        return o;
    }
};

// Stockham stage geometry.  A butterfly of a stage of radix RP (sub-length L = 2^lgL
// already transformed) takes rows q + i*M/RP of column c in block hb and writes rows
// ob + m*L, ob = hb*M + (q/L)*RP*L + (q mod L); every thread owns E/RP butterflies.
struct BflyPos {
    int c, q, hb;
};

// The thread's butterfly k.  Where a column has at least E rows the thread owns the rows
// q0 + j M/E, j < E, of its column and block in every stage (butterfly k sits at
// q0 + k M/E), so a last stage's outputs, reordered in registers (to_rows), are a first
// stage's inputs; shorter columns deal the butterflies out nt apart.
template <int RP, int LGM, int E>
__device__ __forceinline__ BflyPos bfly_pos(int tid, int k, int nt, int lgC) {
    constexpr int LGR = RP == 8 ? 3 : (RP == 4 ? 2 : 1);
    constexpr int LGE = E == 16 ? 4 : 3;
    static_assert(E == 8 || E == 16, "elements of a thread");
    BflyPos p;
    if constexpr (LGM >= LGE) {
        p.c = tid & ((1 << lgC) - 1);
        const int rest = tid >> lgC;
        p.q = (rest & ((1 << (LGM - LGE)) - 1)) + k * (1 << (LGM - LGE));
        p.hb = rest >> (LGM - LGE);
    } else {
        constexpr int lgMq = LGM - LGR;
        const int b = tid + k * nt;
        p.c = b & ((1 << lgC) - 1);
        const int rest = b >> lgC;
        p.q = rest & ((1 << lgMq) - 1);
        p.hb = rest >> lgMq;
    }
    return p;
}

// Outputs of a last stage (butterfly k, output m: row q0 + (k + NB m) M/E) in the order of
// the thread's rows.
template <int LGM, int E, typename C>
__device__ __forceinline__ void to_rows(C* x) {
    constexpr int RL = LGM % 3 == 0 ? 8 : 1 << (LGM % 3), NB = E / RL;
    static_assert((1 << LGM) >= E, "columns of at least E rows");
    C y[E];
#pragma unroll
    for (int k = 0; k < NB; ++k)
#pragma unroll
        for (int m = 0; m < RL; ++m) y[k + NB * m] = x[k * RL + m];
#pragma unroll
    for (int j = 0; j < E; ++j) x[j] = y[j];
}

// Twiddle the inputs of the butterflies in x (stage S, radix RP) and transform.
template <int RP, int E, int LGM, int LGC, int S, typename C>
__device__ __forceinline__ void stage_compute(C* x, const C* __restrict__ tw, int tid, int nt) {
    constexpr int lgC = LGC;
    constexpr int NB = E / RP;
    constexpr int lgL = 3 * S;
#pragma unroll
    for (int k = 0; k < NB; ++k) {
        if (lgL > 0) {
            const BflyPos p = bfly_pos<RP, LGM, E>(tid, k, nt, lgC);
            const int pq = p.q & ((1 << lgL) - 1);
            const C* t = tw + Plan<LGM>::off(S) + pq * (RP - 1);
#pragma unroll
            for (int i = 1; i < RP; ++i) x[k * RP + i] = cmul(x[k * RP + i], t[i - 1]);
        }
        dft_r<RP, false>(x + k * RP);
    }
}

// stage_compute for a last stage whose twiddles the caller holds in registers
// (last_twiddles): rows transformed one after another reuse them.
template <int E, int LGM, typename C>
__device__ __forceinline__ void last_twiddles(C* w, const C* __restrict__ tw, int tid, int nt) {
    constexpr int S = Plan<LGM>::NST - 1, RP = 1 << Plan<LGM>::lgr(S);
#pragma unroll
    for (int k = 0; k < E / RP; ++k) {
        const C* t = tw + Plan<LGM>::off(S) + bfly_pos<RP, LGM, E>(tid, k, nt, 0).q * (RP - 1);
#pragma unroll
        for (int i = 1; i < RP; ++i) w[k * (RP - 1) + i - 1] = t[i - 1];
    }
}
template <int RP, int E, typename C>
__device__ __forceinline__ void stage_compute_held(C* x, const C* w) {
#pragma unroll
    for (int k = 0; k < E / RP; ++k) {
#pragma unroll
        for (int i = 1; i < RP; ++i) x[k * RP + i] = cmul(x[k * RP + i], w[k * (RP - 1) + i - 1]);
        dft_r<RP, false>(x + k * RP);
    }
}

// Outputs of stage S (radix RP) -> LDS in Stockham order (exchange S).
template <int RP, int E, int LGM, int LGC, int S, int EX = EX_TILE, typename C>
__device__ __forceinline__ void stage_write(C* lds, const C* x, int tid, int nt) {
    constexpr int LAY = ex_lay<EX, S>();
    constexpr int NB = E / RP;
    constexpr int LGR = RP == 8 ? 3 : (RP == 4 ? 2 : 1);
    constexpr int lgL = 3 * S;
    constexpr int STRIDE = 1 << (lgL + LGC);
#pragma unroll
    for (int k = 0; k < NB; ++k) {
        const BflyPos p = bfly_pos<RP, LGM, E>(tid, k, nt, LGC);
        const int ob = (p.hb << LGM) + ((p.q >> lgL) << (LGR + lgL)) + (p.q & ((1 << lgL) - 1));
        const int i0 = (ob << LGC) + p.c, pb = lay_ix<LAY>(i0);
        if constexpr (LAY == 1 || LAY == 2 || (LAY == 3 && S == 0)) {
            // exchange 0: i0 = 8q with entries i0 + m (periods 8 and 16); exchange 1 of
            // LAY 2: i0 mod 64 < 8 with entries i0 + 8m (period 64): all within i0's period
#pragma unroll
            for (int m = 0; m < RP; ++m) lds[pb + m * STRIDE] = x[k * RP + m];
        } else {
#pragma unroll
            for (int m = 0; m < RP; ++m) lds[lds_at<STRIDE, LAY>(i0, pb, m)] = x[k * RP + m];
        }
    }
}

// Inputs of a stage of radix RP <- LDS (exchange XS).
template <int RP, int E, int LGM, int LGC, int XS = 0, int EX = EX_TILE, typename C>
__device__ __forceinline__ void stage_read(const C* lds, C* x, int tid, int nt) {
    constexpr int LAY = ex_lay<EX, XS>();
    constexpr int NB = E / RP;
    constexpr int LGR = RP == 8 ? 3 : (RP == 4 ? 2 : 1);
    constexpr int lgMq = LGM - LGR;
    constexpr int STRIDE = 1 << (lgMq + LGC);
#pragma unroll
    for (int k = 0; k < NB; ++k) {
        const BflyPos p = bfly_pos<RP, LGM, E>(tid, k, nt, LGC);
        const int i0 = (((p.hb << LGM) + p.q) << LGC) + p.c, pb = lay_ix<LAY>(i0);
#pragma unroll
        for (int i = 0; i < RP; ++i) x[k * RP + i] = lds[lds_at<STRIDE, LAY>(i0, pb, i)];
    }
}

// Stages 1 .. NST-1: exchange the previous stage's outputs through LDS, then
// twiddle and transform.
// HELD: the last stage takes its twiddles from the registers w.
template <int LGM, int LGC, int S, int E, int EX = EX_TILE, bool HELD = false, typename C>
__device__ __forceinline__ void run_stages(C* x, C* lds, const C* __restrict__ tw, int tid, int nt,
                                           const C* w = nullptr) {
    if constexpr (S < Plan<LGM>::NST) {
        constexpr int RPprev = 1 << Plan<LGM>::lgr(S - 1);
        constexpr int RP = 1 << Plan<LGM>::lgr(S);
        stage_write<RPprev, E, LGM, LGC, S - 1, EX>(lds, x, tid, nt);
        lds_barrier();
        stage_read<RP, E, LGM, LGC, S - 1, EX>(lds, x, tid, nt);
        lds_barrier();
        if constexpr (HELD && S == Plan<LGM>::NST - 1) stage_compute_held<RP, E>(x, w);
        else stage_compute<RP, E, LGM, LGC, S>(x, tw, tid, nt);
        run_stages<LGM, LGC, S + 1, E, EX, HELD>(x, lds, tw, tid, nt, w);
    }
}
