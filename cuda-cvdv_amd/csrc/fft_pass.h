// fft_pass.h - one pass of a register transform over the state: the tile geometry, the
// loads, the pending phases and the output scale, shared by the tile kernels (fft.hip)
// and the row kernel (fft_row.hip).
#pragma once

#include "diag_fast.h"
#include "fft_stages.h"

// ---------------------------------------------------------------- pass descriptor
struct FftPass {
    int lgM, lgC, lgHb;            // tile = [Hb][M][C] (lgM also selects the kernel instance)
    int lgNLoBlk, lgNH2Blk;        // tiles = nH1 * nH2Blk * nLoBlk
    uint64_t nTiles;
    int rowFastOut;                // linear order of the staged store after the column index
    int vecOut;                    // 1: pairs of complex64 stored as one 16-byte access
    int directOut;                 // 1: last stage stores straight to global (coalesced rows)
    int tw4, tw4Shift, tw4HiBits, tw4LogN;
    int tw4Uni;                    // 1: the twiddle's second index is the same over the tile
    int usePre, useScale;
    int conjIn, conjOut;           // inverse = conj . forward . conj, split over the passes
    int conjLoad;                  // conjugate as loaded, before the four-step twiddle (the
                                   // second half of an inverse whose first half ran alone)
    int conjCtl;                   // bit + 1: tiles with this index bit set run the other way
                                   // (conjIn and conjOut flipped; the bit is the tile's); 0: none
    int lgInH1, lgInH2, lgInR;     // every stride is a power of two
    int lgOutH1, lgOutH2, lgOutR;
    double outScale;  // applied as exact v*hi + rounded v*lo (one FMA): an FP32 store stays unbiased
    int genSteps;     // 1: every generic term is affine in the tile's row index (the host checked)
};

__device__ __forceinline__ int tile_conj(const FftPass& d, int conj, uint64_t inBase) {
    return d.conjCtl ? conj ^ (int)((inBase >> (d.conjCtl - 1)) & 1ull) : conj;
}

// The value lane `lane` of the wave holds (`lane` the same on every lane, and
// that lane active).
__device__ __forceinline__ float2 lane_value(float2 v, int lane) {
    return make_float2(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(v.x), lane)),
                       __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v.y), lane)));
}
__device__ __forceinline__ double2 lane_value(double2 v, int lane) {
    auto rd = [lane](double d) {
        const long long b = __double_as_longlong(d);
        const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)b, lane);
        const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), lane);
        return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
    };
    return make_double2(rd(v.x), rd(v.y));
}

// Tile element e (linear) -> (c, row, hb) in the given order.
template <int LGM>
__device__ __forceinline__ void tile_coords(int e, int lgC, int lgHb, int rowFast, int& c, int& row, int& hb) {
    c = e & ((1 << lgC) - 1);
    const int rest = e >> lgC;
    const int lgLo = rowFast ? LGM : lgHb;  // selects, not branches on references (no scratch)
    const int lo = rest & ((1 << lgLo) - 1), hi = rest >> lgLo;
    row = rowFast ? lo : hi;
    hb = rowFast ? hi : lo;
}

// The compiled pending program, staged in LDS so its runtime-length loops read
// LDS instead of forcing a scratch copy of the kernel argument.
struct PreLds {
    DiagTab tab[CVDV_FAST_TABS];
    DiagTerm gen[CVDV_FAST_GEN];
};

// The generic terms over a one-row tile (only the transformed field
// [fs, fs + fn) varies inside it): when every term is affine in that field's
// coordinate m, their sum is a·m + b (mod 1) with per-tile a, b, and one FP64
// product per element replaces the per-term evaluation.  a is reduced mod 1 (m is
// an integer); al is what its rounding left of a bilinear term's slope, and a·m,
// up to 2^(fn-1) revolutions, is reduced before it is rounded.
struct GenFold {
    double a, al, b;
    int ok;
    __device__ __forceinline__ double turn(double m) const { return fma(al, m, fma(a, m, -rint(a * m))); }
    __device__ __forceinline__ void slope(double c, double m) {
        const double p = c * m;
        a += cvdv_frac(p);
        al += fma(c, m, -p);
    }
};

__device__ __forceinline__ bool field_overlaps(int sh, int nb, int fs, int fn) {
    return sh < fs + fn && fs < sh + nb;
}

__device__ __forceinline__ GenFold fold_generic(const DiagTerm* gen, int ngen, double genrev, uint64_t g0, int fs,
                                                int fn) {
    GenFold f{0.0, 0.0, genrev, 1};
    for (int i = 0; i < ngen; ++i) {
        const DiagTerm& T = gen[i];
        if (T.ctrl >= 0 && T.ctrl >= fs && T.ctrl < fs + fn) f.ok = 0;
        const double sg = (T.ctrl >= 0 && ((g0 >> T.ctrl) & 1ull)) ? -1.0 : 1.0;
        const bool in1 = T.sh1 == fs && T.nb1 == fn;
        if (T.kind == DT_BILIN) {
            const bool in2 = T.sh2 == fs && T.nb2 == fn;
            if ((!in1 && field_overlaps(T.sh1, T.nb1, fs, fn)) || (!in2 && field_overlaps(T.sh2, T.nb2, fs, fn)) ||
                (in1 && in2))
                f.ok = 0;
            else if (in1)
                f.slope(sg * T.c1, diag_field_m(g0, T.sh2, T.nb2));
            else if (in2)
                f.slope(sg * T.c1, diag_field_m(g0, T.sh1, T.nb1));
            else
                f.b += cvdv_frac(sg * diag_term_rev(T, g0));
        } else if (T.kind == DT_POLY || T.kind == DT_LINF) {
            if (in1 && T.c2 == 0.0 && T.c3 == 0.0)
                f.a += cvdv_frac(sg * T.c1);
            else if (field_overlaps(T.sh1, T.nb1, fs, fn))
                f.ok = 0;
            else
                f.b += cvdv_frac(sg * diag_term_rev(T, g0));
        } else {
            if (T.sh1 >= fs && T.sh1 < fs + fn) f.ok = 0;
            else f.b += cvdv_frac(sg * diag_term_rev(T, g0));
        }
    }
    f.a = cvdv_frac(f.a);
    f.b = cvdv_frac(f.b);
    return f;
}

// Phase of the generic (untabulated) terms at element g.
template <typename C>
__device__ __forceinline__ C gen_factor(const PreLds& P, const FastDiag& pre, uint64_t g) {
    using R = decltype(C{}.x);
    double r = pre.genrev;
    for (int i = 0; i < pre.ngen; ++i) r += cvdv_frac(diag_term_rev(P.gen[i], g));
    return unit_rev_fast(cvdv_frac(r), R(0));
}

// Stage-0 inputs straight from global memory (issued early: a tile ahead).
template <int RP, int E, int LGM, int LGC, typename C>
__device__ __forceinline__ void stage0_load(const C* __restrict__ in, C* x, const FftPass& d, uint64_t inBase,
                                            int tid, int nt) {
    constexpr int NB = E / RP;
    constexpr int LGR = RP == 8 ? 3 : (RP == 4 ? 2 : 1);
    constexpr int lgMq = LGM - LGR;
#pragma unroll
    for (int k = 0; k < NB; ++k) {
        const BflyPos p = bfly_pos<RP, LGM, E>(tid, k, nt, LGC);
        const uint64_t g0 = inBase + ((uint64_t)p.hb << d.lgInH2) + ((uint64_t)p.q << d.lgInR) + p.c;
#pragma unroll
        for (int i = 0; i < RP; ++i) x[k * RP + i] = in[g0 + ((uint64_t)(i << lgMq) << d.lgInR)];
    }
}

// Pending phases, the four-step twiddle W_N^{j1 k2} of a second pass (row j1 =
// the transformed index, k2 = (g >> tw4Shift) mod 2^tw4HiBits; TW4: the
// instance may carry one) and the input conjugation of an inverse on the loaded
// inputs.  TM, how the phase tables are read:
//   TM_ANY    tables of several columns stage their product by row in LDS when
//             every table allows it, else each element takes its flat index;
//   TM_STAGED every table is read by row (the host checked, tile_tables_by_row())
//             and is staged by row; generic terms go through the free exchange
//             buffer (complex64: their row steps per column and row block;
//             complex128: each element's factor from a rolled loop), which
//             keeps their FP64 temporaries off the other elements' registers.
// TM_NONE: the pass applies no phases (only the four-step twiddle, if TW4).
enum { TM_ANY = 1, TM_STAGED = 2, TM_NONE = 3 };
template <int RP, int E, int LGM, int LGC, bool TW4, int TM, typename C>
__device__ __forceinline__ void stage0_pre(C* x, const FftPass& d, uint64_t inBase, const PreLds& P,
                                           const FastDiag& pre, const C* __restrict__ tw4, int tid, int nt,
                                           C* sRow) {
    constexpr int NB = E / RP;
    constexpr int LGR = RP == 8 ? 3 : (RP == 4 ? 2 : 1);
    constexpr int lgMq = LGM - LGR;
    if (TW4 && d.tw4) {
        // second four-step pass: straight-line, so these loads issue with the
        // tile's input loads and share their wait
        if (d.tw4Uni) {
            // k2 is the tile's (no tile index bit selects it), so W^{k2 (q + i M/RP)} =
            // W^{k2 q} W^{k2 i M/RP} takes one gathered and RP-1 tile-uniform
            // (scalar) loads per butterfly instead of RP gathers
            const uint32_t nmask = (1u << d.tw4LogN) - 1u;
            const uint32_t k2 = (uint32_t)(inBase >> d.tw4Shift) & ((1u << d.tw4HiBits) - 1u);
            C st[RP];
#pragma unroll
            for (int i = 1; i < RP; ++i) st[i] = tw4[(k2 * (uint32_t)(i << lgMq)) & nmask];
#pragma unroll
            for (int k = 0; k < NB; ++k) {
                const BflyPos p = bfly_pos<RP, LGM, E>(tid, k, nt, LGC);
                const C b = tw4[(k2 * (uint32_t)p.q) & nmask];
                x[k * RP] = cmul(x[k * RP], b);
#pragma unroll
                for (int i = 1; i < RP; ++i) x[k * RP + i] = cmul(x[k * RP + i], cmul(b, st[i]));
            }
        } else {
            // k2 differs within the tile (between row blocks or columns): per
            // butterfly, gather W^{k2 q} and
            // w = W^{k2 M/RP}; the powers w^i come from a multiplication tree of
            // depth log2(RP)
#pragma unroll
            for (int k = 0; k < NB; ++k) {
                const BflyPos p = bfly_pos<RP, LGM, E>(tid, k, nt, LGC);
                const uint64_t g0 = inBase + ((uint64_t)p.hb << d.lgInH2) + ((uint64_t)p.q << d.lgInR) + p.c;
                const uint32_t nmask = (1u << d.tw4LogN) - 1u;
                const uint32_t k2 = (uint32_t)(g0 >> d.tw4Shift) & ((1u << d.tw4HiBits) - 1u);
                const C b = tw4[(k2 * (uint32_t)p.q) & nmask];
                C st[RP];
                st[1] = tw4[(k2 << lgMq) & nmask];
#pragma unroll
                for (int i = 2; i < RP; ++i) st[i] = cmul(st[i / 2], st[i - i / 2]);
                x[k * RP] = cmul(x[k * RP], b);
#pragma unroll
                for (int i = 1; i < RP; ++i) x[k * RP + i] = cmul(x[k * RP + i], cmul(b, st[i]));
            }
        }
    }
    if (TM != TM_NONE && d.usePre) {
        int tt = tid;
        auto elem = [&](int k, int i) {
            const BflyPos p = bfly_pos<RP, LGM, E>(tt, k, nt, LGC);
            return inBase + ((uint64_t)p.hb << d.lgInH2) + ((uint64_t)p.q << d.lgInR) + p.c +
                   ((uint64_t)(i << lgMq) << d.lgInR);
        };
        // Table-major: the E entries of one table are loaded together, so a wave
        // has E loads in flight instead of one dependent load per element.  The
        // first table is applied in straight-line code, so its loads issue with
        // the tile's input loads and share their wait (a loop that touches x
        // would wait for x's loads before issuing its first table load).
        // A table whose field misses the tile's column and row-block bits, and
        // holds all or none of its row bits, is read at base + (row << s) with a
        // per-tile base and conjugation: 32-bit indices instead of each element's
        // 64-bit flat index.
        const int rowLo = d.lgInR, rowHi = d.lgInR + LGM;
        auto hits = [](int sh, int nb, int lo, int n) { return n > 0 && sh < lo + n && lo < sh + nb; };
        // Where a table is read through the tile's base: the base, the row shift
        // (31: the row does not index it) and the conjugation.
        struct TabAt {
            DiagTab T;
            bool fast, cj;
            int s;
            const C* tb;
        };
        auto tab_at = [&](const DiagTab& TL) {
            TabAt A;
            // the descriptor is read from LDS into vector registers; it is the
            // same for every lane, so keep it in scalar registers
            DiagTab& T = A.T;
            T.sh = __builtin_amdgcn_readfirstlane(TL.sh);
            T.nb = __builtin_amdgcn_readfirstlane(TL.nb);
            T.ctrl = __builtin_amdgcn_readfirstlane(TL.ctrl);
            T.off = (uint32_t)__builtin_amdgcn_readfirstlane((int)TL.off);
            T.nsel = __builtin_amdgcn_readfirstlane(TL.nsel);
            T.sel = (uint32_t)__builtin_amdgcn_readfirstlane((int)TL.sel);
            const bool rowIn = T.sh <= rowLo && rowHi <= T.sh + T.nb;
            auto varies = [&](int b) {
                return b >= 0 && (b < LGC || (b >= rowLo && b < rowHi) ||
                                  (d.lgHb > 0 && b >= d.lgInH2 && b < d.lgInH2 + d.lgHb));
            };
            bool ctrlVar = varies(T.ctrl);
#pragma unroll
            for (int j = 0; j < CVDV_TAB_SEL; ++j)
                if (j < T.nsel) ctrlVar = ctrlVar || varies(tab_sel(T, j));
            A.fast = !hits(T.sh, T.nb, 0, LGC) && !hits(T.sh, T.nb, d.lgInH2, d.lgHb) &&
                     (rowIn || !hits(T.sh, T.nb, rowLo, LGM)) && !ctrlVar;
            // choice bits are tile-uniform here: they only move the tile's base
            A.tb = (const C*)pre.arena + T.off + (uint32_t)((inBase >> T.sh) & ((1ull << T.nb) - 1ull)) +
                   (T.nsel > 0 ? tab_choice(T, inBase) : 0u);
            A.s = rowIn ? rowLo - T.sh : 31;
            A.cj = T.ctrl >= 0 && ((inBase >> T.ctrl) & 1ull);
            return A;
        };
        auto apply_table = [&](const DiagTab& TL) {
            const TabAt A = tab_at(TL);
            const DiagTab& T = A.T;
            const bool fast = A.fast;
            constexpr int CH = sizeof(C) == 16 ? (RP < 8 ? 2 : 4) : 8;  // entries in flight per batch
            if (fast) {
                const C* tb = A.tb;
                const int s = A.s;
                const bool cj = A.cj;
#pragma unroll
                for (int j0 = 0; j0 < E; j0 += CH) {
                    C e[CH];
#pragma unroll
                    for (int j = 0; j < CH; ++j) {
                        const BflyPos p = bfly_pos<RP, LGM, E>(tt, (j0 + j) / RP, nt, LGC);
                        const uint32_t row = (uint32_t)(p.q + (((j0 + j) % RP) << lgMq));
                        e[j] = tb[s < 31 ? (row << s) : 0u];
                        if (cj) e[j].y = -e[j].y;
                    }
#pragma unroll
                    for (int j = 0; j < CH; ++j) x[j0 + j] = cmul(x[j0 + j], e[j]);
                }
            } else if constexpr (TM == TM_ANY) {
                // per element; the choice bits are tile-uniform (the tables were
                // compiled for this tiling), so the choice is one per tile
                const C* tb = (const C*)pre.arena + T.off + (T.nsel > 0 ? tab_choice(T, inBase) : 0u);
#pragma unroll
                for (int j0 = 0; j0 < E; j0 += CH) {
                    C e[CH];
#pragma unroll
                    for (int j = 0; j < CH; ++j) {
                        const uint64_t g = elem((j0 + j) / RP, (j0 + j) % RP);
                        e[j] = tb[(uint32_t)((g >> T.sh) & ((1ull << T.nb) - 1ull))];
                        if (T.ctrl >= 0 && ((g >> T.ctrl) & 1ull)) e[j].y = -e[j].y;
                    }
#pragma unroll
                    for (int j = 0; j < CH; ++j) x[j0 + j] = cmul(x[j0 + j], e[j]);
                }
            }
        };
        // Generic terms affine in the row index (complex64 staged instances always;
        // otherwise when d.genSteps): a butterfly's rows are q + i M/RP with its
        // column and row block (position j) fixed, so its phases are P(q) + i D_j.
        // The steps e^{2 pi i i D_j} go to the free exchange buffer, RP-1 per
        // position, one sin/cos each; a butterfly then takes one FP64 evaluation,
        // one sin/cos e0 and RP-1 products e0 * step.  The caller puts a barrier
        // before the buffer is written again.
        auto row_steps = [&]() {
            using RR = decltype(C{}.x);
            const int nj = (nt * E) >> LGM;
#pragma unroll 1
            for (int s = tt; s < nj * (RP - 1); s += nt) {
                const int j = s / (RP - 1), i = s - j * (RP - 1) + 1;
                const uint64_t g0 =
                    inBase + ((uint64_t)(j >> LGC) << d.lgInH2) + (uint64_t)(j & ((1 << LGC) - 1));
                const uint64_t g1 = g0 + ((uint64_t)(1 << lgMq) << d.lgInR);
                double dl = 0.0;
                for (int t = 0; t < pre.ngen; ++t)
                    dl += cvdv_frac(diag_term_rev(P.gen[t], g1) - diag_term_rev(P.gen[t], g0));
                sRow[s] = unit_rev_fast(cvdv_frac((double)i * cvdv_frac(dl)), RR(0));
            }
            lds_barrier();
#pragma unroll
            for (int k = 0; k < NB; ++k) {
                const BflyPos p = bfly_pos<RP, LGM, E>(tt, k, nt, LGC);
                const uint64_t g0 = elem(k, 0);
                double p0 = pre.genrev;
                for (int t = 0; t < pre.ngen; ++t) p0 += cvdv_frac(diag_term_rev(P.gen[t], g0));
                const C e0 = unit_rev_fast(cvdv_frac(p0), RR(0));
                const C* st = sRow + (p.c | (p.hb << LGC)) * (RP - 1) - 1;
                x[k * RP] = cmul(x[k * RP], e0);
#pragma unroll
                for (int i = 1; i < RP; ++i) x[k * RP + i] = cmul(x[k * RP + i], cmul(e0, st[i]));
            }
        };
        bool staged = false;
        if constexpr (LGC > 0) {
            // Tiles of several columns: when every table is read by row, their
            // product over the tile's M rows is staged in LDS (one table load per
            // row instead of one per element), and each element takes one LDS
            // read and one product.  The exchange buffer is free before the
            // stages; a barrier hands it back.
            bool byRow = pre.ntab > 0;
            if constexpr (TM == TM_ANY)
                for (int t = 0; t < pre.ntab; ++t) byRow = byRow && tab_at(P.tab[t]).fast;
            if (byRow) {
                for (int r = tid; r < (1 << LGM); r += nt) {
                    C f = cmk<C>(1.0, 0.0);
                    for (int t = 0; t < pre.ntab; ++t) {
                        const TabAt A = tab_at(P.tab[t]);
                        C e = A.tb[A.s < 31 ? ((uint32_t)r << A.s) : 0u];
                        if (A.cj) e.y = -e.y;
                        f = t == 0 ? e : cmul(f, e);
                    }
                    sRow[r] = f;
                }
                lds_barrier();
#pragma unroll
                for (int k = 0; k < NB; ++k) {
                    const BflyPos p = bfly_pos<RP, LGM, E>(tt, k, nt, LGC);
#pragma unroll
                    for (int i = 0; i < RP; ++i) x[k * RP + i] = cmul(x[k * RP + i], sRow[p.q + (i << lgMq)]);
                }
                lds_barrier();
                staged = true;
            }
        }
        if (TM != TM_STAGED && !staged) {
            if (pre.ntab > 0) apply_table(P.tab[0]);
            for (int t = 1; t < pre.ntab; ++t) {
                // opaque: the element indices are recomputed per table, not held
                asm volatile("" : "+v"(tt));
                apply_table(P.tab[t]);
            }
        }
        if constexpr (TM == TM_STAGED && LGC > 0) {
            if (pre.ngen > 0) {
                using RR = decltype(C{}.x);
                if (sizeof(C) == 8 || d.genSteps) {
                    row_steps();
                } else {
                    // complex128 with terms that are not affine in the rows: one
                    // element per iteration, its terms evaluated exactly; its factor
                    // goes to its own slot of the exchange buffer (element-major, so
                    // a wave's writes are consecutive), then every element takes its
                    // product.
#pragma unroll 1
                    for (int k = 0; k < NB; ++k) {
#pragma unroll 1
                        for (int i = 0; i < RP; ++i) {
                            const uint64_t g = elem(k, i);
                            double r = pre.genrev;
                            for (int t = 0; t < pre.ngen; ++t) r += cvdv_frac(diag_term_rev(P.gen[t], g));
                            sRow[(k * RP + i) * nt + tt] = unit_rev_fast(cvdv_frac(r), RR(0));
                        }
                    }
#pragma unroll
                    for (int j = 0; j < E; ++j) x[j] = cmul(x[j], sRow[j * nt + tt]);
                }
                lds_barrier();  // the stages that follow write other threads' slots
            }
        } else if (pre.ngen > 0) {
            asm volatile("" : "+v"(tt));
            // one-row tiles: the terms are affine in the row coordinate
            GenFold gf{0.0, 0.0, 0.0, 0};
            if (LGC == 0 && d.lgHb == 0) gf = fold_generic(P.gen, pre.ngen, pre.genrev, inBase, d.lgInR, LGM);
            if (gf.ok) {
                using R = decltype(C{}.x);
                // A butterfly's rows are q + i M/RP, so its phases are e^{2 pi i (a m0 + b)}
                // times the tile-wide steps e^{2 pi i a 2 i M/RP}: one sin/cos per
                // butterfly, and RP-1 per tile (uniform across the wave).
                C st[RP];
                if (nt >= 64) {
                    // full waves: lane i evaluates step i, the others read it
                    const int li = (int)__builtin_amdgcn_mbcnt_lo(~0u, 0u) & (RP - 1);
                    const C mine = unit_rev_fast(cvdv_frac(gf.turn((double)(2 * (li << lgMq)))), R(0));
#pragma unroll
                    for (int i = 1; i < RP; ++i) st[i] = lane_value(mine, i);
                } else {
#pragma unroll
                    for (int i = 1; i < RP; ++i)
                        st[i] = unit_rev_fast(cvdv_frac(gf.turn((double)(2 * (i << lgMq)))), R(0));
                }
#pragma unroll
                for (int k = 0; k < NB; ++k) {
                    const BflyPos p = bfly_pos<RP, LGM, E>(tt, k, nt, LGC);
                    const double m0 = (double)(2 * p.q + 1 - (1 << LGM));
                    const C e0 = unit_rev_fast(cvdv_frac(gf.turn(m0) + gf.b), R(0));
                    x[k * RP] = cmul(x[k * RP], e0);
#pragma unroll
                    for (int i = 1; i < RP; ++i) x[k * RP + i] = cmul(x[k * RP + i], cmul(e0, st[i]));
                }
            } else if (d.genSteps) {
                // tiles of several columns or row blocks
                row_steps();
                lds_barrier();  // the stages that follow write the exchange buffer
            } else {
#pragma unroll
                for (int k = 0; k < NB; ++k)
#pragma unroll
                    for (int i = 0; i < RP; ++i)
                        x[k * RP + i] = cmul(x[k * RP + i], gen_factor<C>(P, pre, elem(k, i)));
            }
        }
        if (tile_conj(d, d.conjIn, inBase)) {
#pragma unroll
            for (int i = 0; i < E; ++i) x[i].y = -x[i].y;
        }
    } else if (tile_conj(d, d.conjIn, inBase)) {
#pragma unroll
        for (int i = 0; i < E; ++i) x[i].y = -x[i].y;
    }
}

// Output scale and conjugation (inverse), applied to a thread's transformed
// elements before either store path.  Behind uniform branches: the compiler
// would otherwise select per element and pay for the scale even when it is off.
template <int E, typename R, typename C>
__device__ __forceinline__ void out_finish(C* x, const FftPass& d, int conj, R scale, R scaleLo) {
    if (d.useScale) {
#pragma unroll
        for (int i = 0; i < E; ++i) {
            x[i].x = fma(x[i].x, scale, x[i].x * scaleLo);
            x[i].y = fma(x[i].y, scale, x[i].y * scaleLo);
        }
    }
    if (conj) {
#pragma unroll
        for (int i = 0; i < E; ++i) x[i].y = -x[i].y;
    }
}

// Last-stage outputs straight to global memory (rows q + m*M/RP of column c).
template <int RP, int E, int LGM, int LGC, typename R, typename C>
__device__ __forceinline__ void last_store(C* __restrict__ out, const C* v, const FftPass& d, uint64_t outBase,
                                           R scale, R scaleLo, int tid, int nt) {
    constexpr int NB = E / RP;
    constexpr int LGR = RP == 8 ? 3 : (RP == 4 ? 2 : 1);
    constexpr int lgMq = LGM - LGR;
#pragma unroll
    for (int k = 0; k < NB; ++k) {
        const BflyPos p = bfly_pos<RP, LGM, E>(tid, k, nt, LGC);
        const uint64_t g0 = outBase + ((uint64_t)p.hb << d.lgOutH2) + p.c;
#pragma unroll
        for (int m = 0; m < RP; ++m) {
            const int row = p.q + (m << lgMq);
            out[g0 + ((uint64_t)row << d.lgOutR)] = v[k * RP + m];
        }
    }
}
