// fft_chain.hip - several transforms of one register field in one launch.
//
// Where a tile of the state (all M rows of the field x C columns x Hb blocks) fits a
// workgroup's LDS, the transforms that one gate applies to that field run back to
// back on the tile in registers: load, then for each transform its pending phases
// and the Stockham stages (fft_stages.h), then one store.  A squeezing gate's four
// transforms take one launch and one pass over the state instead of four of each.
//
// The phases are evaluated in place in FP64 (one cubic in the row coordinate a
// butterfly, reduced, its sine and cosine rounded once to the state's precision with the
// normalisation folded in), so no table has to be built by a launch of its own.  A tile
// of several columns evaluates each row once when no term of the program varies over
// its columns, and shares the factors through LDS.
//
// Bound by in-CU work: at 2^21 complex128 ([1,10,10]) a launch takes 15 us with one
// transform of the contiguous register (10 of them to load and store) and about 7 more
// with each further one, a third of that the phases; a whole pass with its table build
// took 20.5.  One workgroup alone ([1,10]) takes 4 us and 2.4 a transform.

#include <algorithm>
#include <cmath>

#include "cvdv_internal.h"
#include "fft_stages.h"
#include "phase_eval.h"

// One transform of a chain: phases, direction, normalisation.  Terms [0, nrow): the
// transformed field itself (a cubic, or bilinear with another field), their control
// outside it; the rest vary over the rows in some other way.
struct ChainStep {
    int inv, n, nrow;
    int ctl;        // bit + 1: elements with this index bit set are transformed the other way; 0: none
    int byRow;      // every term has one value per row of a tile
    double grev, scale;
    DiagTerm t[FT_CHAIN_TERMS];
};

struct ChainArgs {
    int m;
    int lgHb, lgNLoBlk;  // blocks of a tile, column groups
    int lgH, lgR, pad;   // element strides of blocks and rows
    ChainStep s[FT_CHAIN_MAX];
};

// Largest tile: 64 KiB of elements, so that two workgroups share a CU.
template <typename R> constexpr int chain_lg_tile() { return sizeof(R) == 8 ? 12 : 13; }
template <typename R, int LGC> constexpr int chain_ex() { return sizeof(R) == 8 && LGC == 0 ? EX_ROWS : EX_TILE; }
// Elements of LDS for one block of rows.
template <typename R, int LGM, int LGC> constexpr int chain_block_lds() {
    constexpr int tile = 1 << (LGM + LGC);
    return tile + (chain_ex<R, LGC>() == EX_ROWS || tile < 32 ? tile / 8 : tile / 32);
}

// The row terms at a thread's elements (fixed column and block) as a + c1 m + c2 m^2 +
// c3 m^3 in the row coordinate m (revolutions; m is an integer, so linear coefficients
// count mod 1).  The linear part is split: a is its multiple of 1/(4N), whose products
// with m are exact (a transform's own twiddle is nothing else), c1 the rest, at most
// 1/(8N).  In one sum the twiddle's hundreds of revolutions would cost the others their
// last digits ([1,1,1,1,12] state transfer: 1.7e-14 off instead of 3e-15).
struct RowCubic {
    double a, c1, c2, c3;
    // (the quadratic and cubic part, a thousand revolutions at the edge, reduced before it is rounded)
    __device__ __forceinline__ double at(double m) const {
        const double m2 = m * m, q = fma(c3, m, c2);
        return cvdv_frac(a * m) + fma(c1, m, fma(q, m2, -rint(q * m2)));
    }
    __device__ __forceinline__ void linear(double c, double n4) {  // n4 = 4N
        c = cvdv_frac(c);
        const double h = rint(c * n4) / n4;
        a += h;
        c1 += c - h;
    }
};

__device__ __forceinline__ double chain_coord(uint32_t g, int sh, int nb) {
    return (double)((int)(2u * ((g >> sh) & ((1u << nb) - 1u))) + 1 - (1 << nb));
}

template <int N>
__device__ __forceinline__ RowCubic row_cubic(const ChainStep& st, uint32_t g, int sh) {
    RowCubic f{0.0, 0.0, 0.0, 0.0};
    const int n = __builtin_amdgcn_readfirstlane(st.nrow);
#pragma unroll 1
    for (int k = 0; k < n; ++k) {
        const DiagTerm& t = st.t[k];
        const int ctrl = __builtin_amdgcn_readfirstlane(t.ctrl);
        const double sg = ctrl >= 0 && ((g >> ctrl) & 1u) ? -1.0 : 1.0;
        if (__builtin_amdgcn_readfirstlane(t.kind) == DT_BILIN) {
            const bool first = __builtin_amdgcn_readfirstlane(t.sh1) == sh;
            const int osh = __builtin_amdgcn_readfirstlane(first ? t.sh2 : t.sh1);
            const int onb = __builtin_amdgcn_readfirstlane(first ? t.nb2 : t.nb1);
            const double c = chain_coord(g, osh, onb), p = t.c1 * c;
            f.linear(sg * p, 4.0 * N);
            f.c1 += sg * fma(t.c1, c, -p);
        } else {
            f.linear(sg * t.c1, 4.0 * N);
            f.c2 += sg * t.c2;
            f.c3 += sg * t.c3;
        }
    }
    f.a = cvdv_frac(f.a);
    return f;
}

// The other terms at element g.
__device__ __forceinline__ double chain_others(const ChainStep& st, uint32_t g) {
    double r = 0.0;
    const int n = __builtin_amdgcn_readfirstlane(st.n);
#pragma unroll 1
    for (int k = __builtin_amdgcn_readfirstlane(st.nrow); k < n; ++k) r += cvdv_frac(diag_term_rev(st.t[k], g));
    return r;
}

// Phase factor and normalisation at rev revolutions past the constant phase.
template <typename R>
__device__ __forceinline__ double2 chain_factor(const ChainStep& st, double rev) {
    const double2 u = unit_turn(cvdv_frac(rev + st.grev), R(0));
    return make_double2(u.x * st.scale, u.y * st.scale);
}

// The factor applied: a complex64 element takes the FP64 factor in FP64 and is rounded
// once, where a factor rounded first would add its own error.
template <typename R, typename C>
__device__ __forceinline__ C chain_apply(const ChainStep& st, double rev, C v) {
    const double2 p = cmul(make_double2((double)v.x, (double)v.y), chain_factor<R>(st, rev));
    return cmk<C>(p.x, p.y);
}

// A thread owns the rows q + j M/8, j < 8, of one column and block in every stage
// (bfly_pos), so no exchange is needed between transforms.  Each block of rows is
// transformed by threads and LDS of its own.
// The steps are read from the kernel's argument segment straight into LDS (a is the
// first argument): indexing the argument at run time would copy it to scratch memory.
template <typename R, int LGM, int LGC> constexpr int chain_threads_max() { return LGM + LGC >= 13 ? 1024 : 512; }
template <typename R, int LGM, int LGC>
__global__ void __launch_bounds__((chain_threads_max<R, LGM, LGC>()), 4)
k_fft_chain(ChainArgs a, typename CT<R>::type* data, const typename CT<R>::type* __restrict__ tw) {
    using C = typename CT<R>::type;
    constexpr int EX = chain_ex<R, LGC>();
    constexpr int M = 1 << LGM, ST = 1 << (LGM + LGC - 3);  // threads of a block
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ ChainStep steps[FT_CHAIN_MAX];
    const int tid = threadIdx.x & (ST - 1), hb = threadIdx.x >> (LGM + LGC - 3);
    C* lds = reinterpret_cast<C*>(smem_raw) + hb * chain_block_lds<R, LGM, LGC>();

    // tiles of part of a 256-byte run (narrow columns) that share it run on one XCD
    // (workgroups go round the eight XCDs in turn): 64-byte columns would fetch and
    // write every 128-byte line from two of them
    uint32_t t = blockIdx.x;
    if ((sizeof(C) << LGC) < 256 && a.lgNLoBlk >= 2 && (gridDim.x & 31u) == 0) {
        const uint32_t xcd = t & 7u, i = t >> 3;
        t = ((((i >> 2) << 3) + xcd) << 2) + (i & 3u);
    }
    const uint32_t loBlk = t & ((1u << a.lgNLoBlk) - 1u), h = (t >> a.lgNLoBlk << a.lgHb) + (uint32_t)hb;
    const uint32_t base = (h << a.lgH) + (loBlk << LGC);  // the block's first element
    const uint32_t own = base + ((uint32_t)(tid >> LGC) << a.lgR) + (uint32_t)(tid & ((1 << LGC) - 1));
    auto elem = [&](int j) { return own + ((uint32_t)(j << (LGM - 3)) << a.lgR); };
    C x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = data[elem(j)];
    {
        typedef const __attribute__((address_space(4))) uint32_t* KArg;
        const KArg src = (KArg)__builtin_amdgcn_kernarg_segment_ptr() + offsetof(ChainArgs, s) / 4;
        const int words = a.m * (int)(sizeof(ChainStep) / 4);
        for (int i = threadIdx.x; i < words; i += blockDim.x) ((uint32_t*)steps)[i] = src[i];
    }
    __syncthreads();

#pragma unroll 1
    for (int s = 0; s < a.m; ++s) {
        const ChainStep& st = steps[s];
        const int ctl = __builtin_amdgcn_readfirstlane(st.ctl);
        int inv = __builtin_amdgcn_readfirstlane(st.inv);
        if (ctl) inv ^= (int)(own >> (ctl - 1)) & 1;
        // an opaque copy of the thread id: index math and twiddles, the same for every
        // step, would otherwise all be held across the steps
        int ti = tid;
        asm volatile("" : "+v"(ti));
        const int q = ti >> LGC;
        const bool other = __builtin_amdgcn_readfirstlane(st.n) > __builtin_amdgcn_readfirstlane(st.nrow);
        auto coord = [](int row) { return (double)(2 * row + 1 - M); };
        bool shared = false;
        if constexpr (LGC > 0) {
            if (__builtin_amdgcn_readfirstlane(st.byRow)) {
                // one factor per row; the exchange buffer is free here
                const RowCubic f = row_cubic<M>(st, base, a.lgR);
#pragma unroll 1
                for (int row = ti; row < M; row += ST) {
                    double r = f.at(coord(row));
                    if (other) r += chain_others(st, base + ((uint32_t)row << a.lgR));
                    const double2 e = chain_factor<R>(st, r);
                    lds[row] = cmk<C>(e.x, e.y);
                }
                lds_barrier();
#pragma unroll
                for (int j = 0; j < 8; ++j) x[j] = cmul(x[j], lds[q + j * (M / 8)]);
                lds_barrier();
                shared = true;
            }
        }
        if (!shared) {
            const RowCubic f = row_cubic<M>(st, own, a.lgR);
            double r[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) r[j] = f.at(coord(q + j * (M / 8)));
            if (other) {
                // one element at a time, through its own slot of the exchange buffer; x is
                // not touched here (a first transform's loads are still in flight)
                double* mine = reinterpret_cast<double*>(lds) + ti * (int)(sizeof(C) / sizeof(double));
#pragma unroll 1
                for (int j = 0; j < 8; ++j) mine[j * ST * (int)(sizeof(C) / sizeof(double))] = chain_others(st, elem(j));
#pragma unroll
                for (int j = 0; j < 8; ++j) r[j] += mine[j * ST * (int)(sizeof(C) / sizeof(double))];
                lds_barrier();
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] = chain_apply<R>(st, r[j], x[j]);
        }
        if (inv) {  // inverse = conj . forward . conj
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j].y = -x[j].y;
        }
        stage_compute<8, 8, LGM, LGC, 0>(x, tw, ti, ST);
        run_stages<LGM, LGC, 1, 8, EX>(x, lds, tw, ti, ST);
        to_rows<LGM, 8>(x);
        if (inv) {
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j].y = -x[j].y;
        }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) data[elem(j)] = x[j];
}

// ---------------------------------------------------------------- planning
// The chain tile of field [sh, sh + nb): lg of columns and blocks; false when the field's
// transforms do not run as chains.
//
// States up to 2^FT_CHAIN_LG_SMALL are bound by launches, table builds and latency, and
// every transform goes through here (gates alone, us, table path against chains: [1,10]
// complex128 135 / 74, [8,8] 432 / 189, [1,10,10] 580 / 442, mixed 509 / 370).  Above,
// HBM passes are the cost: only gates with several transforms of a field whose tile
// keeps whole runs, and no more than 2^12 elements ([1,12,12] complex128 7.22 / 6.59 ms by its
// contiguous register, [14,12] mixed 9.89 / 8.92; runs of 64 bytes lose, [10,14] mixed 2.39 / 2.48, as do
// tiles of 2^13, [14,13] mixed 20.1 / 20.8).  Contiguous rows of row_instance lengths go
// through fft_row.hip there.
static bool chain_tile(const CVDVContext* ctx, int sh, int nb, int& lgC, int& lgHb) {
    const int T = ctx->totalQbt, lgW = ctx->prec == CVDV_C128 ? 4 : 5;
    const bool small = T <= FT_CHAIN_LG_SMALL;
    const int lgTile = small && ctx->prec == CVDV_MIXED ? 13 : 12;
    if (ctx->rec || T > FT_CHAIN_LG_MAX || nb < 3 || nb > lgTile || T < 6) return false;
    // 256 bytes of a row where the tile has room, no less than 64 (or the whole run)
    lgC = std::min({sh, lgW, lgTile - nb});
    if (lgC < sh && lgC < (small ? lgW - 2 : lgW)) return false;
    // a tile of at least 64 threads and at most 2^11 elements over blocks, while more than
    // 512 tiles remain
    lgHb = 0;
    while (nb + lgC + lgHb < 11 && lgHb < T - sh - nb && (nb + lgC + lgHb < 9 || T - nb - lgC - lgHb > 9)) ++lgHb;
    return true;
}

static bool term_idle(const DiagTerm& t) { return t.c1 == 0.0 && t.c2 == 0.0 && t.c3 == 0.0; }

template <typename R, int LGM, int LGC>
static void launch_chain_geom(CVDVContext* ctx, const ChainArgs& a, unsigned tiles) {
    if constexpr (LGM + LGC <= chain_lg_tile<R>()) {
        using C = typename CT<R>::type;
        const int tile = 1 << (LGM + LGC + a.lgHb);
        const size_t lds = ((size_t)chain_block_lds<R, LGM, LGC>() << a.lgHb) * sizeof(C);
        auto kfn = k_fft_chain<R, LGM, LGC>;
        if (tile / 8 > chain_threads_max<R, LGM, LGC>() || tile < 8) throw CvdvError{CVDV_ERR_UNSUPPORTED, "chain tile out of range"};
        if (lds > 64 * 1024)
            HIPCHK(hipFuncSetAttribute((const void*)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        const C* tw = (const C*)fft_stage_table(ctx->tw, LGM, ctx->prec);
        hipLaunchKernelGGL(kfn, dim3(tiles), dim3(tile / 8), lds, ctx->stream, a, (C*)ctx->state(), tw);
    } else {
        throw CvdvError{CVDV_ERR_UNSUPPORTED, "chain tile shape without a kernel instance"};
    }
}

template <typename R, int LGM>
static void launch_chain_lgm(CVDVContext* ctx, const ChainArgs& a, int lgC, unsigned tiles) {
    switch (lgC) {
        case 0: launch_chain_geom<R, LGM, 0>(ctx, a, tiles); break;
        case 1: launch_chain_geom<R, LGM, 1>(ctx, a, tiles); break;
        case 2: launch_chain_geom<R, LGM, 2>(ctx, a, tiles); break;
        case 3: launch_chain_geom<R, LGM, 3>(ctx, a, tiles); break;
        case 4: launch_chain_geom<R, LGM, 4>(ctx, a, tiles); break;
        case 5:
            if constexpr (sizeof(R) == 4) {
                launch_chain_geom<R, LGM, 5>(ctx, a, tiles);
                break;
            }
        default: throw CvdvError{CVDV_ERR_UNSUPPORTED, "chain tile column count out of range"};
    }
}

template <typename R>
static void launch_chain(CVDVContext* ctx, const ChainArgs& a, int nb, int lgC, unsigned tiles) {
    switch (nb) {
#define CVDV_CHAIN_CASE(L) \
    case L: launch_chain_lgm<R, L>(ctx, a, lgC, tiles); break;
        CVDV_CHAIN_CASE(3) CVDV_CHAIN_CASE(4) CVDV_CHAIN_CASE(5) CVDV_CHAIN_CASE(6) CVDV_CHAIN_CASE(7)
        CVDV_CHAIN_CASE(8) CVDV_CHAIN_CASE(9) CVDV_CHAIN_CASE(10) CVDV_CHAIN_CASE(11) CVDV_CHAIN_CASE(12)
        CVDV_CHAIN_CASE(13)
#undef CVDV_CHAIN_CASE
        default: throw CvdvError{CVDV_ERR_UNSUPPORTED, "chain transform length out of range"};
    }
}

void chain_flush(CVDVContext* ctx) {
    FtChain& ch = ctx->chain;
    if (ch.n == 0) return;
    const int sh = ch.sh, nb = ch.nb, m = ch.n;
    ch.n = 0;  // launched or, on an error, dropped
    const bool rows = row_field(ctx, sh, nb);
    if (m == 1 && (rows || ctx->totalQbt > FT_CHAIN_LG_SMALL)) {
        const FtChainStep c = ch.st[0];
        fft_whole(ctx, sh, nb, c.inverse != 0, c.prog, c.scale, c.ctrl);
        return;
    }
    if (rows) {
        FtChainStep st[FT_CHAIN_MAX];  // (compiling may flush)
        std::copy(ch.st, ch.st + m, st);
        fft_row_chain(ctx, nb, st, m);
        return;
    }
    int lgC, lgHb;
    if (!chain_tile(ctx, sh, nb, lgC, lgHb)) throw CvdvError{CVDV_ERR_STATE, "chain without a tile"};
    const int T = ctx->totalQbt;
    ChainArgs a{};
    a.m = m;
    a.lgHb = lgHb;
    a.lgNLoBlk = sh - lgC;
    a.lgR = sh;
    a.lgH = sh + nb;
    const uint64_t within = (1ull << lgC) - 1ull;  // columns
    for (int i = 0; i < m; ++i) {
        const FtChainStep& c = ch.st[i];
        ChainStep& s = a.s[i];
        s.inv = c.inverse;
        s.ctl = c.ctrl + 1;
        s.grev = cvdv_frac(c.prog.grev);
        s.scale = c.scale;
        s.byRow = 1;
        DiagTerm rest[FT_CHAIN_TERMS];
        int nrest = 0;
        for (int k = 0; k < c.prog.n; ++k) {
            const DiagTerm& t = c.prog.t[k];
            if (term_idle(t)) continue;
            const bool in1 = t.sh1 == sh && t.nb1 == nb, in2 = t.sh2 == sh && t.nb2 == nb;
            const bool row = !(t.ctrl >= sh && t.ctrl < sh + nb) &&
                             (t.kind == DT_BILIN ? in1 != in2 : (t.kind == DT_POLY || t.kind == DT_LINF) && in1);
            if (row) s.t[s.nrow++] = t;
            else rest[nrest++] = t;
            uint64_t bits = ((1ull << t.nb1) - 1ull) << t.sh1;
            if (t.kind == DT_BILIN) bits |= ((1ull << t.nb2) - 1ull) << t.sh2;
            if (t.ctrl >= 0) bits |= 1ull << t.ctrl;
            if (bits & within) s.byRow = 0;
        }
        s.n = s.nrow;
        for (int k = 0; k < nrest; ++k) s.t[s.n++] = rest[k];
    }
    const unsigned tiles = 1u << (T - nb - lgC - lgHb);
    const int pid = prof_begin(ctx, lgC == 0 && lgHb == 0 && nb >= 12 ? KK_FFT_ROW : KK_FFT);
    if (ctx->prec == CVDV_C128) launch_chain<double>(ctx, a, nb, lgC, tiles);
    else launch_chain<float>(ctx, a, nb, lgC, tiles);
    HIPCHK(hipGetLastError());
    prof_end(ctx, pid);
}

bool chain_field(const CVDVContext* ctx, int sh, int nb) {
    int lgC, lgHb;
    return row_field(ctx, sh, nb) || chain_tile(ctx, sh, nb, lgC, lgHb);
}

bool chain_accept(CVDVContext* ctx, int sh, int nb, bool inverse, const DiagProg& pre, double outScale,
                  int ctrl) {
    FtChain& ch = ctx->chain;
    const bool one = !ch.open || !ctx->fuseFt;
    const bool rows = row_field(ctx, sh, nb);
    if ((one && (rows || ctx->totalQbt > FT_CHAIN_LG_SMALL)) || !chain_field(ctx, sh, nb)) return false;
    int n = 0;
    for (int k = 0; k < pre.n; ++k) n += !term_idle(pre.t[k]);
    if (rows ? !row_accepts(ctx, nb, pre) : n > FT_CHAIN_TERMS) return false;
    if (ch.n > 0 && (ch.sh != sh || ch.nb != nb || ch.n == FT_CHAIN_MAX)) chain_flush(ctx);
    ch.sh = sh;
    ch.nb = nb;
    ch.st[ch.n++] = FtChainStep{pre, inverse ? 1 : 0, outScale, ctrl};
    if (one) chain_flush(ctx);
    return true;
}
