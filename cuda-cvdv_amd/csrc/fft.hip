// fft.hip - register-axis FFT for gfx950 (replaces the cuFFT plans and the
// outer-block exec loop of src/cuda/context.cu:48-65 and gates.cu:37-52).
//
// A register field [sh, sh+n) of the flat index splits every element index as
//     g = hi * (N*S) + j * S + lo,   S = 2^sh, N = 2^n,
// and the FFT runs over j for every (hi, lo).  A workgroup stages a tile of
// C consecutive lo columns x M rows x Hb consecutive hi blocks in LDS, runs a
// Stockham FFT there (radix 8/4/2 butterflies in registers, per-stage twiddle
// tables generated in FP64), and writes the tile back:
//   * one HBM pass when the tile fits in LDS: C*M elements with C = 32 (c64)
//     or 16 (c128) columns (256 bytes per row) for a strided register, or a
//     whole contiguous register of up to 2^14 (c64) / 2^13 (c128) points in one
//     workgroup (c64 rows of 2^13 and 2^14: fft_row.hip);
//   * otherwise the four-step split N = N1 * N2 (j = j1 + N1 j2):
//       pass 1 (in place):  FFT over j2;
//       pass 2 (out of place, transposing): times W_N^{j1 k2} on load, FFT
//       over j1, written at k2 + N2 k1.
// Pending diagonal phases are applied (compiled, see diag_fast.h) as elements
// are loaded by the first pass and 1/sqrt(N) as they are stored by the last.
// Every tile dimension is a power of two: indices use shifts and masks only.

#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

#include "cvdv_internal.h"
#include "fft_pass.h"
#include "fft_fused.h"
#include "fft_row.h"

static const long double PI_L = 3.141592653589793238462643383279502884L;

// ---------------------------------------------------------------- twiddles
struct TwKey {
    int logM;
    int prec;
    bool operator<(const TwKey& o) const { return logM != o.logM ? logM < o.logM : prec < o.prec; }
};

struct TwiddleCache {
    std::map<TwKey, void*> stage;  // per-stage Stockham tables for length M
    std::map<TwKey, void*> full;   // W_N^e, e in [0, N)
};

void twiddle_cache_free(TwiddleCache* tc) {
    for (auto& kv : tc->stage) (void)hipFree(kv.second);
    for (auto& kv : tc->full) (void)hipFree(kv.second);
    delete tc;
}

// exp(-2 pi i e / N) from an 80-bit evaluation, rounded once to double.
static void host_twiddle(uint64_t e, uint64_t N, double& c, double& s) {
    const long double a = 2.0L * PI_L * (long double)e / (long double)N;
    c = (double)cosl(a);
    s = (double)-sinl(a);
}

struct StagePlan {
    int nst = 0;
    int rad[16];
    int L[16];
    int off[16];
    int total = 0;  // table entries
};

static StagePlan stage_plan(int logM) {
    StagePlan p;
    int rem = logM, L = 1, off = 0;
    while (rem > 0) {
        const int r = rem >= 3 ? 3 : rem;  // radix 8, then a final 4 or 2
        const int R = 1 << r;
        p.rad[p.nst] = R;
        p.L[p.nst] = L;
        p.off[p.nst] = off;
        off += L * (R - 1);
        L *= R;
        rem -= r;
        p.nst++;
    }
    p.total = off;
    return p;
}

// FP32 twiddles: every entry is one of the floats adjacent to (or equal to) the
// exact value, chosen by error diffusion so that sum(|w|^2 - 1) over each
// stage stays near zero.  Rounding each entry to nearest leaves a mean
// |w|^2 - 1 of order -1e-8, which shrinks the norm by ~2e-8 per FFT.
static void round_unit_diffused(const double* re, const double* im, size_t n, float2* out) {
    double acc = 0.0;
    for (size_t i = 0; i < n; ++i) {
        const float c0 = (float)re[i], s0 = (float)im[i];
        const float cs[3] = {nextafterf(c0, -2.f), c0, nextafterf(c0, 2.f)};
        const float ss[3] = {nextafterf(s0, -2.f), s0, nextafterf(s0, 2.f)};
        double bestErr = 0.0, bestScore = 1e300;
        float bc = c0, bs = s0;
        for (int a = 0; a < 3; ++a) {
            if (std::fabs((double)cs[a] - re[i]) > std::fabs((double)nextafterf(c0, 2.f) - (double)c0)) continue;
            for (int b = 0; b < 3; ++b) {
                if (std::fabs((double)ss[b] - im[i]) > std::fabs((double)nextafterf(s0, 2.f) - (double)s0)) continue;
                const double err = (double)cs[a] * cs[a] + (double)ss[b] * ss[b] - 1.0;
                const double score = std::fabs(acc + err);
                if (score < bestScore) {
                    bestScore = score;
                    bestErr = err;
                    bc = cs[a];
                    bs = ss[b];
                }
            }
        }
        acc += bestErr;
        out[i] = make_float2(bc, bs);
    }
}

// Host copy of a table in the state's precision (FP32: error-diffused per segment).
static std::vector<uint8_t> round_table(const std::vector<double>& re, const std::vector<double>& im, int prec,
                                        const std::vector<size_t>& segments = {}) {
    const size_t n = re.size();
    std::vector<uint8_t> bytes;
    if (prec == CVDV_C128) {
        bytes.resize(n * sizeof(double2));
        double2* h = (double2*)bytes.data();
        for (size_t i = 0; i < n; ++i) h[i] = make_double2(re[i], im[i]);
    } else {
        bytes.resize(n * sizeof(float2));
        float2* h = (float2*)bytes.data();
        size_t start = 0;
        std::vector<size_t> seg = segments;
        seg.push_back(n);
        for (size_t end : seg) {
            if (end > start) round_unit_diffused(re.data() + start, im.data() + start, end - start, h + start);
            start = end;
        }
    }
    return bytes;
}

static void* upload_table(const std::vector<double>& re, const std::vector<double>& im, int prec,
                          const std::vector<size_t>& segments = {}) {
    const std::vector<uint8_t> h = round_table(re, im, prec, segments);
    void* d = nullptr;
    HIPCHK(hipMalloc(&d, h.size() ? h.size() : 16));
    if (!h.empty()) HIPCHK(hipMemcpy(d, h.data(), h.size(), hipMemcpyHostToDevice));
    return d;
}

static TwiddleCache* cache(CVDVContext* ctx) {
    if (!ctx->tw) ctx->tw = new TwiddleCache();
    return ctx->tw;
}

// Stockham stage twiddles for length 2^logM: stage s (radix R, sub-length L)
// holds W_{RL}^{ij} at off[s] + j (R-1) + i - 1, j < L, 1 <= i < R.
static void stage_values(int logM, std::vector<double>& re, std::vector<double>& im, std::vector<size_t>& segs) {
    const StagePlan p = stage_plan(logM);
    const uint64_t M = 1ull << logM;
    re.assign(p.total, 0.0);
    im.assign(p.total, 0.0);
    for (int s = 0; s < p.nst; ++s) {
        const int R = p.rad[s], L = p.L[s];
        for (int j = 0; j < L; ++j)
            for (int i = 1; i < R; ++i) {
                // W_{R L}^{i j} = W_M^{i j M / (R L)}
                const uint64_t e = (uint64_t)i * j * (M / ((uint64_t)R * L));
                host_twiddle(e, M, re[p.off[s] + j * (R - 1) + i - 1], im[p.off[s] + j * (R - 1) + i - 1]);
            }
    }
    segs.clear();
    for (int st = 1; st < p.nst; ++st) segs.push_back((size_t)p.off[st]);
}

std::vector<uint8_t> fft_stage_host(int logM, int prec) {
    std::vector<double> re, im;
    std::vector<size_t> segs;
    stage_values(logM, re, im, segs);
    return round_table(re, im, prec, segs);
}

const void* fft_stage_table(TwiddleCache*& tcp, int logM, int prec) {
    if (!tcp) tcp = new TwiddleCache();
    TwiddleCache* tc = tcp;
    auto it = tc->stage.find({logM, prec});
    if (it != tc->stage.end()) return it->second;
    std::vector<double> re, im;
    std::vector<size_t> segs;
    stage_values(logM, re, im, segs);
    void* d = upload_table(re, im, prec, segs);
    tc->stage[{logM, prec}] = d;
    return d;
}

// Twiddles of the row kernel (fft_row.hip), E elements a thread: W_{E^2}^{j p} of the middle
// stage (p < E), then W_M^{j t}, t < M/E, of the last as W_{M/E}^{j a} W_M^{j b}, t = E a + b;
// j-major.
static void row_values(int lgm, int lge, std::vector<double>& re, std::vector<double>& im, std::vector<size_t>& segs) {
    const uint64_t M = 1ull << lgm, E = 1ull << lge, RL = M / (E * E);
    auto put = [&](uint64_t e, uint64_t N) {
        double c, s;
        host_twiddle(e, N, c, s);
        re.push_back(c);
        im.push_back(s);
    };
    for (uint64_t j = 1; j < E; ++j)
        for (uint64_t p = 0; p < E; ++p) put(j * p, E * E);
    segs.push_back(re.size());
    for (uint64_t j = 1; j < RL; ++j)
        for (uint64_t a = 0; a < RL; ++a) put(j * a, M / E);
    segs.push_back(re.size());
    for (uint64_t j = 1; j < RL; ++j)
        for (uint64_t b = 0; b < E; ++b) put(j * b, M);
}

static const void* row_table(CVDVContext* ctx, int lgm, int prec) {
    TwiddleCache* tc = cache(ctx);
    const TwKey key{lgm + 1000, prec};
    auto it = tc->stage.find(key);
    if (it != tc->stage.end()) return it->second;
    if (ctx->capturing) throw CvdvError{CVDV_ERR_UNSUPPORTED, "FFT table not prepared before the graph capture"};
    std::vector<double> re, im;
    std::vector<size_t> segs;
    row_values(lgm, row_lge_of(prec == CVDV_C128), re, im, segs);
    void* d = upload_table(re, im, prec, segs);
    tc->stage[key] = d;
    return d;
}

// Twiddles of the two-stage fused kernel (fft_fused.hip): for each j and q those of a thread's
// two butterflies, side by side.
static const void* fuse2_table(CVDVContext* ctx) {
    TwiddleCache* tc = cache(ctx);
    const TwKey key{FUSE2_LGM + 2000, CVDV_MIXED};
    auto it = tc->stage.find(key);
    if (it != tc->stage.end()) return it->second;
    if (ctx->capturing) throw CvdvError{CVDV_ERR_UNSUPPORTED, "FFT table not prepared before the graph capture"};
    const uint64_t M = 1ull << FUSE2_LGM, Q = M / 16;
    std::vector<double> re, im;
    for (uint64_t j = 1; j < 8; ++j)
        for (uint64_t q = 0; q < Q; ++q)
            for (uint64_t k = 0; k < 2; ++k) {
                double c, s;
                host_twiddle(j * (q + k * Q), M, c, s);
                re.push_back(c);
                im.push_back(s);
            }
    void* d = upload_table(re, im, CVDV_MIXED);
    tc->stage[key] = d;
    return d;
}

static void* stage_table(CVDVContext* ctx, int logM, int prec) {
    if (ctx->capturing && (!ctx->tw || !ctx->tw->stage.count({logM, prec})))
        throw CvdvError{CVDV_ERR_UNSUPPORTED, "FFT table not prepared before the graph capture"};
    return (void*)fft_stage_table(ctx->tw, logM, prec);
}

// W_N^e for e in [0, N) in the given precision (FP32: error-diffused rounding,
// as for the stage tables).  The direct DFT always uses the FP64 table.
static const void* full_table(CVDVContext* ctx, int logN, int prec = CVDV_C128) {
    TwiddleCache* tc = cache(ctx);
    auto it = tc->full.find({logN, prec});
    if (it != tc->full.end()) return it->second;
    if (ctx->capturing) throw CvdvError{CVDV_ERR_UNSUPPORTED, "FFT table not prepared before the graph capture"};
    const uint64_t N = 1ull << logN;
    std::vector<double> re(N), im(N);
    for (uint64_t e = 0; e < N; ++e) host_twiddle(e, N, re[e], im[e]);
    void* d = upload_table(re, im, prec);
    tc->full[{logN, prec}] = d;
    return d;
}

// Device properties the planner asks for on every launch, cached per device.
// Contexts may run on several host threads: the caches are guarded.
static std::mutex g_devCacheMu;

size_t device_max_lds() {
    static std::map<int, size_t> cached;
    int dev = 0;
    HIPCHK(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(g_devCacheMu);
    auto it = cached.find(dev);
    if (it != cached.end()) return it->second;
    int v = 0;
    HIPCHK(hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    cached[dev] = (size_t)v;
    return (size_t)v;
}

// One-row complex64 tiles of 2^13-2^14 points lay out their first two exchanges
// apart from the others (ex_lay); their LDS ends at tile + tile/8.
template <typename R, int LGM, int LGC>
constexpr bool one_row_layouts() {
    return sizeof(R) == 4 && LGC == 0 && LGM >= 13 && Plan<LGM>::lgr(0) == 3 && Plan<LGM>::lgr(1) == 3;
}

// Workgroup size bound: one-row tiles of 2^12 points and more take up to 1024
// threads; every other tile fits 64 KiB of LDS, i.e. at most 512 (complex64) or
// 256 (complex128) threads at 8 elements each.
template <typename R, int LGM, int LGC>
constexpr int tile_threads_max() {
    return (LGC == 0 && LGM >= 12) ? 1024 : (sizeof(R) == 4 ? 512 : 256);
}

template <typename R, int LGM, int LGC, int E>
__global__ void __launch_bounds__((tile_threads_max<R, LGM, LGC>()))
k_fft_tile(const typename CT<R>::type* in, typename CT<R>::type* out, FftPass d, FastDiag pre,
           const typename CT<R>::type* __restrict__ tw, const typename CT<R>::type* __restrict__ tw4) {
    using C = typename CT<R>::type;
    constexpr int NST = Plan<LGM>::NST;
    constexpr int R0 = 1 << Plan<LGM>::lgr(0);
    constexpr int RL = 1 << Plan<LGM>::lgr(NST - 1);
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ PreLds P;
    C* lds = reinterpret_cast<C*>(smem_raw);
    const int tid = threadIdx.x, nt = blockDim.x;
    constexpr int lgC = LGC;  // the tile's column count is part of the instance
    const int lgHb = d.lgHb;
    // one-row complex64 tiles of 2^13-2^14 points: exchanges 0 and 1 in their own
    // layouts, the largest of which ends at tile + tile/8 (the host sizes LDS so)
    constexpr bool ONE = one_row_layouts<R, LGM, LGC>();

    if (d.usePre) {
        // constant indices: the argument is read in place (one entry per thread,
        // or all by thread 0 in a tile with fewer threads than entries)
        if (nt >= CVDV_FAST_TABS + CVDV_FAST_GEN) {
#pragma unroll
            for (int i = 0; i < CVDV_FAST_TABS; ++i)
                if (tid == i && i < pre.ntab) P.tab[i] = pre.tab[i];
#pragma unroll
            for (int i = 0; i < CVDV_FAST_GEN; ++i)
                if (tid == CVDV_FAST_TABS + i && i < pre.ngen) P.gen[i] = pre.gen[i];
        } else if (tid == 0) {
#pragma unroll
            for (int i = 0; i < CVDV_FAST_TABS; ++i)
                if (i < pre.ntab) P.tab[i] = pre.tab[i];
#pragma unroll
            for (int i = 0; i < CVDV_FAST_GEN; ++i)
                if (i < pre.ngen) P.gen[i] = pre.gen[i];
        }
        __syncthreads();
    }

    const R scale = (R)d.outScale;
    const R scaleLo = (R)(d.outScale - (double)scale);
    auto tile_base = [&](uint64_t t, uint64_t& lo0, uint64_t& inBase, uint64_t& outBase) {
        const uint64_t loBlk = t & ((1ull << d.lgNLoBlk) - 1);
        const uint64_t r = t >> d.lgNLoBlk;
        const uint64_t h2Blk = r & ((1ull << d.lgNH2Blk) - 1);
        const uint64_t h1 = r >> d.lgNH2Blk;
        lo0 = loBlk << lgC;
        inBase = (h1 << d.lgInH1) + ((h2Blk << lgHb) << d.lgInH2) + lo0;
        outBase = (h1 << d.lgOutH1) + ((h2Blk << lgHb) << d.lgOutH2) + lo0;
    };
    // Phases of the loaded tile t (their table loads are global loads).
    auto prephase = [&](C* x, uint64_t t, int ti) {
        uint64_t lo0, inBase, outBase;
        tile_base(t, lo0, inBase, outBase);
        stage0_pre<R0, E, LGM, LGC, true, TM_ANY>(x, d, inBase, P, pre, tw4, ti, nt, lds);
    };
    // Transform the phased tile in registers (the last stage's outputs stay in x).
    auto stages = [&](C* x, int ti) {
        stage_compute<R0, E, LGM, LGC, 0>(x, tw, ti, nt);
        run_stages<LGM, LGC, 1, E, ONE ? EX_ONE : EX_TILE>(x, lds, tw, ti, nt);
    };
    // Store the transformed tile t.
    // Staged store, first half: the last stage's outputs into LDS in natural order.
    auto stage_out = [&](C* x, int ti) {
        stage_write<RL, E, LGM, LGC, NST - 1>(lds, x, ti, nt);
        lds_barrier();
    };
    // Staged store, second half: LDS to global memory in the output's contiguous order.
    auto store_lds = [&](uint64_t t, int ti) {
        uint64_t lo0, inBase, outBase;
        tile_base(t, lo0, inBase, outBase);
        auto value = [&](int c, int row, int hb) {
            return lds[lds_ix((((hb << LGM) + row) << lgC) + c)];
        };
        if (sizeof(C) == 8 && d.vecOut) {
#pragma unroll
            for (int j = 0; j < E / 2; ++j) {
                const int e = 2 * ti + j * 2 * nt;
                int c, row, hb, c1, row1, hb1;
                tile_coords<LGM>(e, lgC, lgHb, d.rowFastOut, c, row, hb);
                tile_coords<LGM>(e + 1, lgC, lgHb, d.rowFastOut, c1, row1, hb1);
                const C v0 = value(c, row, hb);
                const C v1 = value(c1, row1, hb1);
                const uint64_t g = outBase + ((uint64_t)hb << d.lgOutH2) + ((uint64_t)row << d.lgOutR) + c;
                *reinterpret_cast<float4*>(out + g) = make_float4((float)v0.x, (float)v0.y, (float)v1.x, (float)v1.y);
            }
        } else {
#pragma unroll
            for (int j = 0; j < E; ++j) {
                const int e = ti + j * nt;
                int c, row, hb;
                tile_coords<LGM>(e, lgC, lgHb, d.rowFastOut, c, row, hb);
                out[outBase + ((uint64_t)hb << d.lgOutH2) + ((uint64_t)row << d.lgOutR) + c] = value(c, row, hb);
            }
        }
    };
    auto store = [&](C* x, uint64_t t, int ti) {
        uint64_t lo0, inBase, outBase;
        tile_base(t, lo0, inBase, outBase);
        out_finish<E>(x, d, tile_conj(d, d.conjOut, inBase), scale, scaleLo);
        if (d.directOut) {
            last_store<RL, E, LGM, LGC>(out, x, d, outBase, scale, scaleLo, ti, nt);
            return;
        }
        stage_out(x, ti);
        store_lds(t, ti);
    };

    // one tile per workgroup
    const uint64_t t = blockIdx.x;
    uint64_t lo0, inBase, outBase;
    tile_base(t, lo0, inBase, outBase);
    C x[E];
    stage0_load<R0, E, LGM, LGC>(in, x, d, inBase, tid, nt);
    if (d.conjLoad) {
#pragma unroll
        for (int i = 0; i < E; ++i) x[i].y = -x[i].y;
    }
    prephase(x, t, tid);
    // an opaque copy of the thread id for the stages and the store: their
    // index math would otherwise be computed early and held across the phases
    // (8-element tiles; the 16-element one-row tile has no register left for it)
    int t2 = tid;
    if constexpr (E == 8) asm volatile("" : "+v"(t2));
    stages(x, t2);
    store(x, t, t2);
}

// Two half transforms of one register field in one in-place pass (FtDefer):
// the pending half of the previous transform (the four-step twiddle on load,
// a length-M transform over the tile's rows), the pending phases, then the
// first half of the next transform (a transform over the same rows), stored
// back in place.  Each half of an inverse is conj . forward half . conj (so a
// half-done inverse is a linear map of the state and commutes with work on
// other bits): conjMid conjugates before and after the pending half, dD.conjIn
// and d.conjOut before and after the next one.
// The phases are evaluated at the natural index of the completed transform:
// dD is the tile geometry seen in that index (row and row-block shifts), and
// swapLo > 0 exchanges the digits of swapLo and swapHi bits at swapSh of the tile
// base (the in-place L half leaves the register's digits exchanged).  Between the
// halves the elements stay in their threads, reordered in registers.
template <typename R, int LGM, int LGC, int E, bool STG>
__global__ void __launch_bounds__((tile_threads_max<R, LGM, LGC>()))
__attribute__((amdgpu_waves_per_eu((STG && sizeof(R) == 4) ? 8 : 1)))
k_fft_fused(typename CT<R>::type* data, FftPass d, FftPass dD, FastDiag pre, int conjMid, int swapSh, int swapLo,
            int swapHi,
            const typename CT<R>::type* __restrict__ tw, const typename CT<R>::type* __restrict__ tw4) {
    using C = typename CT<R>::type;
    constexpr int NST = Plan<LGM>::NST;
    constexpr int R0 = 1 << Plan<LGM>::lgr(0);
    constexpr int RL = 1 << Plan<LGM>::lgr(NST - 1);
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ PreLds P;
    C* lds = reinterpret_cast<C*>(smem_raw);
    const int tid = threadIdx.x, nt = blockDim.x;

    if (dD.usePre) {
        if (nt >= CVDV_FAST_TABS + CVDV_FAST_GEN) {
#pragma unroll
            for (int i = 0; i < CVDV_FAST_TABS; ++i)
                if (tid == i && i < pre.ntab) P.tab[i] = pre.tab[i];
#pragma unroll
            for (int i = 0; i < CVDV_FAST_GEN; ++i)
                if (tid == CVDV_FAST_TABS + i && i < pre.ngen) P.gen[i] = pre.gen[i];
        } else if (tid == 0) {
#pragma unroll
            for (int i = 0; i < CVDV_FAST_TABS; ++i)
                if (i < pre.ntab) P.tab[i] = pre.tab[i];
#pragma unroll
            for (int i = 0; i < CVDV_FAST_GEN; ++i)
                if (i < pre.ngen) P.gen[i] = pre.gen[i];
        }
        __syncthreads();
    }
    const R scale = (R)d.outScale;
    const R scaleLo = (R)(d.outScale - (double)scale);

    const uint64_t t = blockIdx.x;
    const uint64_t loBlk = t & ((1ull << d.lgNLoBlk) - 1);
    const uint64_t rr = t >> d.lgNLoBlk;
    const uint64_t h2Blk = rr & ((1ull << d.lgNH2Blk) - 1);
    const uint64_t h1 = rr >> d.lgNH2Blk;
    const uint64_t base = (h1 << d.lgInH1) + ((h2Blk << d.lgHb) << d.lgInH2) + (loBlk << LGC);
    uint64_t natBase = base;
    if (swapLo > 0) {
        const uint64_t ml = (1ull << swapLo) - 1ull, mh = (1ull << swapHi) - 1ull;
        const uint64_t lo = (base >> swapSh) & ml, hi = (base >> (swapSh + swapLo)) & mh;
        natBase = (base & ~(((mh << swapLo) | ml) << swapSh)) | (((lo << swapHi) | hi) << swapSh);
    }

    C x[E];
    stage0_load<R0, E, LGM, LGC>(data, x, d, base, tid, nt);
    if (conjMid) {  // an inverse's half is conj . forward half . conj
#pragma unroll
        for (int i = 0; i < E; ++i) x[i].y = -x[i].y;
    }
    // pending half: the four-step twiddle (d carries no phases and no input conjugation)
    stage0_pre<R0, E, LGM, LGC, true, TM_NONE>(x, d, base, P, pre, tw4, tid, nt, lds);
    stage_compute<R0, E, LGM, LGC, 0>(x, tw, tid, nt);
    run_stages<LGM, LGC, 1, E>(x, lds, tw, tid, nt);
    if (conjMid) {
#pragma unroll
        for (int i = 0; i < E; ++i) x[i].y = -x[i].y;
    }
    to_rows<LGM, E>(x);  // the last stage's order -> stage 0's
    // phases at the natural index, then the next transform's first half.  An
    // opaque copy of the thread id: index math derived from it (the store
    // addresses above all) would otherwise be computed early and held across
    // the phases in registers that the workgroup size leaves no room for.
    int t2 = tid;
    asm volatile("" : "+v"(t2));
    stage0_pre<R0, E, LGM, LGC, false, STG ? TM_STAGED : TM_ANY>(x, dD, natBase, P, pre, tw4, t2, nt, lds);
    stage_compute<R0, E, LGM, LGC, 0>(x, tw, t2, nt);
    run_stages<LGM, LGC, 1, E>(x, lds, tw, t2, nt);
    out_finish<E>(x, d, d.conjOut, scale, scaleLo);
    last_store<RL, E, LGM, LGC>(data, x, d, base, scale, scaleLo, t2, nt);
}

// Direct DFT for very small states (fewer than 8 elements per tile).
template <typename R, bool INV>
__global__ void k_dft_naive(const typename CT<R>::type* in, typename CT<R>::type* out, uint64_t total,
                            int sh, int nb, FastDiag pre, int usePre, double scale,
                            const double2* __restrict__ twN) {
    using C = typename CT<R>::type;
    const uint64_t M = 1ull << nb, fmask = (M - 1) << sh;
    for (uint64_t g = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; g < total;
         g += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t k = (g >> sh) & (M - 1);
        const uint64_t base = g & ~fmask;
        double ax = 0, ay = 0;
        for (uint64_t j = 0; j < M; ++j) {
            const uint64_t gi = base | (j << sh);
            C v = in[gi];
            if (usePre) v = apply_fast(pre, gi, v);
            const double2 p = mul_w<INV>(make_double2((double)v.x, (double)v.y), twN[(j * k) & (M - 1)]);
            ax += p.x;
            ay += p.y;
        }
        out[g] = cmk<C>(ax * scale, ay * scale);  // accumulated in FP64, rounded once
    }
}

int device_cus() {
    static std::map<int, int> cached;
    int dev = 0;
    HIPCHK(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(g_devCacheMu);
    auto it = cached.find(dev);
    if (it != cached.end()) return it->second;
    int v = 0;
    HIPCHK(hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev));
    cached[dev] = v;
    return v;
}

// ---------------------------------------------------------------- planning
struct PassGeom {
    int M;
    uint64_t nLo, nH2, nH1;
    uint64_t inH1, inH2, inR, outH1, outH2, outR;
};

static int ilog2(uint64_t v) { return 63 - __builtin_clzll(v); }

// Index bits that vary within one tile of a pass: columns, rows, row blocks.
static uint64_t tile_bits(const FftPass& d) {
    auto field = [](int s, int n) { return n > 0 ? (((1ull << n) - 1ull) << s) : 0ull; };
    return field(0, d.lgC) | field(d.lgInR, d.lgM) | field(d.lgInH2, d.lgHb);
}
static size_t lds_bytes(uint64_t tile, size_t esz) { return (tile + tile / 32) * esz; }

// Tile limits: a strided tile stays within 64 KiB of LDS so several workgroups
// share a CU; a whole contiguous register may take one large workgroup.  cfg
// (cvdvFftAutotune) may narrow the rows and change how far a tile grows over
// row blocks.
static bool fit_pass(const PassGeom& g, int prec, FftPass& d, bool allowBig, const FftCfg& cfg) {
    const size_t esz = prec == CVDV_C128 ? 16 : 8;
    // 256 contiguous bytes per row: the measured HBM rate of strided tiles rises
    // from ~4.0 TB/s with 128-byte rows to ~5.1 TB/s with 256-byte rows
    const uint64_t Wmax = prec == CVDV_C128 ? 16 : 32;
    const uint64_t W = cfg.rowElems > 0 && (uint64_t)cfg.rowElems < Wmax ? (uint64_t)cfg.rowElems : Wmax;
    const uint64_t cap = cfg.tileCap > 0 ? (uint64_t)cfg.tileCap : 2048;
    uint64_t C = g.nLo < W ? g.nLo : W;
    const size_t small = 64 * 1024;
    // the passes of a two-step split narrow their rows before giving up (a tall
    // pass of a contiguous register above one tile has M up to 2^12 rows)
    if (!allowBig)
        while (C > 1 && lds_bytes(C * (uint64_t)g.M, esz) > small) C /= 2;
    const uint64_t tileCM = C * (uint64_t)g.M;
    const bool big = allowBig && C == 1 && lds_bytes(tileCM, esz) <= device_max_lds() && tileCM <= 16384;
    if (lds_bytes(tileCM, esz) > small && !big) return false;
    uint64_t Hb = 1;
    while (Hb * 2 <= g.nH2 && tileCM * Hb * 2 <= cap && lds_bytes(tileCM * Hb * 2, esz) <= small) Hb *= 2;
    if (tileCM * Hb < 8) return false;
    const uint64_t tile = tileCM * Hb;
    d.lgM = ilog2(g.M);
    d.lgC = ilog2(C);
    d.lgHb = ilog2(Hb);
    d.lgNLoBlk = ilog2(g.nLo / C);
    d.lgNH2Blk = ilog2(g.nH2 / Hb);
    auto lg0 = [](uint64_t v) { return v ? ilog2(v) : 0; };  // stride 0: that index is always 0
    d.lgInH1 = lg0(g.inH1); d.lgInH2 = lg0(g.inH2); d.lgInR = lg0(g.inR);
    d.lgOutH1 = lg0(g.outH1); d.lgOutH2 = lg0(g.outH2); d.lgOutR = lg0(g.outR);
    d.rowFastOut = g.outR <= g.outH2 ? 1 : 0;
    // 16-byte pairs along the fastest dimension when it is contiguous in memory
    auto vec_ok = [&](int rowFast, uint64_t sR, uint64_t sH) {
        if (esz != 8 || tile < 2) return 0;
        if (C >= 2) return 1;
        if (rowFast) return (sR == 1 && g.M >= 2) ? 1 : 0;
        return (sH == 1 && Hb >= 2) ? 1 : 0;
    };
    d.vecOut = vec_ok(d.rowFastOut, g.outR, g.outH2);
    // last stage writes rows q + m*M/R of column c: coalesced when a full
    // column group is one full-width run or when rows follow the columns directly
    d.directOut = (C == W || g.outR == C) ? 1 : 0;
    return true;
}

// Kernel instances exist for the tile shapes fit_pass can produce: C = 2^LGC
// columns (up to 256 bytes per row) with C*M within 64 KiB of LDS, or one whole
// contiguous row (C = 1) of up to 2^14 complex64 / 2^13 complex128 points.
template <typename R, int LGM, int LGC>
constexpr bool tile_instance() {
    constexpr bool c64 = sizeof(R) == 4;
    if (LGC > (c64 ? 5 : 4)) return false;
    if (LGC == 0 && LGM <= (c64 ? 14 : 13)) return true;
    return LGM + LGC <= (c64 ? 13 : 12);
}

// Every table of the program is read by row in a one-row tile over the field
// [fs, fs + fn): its field holds the whole row field or none of it, and its
// control bit lies outside (the persistent instances compile only that path).
static bool table_by_row(const FastDiag& pre, int fs, int fn) {
    for (int i = 0; i < pre.ntab; ++i) {
        const DiagTab& T = pre.tab[i];
        const bool in = T.sh <= fs && fs + fn <= T.sh + T.nb;
        const bool out = T.sh >= fs + fn || fs >= T.sh + T.nb;
        if (!in && !out) return false;
        if (T.ctrl >= fs && T.ctrl < fs + fn) return false;
        for (int j = 0; j < T.nsel; ++j)
            if (tab_sel(T, j) >= fs && tab_sel(T, j) < fs + fn) return false;
    }
    return true;
}

static bool gen_affine_in_rows(const FastDiag& pre, int rowLo, int rowN);

// What the row kernel takes: whole contiguous rows one after the other; tables read by row
// and generic terms affine in the row coordinate.
static bool row_shape(const FftPass& d) {
    return d.lgHb == 0 && d.lgInR == 0 && d.lgOutR == 0 && d.lgNLoBlk == 0 && d.lgInH2 == d.lgM &&
           d.lgOutH2 == d.lgM && d.nTiles == 1ull << d.lgNH2Blk;
}
static bool row_program(const FastDiag& pre, int lgm) {
    return table_by_row(pre, 0, lgm) && (pre.ngen == 0 || gen_affine_in_rows(pre, 0, lgm));
}

template <typename R, int LGM, int LGC>
static void launch_geom(CVDVContext* ctx, const typename CT<R>::type* in, typename CT<R>::type* out,
                        const FftPass& d, const FastDiag& pre, const typename CT<R>::type* tw,
                        const typename CT<R>::type* tw4, uint64_t blocks, int tile, size_t lds) {
    if constexpr (tile_instance<R, LGM, LGC>()) {
        FftPass dg = d;
        dg.genSteps = d.usePre && pre.ngen > 0 && gen_affine_in_rows(pre, d.lgInR, LGM) ? 1 : 0;
        constexpr bool c128 = sizeof(R) == 8;
        if constexpr (LGC == 0 && row_instance(c128, LGM)) {
            // contiguous whole rows, in place: the row kernel (2^28 complex64: 0.80 ms without
            // phases, 0.98 by a tile of one workgroup a CU).  Rows elsewhere, and programs with a
            // control or a one-bit term inside the row, stay with the tiles.
            if (in == out && row_shape(d) && !d.tw4 && !d.conjLoad && d.conjIn == d.conjOut &&
                (!d.usePre || row_program(pre, LGM))) {
                RowArgs a{};
                a.m = 1;
                a.s[0].pre = d.usePre ? pre : FastDiag{};
                a.s[0].inv = d.conjIn;
                a.s[0].ctl = d.conjCtl;
                a.useScale = d.useScale;
                a.scale = d.outScale;
                a.rows = d.nTiles;
                fft_row_launch(ctx->stream, out, c128, LGM, a, row_table(ctx, LGM, c128 ? CVDV_C128 : CVDV_MIXED));
                return;
            }
        }
        auto go = [&](auto kfn, int E) {
            if (tile / E > tile_threads_max<R, LGM, LGC>())
                throw CvdvError{CVDV_ERR_UNSUPPORTED, "FFT tile larger than its kernel's workgroup bound"};
            if (lds > 64 * 1024)
                HIPCHK(hipFuncSetAttribute((const void*)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
            hipLaunchKernelGGL(kfn, dim3((unsigned)blocks), dim3(tile / E), lds, ctx->stream, in, out, dg, pre, tw, tw4);
        };
        if constexpr (one_row_layouts<R, LGM, LGC>()) {
            if (tile != (1 << LGM))
                throw CvdvError{CVDV_ERR_UNSUPPORTED, "one-row FFT tile of more than one row"};
            lds = (size_t)(tile + tile / 8) * sizeof(typename CT<R>::type);
        }
        if (lds > device_max_lds())
            throw CvdvError{CVDV_ERR_UNSUPPORTED, "FFT tile needs more LDS than the device has"};
        if constexpr (LGM == 14 && LGC == 0 && sizeof(R) == 4) {
            if (tile / 8 > 1024) {
                go(k_fft_tile<R, LGM, LGC, 16>, 16);
                return;
            }
        }
        go(k_fft_tile<R, LGM, LGC, 8>, 8);
    } else {
        throw CvdvError{CVDV_ERR_UNSUPPORTED, "FFT tile shape without a kernel instance"};
    }
}

template <typename R, int LGM>
static void launch_lgm(CVDVContext* ctx, const typename CT<R>::type* in, typename CT<R>::type* out,
                       const FftPass& d, const FastDiag& pre, const typename CT<R>::type* tw,
                       const typename CT<R>::type* tw4, uint64_t blocks, int tile, size_t lds) {
    switch (d.lgC) {
        case 0: launch_geom<R, LGM, 0>(ctx, in, out, d, pre, tw, tw4, blocks, tile, lds); break;
        case 1: launch_geom<R, LGM, 1>(ctx, in, out, d, pre, tw, tw4, blocks, tile, lds); break;
        case 2: launch_geom<R, LGM, 2>(ctx, in, out, d, pre, tw, tw4, blocks, tile, lds); break;
        case 3: launch_geom<R, LGM, 3>(ctx, in, out, d, pre, tw, tw4, blocks, tile, lds); break;
        case 4: launch_geom<R, LGM, 4>(ctx, in, out, d, pre, tw, tw4, blocks, tile, lds); break;
        case 5: launch_geom<R, LGM, 5>(ctx, in, out, d, pre, tw, tw4, blocks, tile, lds); break;
        default: throw CvdvError{CVDV_ERR_UNSUPPORTED, "FFT tile column count out of range"};
    }
}

template <typename R>
static void launch_pass(CVDVContext* ctx, const typename CT<R>::type* in, typename CT<R>::type* out,
                        const FftPass& d, const FastDiag& pre, int prec, uint64_t nH1) {
    using C = typename CT<R>::type;
    const C* tw = (const C*)stage_table(ctx, d.lgM, prec);
    const C* tw4 = d.tw4 ? (const C*)full_table(ctx, d.tw4LogN, prec) : nullptr;
    const int tile = 1 << (d.lgM + d.lgC + d.lgHb);
    if (tile / 16 > 1024 || (tile / 8 > 1024 && d.lgM != 14))
        throw CvdvError{CVDV_ERR_UNSUPPORTED, "FFT tile larger than one workgroup"};
    const uint64_t blocks = nH1 << (d.lgNH2Blk + d.lgNLoBlk);
    FftPass dd = d;
    dd.nTiles = blocks;
    const size_t lds = lds_bytes(tile, sizeof(C));
    const int pid = prof_begin(ctx, (d.lgC == 0 && d.lgHb == 0 && d.lgM >= 12) ? KK_FFT_ROW : KK_FFT);
    switch (d.lgM) {
#define CVDV_LGM_CASE(L) \
    case L: launch_lgm<R, L>(ctx, in, out, dd, pre, tw, tw4, blocks, tile, lds); break;
        CVDV_LGM_CASE(1) CVDV_LGM_CASE(2) CVDV_LGM_CASE(3) CVDV_LGM_CASE(4) CVDV_LGM_CASE(5)
        CVDV_LGM_CASE(6) CVDV_LGM_CASE(7) CVDV_LGM_CASE(8) CVDV_LGM_CASE(9) CVDV_LGM_CASE(10)
        CVDV_LGM_CASE(11) CVDV_LGM_CASE(12) CVDV_LGM_CASE(13) CVDV_LGM_CASE(14)
#undef CVDV_LGM_CASE
        default: throw CvdvError{CVDV_ERR_UNSUPPORTED, "FFT tile length out of range"};
    }
    HIPCHK(hipGetLastError());
    prof_end(ctx, pid);
}

// The four-step split of field [sh, sh+nb) (j = j1 + N1 j2, N1 = 2^(nb/2)):
//   d1: transform over j2 (stride N1 S), columns (j1, lo), in place;
//   d2: twiddle W_N^{j1 k2} on load, transform over j1 (stride S), row blocks
//       k2, written transposed (k2 + N2 k1) out of place;
// and the in-place halves a pending transform completes with:
//   dL:  d2 stored in place (momentum left with its digits exchanged: the low digit,
//        n2 bits, above the high one, n1 bits);
//   d1c: d1 with the twiddle W_N^{j1 j2} (j1 now the tile's) on load.
struct FourStep {
    FftPass d1, d2, dL, d1c;
    uint64_t H;
    int n1, n2;
    bool hasL;
};

static bool four_step_geom(int prec, uint64_t total, int sh, int nb, FourStep& f, const FftCfg& cfg) {
    const uint64_t N = 1ull << nb, S = 1ull << sh;
    const uint64_t H = total / (N * S);
    if (H == 0 || (H & (H - 1)) != 0 || H * N * S != total) return false;
    const int n1 = nb / 2, n2 = nb - n1;
    const uint64_t N1 = 1ull << n1, N2 = 1ull << n2;
    f = FourStep{};
    f.H = H;
    f.n1 = n1;
    f.n2 = n2;
    auto uni = [](const FftPass& d, int s, int n) {
        const uint64_t m = n > 0 ? (((1ull << n) - 1ull) << s) : 0ull;
        return (tile_bits(d) & m) ? 0 : 1;
    };
    PassGeom p1{(int)N2, N1 * S, 1, H, N * S, 0, N1 * S, N * S, 0, N1 * S};
    PassGeom p2{(int)N1, S, N2, H, N * S, N1 * S, S, N * S, S, N2 * S};
    if (!fit_pass(p1, prec, f.d1, false, cfg) || !fit_pass(p2, prec, f.d2, false, cfg)) return false;
    f.d1.tw4 = 0; f.d1.tw4Shift = 0; f.d1.tw4HiBits = 0; f.d1.tw4LogN = 0; f.d1.tw4Uni = 1;
    f.d2.tw4 = 1; f.d2.tw4Shift = sh + n1; f.d2.tw4HiBits = n2; f.d2.tw4LogN = nb;
    f.d2.tw4Uni = uni(f.d2, sh + n1, n2);
    f.d1c = f.d1;
    f.d1c.tw4 = 1; f.d1c.tw4Shift = sh; f.d1c.tw4HiBits = n1; f.d1c.tw4LogN = nb;
    f.d1c.tw4Uni = uni(f.d1c, sh, n1);
    PassGeom pL{(int)N1, S, N2, H, N * S, N1 * S, S, N * S, N1 * S, S};
    f.hasL = fit_pass(pL, prec, f.dL, false, cfg);
    f.dL.tw4 = 1; f.dL.tw4Shift = sh + n1; f.dL.tw4HiBits = n2; f.dL.tw4LogN = nb;
    f.dL.tw4Uni = uni(f.dL, sh + n1, n2);
    return true;
}

// Tile choices for field [sh, sh+nb) of a buffer of `total` elements: the
// context's tuned ones for its own state, the defaults for any other buffer.
static FftCfg field_cfg(const CVDVContext* ctx, uint64_t total, int sh, int nb) {
    if (total != ctx->totalSize) return FftCfg{};
    const auto it = ctx->fftCfg.find(fft_cfg_key(sh, nb));
    return it == ctx->fftCfg.end() ? FftCfg{} : it->second;
}

// Runs the FFT over field [sh, sh+nb) of a buffer of `total` elements, the other way
// where the index bit `ctrl` (>= 0) is set (one-pass plans whose tiles hold one value of it).
// Returns true when the result landed in the buffer returned by tmpFn.
template <typename R, typename TmpFn>
static bool fft_run(CVDVContext* ctx, typename CT<R>::type* data, TmpFn tmpFn, uint64_t total,
                    int sh, int nb, bool inverse, const DiagProg& preProg, double outScale, int prec,
                    int ctrl = -1) {
    using C = typename CT<R>::type;
    const uint64_t N = 1ull << nb, S = 1ull << sh;
    const uint64_t H = total / (N * S);
    if (H == 0 || (H & (H - 1)) != 0 || H * N * S != total)
        throw CvdvError{CVDV_ERR_ARG, "FFT over a buffer whose size is not a power-of-two multiple of the field"};
    bool act = false, folded = false;
    const int inv = inverse ? 1 : 0;
    const FftCfg cfg = field_cfg(ctx, total, sh, nb);
    // The pending phases are compiled once the tiling of the pass that applies
    // them is known: their tables take no choice bit that varies within a tile.
    auto compile_pre = [&](uint64_t tileBits, const DiagProg& prog) {
        const FastDiag f = compile_diag(ctx, prog, act, outScale, &folded, tileBits);
        return f;
    };

    // single pass: rows j (stride S), lo in [0,S), hi blocks in h2 (stride N*S)
    PassGeom g1{(int)N, S, H, 1, 0, N * S, S, 0, N * S, S};
    FftPass d{};
    if (fit_pass(g1, prec, d, true, cfg)) {
        // A persistent complex64 one-row pass folds the linear terms over its row
        // field per butterfly (one sin/cos each): a table would cost a global
        // load per element, queued behind the previous row's stores.
        const bool foldRow = prec == CVDV_MIXED && d.lgC == 0 && d.lgHb == 0 && d.lgM >= 13;
        const FastDiag pre =
            compile_pre(tile_bits(d), foldRow ? diag_fold_linear(preProg, d.lgInR, d.lgM) : preProg);
        const int usePre = act ? 1 : 0;
        d.tw4 = 0; d.tw4Shift = 0; d.tw4HiBits = 0; d.tw4LogN = 0;
        d.usePre = usePre;
        d.useScale = folded ? 0 : 1;
        d.conjIn = inv;
        d.conjOut = inv;
        d.conjCtl = ctrl + 1;
        d.outScale = outScale;
        if (ctrl >= 0 && ((tile_bits(d) >> ctrl) & 1ull))
            throw CvdvError{CVDV_ERR_STATE, "transform direction by a bit that varies within a tile"};
        launch_pass<R>(ctx, data, data, d, pre, prec, 1);
        return false;
    }
    if (ctrl >= 0) throw CvdvError{CVDV_ERR_STATE, "transform direction by a bit outside the one-pass plan"};
    if (total < 4096 || N <= 64) {
        // tiny state: direct DFT, out of place, FP64 accumulation rounded once
        // (per-element table reads: any choice bits)
        const FastDiag pre = compile_pre(0, preProg);
        const int usePre = act ? 1 : 0;
        const double sc = folded ? 1.0 : outScale;
        const double2* twN = (const double2*)full_table(ctx, nb);
        C* tmp = tmpFn();
        uint64_t blocks = (total + 255) / 256;
        const int pid = prof_begin(ctx, KK_FFT);
        if (inverse)
            hipLaunchKernelGGL((k_dft_naive<R, true>), dim3((unsigned)blocks), dim3(256), 0, ctx->stream,
                               data, tmp, total, sh, nb, pre, usePre, sc, twN);
        else
            hipLaunchKernelGGL((k_dft_naive<R, false>), dim3((unsigned)blocks), dim3(256), 0, ctx->stream,
                               data, tmp, total, sh, nb, pre, usePre, sc, twN);
        HIPCHK(hipGetLastError());
        prof_end(ctx, pid);
        return true;
    }
    FourStep f;
    if (!four_step_geom(prec, total, sh, nb, f, cfg))
        throw CvdvError{CVDV_ERR_UNSUPPORTED, "register too large for the two-pass FFT"};
    FftPass d1 = f.d1, d2 = f.d2;
    const FastDiag pre = compile_pre(tile_bits(d1), preProg);
    const int usePre = act ? 1 : 0;
    // inverse: conj(P2(T P1(conj x))) - pass 1 conjugates its input, pass 2 its
    // output; the twiddle T = W_N^{j1 k2} is applied by pass 2 on load, where the
    // pass has memory time to spare (pass 1 also applies the pending phases)
    d1.usePre = usePre;
    d1.useScale = 0;
    d1.conjIn = inv;
    d1.conjOut = 0;
    d1.outScale = 1.0;
    d2.usePre = 0;
    d2.useScale = folded ? 0 : 1;
    d2.conjIn = 0;
    d2.conjOut = inv;
    d2.outScale = outScale;
    C* tmp = tmpFn();
    launch_pass<R>(ctx, data, data, d1, pre, prec, f.H);
    launch_pass<R>(ctx, data, tmp, d2, FastDiag{}, prec, f.H);
    return true;
}

// ---------------------------------------------------------------- half transforms kept pending
// Fused instances exist for digits of 2^FUSE_LGM_MIN .. 2^FUSE_LGM_MAX points
// (registers of 2^8 .. 2^16 points).
#define FUSE_LGM_MIN 4
#define FUSE_LGM_MAX 8

// Every table of the program is read by row in tiles of geometry d (the test
// stage0_pre makes per table, made here on the host): its field misses the
// tile's column and row-block bits and holds all or none of the row bits, and
// no control or choice bit of it varies inside the tile.
static bool tile_tables_by_row(const FastDiag& pre, const FftPass& d) {
    const int rowLo = d.lgInR, rowHi = d.lgInR + d.lgM;
    auto hits = [](int sh, int nb, int lo, int n) { return n > 0 && sh < lo + n && lo < sh + nb; };
    auto varies = [&](int b) {
        return b >= 0 && (b < d.lgC || (b >= rowLo && b < rowHi) ||
                          (d.lgHb > 0 && b >= d.lgInH2 && b < d.lgInH2 + d.lgHb));
    };
    for (int i = 0; i < pre.ntab; ++i) {
        const DiagTab& T = pre.tab[i];
        const bool rowIn = T.sh <= rowLo && rowHi <= T.sh + T.nb;
        bool ctrlVar = varies(T.ctrl);
        for (int j = 0; j < T.nsel; ++j) ctrlVar = ctrlVar || varies(tab_sel(T, j));
        const bool fast = !hits(T.sh, T.nb, 0, d.lgC) && !hits(T.sh, T.nb, d.lgInH2, d.lgHb) &&
                          (rowIn || !hits(T.sh, T.nb, rowLo, d.lgM)) && !ctrlVar;
        if (!fast) return false;
    }
    return true;
}

// Every generic term is affine in the row index of a tile whose rows are the
// bits [rowLo, rowLo + rowN) (column and row-block bits fixed): each field holds
// all of the row bits or none (a bilinear term at most one field with them, a
// polynomial with them only its linear coefficient), and no control or Z bit
// is a row bit.
static bool gen_affine_in_rows(const FastDiag& pre, int rowLo, int rowN) {
    auto rel = [&](int sh, int nb) {  // 0: misses the rows, 1: holds them all, 2: part of them
        if (!(sh < rowLo + rowN && rowLo < sh + nb)) return 0;
        return (sh <= rowLo && rowLo + rowN <= sh + nb) ? 1 : 2;
    };
    for (int i = 0; i < pre.ngen; ++i) {
        const DiagTerm& T = pre.gen[i];
        if (T.ctrl >= rowLo && T.ctrl < rowLo + rowN) return false;
        if (T.kind == DT_POLY || T.kind == DT_LINF) {
            const int r = rel(T.sh1, T.nb1);
            if (r == 2 || (r == 1 && (T.c2 != 0.0 || T.c3 != 0.0))) return false;
        } else if (T.kind == DT_BILIN) {
            const int r1 = rel(T.sh1, T.nb1), r2 = rel(T.sh2, T.nb2);
            if (r1 == 2 || r2 == 2 || (r1 == 1 && r2 == 1)) return false;
        } else if (T.sh1 >= rowLo && T.sh1 < rowLo + rowN) {
            return false;
        }
    }
    return true;
}

template <typename R, int LGM, int LGC>
static void launch_fused_geom(CVDVContext* ctx, typename CT<R>::type* data, const FftPass& d, const FftPass& dD,
                              const FastDiag& pre, int conjMid, int swapSh, int swapLo, int swapHi,
                              const typename CT<R>::type* tw, const typename CT<R>::type* tw4, uint64_t blocks,
                              int tile, size_t lds) {
    if constexpr (tile_instance<R, LGM, LGC>()) {
        if (tile / 8 > tile_threads_max<R, LGM, LGC>())
            throw CvdvError{CVDV_ERR_UNSUPPORTED, "fused FFT tile larger than its kernel's workgroup bound"};
        // tiles of several columns whose tables are all read by row (and, in
        // complex64, whose generic terms are affine in the row index) take the
        // instance that stages them through LDS: fewer registers, more
        // workgroups per CU
        FftPass dDg = dD;
        dDg.genSteps = dD.usePre && pre.ngen > 0 && gen_affine_in_rows(pre, dD.lgInR, LGM) ? 1 : 0;
        // (complex64 digits of 2^7 points in whole runs: fft_fused.hip)
        constexpr bool two = sizeof(R) == 4 && LGM == FUSE2_LGM && LGC == FUSE2_LGC;
        if constexpr (LGC > 0 && !two) {
            const bool gen = sizeof(R) == 8 || pre.ngen == 0 || dDg.genSteps;
            if (!dD.usePre || (tile_tables_by_row(pre, dD) && gen)) {
                hipLaunchKernelGGL((k_fft_fused<R, LGM, LGC, 8, true>), dim3((unsigned)blocks), dim3(tile / 8), lds,
                                   ctx->stream, data, d, dDg, pre, conjMid, swapSh, swapLo, swapHi, tw, tw4);
                return;
            }
        }
        hipLaunchKernelGGL((k_fft_fused<R, LGM, LGC, 8, false>), dim3((unsigned)blocks), dim3(tile / 8), lds,
                           ctx->stream, data, d, dDg, pre, conjMid, swapSh, swapLo, swapHi, tw, tw4);
    } else {
        throw CvdvError{CVDV_ERR_UNSUPPORTED, "fused FFT tile shape without a kernel instance"};
    }
}

template <typename R, int LGM>
static void launch_fused_lgm(CVDVContext* ctx, typename CT<R>::type* data, const FftPass& d, const FftPass& dD,
                             const FastDiag& pre, int conjMid, int swapSh, int swapLo, int swapHi,
                             const typename CT<R>::type* tw, const typename CT<R>::type* tw4, uint64_t blocks,
                             int tile, size_t lds) {
    switch (d.lgC) {
#define CVDV_FUSE_C(L) \
    case L: launch_fused_geom<R, LGM, L>(ctx, data, d, dD, pre, conjMid, swapSh, swapLo, swapHi, tw, tw4, blocks, tile, lds); break;
        CVDV_FUSE_C(0) CVDV_FUSE_C(1) CVDV_FUSE_C(2) CVDV_FUSE_C(3) CVDV_FUSE_C(4) CVDV_FUSE_C(5)
#undef CVDV_FUSE_C
        default: throw CvdvError{CVDV_ERR_UNSUPPORTED, "fused FFT tile column count out of range"};
    }
}

template <typename R>
static void launch_fused(CVDVContext* ctx, const FftPass& d, const FftPass& dD, const FastDiag& pre, int conjMid,
                         int swapSh, int swapLo, int swapHi, uint64_t nH1) {
    using C = typename CT<R>::type;
    const int prec = ctx->prec;
    const C* tw = (const C*)stage_table(ctx, d.lgM, prec);
    const C* tw4 = (const C*)full_table(ctx, d.tw4LogN, prec);
    const int tile = 1 << (d.lgM + d.lgC + d.lgHb);
    const uint64_t blocks = nH1 << (d.lgNH2Blk + d.lgNLoBlk);
    FftPass dd = d;
    dd.nTiles = blocks;
    const size_t lds = lds_bytes(tile, sizeof(C));
    C* data = (C*)ctx->state();
    const int pid = prof_begin(ctx, KK_FFT_FUSED);
    if constexpr (sizeof(R) == 4) {
        // two stages a digit where the instance's rules hold (fft_fused.hip)
        if (d.lgM == FUSE2_LGM) {
            FusedArgs a{dd, dD, conjMid, swapSh, swapLo, swapHi};
            a.dD.genSteps = dD.usePre && pre.ngen > 0 && gen_affine_in_rows(pre, dD.lgInR, d.lgM) ? 1 : 0;
            if ((!dD.usePre || (tile_tables_by_row(pre, dD) && (pre.ngen == 0 || a.dD.genSteps))) &&
                fft_fused2_launch(ctx->stream, data, a, pre, (const float4*)fuse2_table(ctx), tw4, (unsigned)blocks)) {
                HIPCHK(hipGetLastError());
                prof_end(ctx, pid);
                return;
            }
        }
    }
    switch (d.lgM) {
#define CVDV_FUSE_M(L) \
    case L: launch_fused_lgm<R, L>(ctx, data, dd, dD, pre, conjMid, swapSh, swapLo, swapHi, tw, tw4, blocks, tile, lds); break;
        CVDV_FUSE_M(4) CVDV_FUSE_M(5) CVDV_FUSE_M(6) CVDV_FUSE_M(7) CVDV_FUSE_M(8)
#undef CVDV_FUSE_M
        default: throw CvdvError{CVDV_ERR_UNSUPPORTED, "fused FFT digit length out of range"};
    }
    HIPCHK(hipGetLastError());
    prof_end(ctx, pid);
}

static uint64_t bit_field(int sh, int n) { return n > 0 ? (((1ull << n) - 1ull) << sh) : 0ull; }

// The four-step of this register can leave halves pending: fused instances for both
// digits, and tiles that store straight to global memory.  The digits may differ: the
// halves of one transform alternate between them, and a fused pass (L of one transform
// and H of the next, whose high digit is the momentum's, or the twiddle and H of one and
// H of the next) always runs over one digit.
static bool fusable(const CVDVContext* ctx, const FourStep& f, int nb, const FftCfg& cfg) {
    return ctx->fuseFt && cfg.fuse != 0 && !ctx->rec && f.n1 >= FUSE_LGM_MIN && f.n2 <= FUSE_LGM_MAX && f.hasL &&
           f.d1.directOut && f.dL.directOut && nb == f.n1 + f.n2;
}

// Complete the half-done transform D (its record already cleared).
template <typename R>
static void settle_impl(CVDVContext* ctx, const FtDefer D) {
    using C = typename CT<R>::type;
    FourStep f;
    if (!four_step_geom(ctx->prec, ctx->totalSize, D.sh, D.nb, f, field_cfg(ctx, ctx->totalSize, D.sh, D.nb)))
        throw CvdvError{CVDV_ERR_STATE, "half-done register transform without its four-step geometry"};
    C* data = (C*)ctx->state();
    if (D.high) {
        // twiddle W_N^{lo hi} and the transform over hi, in place: natural order
        FftPass d = f.d1c;
        d.usePre = 0;
        d.conjLoad = D.inv;
        d.conjIn = 0;
        d.conjOut = D.inv;
        d.useScale = D.scale != 1.0 ? 1 : 0;
        d.outScale = D.scale;
        launch_pass<R>(ctx, data, data, d, FastDiag{}, ctx->prec, f.H);
    } else {
        // twiddle and the transform over lo, stored transposed into the other buffer
        FftPass d = f.d2;
        d.usePre = 0;
        d.conjLoad = D.inv;
        d.conjIn = 0;
        d.conjOut = D.inv;
        d.useScale = D.scale != 1.0 ? 1 : 0;
        d.outScale = D.scale;
        launch_pass<R>(ctx, data, (C*)ctx->other(), d, FastDiag{}, ctx->prec, f.H);
        ctx->cur = 1 - ctx->cur;
    }
}

static void settle_one(CVDVContext* ctx, FtDefer& rec) {
    chain_flush(ctx);
    const FtDefer D = rec;
    rec = FtDefer{};
    if (ctx->prec == CVDV_C128) settle_impl<double>(ctx, D);
    else settle_impl<float>(ctx, D);
}

void fft_settle(CVDVContext* ctx, bool mayAllocate) {
    chain_flush(ctx);  // (may leave a half pending)
    if (!ctx->defer.any()) return;
    if (!mayAllocate && !ctx->buf[1 - ctx->cur])
        for (const FtDefer& d : ctx->defer.f)
            if (d.on && !d.high)
                throw CvdvError{CVDV_ERR_STATE,
                                "a register transform is half done and completing it needs the second state "
                                "buffer: call cvdvFlush first"};
    for (FtDefer& d : ctx->defer.f)
        if (d.on) settle_one(ctx, d);
}

void fft_settle_bits(CVDVContext* ctx, uint64_t mask) {
    for (FtDefer& d : ctx->defer.f)
        if (d.on && (mask & bit_field(d.sh, d.nb))) settle_one(ctx, d);
}

// A transform of field [sh, sh+nb) that can keep a half pending.  Returns false
// when the ordinary path must run (the caller has settled nothing yet).
template <typename R>
static bool fft_deferred(CVDVContext* ctx, int sh, int nb, bool inverse, const DiagProg& preProg, double outScale) {
    // only where the ordinary path takes the four-step split (fft_run)
    const uint64_t N = 1ull << nb, S = 1ull << sh, total = ctx->totalSize;
    if (total < 4096 || N <= 64 || (total % (N * S)) != 0) return false;
    const FftCfg cfg = field_cfg(ctx, total, sh, nb);
    {
        PassGeom g1{(int)N, S, total / (N * S), 1, 0, N * S, S, 0, N * S, S};
        FftPass d{};
        if (fit_pass(g1, ctx->prec, d, true, cfg)) return false;
    }
    FourStep f;
    if (!four_step_geom(ctx->prec, total, sh, nb, f, cfg) || !fusable(ctx, f, nb, cfg)) return false;
    bool act = false, folded = false;
    if (FtDefer* rec = ctx->defer.find(sh)) {
        FtDefer& D = *rec;
        // fuse the pending half with this transform's first half
        const bool high = D.high != 0;
        FftPass d = high ? f.d1c : f.dL;
        FftPass dD = d;  // the tile in the natural index of the completed transform
        if (!high) {
            dD.lgInR = sh + f.n2;  // rows: the lo digit here is the momentum's hi digit
            dD.lgInH2 = sh;        // row blocks: the hi digit here is the momentum's lo digit
        }
        const uint64_t natBits = tile_bits(dD);
        const double scale = outScale * D.scale;
        if (diag_fits(preProg, natBits)) {
            const FastDiag pre = compile_diag(ctx, preProg, act, scale, &folded, natBits);
            d.usePre = 0;
            d.conjLoad = 0;  // the kernel's conjMid conjugates around the pending half
            d.conjIn = 0;
            d.conjOut = inverse ? 1 : 0;
            d.useScale = folded ? 0 : 1;
            d.outScale = scale;
            dD.tw4 = 0;
            dD.usePre = act ? 1 : 0;
            dD.conjIn = inverse ? 1 : 0;
            launch_fused<R>(ctx, d, dD, pre, D.inv, sh, high ? 0 : f.n1, high ? 0 : f.n2, f.H);
            D = FtDefer{1, sh, nb, high ? 0 : 1, inverse ? 1 : 0, 1.0};
            return true;
        }
        settle_one(ctx, D);
    }
    // first half from the natural order: pending phases on load, transform over hi
    FftPass d = f.d1;
    const FastDiag pre = compile_diag(ctx, preProg, act, outScale, &folded, tile_bits(d));
    d.usePre = act ? 1 : 0;
    d.conjIn = inverse ? 1 : 0;
    d.conjOut = inverse ? 1 : 0;  // a half-done inverse stays a linear map of the state
    d.useScale = folded ? 0 : 1;
    d.outScale = outScale;
    FtDefer* slot = ctx->defer.free_slot();
    if (!slot) throw CvdvError{CVDV_ERR_STATE, "no free record for a half-done register transform"};
    launch_pass<R>(ctx, (typename CT<R>::type*)ctx->state(), (typename CT<R>::type*)ctx->state(), d, pre, ctx->prec,
                   f.H);
    *slot = FtDefer{1, sh, nb, 0, inverse ? 1 : 0, 1.0};
    return true;
}

bool fft_defers(const CVDVContext* ctx, int sh, int nb) {
    const uint64_t N = 1ull << nb, S = 1ull << sh, total = ctx->totalSize;
    if (total < 4096 || N <= 64 || (total % (N * S)) != 0) return false;
    const FftCfg cfg = field_cfg(ctx, total, sh, nb);
    PassGeom g1{(int)N, S, total / (N * S), 1, 0, N * S, S, 0, N * S, S};
    FftPass d{};
    if (fit_pass(g1, ctx->prec, d, true, cfg)) return false;
    FourStep f;
    return four_step_geom(ctx->prec, total, sh, nb, f, cfg) && fusable(ctx, f, nb, cfg);
}

// States whose fields turn in chains alone (elsewhere a one-pass plan does).
static bool turns_in_chains(const CVDVContext* ctx, int sh, int nb) {
    return ctx->totalQbt <= FT_CHAIN_LG_SMALL && !row_field(ctx, sh, nb);
}

uint64_t fft_plan_signature(const CVDVContext* ctx, int sh, int nb, const FftCfg& cfg) {
    const uint64_t N = 1ull << nb, S = 1ull << sh, total = ctx->totalSize;
    if (total % (N * S) != 0) return 0;
    // transforms that run as chains take none of cfg's choices
    if (turns_in_chains(ctx, sh, nb) && chain_field(ctx, sh, nb)) return 500000;
    auto sig = [](const FftPass& d) { return (uint64_t)(d.lgC * 64 + d.lgHb * 4 + d.lgM / 8 + 1); };
    PassGeom g1{(int)N, S, total / (N * S), 1, 0, N * S, S, 0, N * S, S};
    FftPass d{};
    if (fit_pass(g1, ctx->prec, d, true, cfg)) return 1000000 + sig(d);
    if (total < 4096 || N <= 64) return 0;
    FourStep f;
    if (!four_step_geom(ctx->prec, total, sh, nb, f, cfg)) return 0;
    const uint64_t fz = fusable(ctx, f, nb, cfg) ? 1 : 0;
    return 2000000 + ((sig(f.d1) * 4096 + sig(f.d2)) * 4096 + (f.hasL ? sig(f.dL) : 0)) * 2 + fz;
}

// Every twiddle table an FFT of any register of the context can ask for.
void fft_prepare(CVDVContext* ctx) {
    for (int r = 0; r < ctx->numReg; ++r) {
        const int nb = ctx->nq[r];
        if (nb == 0 || nb > 28) continue;  // above 28 qubits the two-pass FFT refuses anyway
        for (int lg = 1; lg <= nb && lg <= 14; ++lg) (void)stage_table(ctx, lg, ctx->prec);
        for (int lg = 12; lg <= nb && lg <= 14; ++lg)
            if (row_instance(ctx->prec == CVDV_C128, lg)) (void)row_table(ctx, lg, ctx->prec);
        (void)full_table(ctx, nb, ctx->prec);                   // four-step twiddles
        if (ctx->prec == CVDV_MIXED) (void)fuse2_table(ctx);
        if (nb <= 12) (void)full_table(ctx, nb, CVDV_C128);     // direct DFT of tiny states
    }
}

// The fields whose gates run as chains of rows.  Small states of 2^12 and 2^13 points stay with
// fft_chain.hip (no table builds); 2^14 points do not fit its tile ([1,14], 12 gates: 380 us
// by single passes, 296 here).
bool row_field(const CVDVContext* ctx, int sh, int nb) {
    if (ctx->rec || sh != 0 || !row_instance(ctx->prec == CVDV_C128, nb)) return false;
    return nb > 13 || ctx->totalQbt > FT_CHAIN_LG_SMALL;
}

// The program as a row's pass compiles it (fft_run's rule).
static DiagProg row_prog(const CVDVContext* ctx, const DiagProg& p, int nb) {
    return ctx->prec == CVDV_MIXED ? diag_fold_linear(p, 0, nb) : p;
}

// Every table is read by row and every generic term is affine in it; no pass of its own for
// terms beyond a program's capacities (it would run ahead of the chain).
bool row_accepts(const CVDVContext* ctx, int nb, const DiagProg& p) {
    const uint64_t row = bit_field(0, nb);
    for (int i = 0; i < p.n; ++i) {
        const DiagTerm& t = p.t[i];
        if (t.c1 == 0.0 && t.c2 == 0.0 && t.c3 == 0.0) continue;
        if (t.ctrl >= 0 && t.ctrl < nb) return false;
        if (t.kind == DT_ZBIT ? t.sh1 < nb : (t.sh1 < nb && (t.sh1 != 0 || t.nb1 != nb))) return false;
        if (t.kind == DT_BILIN && t.sh2 < nb) return false;  // (its fields are in order of their shifts)
    }
    return diag_fits(row_prog(ctx, p, nb), row);
}

void fft_row_chain(CVDVContext* ctx, int nb, const FtChainStep* st, int m) {
    const uint64_t row = bit_field(0, nb);
    int maxNb = 0;
    for (int r = 0; r < ctx->numReg; ++r) maxNb = std::max(maxNb, ctx->nq[r]);
    // the programs' tables side by side; reserved first, since a grown arena starts empty.  Never
    // more than one program may ask for by itself (a capture reserves no more): steps whose
    // tables together exceed that run one by one
    uint64_t entries = 0;
    for (int i = 0; i < m; ++i) entries += diag_entries(row_prog(ctx, st[i].prog, nb), row);
    const size_t need = entries * ctx->elemBytes();
    if (need > diag_arena_bound(maxNb, ctx->elemBytes())) {
        for (int i = 0; i < m; ++i)
            fft_whole(ctx, 0, nb, st[i].inverse != 0, st[i].prog, st[i].scale, st[i].ctrl);
        return;
    }
    arena_reserve(ctx, need);
    RowArgs a{};
    a.m = m;
    a.scale = 1.0;
    a.rows = ctx->totalSize >> nb;
    uint32_t off = 0;
    for (int i = 0; i < m; ++i) {
        bool act = false, folded = false;
        const FastDiag pre =
            compile_diag(ctx, row_prog(ctx, st[i].prog, nb), act, st[i].scale, &folded, row, off, &off);
        if (act && !row_program(pre, nb)) throw CvdvError{CVDV_ERR_STATE, "row chain with a program not read by row"};
        if (act) a.s[i].pre = pre;
        a.s[i].pre.arena = ctx->arena;
        a.s[i].inv = st[i].inverse;
        a.s[i].ctl = st[i].ctrl + 1;
        if (!folded) a.scale *= st[i].scale;
    }
    a.useScale = a.scale != 1.0;
    const int pid = prof_begin(ctx, KK_FFT_ROW);
    fft_row_launch(ctx->stream, ctx->state(), ctx->prec == CVDV_C128, nb, a, row_table(ctx, nb, ctx->prec));
    HIPCHK(hipGetLastError());
    prof_end(ctx, pid);
}

int fft_turn_terms(const CVDVContext* ctx, int sh, int nb) {
    return turns_in_chains(ctx, sh, nb) ? FT_CHAIN_TERMS : CVDV_MAX_TERMS;
}

bool fft_turns(const CVDVContext* ctx, int sh, int nb, int ctrl) {
    if (ctx->rec || (ctrl >= sh && ctrl < sh + nb)) return false;
    if (turns_in_chains(ctx, sh, nb)) return chain_field(ctx, sh, nb);
    const uint64_t N = 1ull << nb, S = 1ull << sh, total = ctx->totalSize;
    const PassGeom g1{(int)N, S, total / (N * S), 1, 0, N * S, S, 0, N * S, S};
    FftPass d{};
    return fit_pass(g1, ctx->prec, d, true, field_cfg(ctx, total, sh, nb)) && !((tile_bits(d) >> ctrl) & 1ull);
}

void fft_register(CVDVContext* ctx, int pshift, int nbits, bool inverse, const DiagProg& pre,
                  double outScale, int ctrl) {
    if (chain_field(ctx, pshift, nbits)) {
        if (FtDefer* rec = ctx->defer.find(pshift)) settle_one(ctx, *rec);
        if (chain_accept(ctx, pshift, nbits, inverse, pre, outScale, ctrl)) return;
    }
    chain_flush(ctx);
    fft_whole(ctx, pshift, nbits, inverse, pre, outScale, ctrl);
}

void fft_whole(CVDVContext* ctx, int sh, int nb, bool inverse, const DiagProg& pre, double outScale, int ctrl) {
    // (halves have one direction: a control goes on to fft_run, which refuses plans without it)
    const bool done = ctrl < 0 && (ctx->prec == CVDV_C128 ? fft_deferred<double>(ctx, sh, nb, inverse, pre, outScale)
                                                          : fft_deferred<float>(ctx, sh, nb, inverse, pre, outScale));
    if (done) return;
    if (FtDefer* rec = ctx->defer.find(sh)) settle_one(ctx, *rec);
    bool swapped;
    if (ctx->prec == CVDV_C128)
        swapped = fft_run<double>(ctx, (double2*)ctx->state(), [ctx] { return (double2*)ctx->other(); },
                                  ctx->totalSize, sh, nb, inverse, pre, outScale, CVDV_C128, ctrl);
    else
        swapped = fft_run<float>(ctx, (float2*)ctx->state(), [ctx] { return (float2*)ctx->other(); },
                                 ctx->totalSize, sh, nb, inverse, pre, outScale, CVDV_MIXED, ctrl);
    if (swapped) ctx->cur = 1 - ctx->cur;
}

void fft_generic_c128(CVDVContext* ctx, double2* data, double2* tmp, uint64_t total, int shift,
                      int nbits, bool inverse, double outScale) {
    if (fft_run<double>(ctx, data, [tmp] { return tmp; }, total, shift, nbits, inverse, DiagProg{},
                        outScale, CVDV_C128))
        HIPCHK(hipMemcpyAsync(data, tmp, total * sizeof(double2), hipMemcpyDeviceToDevice, ctx->stream));
}
