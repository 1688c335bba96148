// fft_row.hip - transforms of contiguous rows of 2^13 and 2^14 complex64 or 2^12 complex128
// points, one workgroup a row, and a gate's transforms of the row one after the other in one
// pass.
//
// A row of 2^14 takes 128 KiB of LDS, a whole CU's: one workgroup, whose loads, stages
// and exchanges then follow each other with nothing beside them.  Here the real and the
// imaginary parts cross LDS one after the other through one buffer of half the size, so
// two workgroups (three of the shorter rows) share a CU and one computes while the other
// waits for memory or exchanges.  A thread holds 32 elements (16 complex128), which is what
// lets a transform be three stages (32 x 32 x 16, 32 x 32 x 8, 16 x 16 x 16) and two exchanges
// instead of five and four (four and three); it owns the same rows before the first stage
// and after the last, so the next transform of a chain starts where the last one ended.
//
// Between HBM and in-CU work.  [14,14] complex64 (4.3 GB a pass; a copy of this shape takes
// 0.74 ms), ms against the tile of 1024 threads that this replaces: one transform without
// phases 0.80 (0.90), with its table 0.86 (1.01); a displacement's two 1.18 (2 x 0.93); a
// conditional rotation's three 1.70 (3 x 1.00); a squeezing gate's four 2.01 (4 x 0.99).
// [14,13]: 0.44, 0.58, 0.84, 0.92.  [13,12] complex128 (1.07 GB, copy 0.20), against one chain
// launch of fft_chain.hip: 0.22 (0.24), 0.29 (0.38), 0.35 (0.50), 0.41 (0.61).  Two
// transforms of a row in one pass of the old tile cost exactly two passes.

#include <algorithm>

#include "cvdv_internal.h"
#include "fft_radix16.h"
#include "fft_row.h"

// 32 inputs in order; output m = m2 + 8 m1 is left at x[m1 + 4 m2] (dft32_slot).
__device__ __forceinline__ constexpr int dft32_slot(int m) { return (m >> 3) + 4 * (m & 7); }
#define SCHED() __builtin_amdgcn_sched_barrier(0)
template <int ST, typename C>
__device__ __forceinline__ void dft8_at(C* x) {
    C y[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) y[j] = x[j * ST];
    dft8<false>(y);
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j * ST] = y[j];
}
template <int K, int M2>
__device__ __forceinline__ void dft32_inner(float2* x) {
    x[K + 4 * M2] = mul_w32<K * M2, true>(x[K + 4 * M2]);
    if constexpr (M2 < 7) dft32_inner<K, M2 + 1>(x);
    else if constexpr (K < 3) dft32_inner<K + 1, 1>(x);
}
__device__ __forceinline__ void dft32(float2* x) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        dft8_at<4>(x + k);
        SCHED();
    }
    dft32_inner<1, 1>(x);
    SCHED();
#pragma unroll
    for (int m = 0; m < 8; ++m) dft4<false>(x[4 * m], x[4 * m + 1], x[4 * m + 2], x[4 * m + 3]);
    SCHED();
}

// A thread's E elements: the first two stages are one DFT of E points a thread.
template <typename R> constexpr int row_lge() { return sizeof(R) == 4 ? 5 : 4; }
__device__ __forceinline__ void dft_own(float2* x) { dft32(x); }
__device__ __forceinline__ void dft_own(double2* x) { dft16<1>(x); }
template <typename R> __device__ __forceinline__ constexpr int own_slot(int m) { return sizeof(R) == 4 ? dft32_slot(m) : m; }

// Butterfly K of the last stage sits at q + K NT: its twiddles are those of butterfly 0
// times W_E^{j K}.
template <int RL, int NB, int J, int K, typename C>
__device__ __forceinline__ void last_twiddle(C* x, C w) {
    x[K + NB * J] = mul_w32<(J * K * (sizeof(C) / 8)) & 31>(cmul(x[K + NB * J], w));
    if constexpr (K + 1 < NB) last_twiddle<RL, NB, J, K + 1>(x, w);
}
template <int RL, int NB, int J, typename C>
__device__ __forceinline__ void last_twiddles_from(C* x, const C* ta, const C* tb) {
    constexpr int E = 1 << row_lge<decltype(C{}.x)>();
    last_twiddle<RL, NB, J, 0>(x, cmul(ta[(J - 1) * RL], tb[(J - 1) * E]));
    if constexpr (J % 2 == 1) SCHED();
    if constexpr (J + 1 < RL) last_twiddles_from<RL, NB, J + 1>(x, ta, tb);
}

// Where a row reads a table: the entry of its first element, index step 1 (over the row) or
// 0 (one factor a row), and the conjugation.
struct RowTab {
    uint32_t off;
    int in;
    int cj;
};
template <int LGM>
__device__ __forceinline__ RowTab row_tab(const DiagTab& T, uint64_t base) {
    RowTab r;
    r.off = T.off + (uint32_t)((base >> T.sh) & ((1ull << T.nb) - 1ull)) + (T.nsel > 0 ? tab_choice(T, base) : 0u);
    r.cj = T.ctrl >= 0 && ((base >> T.ctrl) & 1ull) ? -1 : 1;
    r.in = T.sh <= 0 && LGM <= T.sh + T.nb ? 1 : 0;
    return r;
}

// Each element that took a factor is made opaque there: the products would otherwise be sunk
// below the other groups, whose factors and elements would then all be held at once.
template <typename C>
__device__ __forceinline__ void row_factor(C& x, C e) {
    x = cmul(x, e);
    asm volatile("" : "+v"(x.x), "+v"(x.y));
}

template <int E, typename C>
__device__ __forceinline__ void row_hold(C* x) {
#pragma unroll
    for (int j = 0; j < E; ++j) asm volatile("" : "+v"(x[j].x), "+v"(x[j].y));
}

// A table's factors on a thread's elements, so many loads in flight (complex64: 16 spill in the chain's
// loop, 4 take 0.95 ms where 8 take 0.90).
template <typename R> constexpr int row_batch() { return sizeof(R) == 4 ? 8 : 4; }
template <int LGM, typename C>
__device__ __forceinline__ void row_table(C* x, const RowTab& at, const C* __restrict__ arena, int tid) {
    using R = decltype(C{}.x);
    constexpr int E = 1 << row_lge<R>(), NT = (1 << LGM) / E, B = row_batch<R>();
    const C* tb = arena + (uint32_t)__builtin_amdgcn_readfirstlane((int)at.off);
    const int in = __builtin_amdgcn_readfirstlane(at.in);
    const R cj = (R)at.cj;
    const unsigned own = (unsigned)(tid * in);
#pragma unroll
    for (int j0 = 0; j0 < E; j0 += B) {
        C e[B];
#pragma unroll
        for (int j = 0; j < B; ++j) e[j] = (tb + (j0 + j) * NT * in)[own];
#pragma unroll
        for (int j = 0; j < B; ++j) {
            e[j].y *= cj;
            row_factor(x[j0 + j], e[j]);
        }
        SCHED();
    }
}

template <typename R, int LGM>
__global__ void __launch_bounds__((1 << LGM) >> row_lge<R>(), LGM == 14 ? 4 : 3)
k_fft_row(RowArgs a, typename CT<R>::type* data, const typename CT<R>::type* __restrict__ tw,
          const typename CT<R>::type* __restrict__ arena) {
    using C = typename CT<R>::type;
    constexpr int LGE = row_lge<R>(), E = 1 << LGE, EM = E - 1;
    constexpr int M = 1 << LGM, NT = M / E, RL = M / (E * E), NB = E / RL, TW = row_tw_total(LGM, LGE);
    __shared__ RowStep steps[FT_CHAIN_MAX];
    __shared__ RowTab sAt[FT_CHAIN_MAX * CVDV_FAST_TABS];
    __shared__ C sTw[TW];
    extern __shared__ __align__(16) unsigned char smem_raw[];
    R* ex = reinterpret_cast<R*>(smem_raw);
    const int tid = threadIdx.x;

    // the steps from the argument segment straight into LDS (a is the first argument):
    // indexing the argument at run time would copy it to scratch memory
    {
        typedef const __attribute__((address_space(4))) uint32_t* KArg;
        const KArg src = (KArg)__builtin_amdgcn_kernarg_segment_ptr() + offsetof(RowArgs, s) / 4;
        const int words = a.m * (int)(sizeof(RowStep) / 4);
        for (int i = tid; i < words; i += NT) ((uint32_t*)steps)[i] = src[i];
    }
    for (int e = tid; e < TW; e += NT) sTw[e] = tw[e];
    __syncthreads();
    const R scale = (R)a.scale;
    const R scaleLo = (R)(a.scale - (double)scale);

    for (uint64_t t = blockIdx.x; t < a.rows; t += gridDim.x) {
        const uint64_t base = t << LGM;
        C* row = data + base;
        C x[E];  // rows tid + e NT, in every stage's order of work
        {
            int ti = tid;
            asm volatile("" : "+v"(ti));
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int i = 0; i < E / 4; ++i) x[k + 4 * i] = (row + (k + 4 * i) * NT)[(unsigned)ti];
        }
        SCHED();
        if (tid < a.m * CVDV_FAST_TABS) {
            const FastDiag& p = steps[tid / CVDV_FAST_TABS].pre;
            const int n = tid % CVDV_FAST_TABS;
            if (n < p.ntab) sAt[tid] = row_tab<LGM>(p.tab[n], base);
        }
        lds_barrier();

#pragma unroll 1
        for (int s = 0; s < a.m; ++s) {
            // an opaque copy: index math would otherwise be kept across the steps and rows
            int ti = tid;
            asm volatile("" : "+v"(ti));
            const RowStep& st = steps[s];
            const int ntab = __builtin_amdgcn_readfirstlane(st.pre.ntab);
            const int ngen = __builtin_amdgcn_readfirstlane(st.pre.ngen);
#pragma unroll 1
            for (int n = 0; n < ntab; ++n) row_table<LGM>(x, sAt[s * CVDV_FAST_TABS + n], arena, ti);
            if (ngen > 0) {
                // affine in the row coordinate (the host checked): e^{2 pi i (a m + b)} at one
                // element of each of four groups of rows 4 NT apart, times steps that the whole row
                // shares (lane i evaluates step i)
                const GenFold gf = fold_generic(st.pre.gen, ngen, st.pre.genrev, base, 0, LGM);
                const int li = (int)__builtin_amdgcn_mbcnt_lo(~0u, 0u) & (E / 4 - 1);
                const C mine = unit_rev_fast(cvdv_frac(gf.turn((double)(2 * li * (4 * NT)))), R(0));
                C by[E / 4];
#pragma unroll
                for (int i = 1; i < E / 4; ++i) by[i] = lane_value(mine, i);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const C e0 =
                        unit_rev_fast(cvdv_frac(gf.turn((double)(2 * (ti + k * NT) + 1 - M)) + gf.b), R(0));
                    row_factor(x[k], e0);
#pragma unroll
                    for (int i = 1; i < E / 4; ++i) row_factor(x[k + 4 * i], cmul(e0, by[i]));
                    SCHED();
                }
            }
            const int ctl = __builtin_amdgcn_readfirstlane(st.ctl);
            int inv = __builtin_amdgcn_readfirstlane(st.inv);
            if (ctl) inv ^= (int)(base >> (ctl - 1)) & 1;
            {
                const R sg = inv ? R(-1) : R(1);
#pragma unroll
                for (int j = 0; j < E; ++j) x[j].y *= sg;
            }

            // E points NT apart; output m at m (NT + 1) + thread, so that the writes are
            // consecutive and a reader's stride of NT + 1 covers the banks
            dft_own(x);
            {
                R* wr = ex + ti;
                const R* rd = ex + (ti & EM) * (NT + 1) + (ti >> LGE);
#pragma unroll
                for (int m = 0; m < E; ++m) wr[m * (NT + 1)] = x[own_slot<R>(m)].x;
                lds_barrier();
#pragma unroll
                for (int e = 0; e < E; ++e) x[e].x = rd[e * (NT / E)];
                lds_barrier();
#pragma unroll
                for (int m = 0; m < E; ++m) wr[m * (NT + 1)] = x[own_slot<R>(m)].y;
                lds_barrier();
#pragma unroll
                for (int e = 0; e < E; ++e) x[e].y = rd[e * (NT / E)];
                lds_barrier();
            }
            // E points, each the start of E transformed rows
            {
                const C* w = sTw + (ti & EM);
#pragma unroll
                for (int e = 1; e < E; ++e) {
                    x[e] = cmul(x[e], w[(e - 1) * E]);
                    if (e % 8 == 7) SCHED();
                }
            }
            dft_own(x);
            {
                R* wr = ex + ((ti & ~EM) << LGE) + (ti & EM);
                const R* rd = ex + ti;
#pragma unroll
                for (int m = 0; m < E; ++m) wr[m * E] = x[own_slot<R>(m)].x;
                lds_barrier();
#pragma unroll
                for (int e = 0; e < E; ++e) x[e].x = rd[e * NT];
                lds_barrier();
                SCHED();
#pragma unroll
                for (int m = 0; m < E; ++m) wr[m * E] = x[own_slot<R>(m)].y;
                lds_barrier();
#pragma unroll
                for (int e = 0; e < E; ++e) x[e].y = rd[e * NT];
                lds_barrier();
                SCHED();
            }
            // NB butterflies of RL points E^2 apart
            last_twiddles_from<RL, NB, 1>(x, sTw + row_tw_mid(LGE) + (ti >> LGE),
                                          sTw + row_tw_mid(LGE) + (RL - 1) * RL + (ti & EM));
#pragma unroll
            for (int k = 0; k < NB; ++k) {
                if constexpr (RL == 16) dft16<NB>(x + k);
                else dft8_at<NB>(x + k);
            }
            {
                const R sg = inv ? R(-1) : R(1);
#pragma unroll
                for (int j = 0; j < E; ++j) x[j].y *= sg;
            }
            row_hold<E>(x);
        }
        if (a.useScale) {
#pragma unroll
            for (int e = 0; e < E; ++e) {
                x[e].x = fma(x[e].x, scale, x[e].x * scaleLo);
                x[e].y = fma(x[e].y, scale, x[e].y * scaleLo);
            }
        }
        int to = tid;
        asm volatile("" : "+v"(to));
#pragma unroll
        for (int e = 0; e < E; ++e) (row + e * NT)[(unsigned)to] = x[e];
    }
}

// Workgroups of a CU (LDS: 80 KiB for 2^14 complex64, 48 for 2^13 and for 2^12 complex128).
static int row_groups(int lgm) { return lgm == 14 ? 2 : 3; }

template <typename R, int LGM>
static void launch_row(hipStream_t stream, void* data, const RowArgs& a, const void* tw) {
    using C = typename CT<R>::type;
    constexpr int E = 1 << row_lge<R>(), NT = (1 << LGM) / E;
    auto kfn = k_fft_row<R, LGM>;
    const size_t lds = sizeof(R) * ((1 << LGM) + E);
    HIPCHK(hipFuncSetAttribute((const void*)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const uint64_t grid = std::min<uint64_t>(a.rows, (uint64_t)device_cus() * row_groups(LGM));
    hipLaunchKernelGGL(kfn, dim3((unsigned)grid), dim3(NT), lds, stream, a, (C*)data, (const C*)tw,
                       (const C*)a.s[0].pre.arena);
}

void fft_row_launch(hipStream_t stream, void* data, bool c128, int lgm, const RowArgs& a, const void* tw) {
    if (a.m < 1 || a.m > FT_CHAIN_MAX) throw CvdvError{CVDV_ERR_STATE, "row pass without a transform"};
    if (!c128 && lgm == 14) launch_row<float, 14>(stream, data, a, tw);
    else if (!c128 && lgm == 13) launch_row<float, 13>(stream, data, a, tw);
    else if (c128 && lgm == 12) launch_row<double, 12>(stream, data, a, tw);
    else throw CvdvError{CVDV_ERR_UNSUPPORTED, "row length without a kernel instance"};
}
