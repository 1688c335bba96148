// fft_row.hip - transforms of contiguous complex64 rows of 2^13 and 2^14 points, one
// workgroup a row, and a gate's transforms of the row one after the other in one pass.
//
// A row of 2^14 takes 128 KiB of LDS, a whole CU's: one workgroup, whose loads, stages
// and exchanges then follow each other with nothing beside them.  Here the real and the
// imaginary parts cross LDS one after the other through one buffer of half the size, so
// two workgroups (three of 2^13) share a CU and one computes while the other waits for
// memory or exchanges.  A thread holds 32 elements, which is what lets a transform be three
// stages (32 x 32 x 16, 32 x 32 x 8) and two exchanges instead of five and four; it owns the
// same rows before the first stage and after the last, so the next transform of a chain
// starts where the last one ended.
//
// Between HBM and in-CU work.  [14,14] complex64 (4.3 GB a pass; a copy of this shape takes
// 0.74 ms), ms against the tile of 1024 threads that this replaces: one transform without
// phases 0.80 (0.90), with its table 0.86 (1.01); a displacement's two 1.18 (2 x 0.93); a
// conditional rotation's three 1.70 (3 x 1.00); a squeezing gate's four 2.01 (4 x 0.99).
// [14,13]: 0.44, 0.58, 0.84, 0.92.  Two transforms of a row in one pass of the old tile cost
// exactly two passes.

#include <algorithm>

#include "cvdv_internal.h"
#include "fft_radix16.h"
#include "fft_row.h"

// 32 inputs in order; output m = m2 + 8 m1 is left at x[m1 + 4 m2] (dft32_slot).
__device__ __forceinline__ constexpr int dft32_slot(int m) { return (m >> 3) + 4 * (m & 7); }
#define SCHED() __builtin_amdgcn_sched_barrier(0)
template <int ST>
__device__ __forceinline__ void dft8_at(float2* x) {
    float2 y[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) y[j] = x[j * ST];
    dft8<false>(y);
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j * ST] = y[j];
}
template <int K, int M2>
__device__ __forceinline__ void dft32_inner(float2* x) {
    x[K + 4 * M2] = mul_w32<K * M2>(x[K + 4 * M2]);
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

// Butterfly K of the last stage sits at q + K NT: its twiddles are those of butterfly 0
// times W_32^{j K}.
template <int RL, int NB, int J, int K>
__device__ __forceinline__ void last_twiddle(float2* x, float2 w) {
    x[K + NB * J] = mul_w32<(J * K) & 31>(cmul(x[K + NB * J], w));
    if constexpr (K + 1 < NB) last_twiddle<RL, NB, J, K + 1>(x, w);
}
template <int RL, int NB, int J>
__device__ __forceinline__ void last_twiddles_from(float2* x, const float2* ta, const float2* tb) {
    last_twiddle<RL, NB, J, 0>(x, cmul(ta[(J - 1) * RL], tb[(J - 1) * 32]));
    if constexpr (J % 2 == 1) SCHED();
    if constexpr (J + 1 < RL) last_twiddles_from<RL, NB, J + 1>(x, ta, tb);
}

// Where a row reads a table: the entry of its first element, index step 1 (over the row) or
// 0 (one factor a row), and the conjugation.
struct RowTab {
    uint32_t off;
    int in;
    float cj;
};
template <int LGM>
__device__ __forceinline__ RowTab row_tab(const DiagTab& T, uint64_t base) {
    RowTab r;
    r.off = T.off + (uint32_t)((base >> T.sh) & ((1ull << T.nb) - 1ull)) + (T.nsel > 0 ? tab_choice(T, base) : 0u);
    r.cj = T.ctrl >= 0 && ((base >> T.ctrl) & 1ull) ? -1.f : 1.f;
    r.in = T.sh <= 0 && LGM <= T.sh + T.nb ? 1 : 0;
    return r;
}

// Each element that took a factor is made opaque there: the products would otherwise be sunk
// below the other groups, whose factors and elements would then all be held at once.
__device__ __forceinline__ void row_factor(float2& x, float2 e) {
    x = cmul(x, e);
    asm volatile("" : "+v"(x.x), "+v"(x.y));
}

__device__ __forceinline__ void row_hold(float2* x) {
#pragma unroll
    for (int j = 0; j < 32; ++j) asm volatile("" : "+v"(x[j].x), "+v"(x[j].y));
}

// A table's factors on a thread's elements, ROW_BATCH loads in flight (16 spill in the chain's
// loop, 4 take 0.95 ms where 8 take 0.90).
#define ROW_BATCH 8
template <int LGM>
__device__ __forceinline__ void row_table(float2* x, const RowTab& at, const float2* __restrict__ arena, int tid) {
    constexpr int NT = (1 << LGM) / 32;
    const float2* tb = arena + (uint32_t)__builtin_amdgcn_readfirstlane((int)at.off);
    const int in = __builtin_amdgcn_readfirstlane(at.in);
    const float cj = at.cj;
    const unsigned own = (unsigned)(tid * in);
#pragma unroll
    for (int j0 = 0; j0 < 32; j0 += ROW_BATCH) {
        float2 e[ROW_BATCH];
#pragma unroll
        for (int j = 0; j < ROW_BATCH; ++j) e[j] = (tb + (j0 + j) * NT * in)[own];
#pragma unroll
        for (int j = 0; j < ROW_BATCH; ++j) {
            e[j].y *= cj;
            row_factor(x[j0 + j], e[j]);
        }
        SCHED();
    }
}

template <int LGM>
__global__ void __launch_bounds__((1 << LGM) / 32, LGM == 14 ? 4 : 3)
k_fft_row(RowArgs a, float2* data, const float2* __restrict__ tw, const float2* __restrict__ arena) {
    constexpr int M = 1 << LGM, NT = M / 32, RL = M / 1024, NB = 32 / RL;
    __shared__ RowStep steps[FT_CHAIN_MAX];
    __shared__ RowTab sAt[FT_CHAIN_MAX * CVDV_FAST_TABS];
    __shared__ float2 sTw[row_tw_total(LGM)];
    extern __shared__ __align__(16) unsigned char smem_raw[];
    float* ex = reinterpret_cast<float*>(smem_raw);
    const int tid = threadIdx.x;

    // the steps from the argument segment straight into LDS (a is the first argument):
    // indexing the argument at run time would copy it to scratch memory
    {
        typedef const __attribute__((address_space(4))) uint32_t* KArg;
        const KArg src = (KArg)__builtin_amdgcn_kernarg_segment_ptr() + offsetof(RowArgs, s) / 4;
        const int words = a.m * (int)(sizeof(RowStep) / 4);
        for (int i = tid; i < words; i += NT) ((uint32_t*)steps)[i] = src[i];
    }
    for (int e = tid; e < row_tw_total(LGM); e += NT) sTw[e] = tw[e];
    __syncthreads();
    const float scale = (float)a.scale;
    const float scaleLo = (float)(a.scale - (double)scale);

    for (uint64_t t = blockIdx.x; t < a.rows; t += gridDim.x) {
        const uint64_t base = t << LGM;
        float2* row = data + base;
        float2 x[32];  // rows tid + e NT, in every stage's order of work
        {
            int ti = tid;
            asm volatile("" : "+v"(ti));
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int i = 0; i < 8; ++i) x[k + 4 * i] = (row + (k + 4 * i) * NT)[(unsigned)ti];
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
                // element of each group of 8, M/8 rows apart, times steps that the whole row
                // shares (lane i evaluates step i)
                const GenFold gf = fold_generic(st.pre.gen, ngen, st.pre.genrev, base, 0, LGM);
                const int li = (int)__builtin_amdgcn_mbcnt_lo(~0u, 0u) & 7;
                const float2 mine = unit_rev_fast(cvdv_frac(gf.a * (double)(2 * li * (M / 8))), 0.f);
                float2 by[8];
#pragma unroll
                for (int i = 1; i < 8; ++i) by[i] = lane_value(mine, i);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const float2 e0 =
                        unit_rev_fast(cvdv_frac(fma(gf.a, (double)(2 * (ti + k * NT) + 1 - M), gf.b)), 0.f);
                    row_factor(x[k], e0);
#pragma unroll
                    for (int i = 1; i < 8; ++i) row_factor(x[k + 4 * i], cmul(e0, by[i]));
                    SCHED();
                }
            }
            const int ctl = __builtin_amdgcn_readfirstlane(st.ctl);
            int inv = __builtin_amdgcn_readfirstlane(st.inv);
            if (ctl) inv ^= (int)(base >> (ctl - 1)) & 1;
            {
                const float sg = inv ? -1.f : 1.f;
#pragma unroll
                for (int j = 0; j < 32; ++j) x[j].y *= sg;
            }

            // 32 points NT apart; output m at m (NT + 1) + thread, so that the writes are
            // consecutive and a reader's stride of NT + 1 covers the banks
            dft32(x);
            {
                float* wr = ex + ti;
                const float* rd = ex + (ti & 31) * (NT + 1) + (ti >> 5);
#pragma unroll
                for (int m = 0; m < 32; ++m) wr[m * (NT + 1)] = x[dft32_slot(m)].x;
                lds_barrier();
#pragma unroll
                for (int e = 0; e < 32; ++e) x[e].x = rd[e * (NT / 32)];
                lds_barrier();
#pragma unroll
                for (int m = 0; m < 32; ++m) wr[m * (NT + 1)] = x[dft32_slot(m)].y;
                lds_barrier();
#pragma unroll
                for (int e = 0; e < 32; ++e) x[e].y = rd[e * (NT / 32)];
                lds_barrier();
            }
            // 32 points, each the start of 32 transformed rows
            {
                const float2* w = sTw + (ti & 31);
#pragma unroll
                for (int e = 1; e < 32; ++e) {
                    x[e] = cmul(x[e], w[(e - 1) * 32]);
                    if (e % 8 == 7) SCHED();
                }
            }
            dft32(x);
            {
                float* wr = ex + ((ti & ~31) << 5) + (ti & 31);
                const float* rd = ex + ti;
#pragma unroll
                for (int m = 0; m < 32; ++m) wr[m * 32] = x[dft32_slot(m)].x;
                lds_barrier();
#pragma unroll
                for (int e = 0; e < 32; ++e) x[e].x = rd[e * NT];
                lds_barrier();
                SCHED();
#pragma unroll
                for (int m = 0; m < 32; ++m) wr[m * 32] = x[dft32_slot(m)].y;
                lds_barrier();
#pragma unroll
                for (int e = 0; e < 32; ++e) x[e].y = rd[e * NT];
                lds_barrier();
                SCHED();
            }
            // NB butterflies of RL points 1024 apart
            last_twiddles_from<RL, NB, 1>(x, sTw + row_tw_mid() + (ti >> 5),
                                          sTw + row_tw_mid() + (RL - 1) * RL + (ti & 31));
#pragma unroll
            for (int k = 0; k < NB; ++k) {
                if constexpr (RL == 16) dft16<NB>(x + k);
                else dft8_at<NB>(x + k);
                SCHED();
            }
            {
                const float sg = inv ? -1.f : 1.f;
#pragma unroll
                for (int j = 0; j < 32; ++j) x[j].y *= sg;
            }
            row_hold(x);
        }
        if (a.useScale) {
#pragma unroll
            for (int e = 0; e < 32; ++e) {
                x[e].x = fmaf(x[e].x, scale, x[e].x * scaleLo);
                x[e].y = fmaf(x[e].y, scale, x[e].y * scaleLo);
            }
        }
        int to = tid;
        asm volatile("" : "+v"(to));
#pragma unroll
        for (int e = 0; e < 32; ++e) (row + e * NT)[(unsigned)to] = x[e];
    }
}

template <int LGM>
static void launch_row(hipStream_t stream, float2* data, const RowArgs& a, const float2* tw) {
    constexpr int NT = (1 << LGM) / 32;
    auto kfn = k_fft_row<LGM>;
    const size_t lds = sizeof(float) * ((1 << LGM) + 32);
    HIPCHK(hipFuncSetAttribute((const void*)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const uint64_t grid = std::min<uint64_t>(a.rows, (uint64_t)device_cus() * (LGM == 14 ? 2 : 3));
    hipLaunchKernelGGL(kfn, dim3((unsigned)grid), dim3(NT), lds, stream, a, data, tw,
                       (const float2*)a.s[0].pre.arena);
}

void fft_row_launch(hipStream_t stream, float2* data, int lgm, const RowArgs& a, const float2* tw) {
    if (a.m < 1 || a.m > FT_CHAIN_MAX) throw CvdvError{CVDV_ERR_STATE, "row pass without a transform"};
    if (lgm == 14) launch_row<14>(stream, data, a, tw);
    else if (lgm == 13) launch_row<13>(stream, data, a, tw);
    else throw CvdvError{CVDV_ERR_UNSUPPORTED, "row length without a kernel instance"};
}
