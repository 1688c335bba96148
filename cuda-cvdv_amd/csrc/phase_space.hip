// phase_space.hip - native-grid Wigner and Husimi-Q readouts.
//
// Reference interfaces replaced: src/cuda/bosonic.cu:10-152 and the kernels of
// src/cuda/kernels/bosonic.cuh:7-186; numerical semantics follow
// src/torchCvdv.py:344-404.  Readouts always compute in FP64 (amplitudes of a
// mixed-precision state are widened on load).
//
// Wigner:  rho = X X^H over the slices X[s][j] of register r (a complex
//          Hermitian rank-S product), integrand G[i][k] = rho[i-kd][i+kd] with
//          kd = k - (N-1)/2, an unnormalised inverse FFT along k, and
//          W[jc][i] = Re(e^{-i (N-1) dx p_jc} G[i][(jc+N/2) mod N]) dx / pi,
//          p_jc = (jc - N/2) pi / (N dx)  (bosonic.cuh:39-52, torchCvdv.py:361-368).
// Husimi:  Q[jc][q] = sum_s |FFT_x(psi_s[x] w(q,x))[(jc+N/2) mod N]|^2 / pi with
//          the non-periodic window w(q,x) = pi^-1/4 exp(-((x-q) dx)^2/2) sqrt(dx)
//          (torchCvdv.py:380-397).

#include <cmath>
#include <string>
#include <vector>

#include "cvdv_internal.h"
#include "readout_rows.h"
#include "../../include/cvdv_hip.h"

static const double PI = 3.14159265358979323846;

static unsigned grid_for(uint64_t total, unsigned block = 256) {
    uint64_t b = (total + block - 1) / block;
    if (b > 65536ull * 8) b = 65536ull * 8;
    return (unsigned)(b ? b : 1);
}

// X[s][j] = psi(slice s, logical j) in FP64
template <typename C>
__global__ void k_extract(double2* __restrict__ X, const C* __restrict__ st, uint64_t S, int sh, int n,
                          int refl) {
    const uint64_t N = 1ull << n, tot = S * N, slo = (1ull << sh) - 1ull;
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < tot;
         e += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t s = e >> n, j = e & (N - 1);
        const uint64_t jp = refl ? (N - 1 - j) : j;
        const uint64_t g = ((s & ~slo) << n) | (jp << sh) | (s & slo);
        const C v = st[g];
        X[e] = make_double2((double)v.x, (double)v.y);
    }
}

// rho[a][b] = sum_s X[s][a] conj(X[s][b]); 32x32 output tile per workgroup.
__global__ void __launch_bounds__(256) k_rho(const double2* __restrict__ X, uint64_t S, int N,
                                             double2* __restrict__ rho) {
    __shared__ double2 xa[16][33];
    __shared__ double2 xb[16][33];
    const int tid = threadIdx.x;
    const int a0 = blockIdx.y * 32, b0 = blockIdx.x * 32;
    const int ta = (tid / 16) * 2, tb = (tid % 16) * 2;
    double2 acc[2][2] = {{{0, 0}, {0, 0}}, {{0, 0}, {0, 0}}};
    for (uint64_t s0 = 0; s0 < S; s0 += 16) {
        for (int e = tid; e < 16 * 32; e += 256) {
            const int ks = e / 32, c = e % 32;
            const uint64_t s = s0 + ks;
            const bool ok = s < S;
            xa[ks][c] = (ok && a0 + c < N) ? X[s * N + a0 + c] : make_double2(0, 0);
            xb[ks][c] = (ok && b0 + c < N) ? X[s * N + b0 + c] : make_double2(0, 0);
        }
        __syncthreads();
#pragma unroll 4
        for (int ks = 0; ks < 16; ++ks) {
            const double2 u0 = xa[ks][ta], u1 = xa[ks][ta + 1];
            const double2 v0 = xb[ks][tb], v1 = xb[ks][tb + 1];
            acc[0][0].x += u0.x * v0.x + u0.y * v0.y; acc[0][0].y += u0.y * v0.x - u0.x * v0.y;
            acc[0][1].x += u0.x * v1.x + u0.y * v1.y; acc[0][1].y += u0.y * v1.x - u0.x * v1.y;
            acc[1][0].x += u1.x * v0.x + u1.y * v0.y; acc[1][0].y += u1.y * v0.x - u1.x * v0.y;
            acc[1][1].x += u1.x * v1.x + u1.y * v1.y; acc[1][1].y += u1.y * v1.x - u1.x * v1.y;
        }
        __syncthreads();
    }
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j) {
            const int a = a0 + ta + i, b = b0 + tb + j;
            if (a < N && b < N) rho[(uint64_t)a * N + b] = acc[i][j];
        }
}

__global__ void k_wigner_integrand(double2* __restrict__ G, const double2* __restrict__ rho, int N) {
    const uint64_t tot = (uint64_t)N * N;
    const int h = (N - 1) / 2;
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < tot;
         e += (uint64_t)gridDim.x * blockDim.x) {
        const int i = (int)(e / N), k = (int)(e % N);
        const int kd = k - h, ipy = i + kd, imy = i - kd;
        G[e] = (ipy >= 0 && ipy < N && imy >= 0 && imy < N) ? rho[(uint64_t)imy * N + ipy]
                                                             : make_double2(0, 0);
    }
}

// W[jc][i] = Re(e^{-i (N-1) dx p_jc} G[i][kf]) dx/pi; optionally written as complex
template <bool COMPLEX_OUT>
__global__ void k_wigner_finalize(void* __restrict__ outv, const double2* __restrict__ G, int N, double dx) {
    const uint64_t tot = (uint64_t)N * N;
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < tot;
         e += (uint64_t)gridDim.x * blockDim.x) {
        const int jc = (int)(e / N), i = (int)(e % N);
        const int kf = (jc + N / 2) % N;
        const double2 v = G[(uint64_t)i * N + kf];
        // -(N-1) dx p_jc = -(N-1)(jc - N/2) pi / N  (radians) -> sincospi
        const double a = -(double)(N - 1) * ((double)jc - 0.5 * N) / (double)N;
        const double ar = a - 2.0 * rint(0.5 * a);
        double s, c;
        sincospi(ar, &s, &c);
        const double w = (v.x * c - v.y * s) * dx / PI;
        if (COMPLEX_OUT) ((double2*)outv)[e] = make_double2(w, 0.0);
        else ((double*)outv)[e] = w;
    }
}

// B[q][s][x] = X[s][x] w(q, x) for q in [q0, q0+Qc)
__global__ void k_husimi_window(double2* __restrict__ B, const double2* __restrict__ X, uint64_t S, int n,
                                int q0, int Qc, double dx) {
    const uint64_t N = 1ull << n, tot = (uint64_t)Qc * S * N;
    const double norm = pow(PI, -0.25) * sqrt(dx);
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < tot;
         e += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t x = e & (N - 1);
        const uint64_t sq = e >> n;
        const uint64_t s = sq % S;
        const int q = q0 + (int)(sq / S);
        const double d = ((double)x - (double)q) * dx;
        const double w = norm * exp(-0.5 * d * d);
        const double2 v = X[s * N + x];
        B[e] = make_double2(v.x * w, v.y * w);
    }
}

// acc[q][m] += sum_s |B[q][s][m]|^2 (fixed order over s)
__global__ void k_husimi_accum(double* __restrict__ acc, const double2* __restrict__ B, uint64_t S, int N,
                               int q0, int Qc) {
    const uint64_t tot = (uint64_t)Qc * N;
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < tot;
         e += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t ql = e / N, m = e % N;
        double sum = 0.0;
        for (uint64_t s = 0; s < S; ++s) {
            const double2 v = B[(ql * S + s) * N + m];
            sum += v.x * v.x + v.y * v.y;
        }
        acc[(uint64_t)(q0 + ql) * N + m] = sum;
    }
}

__global__ void k_husimi_finalize(double* __restrict__ Q, const double* __restrict__ acc, int N) {
    const uint64_t tot = (uint64_t)N * N;
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < tot;
         e += (uint64_t)gridDim.x * blockDim.x) {
        const int jc = (int)(e / N), q = (int)(e % N);
        Q[e] = acc[(uint64_t)q * N + (jc + N / 2) % N] / PI;
    }
}

// bosonic.cuh:158-178: spectrum *= exp(-(wq^2 + wp^2)/4)
__global__ void k_husimi_gauss2d(double2* __restrict__ spec, int N, double dx) {
    const uint64_t tot = (uint64_t)N * N;
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < tot;
         e += (uint64_t)gridDim.x * blockDim.x) {
        const int pIdx = (int)(e / N), qIdx = (int)(e % N);
        const int kq = (qIdx <= N / 2) ? qIdx : (qIdx - N);
        const int kp = (pIdx <= N / 2) ? pIdx : (pIdx - N);
        const double Lq = (double)N * dx;
        const double dp = PI / ((double)N * dx);
        const double Lp = (double)N * dp;
        const double wq = 2.0 * PI * kq / Lq, wp = 2.0 * PI * kp / Lp;
        const double g = exp(-0.25 * (wq * wq + wp * wp));
        spec[e] = make_double2(spec[e].x * g, spec[e].y * g);
    }
}

// bosonic.cuh:180-186
__global__ void k_real_clamp(double* __restrict__ out, const double2* __restrict__ in, uint64_t n2,
                             double norm) {
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n2;
         e += (uint64_t)gridDim.x * blockDim.x) {
        const double v = in[e].x / norm;
        out[e] = v < 0.0 ? 0.0 : v;
    }
}

// ---------------------------------------------------------------- row kernels
// Native grids of 2^3 .. 2^13 points: one workgroup builds its rows' integrands in
// registers, transforms them in LDS (fft_stages.h) and writes the picture, so no
// N x N intermediate touches memory.
// Slice s of a contiguous register field, point j (logical), widened to FP64.
template <typename C>
__device__ __forceinline__ double2 slice_at(const C* __restrict__ X, uint64_t s, int lgN, int j, int refl) {
    const C v = X[(s << lgN) + (uint64_t)(refl ? (1 << lgN) - 1 - j : j)];
    return make_double2((double)v.x, (double)v.y);
}

__device__ __forceinline__ void add_product(double2& g, double2 u, double2 v) {  // g += u conj(v)
    g.x += u.x * v.x + u.y * v.y;
    g.y += u.y * v.x - u.x * v.y;
}

// The value of the lane below (above) in the wave; the first (last) lane keeps `edge`.
template <int CTRL>
__device__ __forceinline__ double lane_shift(double v, double edge) {
    const long long a = __double_as_longlong(v), b = __double_as_longlong(edge);
    const int lo = __builtin_amdgcn_update_dpp((int)b, (int)a, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(b >> 32), (int)(a >> 32), CTRL, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double2 from_below(double2 v, double2 edge) {
    return make_double2(lane_shift<0x138>(v.x, edge.x), lane_shift<0x138>(v.y, edge.y));  // wave_shr:1
}
__device__ __forceinline__ double2 from_above(double2 v, double2 edge) {
    return make_double2(lane_shift<0x130>(v.x, edge.x), lane_shift<0x130>(v.y, edge.y));  // wave_shl:1
}

// Products of slices [s, s + K) at distance d for the rows i0 and i0 + 1; d is
// consecutive over the (full) wave.  Points outside the grid count as 0: the caller
// drops the sums of lanes that reach beyond it.
template <int K, typename C>
__device__ __forceinline__ void pair_products(double2& g0, double2& g1, const C* __restrict__ X, uint64_t s, int lgN,
                                              int i0, int d, int refl) {
    const int N = 1 << lgN, lane = threadIdx.x & 63;
    const int a = i0 - d, b = i0 + d, c = lane == 0 ? a + 1 : b + 1;
    const bool edge = (lane == 0 || lane == 63) && c >= 0 && c < N;
    double2 u[K], v[K], w[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        u[k] = a >= 0 && a < N ? slice_at(X, s + k, lgN, a, refl) : make_double2(0.0, 0.0);
        v[k] = b >= 0 && b < N ? slice_at(X, s + k, lgN, b, refl) : make_double2(0.0, 0.0);
        w[k] = make_double2(0.0, 0.0);
    }
    if (edge) {
#pragma unroll
        for (int k = 0; k < K; ++k) w[k] = slice_at(X, s + k, lgN, c, refl);
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        add_product(g0, u[k], v[k]);
        add_product(g1, from_below(u[k], w[k]), from_above(v[k], w[k]));
    }
}

// Wigner rows i = 2a and 2a + 1.  Row i's integrand g(d) = sum_s X_s[i-d] conj(X_s[i+d])
// is Hermitian in d (and g(N/2) = 0: one of i -+ N/2 lies outside the grid), so its
// transform R is real: the two rows go through one complex transform as
// g_2a + i g_2a+1, and only d >= 0 is summed.  Indexing the transform by d mod N
// instead of k = d + (N-1)/2 turns the finalisation e^{-i (N-1) dx p} into the real
// factor cos(pi u / N) at frequency u (|u| <= N/2): W = cos(pi u / N) R dx / pi.
// A row with a non-finite value reads NaN throughout, and leaves its partner alone.
// Bound by the loads of the sum (one a product: the two rows share them) and the 16-byte
// stores of a picture whose rows are momenta: eight neighbouring pairs share each
// 128-byte line, so they run on one XCD (workgroups go round the eight XCDs in turn:
// 172 us without that order, 150 us with it).  [2,2,12]: 520 us as rho, integrand,
// transform and finalisation over N x N complex intermediates, 150 us here; a wave's
// neighbouring lanes share the loads of both rows (186 us with each lane loading its own).
template <int LGM, typename C, bool COMPLEX_OUT>
__global__ void __launch_bounds__(rows_threads<LGM>())
k_wigner_rows(void* __restrict__ outv, const C* __restrict__ X, uint64_t S, int refl, double dx,
              const double2* __restrict__ tw) {
    constexpr int N = 1 << LGM, NT = rows_threads<LGM>(), NST = Plan<LGM>::NST;
    constexpr int R0 = 1 << Plan<LGM>::lgr(0), RL = 1 << Plan<LGM>::lgr(NST - 1);
    constexpr int HB = 1 << rows_lg_hb<LGM>();
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ int bad[2 * HB];
    double2* lds = reinterpret_cast<double2*>(smem_raw);
    const int tid = threadIdx.x;
    uint32_t b = blockIdx.x;
    if (HB == 1 && (gridDim.x & 63u) == 0) {
        const uint32_t xcd = b & 7u, t = b >> 3;
        b = ((((t >> 3) << 3) + xcd) << 3) + (t & 7u);
    }
    const int a0 = (int)b * HB;
    for (int k = tid; k < 2 * HB; k += NT) bad[k] = 0;
    __syncthreads();
#pragma unroll 1
    for (int t = 0; t < 4; ++t) {
        const int e = tid + t * NT, hb = e >> (LGM - 1), d = e & (N / 2 - 1);
        const int i0 = 2 * (a0 + hb), i1 = i0 + 1;
        // row i0 reaches d <= min(i0, N-1-i0), row i1 as far or one further or less
        const bool in = i1 < N, ok0 = in && i0 - d >= 0 && i0 + d < N, ok1 = in && i1 - d >= 0 && i1 + d < N;
        double2 g0 = make_double2(0.0, 0.0), g1 = make_double2(0.0, 0.0);
        if constexpr (LGM >= 7) {
            // a wave holds 64 consecutive d of one pair of rows: X[i1-d] is its
            // neighbour's X[i0-(d-1)], X[i1+d] its other neighbour's X[i0+(d+1)]
            if (__any(ok0 || ok1)) {
                if (S >= 4)
                    for (uint64_t s = 0; s < S; s += 4) pair_products<4>(g0, g1, X, s, LGM, i0, d, refl);
                else
                    for (uint64_t s = 0; s < S; ++s) pair_products<1>(g0, g1, X, s, LGM, i0, d, refl);
            }
            if (!ok0) g0 = make_double2(0.0, 0.0);
            if (!ok1) g1 = make_double2(0.0, 0.0);
        } else if (ok0 || ok1) {
#pragma unroll 4
            for (uint64_t s = 0; s < S; ++s) {
                if (ok0) add_product(g0, slice_at(X, s, LGM, i0 - d, refl), slice_at(X, s, LGM, i0 + d, refl));
                if (ok1) add_product(g1, slice_at(X, s, LGM, i1 - d, refl), slice_at(X, s, LGM, i1 + d, refl));
            }
        }
        if (!isfinite(g0.x) || !isfinite(g0.y)) {
            bad[2 * hb] = 1;
            g0 = make_double2(0.0, 0.0);
        }
        if (!isfinite(g1.x) || !isfinite(g1.y)) {
            bad[2 * hb + 1] = 1;
            g1 = make_double2(0.0, 0.0);
        }
        // the inverse transform is conj . forward . conj: conj(g0 + i g1) at d and at N - d
        const int o = hb << LGM;
        if (d == 0) {
            lds[lay_ix<3>(o)] = make_double2(g0.x, -g1.x);
            lds[lay_ix<3>(o + N / 2)] = make_double2(0.0, 0.0);
        } else {
            lds[lay_ix<3>(o + d)] = make_double2(g0.x - g1.y, -(g0.y + g1.x));
            lds[lay_ix<3>(o + N - d)] = make_double2(g0.x + g1.y, g0.y - g1.x);
        }
    }
    __syncthreads();
    double2 x[8];
    stage_read<R0, 8, LGM, 0, 0, EX_ROWS>(lds, x, tid, NT);
    lds_barrier();
    stage_compute<R0, 8, LGM, 0, 0>(x, tw, tid, NT);
    run_stages<LGM, 0, 1, 8, EX_ROWS>(x, lds, tw, tid, NT);
    const double w = dx / PI;
#pragma unroll
    for (int k = 0; k < 8 / RL; ++k) {
        const BflyPos p = bfly_pos<RL, LGM, 8>(tid, k, NT, 0);
        const bool n0 = bad[2 * p.hb] != 0, n1 = bad[2 * p.hb + 1] != 0;
        if (2 * (a0 + p.hb) >= N) continue;
#pragma unroll
        for (int m = 0; m < RL; ++m) {
            const int kf = p.q + m * (N / RL), u = kf < N / 2 ? kf : kf - N;
            const double c = cospi((double)u / (double)N) * w;
            const double r0 = n0 ? NAN : x[k * RL + m].x * c, r1 = n1 ? NAN : -x[k * RL + m].y * c;
            const uint64_t o = (uint64_t)(kf ^ (N / 2)) * N + 2 * (a0 + p.hb);
            if constexpr (COMPLEX_OUT) {
                ((double2*)outv)[o] = make_double2(r0, 0.0);
                ((double2*)outv)[o + 1] = make_double2(r1, 0.0);
            } else {
                *(double2*)((double*)outv + o) = make_double2(r0, r1);
            }
        }
    }
}

// acc[q][m] = sum_s |FFT_x(X_s[x] w(q, x))[m]|^2 for the rows q of the workgroup's
// tile, summed over the slices in order.  Bound by FP64 arithmetic (VALU issue half of
// the cycles) and the LDS exchanges, with the slices read from L2.  [2,2,12]: 3610 us as
// windowed batches, transforms and sums through HBM (17 GB), 786 us here; 950 us without
// the held last-stage twiddles and with exchanges of one pad entry per 32.
template <int LGM, typename C>
__global__ void __launch_bounds__(rows_threads<LGM>())
k_husimi_rows(double* __restrict__ acc, const C* __restrict__ X, uint64_t S, int refl, double dx,
              const double2* __restrict__ tw) {
    constexpr int N = 1 << LGM, NT = rows_threads<LGM>(), NST = Plan<LGM>::NST;
    constexpr int R0 = 1 << Plan<LGM>::lgr(0), RL = 1 << Plan<LGM>::lgr(NST - 1);
    constexpr int HB = 1 << rows_lg_hb<LGM>();
    extern __shared__ __align__(16) unsigned char smem_raw[];
    double2* lds = reinterpret_cast<double2*>(smem_raw);
    const int tid = threadIdx.x, q0 = blockIdx.x * HB;
    const double norm = pow(PI, -0.25) * sqrt(dx);
    double w[8], sum[8];
#pragma unroll
    for (int k = 0; k < 8 / R0; ++k) {
        const BflyPos p = bfly_pos<R0, LGM, 8>(tid, k, NT, 0);
#pragma unroll
        for (int i = 0; i < R0; ++i) {
            const double d = ((double)(p.q + i * (N / R0)) - (double)(q0 + p.hb)) * dx;
            w[k * R0 + i] = norm * exp(-0.5 * d * d);
            sum[k * R0 + i] = 0.0;
        }
    }
    double2 wl[8 / RL * (RL - 1)];
    if constexpr (NST > 1) last_twiddles<8, LGM>(wl, tw, tid, NT);
#pragma unroll 1
    for (uint64_t s = 0; s < S; ++s) {
        // an opaque copy of the thread id: the other stages' twiddles, the same for every
        // slice, would otherwise all be held in registers (200 of them, one workgroup a CU)
        int ti = tid;
        asm volatile("" : "+v"(ti));
        double2 x[8];
#pragma unroll
        for (int k = 0; k < 8 / R0; ++k) {
            const BflyPos p = bfly_pos<R0, LGM, 8>(ti, k, NT, 0);
#pragma unroll
            for (int i = 0; i < R0; ++i) x[k * R0 + i] = slice_at(X, s, LGM, p.q + i * (N / R0), refl);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = make_double2(x[i].x * w[i], x[i].y * w[i]);
        stage_compute<R0, 8, LGM, 0, 0>(x, tw, ti, NT);
        run_stages<LGM, 0, 1, 8, EX_ROWS, true>(x, lds, tw, ti, NT, wl);
#pragma unroll
        for (int i = 0; i < 8; ++i) sum[i] += x[i].x * x[i].x + x[i].y * x[i].y;
    }
#pragma unroll
    for (int k = 0; k < 8 / RL; ++k) {
        const BflyPos p = bfly_pos<RL, LGM, 8>(tid, k, NT, 0);
        if (q0 + p.hb >= N) continue;
#pragma unroll
        for (int m = 0; m < RL; ++m) acc[(uint64_t)(q0 + p.hb) * N + p.q + m * (N / RL)] = sum[k * RL + m];
    }
}

// Q[jc][q] = acc[q][(jc + N/2) mod N] / pi through 32 x 32 tiles (rows of both
// sides in whole lines; N a multiple of 32).
__global__ void __launch_bounds__(256) k_husimi_turn(double* __restrict__ Q, const double* __restrict__ acc, int N) {
    __shared__ double t[32][33];
    const int c = threadIdx.x & 31, r = threadIdx.x >> 5;
    const int m0 = blockIdx.x * 32, q0 = blockIdx.y * 32;
#pragma unroll
    for (int k = 0; k < 32; k += 8) t[r + k][c] = acc[(uint64_t)(q0 + r + k) * N + m0 + c];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 32; k += 8)
        Q[(uint64_t)((m0 + r + k) ^ (N / 2)) * N + q0 + c] = t[c][r + k] / PI;
}

// ---------------------------------------------------------------- drivers
struct Bufs {
    double2* X;
    uint64_t S;
    int N, n, sh;
};

static Bufs extract_slices(CVDVContext* ctx, int r, double2* X) {
    Bufs b{};
    b.n = ctx->nq[r];
    b.N = 1 << b.n;
    b.sh = ctx->pshift[r];
    b.S = ctx->totalSize >> b.n;
    b.X = X;
    const uint64_t tot = ctx->totalSize;
    if (ctx->prec == CVDV_C128)
        hipLaunchKernelGGL(k_extract<double2>, dim3(grid_for(tot)), dim3(256), 0, ctx->stream, X,
                           (const double2*)ctx->state(), b.S, b.sh, b.n, ctx->refl[r]);
    else
        hipLaunchKernelGGL(k_extract<float2>, dim3(grid_for(tot)), dim3(256), 0, ctx->stream, X,
                           (const float2*)ctx->state(), b.S, b.sh, b.n, ctx->refl[r]);
    HIPCHK(hipGetLastError());
    return b;
}

// The rows kernels read the slices of a contiguous field from the state itself, those
// of any other field from the extracted copy X.  Wigner sums read every slice for every pair
// of rows: from 16 complex64 slices on, widening them once (the copy) costs less than widening
// them at every load ([4,8] 33 us by the copy, 42 directly; [4,12] 145 and 173; [3,8] 34 and 30).
struct RowsIn {
    const void* p;
    bool wide;  // double2 (else float2)
    int refl;
};

static bool rows_direct(const CVDVContext* ctx, int r, bool wigner) {
    const bool widen = wigner && ctx->prec == CVDV_MIXED && (ctx->totalSize >> ctx->nq[r]) >= 16;
    return ctx->pshift[r] == 0 && !widen;
}

static RowsIn rows_input(CVDVContext* ctx, int r, bool wigner, double2* X) {
    if (rows_direct(ctx, r, wigner)) return RowsIn{ctx->state(), ctx->prec == CVDV_C128, ctx->refl[r]};
    extract_slices(ctx, r, X);
    return RowsIn{X, true, 0};
}

// Every pair of rows reads the slices again, where k_rho's tiles share them: with many
// slices for the grid's size the sum is the time, and the tiles win.  Measured (us, rows
// against tiles, integrand, transform and finalisation): N = 2^8: 31 / 40 at 16 slices,
// 168 / 71 at 256; 2^10: 62 / 72 at 64, 199 / 132 at 256; 2^12: 148 / 529 at 16,
// 317 / 722 at 64, 1102 / 1511 at 256.  The line is N/16 slices (16 for small grids).  At 2^5 and
// 2^6 points, whose 2 and 4 workgroups of one wave each sum several rows in turn, it is 8, or 4
// where the slices are extracted first: 33 / 29 and 35 / 32 at 16 slices, 28 / 32 at 8 (33 / 31
// extracted); 2^4 24 / 28 at 16.
static bool wigner_by_rows(const CVDVContext* ctx, int r) {
    const int n = ctx->nq[r];
    const uint64_t N = 1ull << n, S = ctx->totalSize >> n;
    if (n < ROWS_LGM_MIN || n > ROWS_LGM_MAX) return false;
    if (n == 5 || n == 6) return S <= (rows_direct(ctx, r, true) ? 8 : 4);
    return S <= (N > 256 ? N / 16 : 16);
}

// A Husimi row's workgroup transforms its slices one after the other: below 2^9 points there
// are too few rows to fill the chip, and with many slices the windowed batches win.  Measured
// (us, rows against batches, contiguous and extracted fields): 2^3: 47 / 61 at 64 slices, 106 /
// 106 at 256; 2^6: 38 / 43 at 8, 44 / 47 and 49 / 45 at 16, 71 / 58 at 64, 1860 / 380 at 1024; 2^7:
// 49 / 51 and 54 / 48 at 16, 89 / 72 at 64; 2^8: 92 / 92 and 102 / 92 at 64, 278 / 305 and 310 / 304 at
// 256; 2^9: 301 / 897 at 256.
static bool husimi_by_rows(const CVDVContext* ctx, int r) {
    const int n = ctx->nq[r];
    const uint64_t S = ctx->totalSize >> n;
    if (n < ROWS_LGM_MIN || n > ROWS_LGM_MAX) return false;
    if (n >= 9) return true;
    if (rows_direct(ctx, r, false)) return n == 8 || S <= (n == 3 ? 64 : 16);
    return S <= (n == 8 ? 32 : n <= 4 ? 16 : 8);
}

// Device scratch of wigner_device: X (A c128), and rho, G, tmp (N2 c128 each) where
// the rows kernels don't serve the register.
static size_t wigner_scratch(const CVDVContext* ctx, int r) {
    const uint64_t N2 = 1ull << (2 * ctx->nq[r]), A = ctx->totalSize;
    if (wigner_by_rows(ctx, r)) return rows_direct(ctx, r, true) ? 0 : A * 16;
    return A * 16 + 3 * N2 * 16;
}

// Wigner into dev (N*N doubles or complex when asComplex).
static void wigner_device(CVDVContext* ctx, int r, void* dev, bool asComplex, double2* X) {
    ctx_flush(ctx);
    if (wigner_by_rows(ctx, r)) {
        const RowsIn in = rows_input(ctx, r, true, X);
        const uint64_t S = ctx->totalSize >> ctx->nq[r];
        const double2* tw = (const double2*)fft_stage_table(ctx->tw, ctx->nq[r], CVDV_C128);
        rows_dispatch(ctx->nq[r], [&](auto lg) {
            constexpr int L = decltype(lg)::value, HB = 1 << rows_lg_hb<L>();
            const unsigned blocks = (unsigned)(((1 << (L - 1)) + HB - 1) / HB);
            auto go = [&](auto kfn, auto* src) {
                rows_launch_attr(kfn, rows_lds<L>());
                hipLaunchKernelGGL(kfn, dim3(blocks), dim3(rows_threads<L>()), rows_lds<L>(), ctx->stream, dev, src,
                                   S, in.refl, ctx->dx[r], tw);
            };
            if (in.wide) {
                if (asComplex) go(k_wigner_rows<L, double2, true>, (const double2*)in.p);
                else go(k_wigner_rows<L, double2, false>, (const double2*)in.p);
            } else {
                if (asComplex) go(k_wigner_rows<L, float2, true>, (const float2*)in.p);
                else go(k_wigner_rows<L, float2, false>, (const float2*)in.p);
            }
        });
        HIPCHK(hipGetLastError());
        return;
    }
    Bufs b = extract_slices(ctx, r, X);
    const int N = b.N;
    const uint64_t N2 = (uint64_t)N * N;
    double2* rho = X + ctx->totalSize;
    double2* G = rho + N2;
    double2* tmp = G + N2;
    dim3 gr((N + 31) / 32, (N + 31) / 32);
    hipLaunchKernelGGL(k_rho, gr, dim3(256), 0, ctx->stream, X, b.S, N, rho);
    HIPCHK(hipGetLastError());
    hipLaunchKernelGGL(k_wigner_integrand, dim3(grid_for(N2)), dim3(256), 0, ctx->stream, G, rho, N);
    HIPCHK(hipGetLastError());
    // unnormalised inverse FFT along k (rows of G)
    if (b.n > 0) fft_generic_c128(ctx, G, tmp, N2, 0, b.n, true, 1.0);
    if (asComplex)
        hipLaunchKernelGGL(k_wigner_finalize<true>, dim3(grid_for(N2)), dim3(256), 0, ctx->stream, dev, G, N,
                           ctx->dx[r]);
    else
        hipLaunchKernelGGL(k_wigner_finalize<false>, dim3(grid_for(N2)), dim3(256), 0, ctx->stream, dev, G,
                           N, ctx->dx[r]);
    HIPCHK(hipGetLastError());
}

// The readouts below write their N x N result into `out`: host memory (through
// a device scratch copy), or, with outOnDevice, caller device memory directly.
static void finish_out(CVDVContext* ctx, double* out, const double* dev, uint64_t n, bool outOnDevice) {
    if (outOnDevice) HIPCHK(hipStreamSynchronize(ctx->stream));
    else copy_to_host(ctx->stream, out, dev, n * sizeof(double));
}

static void get_wigner(CVDVContext* ctx, int r, double* out, bool outOnDevice) {
    const int N = 1 << ctx->nq[r];
    const uint64_t N2 = (uint64_t)N * N;
    // scratch: wigner_device's | W (N2 doubles)
    const size_t work = wigner_scratch(ctx, r);
    char* base = (char*)ctx_scratch(ctx, work + (outOnDevice ? 0 : N2 * 8));
    double* W = outOnDevice ? out : (double*)(base + work);
    const int pid = prof_begin(ctx, KK_OTHER);  // the readout's device time, first to last kernel
    wigner_device(ctx, r, W, false, (double2*)base);
    prof_end(ctx, pid);
    finish_out(ctx, out, W, N2, outOnDevice);
}

static void get_husimi_overlap(CVDVContext* ctx, int r, double* out, bool outOnDevice) {
    ctx_flush(ctx);
    const int n = ctx->nq[r], N = 1 << n;
    const uint64_t N2 = (uint64_t)N * N, A = ctx->totalSize, S = A >> n;
    if (husimi_by_rows(ctx, r)) {
        // scratch: X (A, when the field is not contiguous) | acc (N2 doubles) | Q (N2 doubles)
        const size_t xb = rows_direct(ctx, r, false) ? 0 : A * 16;
        char* base = (char*)ctx_scratch(ctx, xb + (outOnDevice ? 1 : 2) * N2 * 8);
        double* acc = (double*)(base + xb);
        double* Q = outOnDevice ? out : acc + N2;
        const int pid = prof_begin(ctx, KK_OTHER);
        const RowsIn in = rows_input(ctx, r, false, (double2*)base);
        const double2* tw = (const double2*)fft_stage_table(ctx->tw, n, CVDV_C128);
        rows_dispatch(n, [&](auto lg) {
            constexpr int L = decltype(lg)::value, HB = 1 << rows_lg_hb<L>();
            const unsigned blocks = (unsigned)(((1 << L) + HB - 1) / HB);
            auto go = [&](auto kfn, auto* src) {
                rows_launch_attr(kfn, rows_lds<L>());
                hipLaunchKernelGGL(kfn, dim3(blocks), dim3(rows_threads<L>()), rows_lds<L>(), ctx->stream, acc, src,
                                   S, in.refl, ctx->dx[r], tw);
            };
            if (in.wide) go(k_husimi_rows<L, double2>, (const double2*)in.p);
            else go(k_husimi_rows<L, float2>, (const float2*)in.p);
        });
        HIPCHK(hipGetLastError());
        if (N % 32 == 0)
            hipLaunchKernelGGL(k_husimi_turn, dim3(N / 32, N / 32), dim3(256), 0, ctx->stream, Q, acc, N);
        else
            hipLaunchKernelGGL(k_husimi_finalize, dim3(grid_for(N2)), dim3(256), 0, ctx->stream, Q, acc, N);
        HIPCHK(hipGetLastError());
        prof_end(ctx, pid);
        finish_out(ctx, out, Q, N2, outOnDevice);
        return;
    }
    // q chunk so that the windowed batch stays below 2^26 elements (1 GiB)
    uint64_t Qc = 1;
    while (Qc * 2 <= (uint64_t)N && Qc * 2 * S * N <= (1ull << 26)) Qc *= 2;
    const uint64_t batch = Qc * S * N;
    // scratch: X (A) | B (batch) | tmp (batch) | acc (N2 doubles) | Q (N2 doubles)
    char* base = (char*)ctx_scratch(ctx, A * 16 + 2 * batch * 16 + (outOnDevice ? 1 : 2) * N2 * 8);
    double2* X = (double2*)base;
    double2* B = X + A;
    double2* tmp = B + batch;
    double* acc = (double*)(tmp + batch);
    double* Q = outOnDevice ? out : acc + N2;
    const int pid = prof_begin(ctx, KK_OTHER);
    Bufs b = extract_slices(ctx, r, X);
    for (uint64_t q0 = 0; q0 < (uint64_t)N; q0 += Qc) {
        hipLaunchKernelGGL(k_husimi_window, dim3(grid_for(batch)), dim3(256), 0, ctx->stream, B, X, b.S, n,
                           (int)q0, (int)Qc, ctx->dx[r]);
        HIPCHK(hipGetLastError());
        if (n > 0) fft_generic_c128(ctx, B, tmp, batch, 0, n, false, 1.0);
        hipLaunchKernelGGL(k_husimi_accum, dim3(grid_for(Qc * N)), dim3(256), 0, ctx->stream, acc, B, b.S, N,
                           (int)q0, (int)Qc);
        HIPCHK(hipGetLastError());
    }
    hipLaunchKernelGGL(k_husimi_finalize, dim3(grid_for(N2)), dim3(256), 0, ctx->stream, Q, acc, N);
    HIPCHK(hipGetLastError());
    prof_end(ctx, pid);
    finish_out(ctx, out, Q, N2, outOnDevice);
}

// bosonic.cu:63-101: Wigner -> 2D FFT -> Gaussian -> inverse 2D FFT -> Re/N^2, clamped
static void get_husimi_wigner(CVDVContext* ctx, int r, double* out, bool outOnDevice) {
    const int n = ctx->nq[r], N = 1 << n;
    const uint64_t N2 = (uint64_t)N * N;
    // scratch: Wc | tmp (N2 c128 each) | wigner_device's | Q (N2 doubles)
    const size_t work = wigner_scratch(ctx, r);
    char* base = (char*)ctx_scratch(ctx, 2 * N2 * 16 + work + (outOnDevice ? 0 : N2 * 8));
    double2* Wc = (double2*)base;
    double2* tmp = Wc + N2;
    double* Q = outOnDevice ? out : (double*)(base + 2 * N2 * 16 + work);
    const int pid = prof_begin(ctx, KK_OTHER);
    wigner_device(ctx, r, Wc, true, tmp + N2);
    if (n > 0) {
        fft_generic_c128(ctx, Wc, tmp, N2, 0, n, false, 1.0);  // along q (columns index)
        fft_generic_c128(ctx, Wc, tmp, N2, n, n, false, 1.0);  // along p (rows index)
    }
    hipLaunchKernelGGL(k_husimi_gauss2d, dim3(grid_for(N2)), dim3(256), 0, ctx->stream, Wc, N, ctx->dx[r]);
    HIPCHK(hipGetLastError());
    if (n > 0) {
        fft_generic_c128(ctx, Wc, tmp, N2, 0, n, true, 1.0);
        fft_generic_c128(ctx, Wc, tmp, N2, n, n, true, 1.0);
    }
    hipLaunchKernelGGL(k_real_clamp, dim3(grid_for(N2)), dim3(256), 0, ctx->stream, Q, Wc, N2, (double)N2);
    HIPCHK(hipGetLastError());
    prof_end(ctx, pid);
    finish_out(ctx, out, Q, N2, outOnDevice);
}

// bosonic.cu:13-25: the overlap route holds one N-point window, two N x N double
// arrays, every slice and an N x N complex block per slice; above 80% of the
// free device memory (or when the device cannot say) the FFT2 route runs.  Both
// are FP64; they differ in grid and normalisation (getHusimiQWigner's p spacing
// is pi/(N dx) and its scale that of the Wigner), as in the reference.  The
// overlap route here is chunked and needs far less than that estimate; the
// estimate is kept so the same states take the same route.
static void get_husimi(CVDVContext* ctx, int r, double* out, bool outOnDevice) {
    const uint64_t N = 1ull << ctx->nq[r], N2 = N * N, S = ctx->totalSize >> ctx->nq[r];
    const double need = (double)(N * 16 + 2 * N2 * 8) + (double)S * (double)N * 16.0 + (double)S * (double)N2 * 16.0;
    size_t freeB = ctx->freeMemOverride, totalB = 0;
    bool known = true;
    if (!freeB) known = hipMemGetInfo(&freeB, &totalB) == hipSuccess;
    if (!known || need > 0.8 * (double)freeB) get_husimi_wigner(ctx, r, out, outOnDevice);
    else get_husimi_overlap(ctx, r, out, outOnDevice);
}

#define CVDV_TRY try {
#define CVDV_CATCH()                                                         \
    }                                                                        \
    catch (const CvdvError& e) {                                             \
        cvdv_set_error(e.code, e.msg);                                       \
    }                                                                        \
    catch (...) {                                                            \
        cvdv_set_error(CVDV_ERR_HIP, "unexpected internal error");           \
    }

static bool ps_ok(CVDVContext* ctx, int r, double* out) {
    if (!ctx || !out || refuse_recording(ctx)) return false;
    if (!ctx->initialized) {
        cvdv_set_error(CVDV_ERR_STATE, "State not initialized");
        return false;
    }
    if (r < 0 || r >= ctx->numReg) {
        cvdv_set_error(CVDV_ERR_ARG, "Invalid register index: " + std::to_string(r));
        return false;
    }
    return true;
}

extern "C" {

void cvdvGetWigner(CVDVContext* ctx, int regIdx, double* wignerOut) {
    if (!ps_ok(ctx, regIdx, wignerOut)) return;
    CVDV_TRY get_wigner(ctx, regIdx, wignerOut, false); CVDV_CATCH()
}

void cvdvGetHusimiQ(CVDVContext* ctx, int regIdx, double* husimiOut) {
    if (!ps_ok(ctx, regIdx, husimiOut)) return;
    CVDV_TRY get_husimi(ctx, regIdx, husimiOut, false); CVDV_CATCH()
}

void cvdvGetHusimiQOverlap(CVDVContext* ctx, int regIdx, double* husimiOut) {
    if (!ps_ok(ctx, regIdx, husimiOut)) return;
    CVDV_TRY get_husimi_overlap(ctx, regIdx, husimiOut, false); CVDV_CATCH()
}

void cvdvGetHusimiQWigner(CVDVContext* ctx, int regIdx, double* husimiOut) {
    if (!ps_ok(ctx, regIdx, husimiOut)) return;
    CVDV_TRY get_husimi_wigner(ctx, regIdx, husimiOut, false); CVDV_CATCH()
}

void cvdvGetWignerDevice(CVDVContext* ctx, int regIdx, double* d_out) {
    if (!ps_ok(ctx, regIdx, d_out)) return;
    CVDV_TRY get_wigner(ctx, regIdx, d_out, true); CVDV_CATCH()
}

void cvdvGetHusimiQDevice(CVDVContext* ctx, int regIdx, double* d_out) {
    if (!ps_ok(ctx, regIdx, d_out)) return;
    CVDV_TRY get_husimi(ctx, regIdx, d_out, true); CVDV_CATCH()
}

void cvdvSetFreeMemoryOverride(CVDVContext* ctx, size_t bytes) {
    if (!ctx) return;
    ctx->freeMemOverride = bytes;
}

}  // extern "C"
