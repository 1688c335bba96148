// phase_grid.hip - Wigner and Husimi-Q of one register at arbitrary phase-space
// points, traced over the other registers or one block per slice (per branch of
// the other registers' values).  An addition: the reference evaluates both only
// on its native grid (src/cuda/bosonic.cu:10-152); on that grid these equal
// cvdvGetWigner / cvdvGetHusimiQ.
//
// Wigner.  With x = x_i + t dx (t in [0,1), t = 0 on grid points) and phi_s the
// trigonometric interpolant of slice s sampled at x_j + t dx (one FFT per slice,
// a phase ramp and one inverse FFT per x point), A(d) = sum_s phi_s(i-d)
// conj(phi_s(i+d)) for |d| <= N/2 (zero outside the grid), and
//     W(x, p) = dx/pi Re sum_d A(d) e^{i dx p m(d)},
// m(d) = 2(d + (N-1)/2) - (N-1) (native: the e^{-i (N-1) dx p} finalisation of
// bosonic.cuh:39-52) or m(d) = 2d (the symmetric sum).  A is Hermitian in d and
// A(N/2) = 0, and native's m = 2d - 1 only multiplies the symmetric sum by
// cos(dx p), so
//     W(x, p) = dx/pi [cos(dx p)] (A(0) + 2 sum_{0<d<N/2} Re A(d) cos 2 d dx p - Im A(d) sin 2 d dx p):
// for all points at once a real GEMM of depth N (rocBLAS dgemm), a quarter of the
// operations of the complex GEMM over all d.
// Husimi.  Q(q, p) = dx/pi^(3/2) sum_s |H_s(q,p)|^2 with
//     H_s(q, p) = sum_j e^{-i p x_j} psi_s(x_j) e^{-(x_j-q)^2/2}.
// The grid is symmetric (x_{N-1-j} = -x_j): with g the windowed slice, each pair of
// points adds cos(p x_j) (g_j + g_{N-1-j}) - i sin(p x_j) (g_j - g_{N-1-j}), so the real
// and imaginary parts are real GEMMs of depth N, half the operations of the complex
// one.  Points whose window is exactly 0 in FP64 for every q are left out.  Angles are
// FP64 with range reduction (revolutions, frac, sincospi); all arithmetic is FP64.

#include <rocblas/rocblas.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "cvdv_internal.h"
#include "readout_rows.h"
#include "../../include/cvdv_hip.h"

static const double PI = 3.14159265358979323846;
static const uint64_t GRID_CHUNK = 1ull << 26;  // complex128 elements per intermediate buffer (1 GiB)

static unsigned grid_for(uint64_t total, unsigned block = 256) {
    uint64_t b = (total + block - 1) / block;
    if (b > 65536ull * 8) b = 65536ull * 8;
    return (unsigned)(b ? b : 1);
}

static rocblas_handle blas(CVDVContext* ctx) {
    if (!ctx->blas) {
        rocblas_handle h = nullptr;
        if (rocblas_create_handle(&h) != rocblas_status_success)
            throw CvdvError{CVDV_ERR_HIP, "rocblas_create_handle failed"};
        ctx->blas = h;
    }
    rocblas_handle h = (rocblas_handle)ctx->blas;
    if (rocblas_set_stream(h, ctx->stream) != rocblas_status_success)
        throw CvdvError{CVDV_ERR_HIP, "rocblas_set_stream failed"};
    return h;
}

void blas_release(CVDVContext* ctx) {
    if (ctx->blas) (void)rocblas_destroy_handle((rocblas_handle)ctx->blas);
    ctx->blas = nullptr;
}

static void blas_check(rocblas_status s, const char* what) {
    if (s != rocblas_status_success) throw CvdvError{CVDV_ERR_HIP, std::string(what) + " failed"};
}

// Ccm(m x n, ldc) = alpha Acm^T Bcm for `batch` slices (column-major; A: k x m, B: k x n,
// the same for every slice).
static void dgemm_tn(CVDVContext* ctx, int m, int n, int k, double alpha, const double* A, uint64_t strideA,
                     const double* B, double* C, int ldc, uint64_t strideC, int batch) {
    const double zero = 0.0;
    blas_check(rocblas_dgemm_strided_batched(blas(ctx), rocblas_operation_transpose, rocblas_operation_none, m, n, k,
                                             &alpha, A, k, (rocblas_stride)strideA, B, k, 0, &zero, C, ldc,
                                             (rocblas_stride)strideC, batch),
               "rocblas_dgemm_strided_batched");
}

// The same in complex arithmetic, C = A^T B.
static void zgemm_tn(CVDVContext* ctx, int m, int n, int k, const double2* A, uint64_t strideA, const double2* B,
                     double2* C, int ldc, uint64_t strideC, int batch) {
    const rocblas_double_complex one{1.0, 0.0}, zero{0.0, 0.0};
    blas_check(rocblas_zgemm_strided_batched(blas(ctx), rocblas_operation_transpose, rocblas_operation_none, m, n, k,
                                             &one, (const rocblas_double_complex*)A, k, (rocblas_stride)strideA,
                                             (const rocblas_double_complex*)B, k, 0, &zero,
                                             (rocblas_double_complex*)C, ldc, (rocblas_stride)strideC, batch),
               "rocblas_zgemm_strided_batched");
}

// ---------------------------------------------------------------- kernels
// X[s][j]: slices of register r in the canonical layout (field at sh), FP64.
template <typename C>
__global__ void k_grid_slices(double2* __restrict__ X, const C* __restrict__ st, uint64_t S, int sh, int n) {
    const uint64_t N = 1ull << n, tot = S * N, slo = (1ull << sh) - 1ull;
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < tot;
         e += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t s = e >> n, j = e & (N - 1);
        const C v = st[((s & ~slo) << n) | (j << sh) | (s & slo)];
        X[e] = make_double2((double)v.x, (double)v.y);
    }
}

// Y[x][s][k] = spec[s][k] e^{2 pi i kk t_x / N} / N (kk the signed frequency);
// an inverse FFT along k then samples the interpolant at x_j + t_x dx.
__global__ void k_grid_shift(double2* __restrict__ Y, const double2* __restrict__ spec, uint64_t S, int n,
                             const double* __restrict__ tx, int nxc) {
    const uint64_t N = 1ull << n, per = S * N, tot = per * (uint64_t)nxc;
    const double invN = 1.0 / (double)N;
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < tot;
         e += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t x = e / per, sk = e - x * per, k = sk & (N - 1);
        const int64_t kk = k < N / 2 ? (int64_t)k : (int64_t)k - (int64_t)N;
        const double2 u = unit_rev(cvdv_frac((double)kk * tx[x] * invN), 0.0);
        const double2 c = spec[sk];
        Y[e] = make_double2((c.x * u.x - c.y * u.y) * invN, (c.x * u.y + c.y * u.x) * invN);
    }
}

// Re and Im of A(d) = sum_s (or slice s) phi[x][s][i_x - d] conj(phi[x][s][i_x + d]) at
// A[(s,) x][2d] and [2d+1], 0 <= d < max(1, N/2).
__global__ void k_grid_pairs(double2* __restrict__ A, const double2* __restrict__ phi, uint64_t S, int n,
                             const int* __restrict__ ix, int nxc, int nxa, int perSlice) {
    const int N = 1 << n, nd = N > 1 ? N / 2 : 1;
    const uint64_t blocks = perSlice ? S * (uint64_t)nxa : (uint64_t)nxa;
    const uint64_t tot = blocks * (uint64_t)nd;
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < tot;
         e += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t row = e / nd;
        const int d = (int)(e - row * nd);
        const uint64_t x = perSlice ? row % nxa : row;
        const uint64_t s0 = perSlice ? row / nxa : 0, s1 = perSlice ? s0 + 1 : S;
        const int i = ix[x], a = i - d, b = i + d;
        double re = 0.0, im = 0.0;
        if (a >= 0 && b < N) {
#pragma unroll 4
            for (uint64_t s = s0; s < s1; ++s) {
                const double2 u = phi[(x * S + s) * N + a], v = phi[(x * S + s) * N + b];
                re += u.x * v.x + u.y * v.y;  // u conj(v)
                im += u.y * v.x - u.x * v.y;
            }
        }
        A[e] = make_double2(re, im);
    }
}

// k_grid_shift, the inverse FFT and k_grid_pairs in one launch for N = 2^LGM: a row is
// the interpolant of one slice at one x, built, transformed and multiplied in LDS
// (traced readouts sum the products of their slices, in order, in registers).  Bound by
// writing the operand A (8 bytes a grid point and row) and the transform's exchanges:
// 512 points of [2,2,12] per branch take 177 us, 467 us as three kernels over complex
// intermediates (with all d); the GEMM behind it 535 us instead of 2170 us.
template <int LGM>
__global__ void __launch_bounds__(rows_threads<LGM>())
k_grid_rows(double2* __restrict__ A, const double2* __restrict__ spec, uint64_t S, const int* __restrict__ ix,
            const double* __restrict__ tx, int nxa, int perSlice, const double2* __restrict__ tw) {
    constexpr int N = 1 << LGM, NT = rows_threads<LGM>(), NST = Plan<LGM>::NST, HB = 1 << rows_lg_hb<LGM>();
    constexpr int RL = 1 << Plan<LGM>::lgr(NST - 1);
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ double2 step[HB * 8];
    double2* lds = reinterpret_cast<double2*>(smem_raw);
    const int tid = threadIdx.x;
    const uint64_t rows = perSlice ? S * (uint64_t)nxa : (uint64_t)nxa, row0 = (uint64_t)blockIdx.x * HB;
    // e^{2 pi i kk t / N} with kk = q + i N/8 (- N from N/2 on): one factor per row and i,
    // one per thread's q
    for (int e = tid; e < HB * 8; e += NT) {
        const uint64_t row = row0 + (e >> 3);
        const double t = row < rows ? tx[perSlice ? row % nxa : row] : 0.0;
        const int i = e & 7;
        step[e] = unit_rev(cvdv_frac(0.125 * (double)(i < 4 ? i : i - 8) * t), 0.0);
    }
    __syncthreads();
    const BflyPos p0 = bfly_pos<8, LGM, 8>(tid, 0, NT, 0);
    const uint64_t myRow = row0 + p0.hb;
    const double myT = myRow < rows ? tx[perSlice ? myRow % nxa : myRow] : 0.0;
    const double2 u0 = unit_rev(cvdv_frac((double)p0.q * myT * (1.0 / N)), 0.0);
    double2 sum[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) sum[t] = make_double2(0.0, 0.0);
#pragma unroll 1
    for (uint64_t s1 = 0; s1 < (perSlice ? 1 : S); ++s1) {
        const uint64_t s = perSlice ? myRow / nxa : s1;
        // opaque: the stages' twiddles, the same for every slice, would otherwise be held
        int ti = tid;
        asm volatile("" : "+v"(ti));
        double2 x[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            x[i] = myRow < rows ? spec[(s << LGM) + p0.q + i * (N / 8)] : make_double2(0.0, 0.0);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            // the inverse transform is conj . forward . conj
            const double2 v = cmul(x[i], cmul(u0, step[(p0.hb << 3) + i]));
            x[i] = make_double2(v.x * (1.0 / N), -v.y * (1.0 / N));
        }
        stage_compute<8, 8, LGM, 0, 0>(x, tw, ti, NT);
        run_stages<LGM, 0, 1, 8, EX_ROWS>(x, lds, tw, ti, NT);
        stage_write<RL, 8, LGM, 0, NST - 1, EX_ROWS>(lds, x, ti, NT);
        lds_barrier();
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int e = ti + t * NT, hb = e >> (LGM - 1), d = e & (N / 2 - 1);
            const uint64_t row = row0 + hb;
            if (row >= rows) continue;
            const int i = ix[perSlice ? row % nxa : row], a = i - d, b = i + d;
            if (a >= 0 && b < N) {
                // lds holds the conjugates: phi_a conj(phi_b) = conj(u) v
                const double2 u = lds[lay_ix<3>((hb << LGM) + a)], v = lds[lay_ix<3>((hb << LGM) + b)];
                sum[t].x += u.x * v.x + u.y * v.y;
                sum[t].y += u.x * v.y - u.y * v.x;
            }
        }
        lds_barrier();
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int e = tid + t * NT, hb = e >> (LGM - 1), d = e & (N / 2 - 1);
        if (row0 + hb < rows) A[((row0 + hb) << (LGM - 1)) + d] = sum[t];
    }
}

// E[p][2d], [2d+1] = w cos 2 d dx p, -w sin 2 d dx p (w = 1 at d = 0, else 2; times
// cos(dx p) for native), 0 <= d < nd = max(1, N/2).
__global__ void k_grid_wigner_E(double2* __restrict__ E, const double* __restrict__ ps, int np, int n, double dx,
                                int native) {
    const int N = 1 << n, nd = N > 1 ? N / 2 : 1;
    const uint64_t tot = (uint64_t)np * nd;
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < tot;
         e += (uint64_t)gridDim.x * blockDim.x) {
        const int p = (int)(e / nd), d = (int)(e % nd);
        const double r = cvdv_frac(dx * ps[p] / (2.0 * PI));
        const double2 u = unit_rev(cvdv_frac(r * (double)(2 * d)), 0.0);
        const double w = (d ? 2.0 : 1.0) * (native && N > 1 ? cospi(2.0 * r) : 1.0);
        E[e] = make_double2(u.x * w, -u.y * w);
    }
}

// The pairs of points (j, N-1-j), j = j0 + jj, jj < nj, of the windowed slices
// g = X[s] e^{-(x-q)^2/2}: row 2q (for Re H) holds Re(g_j + g_m), Im(g_j - g_m) at 2jj and
// 2jj + 1, row 2q + 1 (for Im H) holds Im(g_j + g_m), -Re(g_j - g_m).  out[s] is added to
// the first pair (k_grid_outside).  N = 1 has one point, its own mirror image.
__global__ void k_grid_husimi_B(double2* __restrict__ B, const double2* __restrict__ X, uint64_t S, int n,
                                const double* __restrict__ qs, int nqc, double dx, int j0, int nj,
                                const double2* __restrict__ out) {
    const uint64_t N = 1ull << n, tot = S * (uint64_t)nqc * nj;
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < tot;
         e += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t jj = e % nj, sq = e / nj, q = sq % nqc, s = sq / nqc, j = j0 + jj, m = N - 1 - j;
        const double x = ((double)j - 0.5 * (double)(N - 1)) * dx;
        const double a = x - qs[q], b = -x - qs[q];
        const double wa = exp(-0.5 * a * a), wb = N > 1 ? exp(-0.5 * b * b) : 0.0;
        const double2 u = X[s * N + j], v = N > 1 ? X[s * N + m] : make_double2(0.0, 0.0);
        double2 g = make_double2(u.x * wa, u.y * wa);
        const double2 h = make_double2(v.x * wb, v.y * wb);
        if (jj == 0 && out) {
            g.x += out[s].x;
            g.y += out[s].y;
        }
        double2* row = B + (s * nqc + q) * 2 * nj;
        row[jj] = make_double2(g.x + h.x, g.y - h.y);
        row[nj + jj] = make_double2(g.y + h.y, h.x - g.x);
    }
}

// out[s] = sum of 0 * X[s][j] over the points j < j0 and their mirror images: 0, or NaN
// where the window's exact 0 meets a value that is not finite.
__global__ void __launch_bounds__(256) k_grid_outside(double2* __restrict__ out, const double2* __restrict__ X, int n,
                                                      int j0) {
    __shared__ int bad[2];
    if (threadIdx.x < 2) bad[threadIdx.x] = 0;
    __syncthreads();
    const uint64_t N = 1ull << n, s = blockIdx.x;
    for (int j = threadIdx.x; j < j0; j += blockDim.x) {
        const double2 u = X[s * N + j], v = X[s * N + N - 1 - j];
        if (!isfinite(u.x) || !isfinite(v.x)) bad[0] = 1;
        if (!isfinite(u.y) || !isfinite(v.y)) bad[1] = 1;
    }
    __syncthreads();
    if (threadIdx.x == 0) out[s] = make_double2(bad[0] ? NAN : 0.0, bad[1] ? NAN : 0.0);
}

// E2[p][2jj], [2jj+1] = cos(p x_j), sin(p x_j), x_j = (2j - N + 1) dx / 2, j = j0 + jj.
__global__ void k_grid_husimi_E(double2* __restrict__ E, const double* __restrict__ ps, int np, int n, double dx,
                                int j0, int nj) {
    const uint64_t N = 1ull << n, tot = (uint64_t)np * nj;
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < tot;
         e += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t p = e / nj, j = j0 + e % nj;
        const double m = (double)(2 * (int64_t)j - (int64_t)N + 1);
        E[e] = unit_rev(cvdv_frac(cvdv_frac(dx * ps[p] / (4.0 * PI)) * m), 0.0);
    }
}

// The operands of the complex form: B[s][q][j] = X[s][j] e^{-(x_j-q)^2/2}, E[p][j] = e^{-i p x_j}.
__global__ void k_grid_husimi_zB(double2* __restrict__ B, const double2* __restrict__ X, uint64_t S, int n,
                                 const double* __restrict__ qs, int nqc, double dx) {
    const uint64_t N = 1ull << n, tot = S * (uint64_t)nqc * N;
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < tot;
         e += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t j = e & (N - 1), sq = e >> n, q = sq % nqc, s = sq / nqc;
        const double a = ((double)j - 0.5 * (double)(N - 1)) * dx - qs[q], w = exp(-0.5 * a * a);
        const double2 u = X[s * N + j];
        B[e] = make_double2(u.x * w, u.y * w);
    }
}
__global__ void k_grid_husimi_zE(double2* __restrict__ E, const double* __restrict__ ps, int np, int n, double dx) {
    const uint64_t N = 1ull << n, tot = (uint64_t)np << n;
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < tot;
         e += (uint64_t)gridDim.x * blockDim.x) {
        const double m = (double)(2 * (int64_t)(e & (N - 1)) - (int64_t)N + 1);
        E[e] = unit_rev(cvdv_frac(cvdv_frac(-dx * ps[e >> n] / (4.0 * PI)) * m), 0.0);
    }
}

// out[(s,) p][q] = scale * (|H_s|^2, or summed over s in slice order).
__global__ void k_grid_abs2(double* __restrict__ out, const double2* __restrict__ H, uint64_t S, uint64_t per,
                            int perSlice, double scale) {
    const uint64_t tot = perSlice ? S * per : per;
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < tot;
         e += (uint64_t)gridDim.x * blockDim.x) {
        double acc = 0.0;
        if (perSlice) {
            const double2 h = H[e];
            acc = h.x * h.x + h.y * h.y;
        } else {
            for (uint64_t s = 0; s < S; ++s) {
                const double2 h = H[s * per + e];
                acc += h.x * h.x + h.y * h.y;
            }
        }
        out[e] = acc * scale;
    }
}

// ---------------------------------------------------------------- drivers
// x -> (i, t) with x = x_i + t dx; within 1e-9 of a grid point: t = 0.
static void grid_split(double x, int N, double dx, int& i, double& t) {
    const double u = (x + 0.5 * (double)(N - 1) * dx) / dx;
    const double r = std::nearbyint(u);
    if (std::fabs(u - r) < 1e-9) {
        i = (int)r;
        t = 0.0;
    } else {
        const double f = std::floor(u);
        i = (int)f;
        t = u - f;
    }
    if (i < 0 || !std::isfinite(u)) {
        i = 0;
        t = 0.0;
    }
    if (i > N - 1) {
        i = N - 1;
        t = 0.0;
    }
}

// Canonical slices of register r (pending phases applied, lazy layout undone).
static double2* grid_slices(CVDVContext* ctx, int r, double2* X) {
    ctx_materialize(ctx);
    const int n = ctx->nq[r];
    const uint64_t S = ctx->totalSize >> n, tot = ctx->totalSize;
    if (ctx->prec == CVDV_C128)
        hipLaunchKernelGGL(k_grid_slices<double2>, dim3(grid_for(tot)), dim3(256), 0, ctx->stream, X,
                           (const double2*)ctx->state(), S, ctx->flw[r], n);
    else
        hipLaunchKernelGGL(k_grid_slices<float2>, dim3(grid_for(tot)), dim3(256), 0, ctx->stream, X,
                           (const float2*)ctx->state(), S, ctx->flw[r], n);
    HIPCHK(hipGetLastError());
    return X;
}

// Device scratch carved in order; the host arrays behind `up` go over in one copy.
struct GridScratch {
    char* base;
    size_t off = 0;
    template <typename T> T* take(size_t n) {
        T* p = (T*)(base + off);
        off += (n * sizeof(T) + 15) & ~(size_t)15;
        return p;
    }
};

// Traced pictures sum the slices one after the other in every row's workgroup: with more than
// a few slices that serial chain is the time, unless the rows alone fill the chip, and the
// batched transforms of k_grid_shift and k_grid_pairs win.  Measured (us, rows against
// batches): 32 points of N = 2^6: 77 / 73 at 16 slices, 163 / 90 at 64, 1840 / 435 at 1024;
// of 2^10: 114 / 109 at 16, 256 / 141 at 64; 128 points of 2^10: 279 / 221 at 64; 256 of 2^10:
// 286 / 327 at 64, 853 / 1003 at 256; 128 of 2^12: 655 / 770 at 64; 256 of 2^9: 225 / 215 at 64,
// 2331 / 2532 at 1024; 16 of 2^3: 73 / 77 at 32, 99 / 87 at 64.
static bool wigner_grid_by_rows(int n, uint64_t S, int nx, int perSlice) {
    if (n < ROWS_LGM_MIN || n > ROWS_LGM_MAX) return false;
    const uint64_t work = (uint64_t)nx << n;
    return perSlice || S <= (n == 3 ? 32 : 16) || (nx >= 256 && work >= (1ull << 17)) ||
           (nx >= 128 && work >= (1ull << 18));
}

static void get_wigner_grid(CVDVContext* ctx, int r, const double* xs, int nx, const double* ps, int np,
                            int perSlice, int native, double* out) {
    const int n = ctx->nq[r], N = 1 << n, nd = N > 1 ? N / 2 : 1, K = 2 * nd;
    const double dx = ctx->dx[r];
    const uint64_t A = ctx->totalSize, S = A >> n;
    const uint64_t outBlocks = perSlice ? S : 1;
    const bool rows = wigner_grid_by_rows(n, S, nx, perSlice);
    // x chunk: a power of two (the batched FFT over the chunk's S rows per point
    // needs a power-of-two row count); the last chunk is padded with t = 0 rows.
    // The row kernels have no intermediate but the operand A.
    int nxc = 1;
    while (nxc < nx && (rows || (uint64_t)nxc * 2 * S * N <= GRID_CHUNK) &&
           (uint64_t)nxc * 2 * nd * outBlocks <= GRID_CHUNK)
        nxc *= 2;
    const int nChunks = (nx + nxc - 1) / nxc;
    const int nxPad = nChunks * nxc;
    // ps | t of every x | grid index of every x
    std::vector<double> up((size_t)np + nxPad + (nxPad + 1) / 2, 0.0);
    std::copy(ps, ps + np, up.begin());
    double* ht = up.data() + np;
    int* hi = (int*)(ht + nxPad);
    for (int x = 0; x < nx; ++x) grid_split(xs[x], N, dx, hi[x], ht[x]);
    // scratch: spec | Y (nxc S N, general lengths) | tmp | operand A | E | out | the uploads
    const uint64_t nY = rows ? 0 : (uint64_t)nxc * S * N, nA = outBlocks * nxc * nd, nE = (uint64_t)np * nd;
    const uint64_t nZ = outBlocks * (uint64_t)np * nx;
    const uint64_t nTmp = std::max(nY, A);
    GridScratch g{(char*)ctx_scratch(ctx, (A + nY + nTmp + nA + nE) * 16 + (nZ + up.size()) * 8 + 256)};
    double2* spec = g.take<double2>(A);
    double2* Y = g.take<double2>(nY);
    double2* tmp = g.take<double2>(nTmp);
    double2* Ap = g.take<double2>(nA);
    double2* E = g.take<double2>(nE);
    double* dout = g.take<double>(nZ);
    double* dps = g.take<double>(up.size());
    const double* dtx = dps + np;
    const int* dix = (const int*)(dtx + nxPad);
    // spectra of the slices (unnormalised forward FFT)
    grid_slices(ctx, r, spec);
    HIPCHK(hipMemcpyAsync(dps, up.data(), up.size() * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    if (n > 0) fft_generic_c128(ctx, spec, tmp, A, 0, n, false, 1.0);
    hipLaunchKernelGGL(k_grid_wigner_E, dim3(grid_for(nE)), dim3(256), 0, ctx->stream, E, dps, np, n, dx, native);
    HIPCHK(hipGetLastError());
    const double2* tw = rows ? (const double2*)fft_stage_table(ctx->tw, n, CVDV_C128) : nullptr;
    for (int x0 = 0; x0 < nx; x0 += nxc) {
        const int c = nx - x0 < nxc ? nx - x0 : nxc;
        if (rows) {
            rows_dispatch(n, [&](auto lg) {
                constexpr int L = decltype(lg)::value, HB = 1 << rows_lg_hb<L>();
                const uint64_t blocks = (outBlocks * c + HB - 1) / HB;
                rows_launch_attr(k_grid_rows<L>, rows_lds<L>());
                hipLaunchKernelGGL(k_grid_rows<L>, dim3((unsigned)blocks), dim3(rows_threads<L>()), rows_lds<L>(),
                                   ctx->stream, Ap, spec, S, dix + x0, dtx + x0, c, perSlice, tw);
            });
            HIPCHK(hipGetLastError());
        } else {
            hipLaunchKernelGGL(k_grid_shift, dim3(grid_for(nY)), dim3(256), 0, ctx->stream, Y, spec, S, n, dtx + x0,
                               nxc);  // padded rows keep the FFT's row count a power of two
            HIPCHK(hipGetLastError());
            if (n > 0) fft_generic_c128(ctx, Y, tmp, nY, 0, n, true, 1.0);
            hipLaunchKernelGGL(k_grid_pairs, dim3(grid_for(outBlocks * c * nd)), dim3(256), 0, ctx->stream, Ap, Y, S,
                               n, dix + x0, nxc, c, perSlice);
            HIPCHK(hipGetLastError());
        }
        // out[(s,) p][x0 + x] = dx/pi sum_k E[p][k] A[(s,) x][k]
        dgemm_tn(ctx, c, np, K, dx / PI, (const double*)Ap, (uint64_t)c * K, (const double*)E, dout + x0, nx,
                 (uint64_t)np * nx, (int)outBlocks);
    }
    copy_to_host(ctx->stream, out, dout, nZ * sizeof(double));
}

// Many slices of a short register on a large window: the output of the product is its time, and
// the library's real kernels (tiles of depth 32) write it more slowly than its complex ones.  Us,
// real against complex, 256 x 256 points: 2^4 points 912 / 798 under 1024 slices, 269 / 274 under 256;
// 2^5 1028 / 918; 2^6 1154 / 1145; 2^7 1481 / 1650.  8 x 8: 2^4 points 72 / 83 under 1024 slices; 64 x 64:
// 2^3 309 / 310, 2^2 359 / 331; 32 x 32: 2^3 355 / 329.
static bool husimi_grid_complex(int n, uint64_t S, uint64_t points) {
    return n <= 5 && S >= 512 && points >= (n <= 3 ? 1u << 10 : 1u << 14);
}

static void get_husimi_grid(CVDVContext* ctx, int r, const double* qs, int nq, const double* ps, int np,
                            int perSlice, double* out) {
    const int n = ctx->nq[r], N = 1 << n, half = N > 1 ? N / 2 : 1;
    const double dx = ctx->dx[r];
    const uint64_t A = ctx->totalSize, S = A >> n;
    // e^{-d^2/2} is exactly 0 in FP64 beyond |d| = 38.61: pairs of points further than
    // that from every q take no part.  A multiple of 16 pairs keeps the GEMM's depth even.
    double far = 0.0;
    for (int i = 0; i < nq; ++i) far = std::max(far, std::fabs(qs[i]));
    const double outside = 0.5 * (double)(N - 1) - (far + 38.7) / dx;  // points j below this
    const int j0 = outside >= 16.0 ? std::min((int)std::floor(outside), half - 1) & ~15 : 0;
    const bool cplx = husimi_grid_complex(n, S, (uint64_t)np * nq);
    const int nj = cplx ? N : half - j0, K = cplx ? N : 2 * nj;
    int nqc = nq;
    while (nqc > 1 && (uint64_t)nqc * S * K > GRID_CHUNK) nqc = (nqc + 1) / 2;
    const uint64_t nB = (uint64_t)nqc * S * K, nE = (uint64_t)np * nj, nH = S * (uint64_t)np * nq;
    const uint64_t nOut = (perSlice ? S : 1) * (uint64_t)np * nq;
    std::vector<double> up(qs, qs + nq);
    up.insert(up.end(), ps, ps + np);
    GridScratch g{(char*)ctx_scratch(ctx, (A + nB + nE + nH + S) * 16 + (up.size() + nOut) * 8 + 256)};
    double2* X = g.take<double2>(A);
    double2* B = g.take<double2>(nB);
    double2* E = g.take<double2>(nE);
    double2* H = g.take<double2>(nH);
    double2* nil = g.take<double2>(S);
    double* dqs = g.take<double>(up.size());
    const double* dps = dqs + nq;
    double* dout = g.take<double>(nOut);
    grid_slices(ctx, r, X);
    HIPCHK(hipMemcpyAsync(dqs, up.data(), up.size() * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    if (cplx)
        hipLaunchKernelGGL(k_grid_husimi_zE, dim3(grid_for(nE)), dim3(256), 0, ctx->stream, E, dps, np, n, dx);
    else
        hipLaunchKernelGGL(k_grid_husimi_E, dim3(grid_for(nE)), dim3(256), 0, ctx->stream, E, dps, np, n, dx, j0, nj);
    HIPCHK(hipGetLastError());
    if (j0 > 0) {
        hipLaunchKernelGGL(k_grid_outside, dim3((unsigned)S), dim3(256), 0, ctx->stream, nil, X, n, j0);
        HIPCHK(hipGetLastError());
    }
    for (int q0 = 0; q0 < nq; q0 += nqc) {
        const int c = nq - q0 < nqc ? nq - q0 : nqc;
        if (cplx) {
            hipLaunchKernelGGL(k_grid_husimi_zB, dim3(grid_for((uint64_t)c * S * N)), dim3(256), 0, ctx->stream, B, X,
                               S, n, dqs + q0, c, dx);
            HIPCHK(hipGetLastError());
            // H_s[p][q0 + q] = sum_j E[p][j] B[s][q][j]
            zgemm_tn(ctx, c, np, N, B, (uint64_t)c * N, E, H + q0, nq, (uint64_t)np * nq, (int)S);
            continue;
        }
        hipLaunchKernelGGL(k_grid_husimi_B, dim3(grid_for((uint64_t)c * S * nj)), dim3(256), 0, ctx->stream, B, X, S,
                           n, dqs + q0, c, dx, j0, nj, j0 > 0 ? nil : nullptr);
        HIPCHK(hipGetLastError());
        // Re and Im of H_s[p][q0 + q] = sum_k E[p][k] B[s][2q (+1)][k]
        dgemm_tn(ctx, 2 * c, np, K, 1.0, (const double*)B, (uint64_t)2 * c * K, (const double*)E,
                 (double*)(H + q0), 2 * nq, (uint64_t)2 * np * nq, (int)S);
    }
    hipLaunchKernelGGL(k_grid_abs2, dim3(grid_for(nOut)), dim3(256), 0, ctx->stream, dout, H, S,
                       (uint64_t)np * nq, perSlice, dx / (PI * std::sqrt(PI)));
    HIPCHK(hipGetLastError());
    copy_to_host(ctx->stream, out, dout, nOut * sizeof(double));
}

static bool grid_ok(CVDVContext* ctx, int r, const double* a, int na, const double* b, int nb, double* out) {
    if (!ctx || !out || refuse_recording(ctx)) return false;
    if (!ctx->initialized) {
        cvdv_set_error(CVDV_ERR_STATE, "State not initialized");
        return false;
    }
    if (r < 0 || r >= ctx->numReg) {
        cvdv_set_error(CVDV_ERR_ARG, "Invalid register index: " + std::to_string(r));
        return false;
    }
    if (!a || !b || na <= 0 || nb <= 0) {
        cvdv_set_error(CVDV_ERR_ARG, "grid readout: empty point list");
        return false;
    }
    for (int i = 0; i < na; ++i)
        if (!std::isfinite(a[i])) {
            cvdv_set_error(CVDV_ERR_ARG, "grid readout: non-finite coordinate");
            return false;
        }
    for (int i = 0; i < nb; ++i)
        if (!std::isfinite(b[i])) {
            cvdv_set_error(CVDV_ERR_ARG, "grid readout: non-finite coordinate");
            return false;
        }
    return true;
}

#define GRID_TRY try {
#define GRID_CATCH()                                                         \
    }                                                                        \
    catch (const CvdvError& e) {                                             \
        cvdv_set_error(e.code, e.msg);                                       \
    }                                                                        \
    catch (...) {                                                            \
        cvdv_set_error(CVDV_ERR_HIP, "unexpected internal error");           \
    }

extern "C" {

void cvdvGetWignerGrid(CVDVContext* ctx, int regIdx, const double* xs, int nx, const double* ps, int np,
                       int perSlice, int native, double* out) {
    if (!grid_ok(ctx, regIdx, xs, nx, ps, np, out)) return;
    GRID_TRY get_wigner_grid(ctx, regIdx, xs, nx, ps, np, perSlice ? 1 : 0, native ? 1 : 0, out); GRID_CATCH()
}

void cvdvGetHusimiQGrid(CVDVContext* ctx, int regIdx, const double* qs, int nq, const double* ps, int np,
                        int perSlice, double* out) {
    if (!grid_ok(ctx, regIdx, qs, nq, ps, np, out)) return;
    GRID_TRY get_husimi_grid(ctx, regIdx, qs, nq, ps, np, perSlice ? 1 : 0, out); GRID_CATCH()
}

}  // extern "C"
