// fft_radix16.h - DFTs of 16 points in registers and the constants W_32^e, shared by the row
// kernel (fft_row.hip) and the fused four-step kernel (fft_fused.hip).
#pragma once

#include "fft_bfly.h"

// e^{-2 pi i E / 32} as float constants.  Nearest roundings of cos and sin leave |w|^2 - 1
// of up to 6e-8, which an inner product of 21 fixed constants per stage would turn into a
// drift of the norm; each pair below is within an ulp of the exact value, and the uses of
// one stage sum to 4e-8 over 32 elements.  A localised state reaches a stage through one of
// its inputs alone, so the constants that one input meets have to balance too: between the two
// steps of 32 points (INNER) W^15 is the pair of the other side, since the products of input 3,
// W^{3 m}, had summed to 8e-8 (now -3e-8, as those of input 1; input 2 -1e-8).
template <typename R, int E, bool INNER> struct W32;
template <int E, bool INNER> struct W32<float, E, INNER> {
    static constexpr int q = (E >> 3) & 3, r = E & 7;
    static constexpr float c1 =
        (E & 31) == 1 || (INNER && (E & 31) == 15) ? 0.9807852506637573f : 0.9807853102684021f;
    static constexpr float s1 = 0.19509032368659973f;
    static constexpr float c2 = (E & 31) == 6 || (E & 31) == 14 ? 0.9238795042037964f : 0.9238795638084412f;
    static constexpr float s2 = 0.3826834261417389f;
    static constexpr float c3 = 0.8314695954322815f, s3 = 0.5555702447891235f;
    static constexpr float c = r == 1 ? c1 : r == 2 ? c2 : r == 3 ? c3 : r == 5 ? s3 : r == 6 ? s2 : s1;
    static constexpr float s = r == 1 ? s1 : r == 2 ? s2 : r == 3 ? s3 : r == 5 ? c3 : r == 6 ? c2 : c1;
};

template <int E, bool INNER> struct W32<double, E, INNER> {
    static constexpr int q = (E >> 3) & 3, r = E & 7;
    static constexpr double c1 = 0.98078528040323044913, s1 = 0.19509032201612826785;
    static constexpr double c2 = 0.92387953251128675613, s2 = 0.38268343236508977173;
    static constexpr double c3 = 0.83146961230254523708, s3 = 0.55557023301960222474;
    static constexpr double c = r == 1 ? c1 : r == 2 ? c2 : r == 3 ? c3 : r == 5 ? s3 : r == 6 ? s2 : s1;
    static constexpr double s = r == 1 ? s1 : r == 2 ? s2 : r == 3 ? s3 : r == 5 ? c3 : r == 6 ? c2 : c1;
};

template <int E, bool INNER = false, typename C>
__device__ __forceinline__ C mul_w32(C a) {
    using W = W32<decltype(C{}.x), E, INNER>;
    C t = a;
    if constexpr (W::r == 4) {
        t.x = mul_rsqrt2(a.x + a.y);
        t.y = mul_rsqrt2(a.y - a.x);
    } else if constexpr (W::r != 0) {
        t.x = fma(a.x, W::c, a.y * W::s);
        t.y = fma(a.y, W::c, -(a.x * W::s));
    }
    C u;
    u.x = W::q == 0 ? t.x : W::q == 1 ? t.y : W::q == 2 ? -t.x : -t.y;
    u.y = W::q == 0 ? t.y : W::q == 1 ? -t.x : W::q == 2 ? -t.y : t.x;
    return u;
}

// Inputs x[0], x[ST], .. x[15 ST] in order, outputs in order.
template <int ST, typename C>
__device__ __forceinline__ void dft16(C* x) {
#pragma unroll
    for (int j = 0; j < 4; ++j) dft4<false>(x[j * ST], x[(j + 4) * ST], x[(j + 8) * ST], x[(j + 12) * ST]);
    // x[(j + 4 m) ST] is output m of group j
    x[5 * ST] = mul_w32<2>(x[5 * ST]);
    x[6 * ST] = mul_w32<4>(x[6 * ST]);
    x[7 * ST] = mul_w32<6>(x[7 * ST]);
    x[9 * ST] = mul_w32<4>(x[9 * ST]);
    x[10 * ST] = mul_w32<8>(x[10 * ST]);
    x[11 * ST] = mul_w32<12>(x[11 * ST]);
    x[13 * ST] = mul_w32<6>(x[13 * ST]);
    x[14 * ST] = mul_w32<12>(x[14 * ST]);
    x[15 * ST] = mul_w32<18>(x[15 * ST]);
#pragma unroll
    for (int m = 0; m < 4; ++m) dft4<false>(x[4 * m * ST], x[(4 * m + 1) * ST], x[(4 * m + 2) * ST], x[(4 * m + 3) * ST]);
    // x[(4 m + m1) ST] is output m + 4 m1: transpose
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int n = m + 1; n < 4; ++n) {
            const C t = x[(4 * m + n) * ST];
            x[(4 * m + n) * ST] = x[(4 * n + m) * ST];
            x[(4 * n + m) * ST] = t;
        }
}
