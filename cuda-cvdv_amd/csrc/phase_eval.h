// phase_eval.h - phase factors evaluated in place (chains, small states) instead of
// read from tables built by a launch of their own.
#pragma once

#include "cvdv_internal.h"

// (c, s) turned by n quarter turns.
__device__ __forceinline__ double2 quarter_turn(int n, double s, double c) {
    const double a = (n & 1) ? s : c, b = (n & 1) ? c : s;
    return make_double2(((n + 1) & 2) ? -a : a, (n & 2) ? -b : b);
}

// e^{2 pi i f}, |f| <= 1/2 (revolutions), as sine and cosine of pi r on r in [-1/4, 1/4]
// after taking off quarter turns (exact): Taylor sums to below 2^-53 with pi as hi + lo, so
// both are the nearest double or its neighbour.  24 FP64 operations, half of sincospi's,
// which has to serve any argument.
__device__ __forceinline__ double2 unit_turn(double f, double) {
    const double n = rint(4.0 * f);
    const double r = fma(-0.5, n, 2.0 * f), z = r * r;
    double p = 7.952054001475513e-07;
    p = fma(p, z, -2.1915353447830217e-05);
    p = fma(p, z, 0.00046630280576761255);
    p = fma(p, z, -0.0073704309457143504);
    p = fma(p, z, 0.08214588661112823);
    p = fma(p, z, -0.5992645293207921);
    p = fma(p, z, 2.5501640398773455);
    p = fma(p, z, -5.16771278004997);
    double q = 4.303069587032947e-06;
    q = fma(q, z, -0.0001046381049248457);
    q = fma(q, z, 0.0019295743094039231);
    q = fma(q, z, -0.02580689139001406);
    q = fma(q, z, 0.2353306303588932);
    q = fma(q, z, -1.3352627688545895);
    q = fma(q, z, 4.0587121264167685);
    q = fma(q, z, -4.934802200544679);
    const double s = fma(r, 3.141592653589793, r * fma(z, p, 1.2246467991473532e-16)), c = fma(z, q, 1.0);
    return quarter_turn((int)n, s, c);
}
// To FP32 accuracy with margin (2^-36), for factors that are rounded to float once.
__device__ __forceinline__ double2 unit_turn(double f, float) {
    const double n = rint(4.0 * f);
    const double r = fma(-0.5, n, 2.0 * f), z = r * r;
    double p = -0.0073704309457143504;
    p = fma(p, z, 0.08214588661112823);
    p = fma(p, z, -0.5992645293207921);
    p = fma(p, z, 2.5501640398773455);
    p = fma(p, z, -5.16771278004997);
    double q = 0.0019295743094039231;
    q = fma(q, z, -0.02580689139001406);
    q = fma(q, z, 0.2353306303588932);
    q = fma(q, z, -1.3352627688545895);
    q = fma(q, z, 4.0587121264167685);
    q = fma(q, z, -4.934802200544679);
    const double s = r * fma(z, p, 3.141592653589793), c = fma(z, q, 1.0);
    return quarter_turn((int)n, s, c);
}
