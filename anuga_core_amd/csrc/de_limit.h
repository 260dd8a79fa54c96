// The limiter's least ratio, for the device and for CPU tests.
#pragma once

#include <math.h>

#if defined(__HIPCC__)
#define DE_LIMIT_FN __host__ __device__ __forceinline__
#else
#define DE_LIMIT_FN static inline
#endif

// The r of limit_gradient (sw_domain_orig.c:1306-1326) for the provisional
// jumps d: the least of 1000 and, edge by edge, qmin / d (d < -tiny) or
// qmax / d (d > tiny); an edge without either repeats the edge before it, the
// first edge counts 1. qmin <= 0 <= qmax.
//
// Two divisions instead of three: qmax / d falls as d grows, rounding keeps
// that order, so the least of the ratios to qmax is the one to the greatest
// jump, and the least of those to qmin the one to the least jump, in the same
// bits. fmax and fmin drop a NaN jump as the comparisons do; a ratio of two
// infinities is dropped by fmin.
//
// An FP64 division is 11 instructions, a triangle has four limiters, and the
// fused kernel is bound by instruction issue: 213.8 -> 206.5 us substep 0 and
// 235.8 -> 228.0 us substep 1 at 4M triangles, a DE0 step of 40k 16.5 -> 16.1.
DE_LIMIT_FN double de_limit_ratio(const double d[3], double qmin, double qmax)
{
    const double tiny = 1.0e-100;
    const double up = fmax(d[0], fmax(d[1], d[2])), down = fmin(d[0], fmin(d[1], d[2]));
    const double x = qmax / up, y = qmin / down;
    const double r = d[0] < -tiny || d[0] > tiny ? 1000.0 : 1.0;
    return fmin(fmin(up > tiny ? x : r, down < -tiny ? y : r), r);
}
