// fp64_inrange.h -- IEEE square root and division of FP64 operands known to
// lie well inside the exponent range.
//
// The compiler's expansions of sqrt and / carry steps for operands near the
// ends of the range (scale, class and fix-up instructions; the division's go
// through the one VCC register, which keeps independent divisions of a lane
// from overlapping).  Inside the range the remaining steps give the same
// correctly rounded results on their own.  Issue cost per wave64 on MI355X:
// the compiler's sqrt 86 cycles and division 61 (measured), these about 59
// and 38 by their instructions at the measured rates.
#pragma once

#include <hip/hip_runtime.h>

namespace gs {

// r2 in [2^-400, 2^400): the operands r2_in_range accepts.
constexpr unsigned R2_HI_MIN = (1023u - 400u) << 20;
constexpr unsigned R2_HI_SPAN = 800u << 20;

// G in [2^-300, 2^300) in magnitude
__device__ __forceinline__ bool numerator_in_range(double G)
{
    const unsigned e = static_cast<unsigned>(__double_as_longlong(G) >> 32) & 0x7fffffffu;
    return e - ((1023u - 300u) << 20) < (600u << 20);
}

// False for zeros, subnormals, infinities, NaN and negative values too.
__device__ __forceinline__ bool r2_in_range(double r2)
{
    return static_cast<unsigned>(__double_as_longlong(r2) >> 32) - R2_HI_MIN < R2_HI_SPAN;
}

// t[u] = fl(G / fl(fl(r * r) * r)) with r = fl(sqrt(r2[u])), for
// r2_in_range(r2[u]) and numerator_in_range(G).  Square root: Goldschmidt
// steps from v_rsq_f64, then two residual corrections (fma(-s, s, x) is
// exact).  Division by d = r^3: the half reciprocal root h gives 1/d to about
// 2^-49 as (2 h)^3, one Newton step brings it to half an ulp, and the
// quotient's exact remainder corrects the quotient (Markstein's theorem).
// K independent values step by step: an FP64 result is ready 12 cycles after
// its issue and issues every 4 to 5, so one chain alone leaves the unit idle.
template <int K>
__device__ __forceinline__ void over_r3(double G, const double (&r2)[K], double (&t)[K])
{
    double h[K], s[K], e[K], d[K], y[K], q[K];
#define GS_EACH _Pragma("unroll") for (int u = 0; u < K; u++)
    GS_EACH y[u] = __builtin_amdgcn_rsq(r2[u]);
    GS_EACH h[u] = 0.5 * y[u];
    GS_EACH s[u] = r2[u] * y[u];
    GS_EACH e[u] = __builtin_fma(-h[u], s[u], 0.5);
    GS_EACH h[u] = __builtin_fma(h[u], e[u], h[u]);
    GS_EACH s[u] = __builtin_fma(s[u], e[u], s[u]);
    GS_EACH e[u] = __builtin_fma(-s[u], s[u], r2[u]);
    GS_EACH s[u] = __builtin_fma(e[u], h[u], s[u]);
    GS_EACH e[u] = __builtin_fma(-s[u], s[u], r2[u]);
    GS_EACH s[u] = __builtin_fma(e[u], h[u], s[u]);
    GS_EACH h[u] = h[u] + h[u];
    GS_EACH d[u] = s[u] * s[u];
    GS_EACH y[u] = h[u] * h[u];
    GS_EACH d[u] = d[u] * s[u];
    GS_EACH y[u] = y[u] * h[u];
    GS_EACH e[u] = __builtin_fma(-d[u], y[u], 1.0);
    GS_EACH y[u] = __builtin_fma(y[u], e[u], y[u]);
    GS_EACH q[u] = G * y[u];
    GS_EACH e[u] = __builtin_fma(-d[u], q[u], G);
    GS_EACH t[u] = __builtin_fma(e[u], y[u], q[u]);
#undef GS_EACH
}

// The same for any operands.
__device__ __forceinline__ double over_r3_any(double G, double r2)
{
    const double r = __builtin_sqrt(r2);
    return G / ((r * r) * r);
}

// z / b for a constant b > 1 with y = RN(1 / b), correctly rounded with one
// multiply and two FMAs instead of a full division (Markstein's theorem: with
// q = RN(z y) within an ulp of z / b, the remainder r = z - b q is exact and
// RN(q + r y) = RN(z / b)); div_const_ready(z) must hold, which excludes
// quotients near the subnormal range, where the remainder can be inexact,
// infinities and NaN.
__device__ __forceinline__ double div_const(double z, double b, double y)
{
    const double q = z * y;
    const double r = __builtin_fma(-q, b, z);
    return __builtin_fma(r, y, q);
}

__device__ __forceinline__ bool div_const_ready(double z)
{
    const double az = fabs(z);
    return az >= 0x1p-900 && az < 0x1p1000;
}

// any z
#define GS_DIVC(z, b) \
    (::gs::div_const_ready(z) ? ::gs::div_const((z), (b), 1.0 / (b)) : (z) / (b))

// Zero or in [2^-400, 2^300): differences of two such values are zero or at
// least 2^-453.
__device__ __forceinline__ bool coordinate_in_range(double a)
{
    const unsigned u = static_cast<unsigned>(__double_as_longlong(a) >> 32) & 0x7fffffffu;
    return a == 0.0 || u - ((1023u - 400u) << 20) < (700u << 20);
}

// q[u][d] = fl(fl(gm[u] t[u][d]) / fl(fl(fl(r r) r) + eps3)), r = fl(sqrt(
// t[u].t[u])) summed left to right: one square root (Goldschmidt's iteration
// with residual corrections, as in over_r3) and three divisions by the same
// value, whose reciprocal is formed once (v_rcp_f64 and two Newton steps);
// each quotient is corrected by its exact remainder (Markstein's theorem).  K
// of them step by step, so that their chains overlap.  `fast` promises t[u][d] zero or in
// [2^-453, 2^301), gm[u] in [2^-300, 2^300) and 0 <= eps3 < 2^300; |t|^2 is
// checked here.  Zero numerators keep their sign (the corrections would turn
// -0 into +0).
template <int K>
__device__ __forceinline__ void pull3(const double (&t)[K][3], const double (&gm)[K], double eps3,
                                      bool fast, double (&q)[K][3])
{
#define GS_EACH _Pragma("unroll") for (int u = 0; u < K; u++)
    double r2[K];
    GS_EACH
    {
        r2[u] = t[u][0] * t[u][0] + t[u][1] * t[u][1] + t[u][2] * t[u][2];
        const unsigned hi = static_cast<unsigned>(__double_as_longlong(r2[u]) >> 32);
        fast = fast && hi - ((1023u - 100u) << 20) < (200u << 20);
    }
    if (__all(fast)) {
        double h[K], s[K], e[K], c[K], y[K];
        GS_EACH y[u] = __builtin_amdgcn_rsq(r2[u]);
        GS_EACH h[u] = 0.5 * y[u];
        GS_EACH s[u] = r2[u] * y[u];
        GS_EACH e[u] = __builtin_fma(-h[u], s[u], 0.5);
        GS_EACH h[u] = __builtin_fma(h[u], e[u], h[u]);
        GS_EACH s[u] = __builtin_fma(s[u], e[u], s[u]);
        GS_EACH e[u] = __builtin_fma(-s[u], s[u], r2[u]);
        GS_EACH s[u] = __builtin_fma(e[u], h[u], s[u]);
        GS_EACH e[u] = __builtin_fma(-s[u], s[u], r2[u]);
        GS_EACH s[u] = __builtin_fma(e[u], h[u], s[u]);
        GS_EACH c[u] = (s[u] * s[u] * s[u]) + eps3;
        GS_EACH y[u] = __builtin_amdgcn_rcp(c[u]);
        GS_EACH e[u] = __builtin_fma(-c[u], y[u], 1.0);
        GS_EACH y[u] = __builtin_fma(e[u], y[u], y[u]);
        GS_EACH e[u] = __builtin_fma(-c[u], y[u], 1.0);
        GS_EACH y[u] = __builtin_fma(e[u], y[u], y[u]);
        GS_EACH
        {
#pragma unroll
            for (int d = 0; d < 3; d++) {
                const double a = gm[u] * t[u][d];
                const double q0 = a * y[u];
                q[u][d] = __builtin_copysign(__builtin_fma(__builtin_fma(-c[u], q0, a), y[u], q0), a);
            }
        }
    } else {
        GS_EACH
        {
            const double n = __builtin_sqrt(r2[u]);
            const double c = (n * n * n) + eps3;
#pragma unroll
            for (int d = 0; d < 3; d++) q[u][d] = gm[u] * t[u][d] / c;
        }
    }
#undef GS_EACH
}

}  // namespace gs
